"""nb_block_codebooks' 16-lane sorting kernel at the edges of its block sizes
(16 R values a row, R = 4, 8, 16), against the CPU's torch.quantile bit for
bit: partial blocks, rows past the last block, unaligned weights, repeated
values, zeros of both signs, many entries."""
import pytest
import torch

from nativebit_amd import ops

pytestmark = pytest.mark.gpu


def _want(w, ne, bs):
    q = torch.linspace(0, 1, ne)
    return torch.stack([torch.quantile(w[i:i + bs], q) for i in range(0, w.numel(), bs)])


@pytest.mark.parametrize("bs", [1, 4, 63, 64, 65, 127, 128, 129, 255, 256])
@pytest.mark.parametrize("ne,blocks,shift", [(8, 17, 0), (16, 5, 1), (40, 33, 0), (17, 3, 0),
                                             (64, 9, 1), (256, 18, 0)])
def test_row_sort(dev, bs, ne, blocks, shift):
    g = torch.Generator().manual_seed(bs * ne)
    w = torch.randn(blocks * bs - bs // 3 + shift, generator=g) * 0.02
    w[::7] = w[3 % w.numel()]
    w[1::9] = 0.0
    w[2::9] = -0.0
    got = ops.block_codebooks(w.to(dev)[shift:], ne, bs).cpu()
    assert torch.equal(got, _want(w[shift:], ne, bs))


@pytest.mark.parametrize("ne", [16, 100])
def test_more_blocks_than_rows_of_the_grid(dev, ne):
    """Every workgroup takes several rounds of blocks (the grid has at most 16
    rows for each of 8 workgroups a CU)."""
    blocks = 16 * 8 * torch.cuda.get_device_properties(dev).multi_processor_count + 37
    w = torch.randn(2 * blocks, 4, generator=torch.Generator().manual_seed(ne))
    got = ops.block_codebooks(w.to(dev).reshape(-1), ne, 4).cpu()
    assert torch.equal(got, torch.quantile(w, torch.linspace(0, 1, ne), dim=1).T)
