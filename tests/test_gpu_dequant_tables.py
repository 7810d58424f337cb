"""nb_dequant through LDS tables (2^bits entries, bits 2..4) against the
numpy gather and against the general kernel (which an unaligned codebook
takes), bit for bit, at edges of chunks, waves and blocks."""
import numpy as np
import pytest
import torch

from nativebit_amd import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("total,bs", [(32, 32), (33, 32), (2048, 64), (2080, 96), (70_001, 128),
                                      (4096 * 70, 256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_tables_equal_gather(dev, bits, total, bs, dtype):
    ne = 1 << bits
    rng = np.random.default_rng(bits * total + bs)
    nb = -(-total // bs)
    idx = rng.integers(0, ne, nb * bs, dtype=np.uint8)
    cb = rng.standard_normal((nb, ne)).astype(np.float32)
    p = torch.from_numpy(O.pack(idx, bits)).to(dev)
    c = torch.from_numpy(cb).to(dev)
    got = ops.dequant(p, c, total, bits, bs, dtype)
    want = torch.from_numpy(cb[np.arange(total) // bs, idx[:total]]).to(dtype)
    assert torch.equal(got.cpu(), want)
    off = torch.empty(nb * ne + 1, device=dev)[1:].view(nb, ne).copy_(c)
    assert torch.equal(ops.dequant(p, off, total, bits, bs, dtype), got)
