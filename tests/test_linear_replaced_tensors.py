"""PackedLinear reads its tensors as attributes on each call (no GPU: the
kernels' wrappers are replaced): a codebook or stream that was replaced by a
Parameter, parametrized or passed to functional_call is the one that every
row count multiplies with."""
import pytest
import torch
from torch.nn.utils import parametrize

from nativebit_amd import PackedLinear, ops

N, K = 4, 128


def _layer(n_entries=8):
    bits = ops.bits_for_entries(n_entries)
    return PackedLinear(torch.zeros(ops.packed_nbytes(N * K, bits), dtype=torch.uint8),
                        torch.zeros(N, n_entries), N, K)


@pytest.fixture
def seen(monkeypatch):
    """(packed, codebook) of each call of a kernel wrapper."""
    calls = []

    def call(x, packed, codebook, n, k, **kw):
        calls.append((packed, codebook))
        return torch.zeros(x.shape[0], n)

    def dequant(packed, codebook, total, *a):
        calls.append((packed, codebook))
        return torch.zeros(total)

    for name in ("gemv", "gemm_prefill", "gemm_prefill_f32"):
        monkeypatch.setattr(ops, name, call)
    monkeypatch.setattr(ops, "dequant", dequant)
    return calls


class WithProperty(PackedLinear):
    @property
    def codebook(self):
        return self._buffers["codebook"] + 7


class Doubled(torch.nn.Module):
    def forward(self, t):
        return 2 * t


@pytest.mark.parametrize("rows,dtype,n_entries", [
    (1, torch.float32, 8), (16, torch.float32, 8), (17, torch.float32, 8),
    (17, torch.bfloat16, 8), (17, torch.float32, 16)])
def test_replaced_tensors_are_used(seen, rows, dtype, n_entries):
    x = torch.zeros(rows, K, dtype=dtype)

    layer = _layer(n_entries)
    layer.codebook = torch.nn.Parameter(torch.ones(N, n_entries))
    assert "codebook" not in layer._buffers
    layer(x)
    assert seen.pop()[1] is layer.codebook

    layer = _layer(n_entries)
    del layer.packed_indices
    layer.packed_indices = torch.ones(ops.packed_nbytes(N * K, layer.bits), dtype=torch.uint8)
    layer(x)
    assert seen.pop()[0] is layer.packed_indices

    layer = _layer(n_entries)
    layer.codebook += 3
    parametrize.register_parametrization(layer, "codebook", Doubled())
    layer(x)
    assert (seen.pop()[1] == 6).all()

    layer = _layer(n_entries)
    layer.__class__ = WithProperty
    layer(x)
    assert (seen.pop()[1] == 7).all()

    layer, other = _layer(n_entries), torch.full((N, n_entries), 5.0)
    torch.func.functional_call(layer, {"codebook": other}, (x,))
    assert seen.pop()[1] is other
