"""nb_gemm_prefill_f32 in one kernel (x and W as bf16 hi + lo parts, three
products a step) and its few-rows route, at edges of tiles, blocks and K
ranges, against fp64.

Bound: hi + lo is x, and W, to 2^-18, and lo.lo (at most 2^-18 |x w|) is
dropped: 3 * 2^-18 sum |x w|; the fp32 sums run over 3 K / 32 MFMAs, their
32 products and at most 16 K ranges: (3 K / 32 + 48) 2^-24 sum |x w|."""
import numpy as np
import pytest
import torch

from nativebit_amd import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _case(dev, m, n, k, pad=0, seed=0):
    rng = np.random.default_rng(seed + m + n + k)
    nb = n * k // 128
    idx = rng.integers(0, 8, n * k, dtype=np.uint8)
    cb = (rng.standard_normal((nb, 8)) * 0.02).astype(np.float32)
    x = rng.standard_normal((m, k)).astype(np.float32)
    xd = torch.zeros(m, k + pad, device=dev)
    xd[:, pad:] = torch.from_numpy(x).to(dev)
    y = ops.gemm_prefill_f32(xd[:, pad:], torch.from_numpy(O.pack(idx, 3)).to(dev),
                             torch.from_numpy(cb).to(dev), n, k).cpu().numpy()
    w = O.dequant(idx, cb, 128, n * k).reshape(n, k).astype(np.float64)
    x = x.astype(np.float64)
    bound = (3 * 2.0 ** -18 + (3 * k / 32 + 48) * 2.0 ** -24) * (np.abs(x) @ np.abs(w).T)
    return np.abs(y - x @ w.T) / bound


@pytest.mark.parametrize("m,n,k", [
    (17, 5, 128),            # few rows: the exact products
    (64, 16384, 384),        # just over that route's size
    (65, 6200, 1024), (129, 130, 2560), (130, 4097, 768), (257, 3000, 640),
    (300, 1000, 1024), (70, 2560, 8192), (1000, 2561, 256), (520, 7000, 256)])
def test_f32_edges(dev, m, n, k):
    print(f"[case] prefill f32 {m}x{n}x{k}", flush=True)
    assert _case(dev, m, n, k).max() <= 1.0


@pytest.mark.parametrize("pad", [1, 4])
def test_f32_strided_rows(dev, pad):
    """Rows of x with and without 16-byte alignment."""
    assert _case(dev, 200, 3000, 1024, pad).max() <= 1.0
    assert _case(dev, 20, 300, 256, pad).max() <= 1.0
