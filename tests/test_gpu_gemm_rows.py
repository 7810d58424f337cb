"""The fp32 multi-row kernel of nb_gemv and nb_gemm_prefill_f32
(nb_gemm_rows.hip): exact codebook values, fp32 activations, at the edges of
its 16-row tiles, 128-column units and wave splits, against fp64.

Bound: a product passes at most 8 roundings in its accumulator (32 over 16
rows), 4 in the unit's tree, one per unit of the wave's sum and one of the
workgroup's (formed in fp64), so |error| <= n 2^-24 sum |x w| with n = 13 + K /
128 (37 + K / 128 over 16 rows; first order; 1 % is added for the higher
ones)."""
import numpy as np
import pytest
import torch

from nativebit_amd import PackedLinear, ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _layer(n, k, bits, bs, seed):
    rng = np.random.default_rng(seed)
    nb = -(-n * k // bs)
    idx = rng.integers(0, 1 << bits, nb * bs, dtype=np.uint8)
    cb = (rng.standard_normal((nb, 1 << bits)) * 0.02).astype(np.float32)
    return O.pack(idx, bits), cb, O.dequant(idx, cb, bs, n * k).reshape(n, k)


def _check(y, x, w, k, slack=0.0, roundings=13):
    x, w = x.astype(np.float64), w.astype(np.float64)
    ref, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    bound = 1.01 * (roundings + k / 128) * 2.0 ** -24 * mag + slack * np.abs(ref)
    assert np.all(np.abs(y - ref) <= bound), float((np.abs(y - ref) / bound).max())


@pytest.mark.parametrize("bits,bs", [(2, 64), (2, 256), (3, 64), (3, 128), (4, 128), (4, 256)])
@pytest.mark.parametrize("n,k,m", [(1, 256, 2), (15, 256, 16), (17, 768, 15), (130, 2560, 3),
                                   (513, 1280, 9), (64, 8448, 2), (4097, 256, 5),
                                   (64, 2048, 16)])   # the last: 16 waves of one unit
def test_rows_vs_f64(dev, bits, bs, n, k, m):
    print(f"[case] rows bits={bits} bs={bs} {n}x{k} m={m}", flush=True)
    packed, cb, w = _layer(n, k, bits, bs, n + k + m)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    y = ops.gemv(torch.from_numpy(x).to(dev), torch.from_numpy(packed).to(dev),
                 torch.from_numpy(cb).to(dev), n, k, bits=bits, block_size=bs)
    _check(y.cpu().numpy(), x, w, k)


# 2..4 activation tiles (nb_gemm_prefill_f32 up to 4e8 products, 3-bit / BS
# 128): full and ragged ones; two units a wave, one or two, 6-7 and 12-13
@pytest.mark.parametrize("m", [17, 31, 32, 33, 48, 49, 63, 64])
@pytest.mark.parametrize("n,k", [(2561, 2304), (2561, 1408), (15, 6272), (300, 12928), (40, 128)])
def test_rows_of_several_tiles_vs_f64(dev, n, k, m):
    """The exact products: a bound of fp32 roundings alone, far below the
    2^-16 of the three bf16 products that larger sizes run on."""
    print(f"[case] rows tiles {n}x{k} m={m}", flush=True)
    assert m * n * k <= 400_000_000
    packed, cb, w = _layer(n, k, 3, 128, n + k + m)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    y = ops.gemm_prefill_f32(torch.from_numpy(x).to(dev), torch.from_numpy(packed).to(dev),
                             torch.from_numpy(cb).to(dev), n, k)
    _check(y.cpu().numpy(), x, w, k, roundings=37)


def test_rows_one_row_odd_units_and_forms(dev):
    """K an odd multiple of 128 (one row), strided x and y, bf16 y, and an x
    view without 16-byte rows (the general kernel) agree with fp64."""
    n, k = 100, 1152
    packed, cb, w = _layer(n, k, 3, 128, 1)
    p, c = torch.from_numpy(packed).to(dev), torch.from_numpy(cb).to(dev)
    x = np.random.default_rng(2).standard_normal((7, k)).astype(np.float32)
    xd = torch.from_numpy(x).to(dev)
    _check(PackedLinear(p, c, n, k)(xd[:1]).cpu().numpy(), x[:1], w, k)
    wide = torch.zeros(7, k + 12, device=dev)
    wide[:, 4:k + 4] = xd
    out = torch.full((7, n + 3), 9.0, device=dev)
    ops.gemv(wide[:, 4:k + 4], p, c, n, k, out=out[:, :n])
    _check(out[:, :n].cpu().numpy(), x, w, k)
    assert (out[:, n:] == 9).all()
    wide[:, 3:k + 3] = xd
    _check(ops.gemv(wide[:, 3:k + 3], p, c, n, k).cpu().numpy(), x, w, k)
    y16 = ops.gemv(xd, p, c, n, k, out_dtype=torch.bfloat16)
    _check(y16.float().cpu().numpy(), x, w, k, slack=2.0 ** -8)


def test_rows_infinite_and_nan_rows_stay_apart(dev):
    """An infinity or NaN in one activation row reaches that row only."""
    n, k = 40, 256
    packed, cb, w = _layer(n, k, 3, 128, 3)
    x = np.random.default_rng(4).standard_normal((5, k)).astype(np.float32)
    x[1, 3], x[3, 200] = np.inf, np.nan
    y = ops.gemv(torch.from_numpy(x).to(dev), torch.from_numpy(packed).to(dev),
                 torch.from_numpy(cb).to(dev), n, k).cpu().numpy()
    ok = [0, 2, 4]
    _check(y[ok], x[ok], w, k)
    assert np.isinf(y[1]).all() and np.isnan(y[3]).all()


def test_rows_subnormal_products(dev):
    """Products below the normal range keep their value (no flush)."""
    n, k = 16, 128
    packed, cb, w = _layer(n, k, 3, 128, 5)
    x = (np.random.default_rng(6).standard_normal((4, k)) * 2.0 ** -124).astype(np.float32)
    y = ops.gemv(torch.from_numpy(x).to(dev), torch.from_numpy(packed).to(dev),
                 torch.from_numpy(cb).to(dev), n, k).cpu().numpy()
    ref = x.astype(np.float64) @ w.T.astype(np.float64)
    assert np.abs(y - ref).max() <= 200 * 2.0 ** -149 + 1e-5 * np.abs(ref).max()
