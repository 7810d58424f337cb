"""nb_attention_rows on fp32 MFMAs (nb_attention_mfma.hip) at the edges of its
16-query and 64-key tiles, wave splits and head groups, against fp64.

Bound: a score is a sum of D products of fp32 numbers (relative error at most
D 2^-24 of sum |q k|), v_exp_f32 and its argument's scaling add about
2^-22 (1 + |s|), so an output is off by at most about
(D max sum |q k| + 8 + 4 max |s|) 2^-24 + n 2^-24 of max |v|; 2e-5 covers the
inputs below (|s| up to 12, sum |q k| up to 20, n up to 1024)."""
import ctypes

import pytest
import torch

from nativebit_amd import _lib

pytestmark = pytest.mark.gpu


def P(t):
    return ctypes.c_void_p(t.data_ptr())


def run(dev, q, kc, vc, pos0, H, D, ctx):
    T = q.shape[0]
    out = torch.empty(T, H * D, device=dev)
    qd, kd, vd = q.to(dev), kc.to(dev), vc.to(dev)
    _lib.check(_lib.load().nb_attention_rows(
        P(qd), P(kd), P(vd), pos0, T, P(out), _lib.NB_F32, H, D, ctx,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return out.cpu()


def reference(q, kc, vc, pos0, H, D):
    T = q.shape[0]
    n = pos0 + T
    s = q.double().reshape(T, H, D).transpose(0, 1) @ kc[:, :, :n].double()
    mask = torch.arange(n)[None, :] <= (pos0 + torch.arange(T))[:, None]
    p = s.masked_fill(~mask[None], float("-inf")).softmax(-1)
    return (p @ vc[:, :n].double()).transpose(0, 1).reshape(T, H * D)


def inputs(H, D, ctx, T, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(T, H * D, generator=g) * D ** -0.5 * 2,
            torch.randn(H, D, ctx, generator=g), torch.randn(H, ctx, D, generator=g))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,ctx,pos0,T", [
    (2, 64, 0, 64), (3, 68, 0, 65), (1, 128, 63, 1), (1, 128, 64, 1), (2, 260, 47, 17),
    (25, 132, 100, 16), (49, 80, 48, 31), (2, 1024, 1007, 17), (1, 320, 255, 33), (2, 300, 0, 300),
    (130, 32, 3, 9),
    (2, 66, 40, 20)])   # the last: rows of keys without 16-byte alignment
def test_tile_edges(dev, D, H, ctx, pos0, T):
    print(f"[case] attention mfma D={D} H={H} ctx={ctx} pos0={pos0} T={T}", flush=True)
    q, kc, vc = inputs(H, D, ctx, T, H + D + ctx + pos0 + T)
    kc[:, :, pos0 + T:] = float("nan")
    vc[:, pos0 + T:] = float("nan")
    out = run(dev, q, kc, vc, pos0, H, D, ctx)
    ref = reference(q, kc, vc, pos0, H, D)
    assert (out - ref).abs().max() <= 2e-5 * vc[:, :pos0 + T].abs().max()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("at", [70, 81, 95])
def test_non_finite_values_reach_only_queries_that_see_them(dev, D, at):
    """A NaN or infinity in a cached value: earlier queries of the same tile
    keep their finite results, later ones take it in its dimension only."""
    H, ctx, pos0, T = 2, 128, 64, 48
    q, kc, vc = inputs(H, D, ctx, T, at)
    vc[0, at, 5], vc[1, at, 7] = float("inf"), float("nan")
    out = run(dev, q, kc, vc, pos0, H, D, ctx).view(T, H, D)
    clean = vc.clone()
    clean[:, at] = torch.where(clean[:, at].isfinite(), clean[:, at], torch.zeros(()))
    ref = reference(q, kc, clean, pos0, H, D).view(T, H, D)
    sees = torch.arange(T) + pos0 >= at
    for h, d in ((0, 5), (1, 7)):
        hit = torch.zeros(T, D, dtype=torch.bool)
        hit[sees, d] = True
        o = out[:, h]
        assert not o[hit].isfinite().any()
        assert (o - ref[:, h])[~hit].abs().max() <= 2e-5 * clean.abs().max()
    assert (out[sees, 0, 5] == float("inf")).all()


def test_nan_and_infinite_scores(dev):
    """A NaN key makes NaN of the queries that see it and of no other; a
    score of -inf has no weight."""
    H, D, ctx, pos0, T = 1, 128, 128, 60, 40
    q, kc, vc = inputs(H, D, ctx, T, 1)
    kc[0, 3, 80] = float("nan")
    out = run(dev, q, kc, vc, pos0, H, D, ctx)
    sees = torch.arange(T) + pos0 >= 80
    assert out[sees].isnan().all() and out[~sees].isfinite().all()
    kc[0, 3, 80] = 0.0
    q[:, 9] = 1.0
    kc[0, 9, 70] = float("-inf")
    out = run(dev, q, kc, vc, pos0, H, D, ctx)
    assert (out - reference(q, kc, vc, pos0, H, D)).abs().max() <= 2e-5 * vc.abs().max()


@pytest.mark.parametrize("D", [64, 128])
def test_weight_zero_times_infinite_value(dev, D):
    """A key that a query sees with a score of -inf has the weight 0, and 0
    times an infinite value is NaN, also where its whole key tile (one wave's)
    scores -inf; keys alone at -inf leave 0 / 0."""
    H, ctx, pos0, T = 1, 256, 200, 3
    q, kc, vc = inputs(H, D, ctx, T, 2)
    q[:, 9] = 1.0
    kc[0, 9, :64] = float("-inf")
    vc[0, 10, 5] = float("inf")
    out = run(dev, q, kc, vc, pos0, H, D, ctx)
    assert out[:, 5].isnan().all()
    clean = vc.clone()
    clean[0, 10, 5] = 0.0
    ref = reference(q, kc, clean, pos0, H, D)
    rest = torch.arange(D) != 5
    assert (out - ref)[:, rest].abs().max() <= 2e-5 * clean.abs().max()
    kc[0, 9] = float("-inf")
    assert run(dev, q, kc, clean, pos0, H, D, ctx).isnan().all()
