"""The row kernels over a batch, at their tile edges: nb_rope_kv_batch and
nb_attention_batch equal the per-sequence calls bit for bit, nb_silu_mul_rows
and the vector and scalar forms of nb_rmsnorm_rows against torch in fp64."""
import ctypes

import pytest
import torch

from nativebit_amd import _lib
from nativebit_amd.model import precompute_rope

pytestmark = pytest.mark.gpu


def P(t):
    return ctypes.c_void_p(t.data_ptr())


def stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("B,H,D,ctx,pos0,T", [
    (3, 5, 128, 96, 40, 1), (2, 3, 128, 132, 0, 33), (3, 2, 64, 100, 31, 64), (2, 3, 32, 72, 7, 31),
    (2, 2, 128, 40, 0, 20), (2, 2, 6, 70, 1, 65),
    # the batch through LDS, a sequence a wave per token and head; one token of many heads
    (3, 5, 128, 132, 3, 120), (2, 3, 64, 840, 0, 800), (40, 64, 64, 8, 5, 1)])
def test_batch_equals_sequences(dev, B, H, D, ctx, pos0, T):
    print(f"[case] rows batch B={B} H={H} D={D} ctx={ctx} pos0={pos0} T={T}", flush=True)
    lib, C = _lib.load(), H * D
    g = torch.Generator(device=dev).manual_seed(B + H + D + T)
    qkv = torch.randn(B, T, 3 * C, generator=g, device=dev)
    k0 = torch.randn(B, H, D, ctx, generator=g, device=dev)
    v0 = torch.randn(B, H, ctx, D, generator=g, device=dev)
    cos, sin = (t.to(dev).contiguous() for t in precompute_rope(D, ctx))
    got = []
    for batched in (True, False):
        k, v = k0.clone(), v0.clone()
        q = torch.empty(B, T, C, device=dev)
        out = torch.empty(B, T, C, dtype=torch.bfloat16, device=dev)
        if batched:
            _lib.check(lib.nb_rope_kv_batch(P(qkv), P(k), P(v), P(cos), P(sin), pos0, T, P(q), B, H,
                                            D, ctx, stream()))
            _lib.check(lib.nb_attention_batch(P(q), P(k), P(v), pos0, T, P(out), _lib.NB_BF16, B, H,
                                              D, ctx, stream()))
        else:
            for b in range(B):
                _lib.check(lib.nb_rope_kv_rows(P(qkv[b]), P(k[b]), P(v[b]), P(cos), P(sin), pos0, T,
                                               P(q[b]), H, D, ctx, stream()))
                _lib.check(lib.nb_attention_rows(P(q[b]), P(k[b]), P(v[b]), pos0, T, P(out[b]),
                                                 _lib.NB_BF16, H, D, ctx, stream()))
        got.append((q, k, v, out))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    q, k, v, out = got[0]
    span = slice(pos0, pos0 + T)
    assert torch.equal(v[:, :, span], qkv[..., 2 * C:].reshape(B, T, H, D).transpose(1, 2))
    keep = [p for p in range(ctx) if not pos0 <= p < pos0 + T]
    assert torch.equal(k[..., keep], k0[..., keep]) and torch.equal(v[:, :, keep], v0[:, :, keep])
    kk = qkv[..., C:2 * C].reshape(B, T, H, D // 2, 2).permute(0, 2, 3, 4, 1).double()
    c, s = cos[span].T.double(), sin[span].T.double()
    rot = torch.stack((kk[:, :, :, 0] * c - kk[:, :, :, 1] * s,
                       kk[:, :, :, 1] * c + kk[:, :, :, 0] * s), 3).reshape(B, H, D, T)
    assert (k[..., span] - rot).abs().max() <= 4 * 2.0 ** -24 * kk.abs().max()


@pytest.mark.parametrize("D,ctx,pos0", [(32, 40, 20), (128, 40, 20), (128, 40, 36), (128, 41, 20)])
def test_a_batch_is_one_launch(dev, D, ctx, pos0):
    """nb_rope_kv_batch and nb_attention_batch are one graph node each, on
    every kernel that they choose from (heads of 32, few positions, the MFMA
    kernel, rows of keys without 16-byte alignment)."""
    lib, B, H = _lib.load(), 5, 2
    qkv = torch.randn(B, 1, 3 * H * D, device=dev)
    k, v = torch.zeros(B, H, D, ctx, device=dev), torch.zeros(B, H, ctx, D, device=dev)
    q, out = torch.empty(B, 1, H * D, device=dev), torch.empty(B, 1, H * D, device=dev)
    cos, sin = (t.to(dev).contiguous() for t in precompute_rope(D, ctx))
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        _lib.check(lib.nb_rope_kv_batch(P(qkv), P(k), P(v), P(cos), P(sin), pos0, 1, P(q), B, H, D,
                                        ctx, stream()))
        _lib.check(lib.nb_attention_batch(P(q), P(k), P(v), pos0, 1, P(out), _lib.NB_F32, B, H, D,
                                          ctx, stream()))
    nodes = ctypes.c_size_t(0)
    get_nodes = lib.hipGraphGetNodes   # (of the HIP runtime that the library is linked to)
    get_nodes.restype, get_nodes.argtypes = ctypes.c_int, [ctypes.c_void_p] * 3
    assert get_nodes(graph.raw_cuda_graph(), None, ctypes.byref(nodes)) == 0
    assert nodes.value == 2


@pytest.mark.parametrize("n", [1, 5, 1024, 4097])
@pytest.mark.parametrize("shift", [0, 1])
def test_silu_mul_rows(dev, n, shift):
    """2^-20 covers v_exp_f32 and the division (a few 2^-23 each)."""
    g = torch.randn(n + 1, device=dev)[shift:n + shift] * 4
    u = torch.randn(n + 1, device=dev)[shift:n + shift]
    want = torch.nn.functional.silu(g.double()) * u.double()
    for dt, code, tol in ((torch.float32, _lib.NB_F32, 2.0 ** -20),
                          (torch.bfloat16, _lib.NB_BF16, 2.0 ** -8)):
        act = torch.empty(n, dtype=dt, device=dev)
        _lib.check(_lib.load().nb_silu_mul_rows(P(g), P(u), P(act), code, n, stream()))
        assert ((act.double() - want).abs() <= tol * want.abs() + 1e-30).all()


@pytest.mark.parametrize("C", [4, 1000, 1001, 2560, 4096, 4100])
def test_rmsnorm_rows_vector_and_scalar(dev, C):
    """Squares summed over at most C terms: C 2^-24 / 2 relative at most."""
    T = 5
    x, add, w = (torch.randn(*s, device=dev) for s in ((T, C), (T, C), (C,)))
    for hd, code, tol in ((torch.float32, _lib.NB_F32, 4e-6 + C * 2.0 ** -25),
                          (torch.bfloat16, _lib.NB_BF16, 2.0 ** -8 + 4e-4)):
        xd, h = x.clone(), torch.empty(T, C, dtype=hd, device=dev)
        _lib.check(_lib.load().nb_rmsnorm_rows(P(xd), P(add), None, None, 0, P(w), P(h), code, T, C,
                                               1e-6, stream()))
        s = (x + add).double()
        want = s / (s.square().mean(-1, keepdim=True) + 1e-6).sqrt() * w.double()
        assert torch.equal(xd, x + add)
        assert ((h.double() - want).abs() <= tol * want.abs() + 1e-30).all()
