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


@pytest.mark.parametrize("kind,D,T,ctx,B", [
    ("rope", 2, 33, 36, 8400),        # 2 workgroups a head: the second launch from head 8388607
    ("attention", 2, 1, 4, 16800),    # the vector kernel: from head 16777215
    ("attention", 64, 1, 4, 16800)])  # the MFMA kernel: from head 16777215
def test_more_workgroups_than_a_launch_takes(dev, kind, D, T, ctx, B):
    """2^24 workgroups of 256 threads are one launch too many (2^32
    work-items): the call covers every head with several, as the sequences
    around the seam, the first and the last ones show."""
    H = 1000
    need = 4 * B * H * D * (T * (4 if kind == "rope" else 2) + ctx * 2)
    if torch.cuda.mem_get_info()[0] < 1.2 * need:
        pytest.skip("not enough free memory")
    print(f"[case] rows launches {kind} D={D} T={T} B={B} ({need >> 30} GiB)", flush=True)
    lib, C = _lib.load(), H * D
    cos, sin = (t.to(dev).contiguous() for t in precompute_rope(D, ctx))

    def call(n, x, k, v):
        out = torch.empty(n, T, C, device=dev)
        if kind == "rope":
            _lib.check(lib.nb_rope_kv_batch(P(x), P(k), P(v), P(cos), P(sin), 0, T, P(out), n, H, D,
                                            ctx, stream()))
            return out, k, v
        _lib.check(lib.nb_attention_batch(P(x), P(k), P(v), 0, T, P(out), _lib.NB_F32, n, H, D, ctx,
                                          stream()))
        return (out,)

    def caches(n):
        if kind == "rope":
            return torch.zeros(n, H, D, ctx, device=dev), torch.zeros(n, H, ctx, D, device=dev)
        return k_all[:n], k_all[:n].view(n, H, ctx, D)   # (any numbers)

    x = torch.empty(B, T, (3 if kind == "rope" else 1) * C, device=dev).normal_()
    if kind == "attention":
        k_all = torch.empty(B, H, D, ctx, device=dev).normal_()
    got = call(B, x, *caches(B))
    for b in {0, (2 ** 24 - 1) // (2 if kind == "rope" else 1) // H, B - 1}:
        if kind == "rope":
            one = call(1, x[b:b + 1].clone(), *caches(1))
        else:
            one = call(1, x[b:b + 1].clone(), k_all[b:b + 1].clone(),
                       k_all[b:b + 1].clone().view(1, H, ctx, D))
        assert all(torch.equal(g[b], o[0]) for g, o in zip(got, one))
        assert one[0].abs().sum() > 0


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
