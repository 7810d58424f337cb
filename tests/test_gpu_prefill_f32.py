"""nb_gemm_prefill_f32 in one kernel (x and W as bf16 hi + lo parts, three
products a step) at edges of tiles, blocks and K ranges, against fp64, and
the way to its few-rows route (whose kernel has tests and a bound of its own).

Bound: hi + lo is x, and W, to 2^-18, and lo.lo (at most 2^-18 |x w|) is
dropped: 3 * 2^-18 sum |x w|; the fp32 sums run over 3 K / 32 MFMAs, their
32 products and at most 16 K ranges: (3 K / 32 + 48) 2^-24 sum |x w|."""
import numpy as np
import pytest
import torch

from nativebit_amd import _lib, ops
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


def _entry(f32, best):
    """(the call, its workspace size) of an entry point; the call takes x,
    packed, codebook, y, m, n, k, workspace and its size."""
    lib, name = _lib.load(), "nb_gemm_prefill_f32" if f32 else "nb_gemm_prefill_split"
    name += "_best" if best else ""
    size, f = getattr(lib, name + "_ws_bytes"), getattr(lib, name)

    def call(x, packed, cb, y, m, n, k, ws, nbytes):
        dtype = () if f32 else (_lib.NB_F32,)
        _lib.check(f(x.data_ptr(), k, packed.data_ptr(), cb.data_ptr(), y.data_ptr(), *dtype, n, m,
                     n, k, ws.data_ptr() if ws is not None else None, nbytes,
                     torch.cuda.current_stream().cuda_stream))
    return call, size


def _operands(dev, f32, m, n, k):
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    idx = torch.randint(0, 8, (n * k,), generator=g, device=dev, dtype=torch.uint8)
    cb = torch.randn(n * k // 128, 8, generator=g, device=dev) * 0.02
    x = torch.randn(m, k, generator=g, device=dev)
    if not f32:
        x, cb = x.bfloat16(), cb.bfloat16().float()
    return idx, ops.pack(idx, 3), cb, x


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("m,n,k", [
    (500, 7680, 2560), (290, 6912, 1280), (1000, 2560, 6912), (257, 2561, 4096), (40, 128, 384)])
def test_plans_of_both_workspaces(dev, f32, m, n, k):
    """The fastest plan (the *_best entry points) and the one of the least
    workspace write only their workspace and y.  fp32: the bound above; bf16:
    exact products of bf16 values in fp32 sums, (K / 32 + 40) 2^-24 sum |x w|."""
    print(f"[case] prefill plans {m}x{n}x{k} f32={f32}", flush=True)
    idx, packed, cb, x = _operands(dev, f32, m, n, k)
    w = cb.double().gather(1, idx.view(-1, 128).long()).view(n, k)
    ref, size = x.double() @ w.T, x.double().abs() @ w.T.abs()
    bound = (3 * 2.0 ** -18 + (3 * k / 32 + 48) * 2.0 ** -24 if f32 else (k / 32 + 40) * 2.0 ** -24) * size
    assert _entry(f32, True)[1](m, n, k) >= _entry(f32, False)[1](m, n, k)
    for best in (False, True):
        call, ws_bytes = _entry(f32, best)
        nbytes = ws_bytes(m, n, k)
        ws = torch.full((nbytes + 4096,), 0xff, dtype=torch.uint8, device=dev)
        y = torch.empty(m + 1, n, device=dev)
        y[m] = 7.0
        call(x, packed, cb, y, m, n, k, ws, nbytes)
        assert (ws[nbytes:] == 0xff).all() and (y[m] == 7.0).all()
        assert ((y[:m].double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("m,n,k", [(1024, 2560, 6912), (500, 7680, 2560), (867, 8716, 3840),
                                   (64, 2560, 2560)])
def test_a_larger_workspace_changes_nothing(dev, f32, m, n, k):
    """Bytes past *_ws_bytes are not touched -- none at all where that is 0,
    so that calls on several streams may share them -- and the result's bits
    do not depend on the workspace's size."""
    print(f"[case] prefill workspace {m}x{n}x{k} f32={f32}", flush=True)
    _, packed, cb, x = _operands(dev, f32, m, n, k)
    most = _entry(f32, True)[1](m, n, k)
    for best in (False, True):
        call, ws_bytes = _entry(f32, best)
        need = ws_bytes(m, n, k)
        ys = []
        for nbytes in (need, need + 512, most + (160 << 20)):
            ws = torch.full((nbytes,), 0xff, dtype=torch.uint8, device=dev) if nbytes else None
            ys.append(torch.empty(m, n, device=dev))
            call(x, packed, cb, ys[-1], m, n, k, ws, nbytes)
            assert ws is None or (ws[need:] == 0xff).all()
        assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])
