"""fmlp_copy_dense: a call's views to dense buffers in one launch, at the edges of the 16-byte pieces, the
256-piece workgroups and the rows, between sentinel guards; and the wrappers' results for
views through it (bit-identical to dense calls, one launch for all of a call's views)."""
import ctypes
import sys

import pytest
import torch

import flashmlp_amd as fm
from flashmlp_amd import _lib
from oracle.inputs import make_inputs
from test_gpu_odd_e import _check_guards, _guarded, _stream

pytestmark = pytest.mark.gpu


def _copy(ts):
    """the tensors' dense copies through one call"""
    n = len(ts)
    bufs = [_guarded(tuple(t.shape), t.dtype) for t in ts]
    arr = lambda vals: (ctypes.c_void_p * 4)(*vals)
    flat = lambda rows: (ctypes.c_int64 * 12)(*[v for r in rows for v in r])
    st = _lib.lib().fmlp_copy_dense(n, arr([t.data_ptr() for t in ts]), arr([o.data_ptr() for _, o in bufs]),
                                    flat([t.shape for t in ts]), flat([t.stride() for t in ts]), ts[0].element_size(),
                                    _stream())
    _lib.check(st, "copy")
    torch.cuda.synchronize()
    for b, o in bufs:
        _check_guards(b, o.numel())
    return [o for _, o in bufs]


def _views(H, B, D, dt):
    base = torch.randn(H, B + 1, D + 5, device="cuda").to(dt)
    yield base[:, :B, 2:2 + D]  # padded rows, a base that is not 16-byte aligned
    yield torch.randn(B, H, D, device="cuda").to(dt).transpose(0, 1)  # heads inside the rows
    yield torch.randn(H, D, B, device="cuda").to(dt).transpose(1, 2)  # columns inside out
    yield torch.randn(D, B, H, device="cuda").to(dt).permute(2, 1, 0)
    yield torch.randn(H, 1, D, device="cuda").to(dt).expand(H, B, D)  # a stride of zero
    yield torch.randn(1, 1, 1, device="cuda").to(dt).expand(H, B, D)


@pytest.mark.parametrize("H,B,D", [(1, 1, 1), (1, 1, 7), (1, 3, 8), (2, 5, 3), (3, 129, 17), (1, 1, 2049), (2, 1024, 8),
                                   (5, 33, 250), (16, 64, 64)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_copies(H, B, D, dt):
    print(f"[copy] {H}x{B}x{D} {dt}", flush=True)
    vs = list(_views(H, B, D, dt))
    for v in vs:
        assert torch.equal(_copy([v])[0], v)
    for k in (2, 3, 4):  # several at once, of different sizes
        ts = [vs[0], vs[2].transpose(1, 2), vs[4][:, :1], vs[1]][:k]
        for got, t in zip(_copy(ts), ts):
            assert torch.equal(got, t)


def test_rejected_arguments():
    L = _lib.lib()
    vp, i64 = ctypes.c_void_p * 4, ctypes.c_int64 * 12
    p, z, s = vp(0x1000, 0x1000, 0x1000, 0x1000), i64(2, 3, 4), i64(12, 4, 1)
    call = lambda n=1, a=p, b=p, z=z, s=s, es=2: L.fmlp_copy_dense(n, a, b, z, s, es, None)
    assert call(n=0) == 0 and call(z=i64(2, 0, 4)) == 0  # nothing to copy
    assert call(n=5) == 1 and call(n=-1) == 1 and call(a=None) == 1 and call(s=None) == 1
    assert call(es=8) == 2 and call(z=i64(1 << 20, 1 << 11, 1)) == 2
    assert call(z=i64(-1, 3, 4)) == 1 and call(s=i64(12, -4, 1)) == 1
    assert call(a=vp(0x1001)) == 1 and call(b=vp(0x1008)) == 1 and call(a=vp(None)) == 1


@pytest.mark.parametrize("H,B,D,E,dt", [(2, 33, 32, 64, torch.bfloat16), (3, 70, 128, 264, torch.float16),
                                        (2, 40, 64, 45, torch.float32), (4, 3000, 128, 520, torch.bfloat16)])
def test_views_through_the_wrappers(H, B, D, E, dt):
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=B))
    xt = x.transpose(0, 1).contiguous().transpose(0, 1)
    w1t = w1.transpose(1, 2).contiguous().transpose(1, 2)
    w2p = torch.empty(H, E, D + 3, dtype=dt, device="cuda")[:, :, 1:1 + D].copy_(w2)
    row = do[:, :1].expand(H, B, D)
    neg = torch._neg_view(do.transpose(0, 1).contiguous().transpose(0, 1))
    for xv, av, bv, dv in ((xt, w1, w2, do), (x, w1t, w2, do), (x, w1, w2p, do), (x, w1, w2, row), (xt, w1t, w2p, row),
                           (x, w1, w2, neg)):
        ref = (fm.flashmlp_fwd(x, w1, w2, "silu"), *fm.flashmlp_bwd(x, w1, w2, dv.resolve_neg().contiguous(), "silu"))
        got = (fm.flashmlp_fwd(xv, av, bv, "silu"), *fm.flashmlp_bwd(xv, av, bv, dv, "silu"))
        for a, b in zip(got, ref):
            assert a.is_contiguous() and torch.equal(a, b)


def test_one_launch_for_all_views():
    H, B, D, E, dt = 2, 33, 32, 64, torch.bfloat16
    x, w1, w2, _ = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=1))
    xt = x.transpose(0, 1).contiguous().transpose(0, 1)
    w1t = w1.transpose(1, 2).contiguous().transpose(1, 2)
    w2p = torch.empty(H, E, D + 3, dtype=dt, device="cuda")[:, :, :D].copy_(w2)
    run = lambda: fm.flashmlp_fwd(xt, w1t, w2p, "silu")
    run()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        run()
        torch.cuda.synchronize()
    kernels = [e.name for e in prof.events() if "kernel" in e.name.lower() and e.device_type == torch.autograd.DeviceType.CUDA]
    assert len(kernels) == 2 and "copy_dense" in kernels[0], kernels


@pytest.mark.parametrize("D,E,dt", [(32, 64, torch.bfloat16), (64, 45, torch.float32), (128, 45, torch.float16),
                                    (64, 64, torch.bfloat16)])
def test_views_whose_copies_do_not_fit(monkeypatch, D, E, dt):
    """Shapes whose views the generic kernels take are read in place then; the others raise, as before."""
    mod = sys.modules["flashmlp_amd.flashmlp"]
    H, B = 2, 70
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=B))
    xt = x.transpose(0, 1).contiguous().transpose(0, 1)
    w2p = torch.empty(H, E, D + 3, dtype=dt, device="cuda")[:, :, 1:1 + D].copy_(w2)
    ref = (fm.flashmlp_fwd(x, w1, w2, "silu"), *fm.flashmlp_bwd(x, w1, w2, do, "silu"))

    def full(t):
        raise torch.OutOfMemoryError("no room for the copy")

    monkeypatch.setattr(mod, "_fast", None)
    monkeypatch.setattr(mod, "_dense", full)
    call = lambda: (fm.flashmlp_fwd(xt, w1, w2p, "silu"), *fm.flashmlp_bwd(xt, w1, w2p, do, "silu"))
    if _lib.lib().fmlp_shape_tuned(D, E, {torch.bfloat16: 1, torch.float16: 0, torch.float32: 2}[dt]):
        with pytest.raises(torch.OutOfMemoryError):
            call()
        return
    for a, b in zip(call(), ref):  # other kernels: sums in another order, results rounded to dt
        assert ((a - b).float().norm() / b.float().norm()).item() <= {torch.float32: 1e-6}.get(dt, 2.0 ** -8)
