"""x and do of dense rows whose heads lie any multiple of 16 bytes apart (0: one matrix expanded to
every head) are read in place: bit-identical to the same values passed densely, with no copy of
them allocated; other views are copied as before.
"""
import ctypes

import pytest
import torch

import flashmlp_amd as fm
from flashmlp_amd import _lib
from oracle.inputs import make_inputs
from test_gpu_narrow import _generic
from test_gpu_odd_e import _DT, _p, _rel, _stream

pytestmark = pytest.mark.gpu

SHAPES = [(4, 300, 128, 256, torch.bfloat16), (4, 1025, 64, 683, torch.float16), (3, 129, 256, 264, torch.bfloat16),
          (5, 200, 32, 96, torch.float16), (3, 77, 16, 45, torch.bfloat16), (3, 257, 64, 100, torch.float32),
          (1, 4096, 128, 1024, torch.bfloat16), (2, 130, 256, 40, torch.float32), (12, 1024, 64, 768, torch.float16)]


def _views(t, pad):
    """t with its heads `pad` elements further apart than dense"""
    H, B, D = t.shape
    buf = torch.full((H, B * D + pad), float("nan"), dtype=t.dtype, device=t.device)
    v = buf[:, :B * D].view(H, B, D)
    v.copy_(t)
    return v


@pytest.mark.parametrize("H,B,D,E,dt", SHAPES)
def test_views_match_dense(H, B, D, E, dt):
    print(f"[heads] H={H} B={B} D={D} E={E} {dt}", flush=True)
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=B))
    xe, de = x[:1].expand(H, B, D), do[:1].expand(H, B, D)
    cases = [(xe, de), (_views(x, 8), do), (x, _views(do, 16)), (_views(x, 24), de),
             (_views(x, 3), do),  # heads not 16-byte aligned: copied
             (x.transpose(0, 1).contiguous().transpose(0, 1), do)]  # rows not dense: copied
    for xv, dv in cases:
        for kw in ({}, {"accurate_dw": True}, {"recompute": True}):
            ref = (fm.flashmlp_fwd(xv.contiguous(), w1, w2, "silu"),
                   *fm.flashmlp_bwd(xv.contiguous(), w1, w2, dv.contiguous(), "silu", **kw))
            got = (fm.flashmlp_fwd(xv, w1, w2, "silu"), *fm.flashmlp_bwd(xv, w1, w2, dv, "silu", **kw))
            for name, a, b in zip(("o", "dx", "dw1", "dw2"), got, ref):
                assert a.is_contiguous() and torch.equal(a, b), (name, xv.stride(), dv.stride(), kw)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_shared_input_module(dt):
    # the module's 2-D input: gradients bit-identical to autograd's mean over dense copies
    torch.manual_seed(0)
    m = fm.FlashMLP(6, 64, 256, activation="silu", dtype=dt)
    x = torch.randn(700, 64, device="cuda", dtype=dt, requires_grad=True)
    g = torch.randn(700, 64, device="cuda", dtype=dt)
    got = torch.autograd.grad(m(x), (x, m.w1, m.w2), g)
    o = fm.FlashMLPFunction.apply(x.unsqueeze(0).expand(6, -1, -1).contiguous(), m.w1, m.w2, "silu").mean(dim=0)
    ref = torch.autograd.grad(o, (x, m.w1, m.w2), g)
    assert torch.equal(m(x), o)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
    with torch.no_grad():
        assert torch.equal(m(x), o)


def test_no_copy_is_allocated():
    H, B, D, E = 16, 4096, 128, 64
    x = torch.randn(B, D, device="cuda", dtype=torch.bfloat16)
    w1 = torch.randn(H, D, E, device="cuda", dtype=torch.bfloat16)
    w2 = torch.randn(H, E, D, device="cuda", dtype=torch.bfloat16)
    xe = x.expand(H, B, D)
    fm.flashmlp_fwd(xe, w1, w2, "silu")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    o = fm.flashmlp_fwd(xe, w1, w2, "silu")
    assert torch.cuda.max_memory_allocated() - before < o.numel() * 2 * 1.5  # the output alone


def _strided(x, w1, w2, do, act, code, st, ws_bytes=0):
    """o, dx, dw1, dw2 (fp32 sums) through the strided C entry points with these stride arrays"""
    L = _lib.lib()
    (H, B, D), E = x.shape, w1.shape[2]
    code |= _lib.FMLP_OUT_F32
    outs = [torch.full(s, float("nan"), device="cuda") for s in ((H, B, D), (H, B, D), (H, D, E), (H, E, D))]
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device="cuda") if ws_bytes else None
    _lib.check(L.fmlp_fwd_strided(_p(x), _p(w1), _p(w2), _p(outs[0]), H, B, D, E, *st[:3], code, _lib.ACT_CODES[act],
                                  _stream()), "forward")
    _lib.check(L.fmlp_bwd_strided(_p(x), _p(w1), _p(w2), _p(do), *(_p(t) for t in outs[1:]), H, B, D, E, *st, code,
                                  _lib.ACT_CODES[act], _p(ws), ws_bytes, _stream()), "backward")
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("B,D,E,which", [(2048, 128, 256, w) for w in range(4)] + [(1, 128, 2048, 0), (1, 128, 2048, 3)])
def test_one_head_with_any_head_stride_accepts_any_workspace(B, D, E, which):
    """A lone head (or row) of a view may carry any stride in that dimension; fmlp_bwd_strided takes such
    a call without a workspace, whatever the dense call's plan needs."""
    L = _lib.lib()
    H, dt, act = 1, torch.bfloat16, "silu"
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=B + E))
    n = L.fmlp_bwd_workspace_bytes(H, B, D, E, _DT[dt])
    print(f"[heads] lone head B={B} D={D} E={E} tensor {which} workspace {n}", flush=True)
    assert n > 0 and L.fmlp_shape_tuned(D, E, _DT[dt]) == 1
    assert L.fmlp_bwd(_p(x), _p(w1), _p(w2), _p(do), _p(torch.empty_like(x)), _p(torch.empty_like(w1)),
                      _p(torch.empty_like(w2)), H, B, D, E, _DT[dt], _lib.ACT_CODES[act], None, 0, _stream()) == 4
    st = [_lib.strides(t) for t in (x, w1, w2, do)]
    ref = _strided(x, w1, w2, do, act, _DT[dt], st, n)
    st[which] = (ctypes.c_int64 * 3)(x[0].numel() + 16, D if B > 1 else 3 * D, 1) if which in (0, 3) else \
        (ctypes.c_int64 * 3)(w1[0].numel() + 16, E if which == 1 else D, 1)
    got = _strided(x, w1, w2, do, act, _DT[dt], st)
    for name, a, r in zip(("o", "dx", "dw1", "dw2"), got, ref):
        assert _rel(a, r) <= 1e-4, name


@pytest.mark.parametrize("H,B,D,E", [(2, 96, 64, 288), (2, 300, 64, 96), (2, 96, 64, 160), (3, 4096, 64, 544),
                                     (2, 96, 128, 288), (2, 96, 128, 96)])
@pytest.mark.parametrize("what", ["x", "w1"])
def test_infinities_in_views_stay_where_the_generic_kernels_have_them(H, B, D, E, what):
    """Views whose heads lie apart, with whole tiles of E (inside a cut one both kernel sets multiply
    zeros): the chunks that an E part does not have, and the subtiles that a row set does not, must not
    turn an infinite input's saturated sigmoid into NaN."""
    dt, act = torch.float16, "sigmoid"
    print(f"[heads] infinite {what} H={H} B={B} D={D} E={E}", flush=True)
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=3))
    w1[w1 == 0] = 0.125  # inf * 0 is the oracle's NaN
    x[x == 0] = 0.125
    if what == "x":
        x[H - 1, 5, 3] = float("inf")
    else:
        w1[H - 1, 5, 3] = float("inf")
    n = _lib.lib().fmlp_bwd_workspace_bytes(H, B, D, E, _DT[dt])
    gen = _generic(x, w1, w2, do, act, 0)
    xv = _views(x, 8)
    st = [_lib.strides(t) for t in (xv, w1, w2, do)]
    assert gen[0].isfinite().all()
    for ws in (0, n):
        got = _strided(xv, w1, w2, do, act, _DT[dt], st, ws)
        for name, a, r in zip(("o", "dx", "dw1", "dw2"), got, gen):
            fin = r.isfinite()
            assert torch.equal(a.isfinite(), fin), (name, ws)
            assert _rel(a[fin], r[fin]) <= 1e-4, (name, ws)
