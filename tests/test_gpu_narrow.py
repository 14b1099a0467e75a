"""D = 16 and 32 on the fused programs (32-column tiles; at D = 16 their upper half is zeros).

Against the generic kernels, which the same values reach with W2 as a view of padded rows: the unrounded
fp32 sums (FMLP_OUT_F32) within 1e-4 normwise, the bar of the other fp32-sum tests. Sizes at the
edges of the tiles (32 columns of E, 64 / 128 rows, 32-row subtiles and the B split of the dW
programs, the forward's E split and its whole grids), with guards around every output.
"""

import pytest
import torch

from flashmlp_amd import _lib
from oracle.inputs import make_inputs
from test_gpu_odd_e import _DT, _bwd, _check_guards, _guarded, _p, _rel, _stream

pytestmark = pytest.mark.gpu

CASES = [
    # H, B, D, E, dtype, act
    (2, 1, 16, 8, torch.bfloat16, "silu"), (2, 33, 32, 40, torch.float16, "leaky_relu"),
    (3, 127, 16, 96, torch.float16, "silu"), (3, 129, 32, 264, torch.bfloat16, "sigmoid"),
    (2, 4097, 16, 200, torch.bfloat16, ""), (2, 4097, 32, 136, torch.float16, "sigmoid"),
    (40, 1000, 32, 72, torch.bfloat16, "silu"), (40, 1000, 16, 1096, torch.bfloat16, "leaky_relu"),
    (5, 300, 32, 45, torch.bfloat16, "silu"), (5, 300, 16, 3, torch.float16, "silu"),
]


def _generic(x, w1, w2, do, act, flags):
    """forward and backward on the generic kernels: W2 with padded rows, which the others do not read"""
    L = _lib.lib()
    H, B, D = x.shape
    E = w1.shape[2]
    w2v = torch.empty(H, E, D + 8, dtype=x.dtype, device="cuda")[:, :, :D].copy_(w2)
    assert E > 1  # (a single row's pitch is no layout of its own)
    code = _DT[x.dtype] | _lib.FMLP_OUT_F32
    outs = [torch.empty(s, device="cuda") for s in ((H, B, D), (H, B, D), (H, D, E), (H, E, D))]
    st = [_lib.strides(t) for t in (x, w1, w2v, do)]
    _lib.check(L.fmlp_fwd_strided(_p(x), _p(w1), _p(w2v), _p(outs[0]), H, B, D, E, *st[:3], code, _lib.ACT_CODES[act],
                                  _stream()), "forward")
    _lib.check(L.fmlp_bwd_strided(_p(x), _p(w1), _p(w2v), _p(do), *(_p(t) for t in outs[1:]), H, B, D, E, *st,
                                  code | flags, _lib.ACT_CODES[act], None, 0, _stream()), "backward")
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("H,B,D,E,dt,act", CASES)
def test_against_the_generic_kernels(H, B, D, E, dt, act):
    print(f"[narrow] H={H} B={B} D={D} E={E} {dt} act='{act}'", flush=True)
    L = _lib.lib()
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=B + E))
    f32, code = _lib.FMLP_OUT_F32, _DT[dt] | _lib.FMLP_OUT_F32
    gen = _generic(x, w1, w2, do, act, 0)
    gen_hilo = _generic(x, w1, w2, do, act, _lib.FMLP_DW_HILO)
    n = L.fmlp_fwd_workspace_bytes(H, B, D, E, code)
    buf, o = _guarded((H, B, D), torch.float32)
    ws = torch.full((max(n, 16),), 0xFF, dtype=torch.uint8, device="cuda")
    _lib.check(L.fmlp_fwd_ws(_p(x), _p(w1), _p(w2), _p(o), H, B, D, E, code, _lib.ACT_CODES[act], _p(ws), n,
                             _stream()), "forward")
    torch.cuda.synchronize()
    _check_guards(buf, o.numel())
    assert _rel(o, gen[0]) <= 1e-4
    buf, oi = _guarded((H, B, D), dt)
    _lib.check(L.fmlp_fwd_ws(_p(x), _p(w1), _p(w2), _p(oi), H, B, D, E, _DT[dt], _lib.ACT_CODES[act], _p(ws), n,
                             _stream()), "forward")
    torch.cuda.synchronize()
    _check_guards(buf, oi.numel())
    assert torch.equal(oi, o.to(dt))
    for flags in (0, _lib.FMLP_BWD_RECOMPUTE, _lib.FMLP_BWD_STORE_DZ, _lib.FMLP_DW_HILO, _lib.FMLP_BWD_NO_DX,
                  _lib.FMLP_BWD_NO_DW):
        nb = L.fmlp_bwd_workspace_bytes(H, B, D, E, code | flags)
        own = _bwd(x, w1, w2, do, act, f32 | flags, nb, torch.float32)
        io = _bwd(x, w1, w2, do, act, flags, nb, dt)
        ref = (gen_hilo if flags & _lib.FMLP_DW_HILO else gen)[1:]
        for name, a, i, r in zip(("dx", "dw1", "dw2"), own, io, ref):
            if a is not None:
                assert _rel(a, r) <= 1e-4, (hex(flags), name)
                assert torch.equal(i, a.to(dt)), (hex(flags), name)
    # any workspace is accepted where E needs no padded W1 copy: dX is the same bits
    if E % 8 == 0:
        full = _bwd(x, w1, w2, do, act, f32, L.fmlp_bwd_workspace_bytes(H, B, D, E, code), torch.float32)
        none = _bwd(x, w1, w2, do, act, f32, 0, torch.float32)
        assert torch.equal(full[0], none[0])
        assert _rel(none[1], full[1]) <= 1e-5 and _rel(none[2], full[2]) <= 1e-5  # the dW split's order


@pytest.mark.parametrize("D,E", [(16, 96), (32, 288), (32, 64)])
@pytest.mark.parametrize("what", ["x", "w1"])
def test_infinities_stay_where_the_generic_kernels_have_them(D, E, what):
    """A saturating activation keeps results finite next to an infinite input; the zeros behind the
    last chunk of an E part or the last subtile of a row set must not turn them into NaN. (E and B
    are multiples of 32: inside a cut tile both kernel sets multiply zeros.)"""
    H, B, dt, act = 2, 96, torch.float16, "sigmoid"
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=3))
    (x if what == "x" else w1)[1, 5, 3] = float("inf")
    L = _lib.lib()
    code = _DT[dt] | _lib.FMLP_OUT_F32
    gen = _generic(x, w1, w2, do, act, 0)
    o = torch.empty(H, B, D, device="cuda")
    _lib.check(L.fmlp_fwd(_p(x), _p(w1), _p(w2), _p(o), H, B, D, E, code, _lib.ACT_CODES[act], _stream()), "forward")
    own = [o, *_bwd(x, w1, w2, do, act, _lib.FMLP_OUT_F32, L.fmlp_bwd_workspace_bytes(H, B, D, E, code), torch.float32)]
    for name, a, r in zip(("o", "dx", "dw1", "dw2"), own, gen):
        assert torch.equal(a.isfinite(), r.isfinite()), name
        fin = r.isfinite()
        assert _rel(a[fin], r[fin]) <= 1e-4, name
