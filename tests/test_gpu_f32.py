"""fp32 io on the dense kernels (fmlp_f32.hip) at the edges of their tiles, against 64-bit torch.

Bound: rounding in a chain of n fp32 additions moves a sum by about sqrt(n) 2^-24 of its size. Z is
a chain of D / 2 steps of the matrix instruction; O, dX, dW1 and dW2 are chains of 16 steps and then
one per 32 columns of E (rows of B), and carry Z's (dH's) error; three more units cover the
hardware exponential and reciprocal of the activation and its derivative.
"""

import pytest
import torch

from flashmlp_amd import _lib
from oracle.inputs import make_inputs
from test_gpu_odd_e import _check_guards, _guarded, _p, _rel, _stream

pytestmark = pytest.mark.gpu
F32 = _lib.FMLP_DTYPE_F32


def _act64(act, z):
    s = torch.sigmoid(z)
    if act == "silu":
        return z * s, s * (1 + z * (1 - s))
    if act == "sigmoid":
        return s, s * (1 - s)
    if act == "leaky_relu":
        return torch.where(z > 0, z, 0.01 * z), torch.where(z > 0, 1.0, 0.01).double()
    return z, torch.ones_like(z)


def _exact(x, w1, w2, do, act):
    x, w1, w2, do = (t.double() for t in (x, w1, w2, do))
    t = lambda a: a.transpose(1, 2).contiguous()
    h, d = _act64(act, torch.matmul(x, w1))
    dz = torch.matmul(do, t(w2)) * d
    return torch.matmul(h, w2), torch.matmul(dz, t(w1)), torch.matmul(t(x), dz), torch.matmul(t(h), do)


def _bound(D, n):
    return ((D / 2) ** 0.5 + (16 + n / 32) ** 0.5 + 3) * 2.0 ** -24


def _run(x, w1, w2, do, act, flags, ws_bytes, strided=None):
    """o, dx, dw1, dw2 through the C entry points, guards checked (strided: X as this view)"""
    L = _lib.lib()
    H, B, D = x.shape
    E = w1.shape[2]
    shapes = ((H, B, D), (H, B, D), (H, D, E), (H, E, D))
    bufs = [_guarded(s, torch.float32) for s in shapes]
    ws = torch.full((max(ws_bytes, 16),), 0xFF, dtype=torch.uint8, device="cuda")
    w = (_p(ws) if ws_bytes else None, ws_bytes)
    o, dx, dw1, dw2 = (b[1] for b in bufs)
    if strided is None:
        _lib.check(L.fmlp_fwd_ws(_p(x), _p(w1), _p(w2), _p(o), H, B, D, E, F32, _lib.ACT_CODES[act], *w, _stream()), "fwd")
        _lib.check(L.fmlp_bwd(_p(x), _p(w1), _p(w2), _p(do), _p(dx), _p(dw1), _p(dw2), H, B, D, E, F32 | flags,
                              _lib.ACT_CODES[act], *w, _stream()), "bwd")
    else:
        st = [_lib.strides(t) for t in (strided, w1, w2, do)]
        _lib.check(L.fmlp_fwd_strided(_p(strided), _p(w1), _p(w2), _p(o), H, B, D, E, *st[:3], F32, _lib.ACT_CODES[act],
                                      _stream()), "fwd")
        _lib.check(L.fmlp_bwd_strided(_p(strided), _p(w1), _p(w2), _p(do), _p(dx), _p(dw1), _p(dw2), H, B, D, E, *st,
                                      F32 | flags, _lib.ACT_CODES[act], *w, _stream()), "bwd")
    torch.cuda.synchronize()
    for b, t in bufs:
        _check_guards(b, t.numel())
    return [t for _, t in bufs]


CASES = [
    # H, B, D, E, act
    (2, 1, 16, 1, "silu"), (2, 31, 32, 3, "sigmoid"), (3, 33, 64, 31, "leaky_relu"), (2, 129, 128, 33, "silu"),
    (1, 257, 16, 100, ""), (5, 1025, 32, 260, "silu"), (2, 2050, 64, 683, "silu"), (1, 1030, 128, 1022, "sigmoid"),
    (40, 300, 64, 96, "silu"), (70, 64, 16, 36, "leaky_relu"), (1, 5000, 64, 128, "silu"), (9, 700, 128, 96, "silu"),
]


@pytest.mark.parametrize("H,B,D,E,act", CASES)
def test_against_64_bits(H, B, D, E, act):
    print(f"[f32] H={H} B={B} D={D} E={E} act='{act}'", flush=True)
    L = _lib.lib()
    assert L.fmlp_shape_dense(D, E, F32) == 1
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, torch.float32, seed=B + E))
    ref = _exact(x, w1, w2, do, act)
    n = max(L.fmlp_bwd_workspace_bytes(H, B, D, E, F32), L.fmlp_fwd_workspace_bytes(H, B, D, E, F32))
    pad = (H * D * ((E + 3) // 4 * 4) * 4 + 255) // 256 * 256 if E % 4 else 0
    full = _run(x, w1, w2, do, act, 0, n)
    sums = (E, E, B, B)
    for name, a, r, k in zip(("o", "dx", "dw1", "dw2"), full, ref, sums):
        assert _rel(a, r) <= _bound(D, k), name
    # with room for the padded W1 copy alone B is not split: dX is the same bits
    lean = _run(x, w1, w2, do, act, 0, pad)
    assert torch.equal(lean[0], full[0]) and torch.equal(lean[1], full[1])
    for a, r in zip(lean[2:], ref[2:]):
        assert _rel(a, r) <= _bound(D, B)
    for flags in (_lib.FMLP_BWD_RECOMPUTE, _lib.FMLP_BWD_STORE_DZ, _lib.FMLP_DW_HILO, _lib.FMLP_OUT_F32):
        nf = max(L.fmlp_bwd_workspace_bytes(H, B, D, E, F32 | flags), n)
        f = _run(x, w1, w2, do, act, flags, nf)
        assert torch.equal(f[1], full[1]), hex(flags)  # dX is the same bits in every form
        for a, r in zip(f[2:], ref[2:]):
            assert _rel(a, r) <= _bound(D, B), hex(flags)


@pytest.mark.parametrize("H,B,D,E", [(2, 1030, 64, 683), (1, 4096, 128, 256)])
def test_partial_backward(H, B, D, E):
    L = _lib.lib()
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, torch.float32, seed=4))
    act = _lib.ACT_CODES["silu"]
    n = L.fmlp_bwd_workspace_bytes(H, B, D, E, F32)
    full = _run(x, w1, w2, do, "silu", 0, n)
    for flag in (_lib.FMLP_BWD_NO_DX, _lib.FMLP_BWD_NO_DW):
        nb = L.fmlp_bwd_workspace_bytes(H, B, D, E, F32 | flag)
        ws = torch.empty(max(nb, 16), dtype=torch.uint8, device="cuda")
        outs = [torch.empty_like(t) for t in (x, w1, w2)]
        keep = (False, True, True) if flag == _lib.FMLP_BWD_NO_DX else (True, False, False)
        _lib.check(L.fmlp_bwd(_p(x), _p(w1), _p(w2), _p(do), *(_p(o) if k else None for o, k in zip(outs, keep)), H, B,
                              D, E, F32 | flag, act, _p(ws), nb, _stream()), "bwd")
        torch.cuda.synchronize()
        for o, k, f in zip(outs, keep, full[1:]):
            assert not k or torch.equal(o, f), hex(flag)
    outs = [torch.empty_like(t) for t in (x, w1, w2)]
    _lib.check(L.fmlp_bwd_noalloc(_p(x), _p(w1), _p(w2), _p(do), *(_p(o) for o in outs), H, B, D, E, F32, act,
                                  _stream()), "bwd (no-alloc)")
    torch.cuda.synchronize()
    assert torch.equal(outs[0], full[1])
    ref = _exact(x, w1, w2, do, "silu")
    for a, r in zip(outs[1:], ref[2:]):
        assert _rel(a, r) <= _bound(D, B)


@pytest.mark.parametrize("what", ["x", "w1"])
def test_infinities_stay_where_the_generic_kernels_have_them(what):
    H, B, D, E = 2, 96, 32, 288  # whole tiles: inside a cut one both kernel sets multiply zeros
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, torch.float32, seed=3))
    (x if what == "x" else w1)[1, 5, 3] = float("inf")
    n = _lib.lib().fmlp_bwd_workspace_bytes(H, B, D, E, F32)
    own = _run(x, w1, w2, do, "sigmoid", 0, n)
    gen = _run(x, w1, w2, do, "sigmoid", 0, 0, strided=x.transpose(1, 2).contiguous().transpose(1, 2))
    for name, a, r in zip(("o", "dx", "dw1", "dw2"), own, gen):
        assert torch.equal(a.isfinite(), r.isfinite()), name
        fin = r.isfinite()
        assert _rel(a[fin], r[fin]) <= 1e-6, name  # two results within the bound of each other
