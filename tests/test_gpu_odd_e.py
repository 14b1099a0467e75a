"""E that is no multiple of 8 on the tuned kernels (W1 through its padded copy in the workspace).

The same call without room for the copy runs on the generic kernels, so every form is compared
with them: the unrounded fp32 sums (FMLP_OUT_F32) within 1e-4 normwise, the bar of the other
fp32-sum tests (another summation order, and the rare one-ulp flip of an io-rounded h or dZ).
Outputs lie between sentinel guards, which must stay untouched (dW1's rows are no longer vectors,
and E cuts the kernels' column groups).
"""
import ctypes
import sys

import pytest
import torch

from flashmlp_amd import _lib
from oracle import emulate
from oracle.inputs import make_inputs

pytestmark = pytest.mark.gpu

_DT = {torch.float16: _lib.FMLP_DTYPE_F16, torch.bfloat16: _lib.FMLP_DTYPE_BF16}
GUARD = 64  # elements on each side of an output
SENTINEL = 0x5A


def _p(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _guarded(shape, dtype):
    """(whole buffer, the output inside it filled with NaN bytes)"""
    n = 1
    for s in shape:
        n *= s
    buf = torch.empty(n + 2 * GUARD, dtype=dtype, device="cuda")
    buf.view(torch.uint8).fill_(SENTINEL)
    out = buf[GUARD:GUARD + n].view(shape)
    out.view(torch.uint8).fill_(0xFF)
    return buf, out


def _check_guards(buf, n):
    b = buf.view(torch.uint8)
    es = buf.element_size()
    assert bool((b[:GUARD * es] == SENTINEL).all()) and bool((b[(GUARD + n) * es:] == SENTINEL).all()), "guard written"


def _rel(a, b):
    a, b = a.double(), b.double()
    return ((a - b).norm() / b.norm().clamp_min(1e-30)).item()


def _bwd(x, w1, w2, do, act, flags, ws_bytes, dtype_out):
    L = _lib.lib()
    H, B, D = x.shape
    E = w1.shape[2]
    bufs = [_guarded(s, dtype_out) for s in ((H, B, D), (H, D, E), (H, E, D))]
    want = (not flags & _lib.FMLP_BWD_NO_DX, not flags & _lib.FMLP_BWD_NO_DW, not flags & _lib.FMLP_BWD_NO_DW)
    ws = torch.full((ws_bytes,), 0xFF, dtype=torch.uint8, device="cuda") if ws_bytes else None
    st = L.fmlp_bwd(_p(x), _p(w1), _p(w2), _p(do), *(_p(o) if k else None for (_, o), k in zip(bufs, want)), H, B, D, E,
                    _DT[x.dtype] | flags, _lib.ACT_CODES[act], _p(ws), ws_bytes, _stream())
    _lib.check(st, "backward")
    torch.cuda.synchronize()
    for b, o in bufs:
        _check_guards(b, o.numel())
    return [o if k else None for (_, o), k in zip(bufs, want)]


CASES = [
    # H, B, D, E: E below one vector, one past a tile, E % 4 == 0, E % 2 == 0, odd; B tails
    (2, 33, 64, 3), (3, 300, 128, 33), (2, 257, 256, 129), (2, 1000, 64, 100), (1, 4097, 128, 1022),
    (4, 1025, 128, 683), (2, 3000, 256, 45), (8, 4097, 64, 130),
]


@pytest.mark.parametrize("H,B,D,E", CASES)
@pytest.mark.parametrize("dt,act", [(torch.bfloat16, "silu"), (torch.float16, "sigmoid")], ids=["bf16", "fp16"])
def test_against_the_generic_kernels(H, B, D, E, dt, act):
    print(f"[odd E] H={H} B={B} D={D} E={E} {dt} act='{act}'", flush=True)
    sys.stdout.flush()
    L = _lib.lib()
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=E))
    code = _DT[dt] | _lib.FMLP_OUT_F32
    assert L.fmlp_shape_dense(D, E, code) == 1 and L.fmlp_shape_tuned(D, E, code) == 0
    n = L.fmlp_fwd_workspace_bytes(H, B, D, E, code)
    assert n >= H * D * ((E + 7) // 8 * 8) * 2
    outs = []
    for size in (n, 0):  # with the padded copy; without a workspace: the generic kernels
        buf, o = _guarded((H, B, D), torch.float32)
        ws = torch.full((n,), 0xFF, dtype=torch.uint8, device="cuda")
        _lib.check(L.fmlp_fwd_ws(_p(x), _p(w1), _p(w2), _p(o), H, B, D, E, code, _lib.ACT_CODES[act],
                                 _p(ws) if size else None, size, _stream()), "forward")
        torch.cuda.synchronize()
        _check_guards(buf, o.numel())
        outs.append(o)
    assert _rel(outs[0], outs[1]) <= 1e-4
    f32 = _lib.FMLP_OUT_F32
    gen = _bwd(x, w1, w2, do, act, f32, 0, torch.float32)
    gen_hilo = _bwd(x, w1, w2, do, act, f32 | _lib.FMLP_DW_HILO, 0, torch.float32)
    for flags in (0, _lib.FMLP_BWD_RECOMPUTE, _lib.FMLP_BWD_STORE_DZ, _lib.FMLP_DW_HILO, _lib.FMLP_BWD_NO_DX,
                  _lib.FMLP_BWD_NO_DW):
        nb = L.fmlp_bwd_workspace_bytes(H, B, D, E, code | flags)
        own = _bwd(x, w1, w2, do, act, f32 | flags, nb, torch.float32)
        ref = gen_hilo if flags & _lib.FMLP_DW_HILO else gen
        for name, a, r in zip(("dx", "dw1", "dw2"), own, ref):
            if a is not None:
                assert _rel(a, r) <= 1e-4, (hex(flags), name)
        io = _bwd(x, w1, w2, do, act, flags, nb, dt)  # the io-dtype stores of the same sums
        for name, a, r in zip(("dx", "dw1", "dw2"), io, own):
            if a is not None:
                assert torch.equal(a, r.to(dt)), (hex(flags), name)


def test_workspace_between_the_copy_and_the_plan():
    # room for the padded copy but not for the plan's partials: a plan that fits, same results
    H, B, D, E, act = 2, 4096, 128, 203, "silu"
    L = _lib.lib()
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, torch.bfloat16, seed=5))
    code = _DT[torch.bfloat16] | _lib.FMLP_OUT_F32
    n = L.fmlp_bwd_workspace_bytes(H, B, D, E, code)
    pad = (H * D * 208 * 2 + 255) // 256 * 256
    assert n > pad + 4096
    gen = _bwd(x, w1, w2, do, act, _lib.FMLP_OUT_F32, 0, torch.float32)
    for size in (pad - 16, pad, pad + 4096, n):
        own = _bwd(x, w1, w2, do, act, _lib.FMLP_OUT_F32, size, torch.float32)
        for a, r in zip(own, gen):
            assert _rel(a, r) <= 1e-4, size
    bufs = [_guarded(s, torch.float32) for s in ((H, B, D), (H, D, E), (H, E, D))]
    st = L.fmlp_bwd_noalloc(_p(x), _p(w1), _p(w2), _p(do), *(_p(o) for _, o in bufs), H, B, D, E, code,
                            _lib.ACT_CODES[act], _stream())
    _lib.check(st, "backward (no-alloc)")
    torch.cuda.synchronize()
    for (b, o), r in zip(bufs, gen):
        _check_guards(b, o.numel())
        assert _rel(o, r) <= 1e-4


@pytest.mark.parametrize("H,B,D,E", [(2, 96, 128, 45), (2, 32, 64, 683), (2, 96, 64, 45), (1, 1056, 128, 683),
                                     (3, 160, 64, 100), (2, 96, 256, 45)])
def test_infinite_weights_stay_where_the_generic_kernels_have_them(H, B, D, E):
    """A row range with an odd number of 32-row subtiles: the row sets without one of their own must not
    add the NaN that an infinite weight makes of the zeros behind the last row."""
    dt, act = torch.float16, "sigmoid"
    print(f"[odd E] infinite w1 H={H} B={B} D={D} E={E}", flush=True)
    L = _lib.lib()
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=3))
    w1[H - 1, 5, 3] = float("inf")
    f32 = _lib.FMLP_OUT_F32
    gen = _bwd(x, w1, w2, do, act, f32, 0, torch.float32)
    assert gen[2].isfinite().all() and not gen[0].isfinite().all()
    for flags in (0, _lib.FMLP_BWD_RECOMPUTE, _lib.FMLP_BWD_STORE_DZ, _lib.FMLP_DW_HILO, _lib.FMLP_BWD_NO_DX):
        n = L.fmlp_bwd_workspace_bytes(H, B, D, E, _DT[dt] | f32 | flags)
        own = _bwd(x, w1, w2, do, act, f32 | flags, n, torch.float32)
        for name, a, r in zip(("dx", "dw1", "dw2"), own, gen):
            if a is not None:
                fin = r.isfinite()
                assert torch.equal(a.isfinite(), fin), (hex(flags), name)
                # (HILO carries h and dZ with twice the bits: the io type's rounding apart)
                assert _rel(a[fin], r[fin]) <= (5e-3 if flags & _lib.FMLP_DW_HILO else 1e-4), (hex(flags), name)


@pytest.mark.parametrize("E", [1, 45, 100, 88, 130])
def test_d256_one_row_range(E):
    """D = 256 and at most 32 rows: one program per E tile writes dW1 and dW2 themselves (no partials), as
    vectors where E % 4 == 0 and else element by element. The unrounded sums against the generic kernels,
    the io-dtype outputs bitwise the rounding of those sums, guards untouched."""
    H, B, D, dt, act = 3, 28, 256, torch.bfloat16, "silu"
    print(f"[odd E] one row range H={H} B={B} D={D} E={E}", flush=True)
    L = _lib.lib()
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=E))
    f32 = _lib.FMLP_OUT_F32
    # (E % 8 == 0 needs no workspace for kernels of its own: the oracle below bounds that call as well)
    gen = _bwd(x, w1, w2, do, act, f32, 0, torch.float32)
    for flags in (0, _lib.FMLP_BWD_RECOMPUTE, _lib.FMLP_BWD_NO_DX):
        n = L.fmlp_bwd_workspace_bytes(H, B, D, E, _DT[dt] | f32 | flags)
        own = _bwd(x, w1, w2, do, act, f32 | flags, n, torch.float32)
        io = _bwd(x, w1, w2, do, act, flags, n, dt)
        for name, a, r, o in zip(("dx", "dw1", "dw2"), own, gen, io):
            if a is not None:
                assert _rel(a, r) <= 1e-4, (hex(flags), name)
                assert torch.equal(o, a.to(dt)), (hex(flags), name)
    ref = emulate.emu_bwd(*(t.cpu() for t in (x, w1, w2, do)), act, dt, round_out=False)
    for name, a, r in zip(("dx", "dw1", "dw2"), gen, ref):
        assert _rel(a.cpu(), r) <= 1e-4, name
