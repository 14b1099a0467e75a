"""The generic kernels (fmlp_gen.hip) against the CPU oracle, through the C ABI calls that reach them.

Dense tensors of nearly every shape run on kernels of their own (fmlp_shape_dense). The generic
kernels take what is left: views (here W2 with padded rows, which no other kernel reads), bases that
are not 16-byte aligned, E % 8 != 0 without room for the padded copy of W1, and fp32 at D = 256. The
tests of the other kernels compare with them, so their own parity is pinned here: every D and dtype,
cut tiles of E and B, the B split of the dW programs, the hi/lo dW mode, the unrounded sums, and
views of every input read in place. Bars: tests/test_gpu_generic.py's.
"""
import pytest
import torch

from flashmlp_amd import _lib
from oracle import emulate, reference
from oracle.inputs import make_inputs
from test_gpu_generic import _fail_frac, _normrel
from test_gpu_odd_e import _p, _stream

pytestmark = pytest.mark.gpu

CODE = {torch.float16: _lib.FMLP_DTYPE_F16, torch.bfloat16: _lib.FMLP_DTYPE_BF16, torch.float32: _lib.FMLP_DTYPE_F32}


def _padded_rows(t, by=8):
    return torch.empty(*t.shape[:2], t.shape[2] + by, dtype=t.dtype, device="cuda")[:, :, :t.shape[2]].copy_(t)


def _call(x, w1, w2, do, act, flags=0, ws_bytes=0):
    """o, dx, dw1, dw2 through the strided entry points, from outputs that start as NaN"""
    L = _lib.lib()
    (H, B, D), E = x.shape, w1.shape[2]
    code, a = CODE[x.dtype] | flags, _lib.ACT_CODES[act]
    out = torch.float32 if flags & _lib.FMLP_OUT_F32 else x.dtype
    outs = [torch.full(s, float("nan"), dtype=out, device="cuda") for s in ((H, B, D), (H, B, D), (H, D, E), (H, E, D))]
    ws = torch.full((ws_bytes,), 0xFF, dtype=torch.uint8, device="cuda") if ws_bytes else None
    st = [_lib.strides(t) for t in (x, w1, w2, do)]
    _lib.check(L.fmlp_fwd_strided(_p(x), _p(w1), _p(w2), _p(outs[0]), H, B, D, E, *st[:3],
                                  code & ~_lib.FMLP_DW_HILO, a, _stream()), "forward")
    _lib.check(L.fmlp_bwd_strided(_p(x), _p(w1), _p(w2), _p(do), *(_p(t) for t in outs[1:]), H, B, D, E, *st, code, a,
                                  _p(ws), ws_bytes, _stream()), "backward")
    torch.cuda.synchronize()
    return outs


def _inputs(H, B, D, E, dt, seed):
    """the oracle's tensors and the GPU's, W2 as a view of padded rows"""
    cpu = make_inputs(H, B, D, E, dt, seed=seed)
    x, w1, w2, do = (t.cuda() for t in cpu)
    return cpu, (x, w1, _padded_rows(w2), do)


def _check16(cpu, got, act, dt):
    ro, rdx, rdw1, rdw2 = reference.autograd_grads(*cpu, act)
    eo = emulate.emu_fwd(*cpu[:3], act, dt)
    _, edw1, edw2 = emulate.emu_bwd(*cpu, act, dt)
    o, dx, dw1, dw2 = (t.cpu() for t in got)
    assert _fail_frac(o, ro) == 0 and _fail_frac(o, eo) == 0 and _fail_frac(dx, rdx) == 0
    assert _fail_frac(dw1, edw1) == 0 and _fail_frac(dw2, edw2) == 0
    assert _normrel(dw1, rdw1) <= 1e-2 and _normrel(dw2, rdw2) <= 1e-2


def _kernels(run):
    run()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        run()
        torch.cuda.synchronize()
    return [e.name for e in prof.events() if e.device_type == torch.autograd.DeviceType.CUDA and "fmlp" in e.name]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_the_calls_reach_the_generic_kernels(dt):
    H, B, D, E = 2, 70, 64, 45
    _, (x, w1, w2v, do) = _inputs(H, B, D, E, dt, 1)
    w2 = w2v.contiguous()
    off = torch.empty(x.numel() + 1, dtype=dt, device="cuda")[1:].view_as(x).copy_(x)
    for args in ((x, w1, w2v, do), (off, w1, w2, do), (x, w1, w2, do)):  # a view, a misaligned base, no workspace
        names = _kernels(lambda: _call(*args, "silu"))
        assert len(names) == 3 and all("gen_" in n for n in names), names


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("act", ["silu", "leaky_relu", "sigmoid", ""])
def test_16bit(D, dt, act):
    H, B, E = 2, 77, 45  # cut tiles of B and E
    print(f"[gen] H={H} B={B} D={D} E={E} {dt} act='{act}'", flush=True)
    cpu, args = _inputs(H, B, D, E, dt, D)
    _check16(cpu, _call(*args, act), act, dt)


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("act", ["silu", "leaky_relu", "sigmoid", ""])
def test_fp32(D, act):
    H, B, E = 2, 150, 200
    print(f"[gen] fp32 H={H} B={B} D={D} E={E} act='{act}'", flush=True)
    cpu, args = _inputs(H, B, D, E, torch.float32, 7)
    for g, r in zip(_call(*args, act), reference.autograd_grads(*cpu, act)):
        assert _normrel(g.cpu(), r) <= 1e-4


@pytest.mark.parametrize("D,dt,act", [(16, torch.float16, "silu"), (32, torch.bfloat16, "silu"),
                                      (128, torch.bfloat16, "leaky_relu"), (256, torch.float16, "sigmoid"),
                                      (64, torch.float32, "leaky_relu"), (256, torch.float32, "silu")])
def test_b_split(D, dt, act):
    """dW programs of a B range each with fp32 partials in the workspace, against the oracle and the
    unsplit call; dX does not depend on the split."""
    H, B, E = 2, 3000, 136
    print(f"[gen] B split H={H} B={B} D={D} E={E} {dt} act='{act}'", flush=True)
    cpu, args = _inputs(H, B, D, E, dt, 81)
    f32 = _lib.FMLP_OUT_F32
    split, whole = _call(*args, act, f32, 64 << 20), _call(*args, act, f32, 0)
    assert torch.equal(split[1], whole[1])
    for a, b in zip(split[2:], whole[2:]):
        assert not torch.equal(a, b) and _normrel(a, b) <= 1e-5  # another order of 3000 fp32 additions
    got = _call(*args, act, 0, 64 << 20)
    if dt == torch.float32:
        for g, r in zip(got, reference.autograd_grads(*cpu, act)):
            assert _normrel(g.cpu(), r) <= 1e-4
        return
    _check16(cpu, got, act, dt)
    _, edw1, edw2 = emulate.emu_bwd(*cpu, act, dt, round_out=False)
    for a, e in zip(split[2:], (edw1, edw2)):
        assert _normrel(a.cpu(), e) <= 1e-4  # the fp32-sum bar: rounding flips of h and dZ


@pytest.mark.parametrize("ws_bytes", [0, 64 << 20])
@pytest.mark.parametrize("D", [32, 256])
def test_accurate_dw(D, ws_bytes):
    H, B, E = 2, 3000, 40
    cpu, args = _inputs(H, B, D, E, torch.bfloat16, 13)
    got = _call(*args, "silu", _lib.FMLP_DW_HILO, ws_bytes)
    assert torch.equal(got[1], _call(*args, "silu", 0, ws_bytes)[1])
    _, _, rdw1, rdw2 = reference.autograd_grads(*cpu, "silu")
    assert _fail_frac(got[2].cpu(), rdw1) == 0 and _fail_frac(got[3].cpu(), rdw2) == 0


@pytest.mark.parametrize("D", [16, 32, 128, 256])
def test_unrounded_sums(D):
    H, B, E = 2, 90, 72
    cpu, args = _inputs(H, B, D, E, torch.bfloat16, 12)
    got = _call(*args, "silu", _lib.FMLP_OUT_F32)
    ref = (emulate.emu_fwd(*cpu[:3], "silu", torch.bfloat16, round_out=False),
           *emulate.emu_bwd(*cpu, "silu", torch.bfloat16, round_out=False))
    for a, b in zip(got, ref):
        assert _normrel(a.cpu(), b) <= 1e-4


@pytest.mark.parametrize("D,dt", [(32, torch.bfloat16), (256, torch.float16), (64, torch.float32), (128, torch.bfloat16)])
def test_views_are_read_in_place(D, dt):
    """Views of every input, bit-identical to the same values through the other views."""
    H, B, E = 3, 70, 44
    _, (x, w1, w2v, do) = _inputs(H, B, D, E, dt, 8)
    ref = _call(x, w1, w2v, do, "silu", 0, 64 << 20)
    xt = x.transpose(0, 1).contiguous().transpose(0, 1)  # heads inside the rows
    xc = x.transpose(1, 2).contiguous().transpose(1, 2)  # columns inside out
    w1w = torch.full((H, D, E + 24), float("nan"), dtype=dt, device="cuda")[:, :, 5:5 + E]  # not 16-byte aligned
    w1w.copy_(w1)
    w1t = w1.transpose(1, 2).contiguous().transpose(1, 2)
    w2t = w2v.transpose(1, 2).contiguous().transpose(1, 2)
    dt_ = do.transpose(0, 1).contiguous().transpose(0, 1)
    for args in ((xt, w1, w2v, do), (xc, w1w, w2v, do), (x, w1t, w2t, dt_), (xt, w1w, w2t, do.clone())):
        for a, b in zip(_call(*args, "silu", 0, 64 << 20), ref):
            assert torch.equal(a, b)
    row = do[:, :1].expand(H, B, D)  # the gradient of a sum over rows: a stride of zero
    one = x[:1].expand(H, B, D)      # one input for every head
    for a, b in zip(_call(one, w1, w2v, row, "silu"), _call(one.contiguous(), w1, w2v, row.contiguous(), "silu")):
        assert torch.equal(a, b)
