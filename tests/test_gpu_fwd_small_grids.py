"""The D = 128 and D = 256 forward on grids that leave half the CUs idle: 128-row tiles of two E parts
(D = 128), and every tile split over workgroups when E is long enough, at the edges of rows, chunks
and parts, with and without a workspace, from outputs and workspaces that start as NaN."""
import pytest
import torch

from flashmlp_amd import _lib
from oracle import emulate
from oracle.inputs import make_inputs
from test_gpu_fwd_split import _DT, _cus, _fwd, _normrel

pytestmark = pytest.mark.gpu

CASES = [
    # H, B, D, E: one chunk, one chunk per part, uneven parts, ragged rows and chunks, one workgroup
    # split over many, all tiles split, the line at half the CUs (None: B from the CU count)
    (1, 1, 128, 8), (2, 129, 128, 64), (3, 255, 128, 96), (2, 33, 128, 296), (1, 300, 128, 683), (4, 257, 128, 2040),
    (16, 1000, 128, 1024), (1, None, 128, 72), (1, 1, 256, 8), (2, 129, 256, 96), (1, 33, 256, 683), (4, 257, 256, 2040),
    (1, None, 256, 72),
]


@pytest.mark.parametrize("H,B,D,E", CASES)
@pytest.mark.parametrize("dt,act", [(torch.bfloat16, "silu"), (torch.float16, "sigmoid")], ids=["bf16", "fp16"])
def test_small_grid_forward(H, B, D, E, dt, act):
    rows = 256 if D == 128 else 128
    B = _cus() // 2 * rows if B is None else B
    print(f"[fwd-small] H={H} B={B} D={D} E={E} {dt} act='{act}'", flush=True)
    L = _lib.lib()
    code = _DT[dt]
    n = L.fmlp_fwd_workspace_bytes(H, B, D, E, code)
    if E >= 2040:
        assert n > 0, "a long E must be split over workgroups"
    x, w1, w2, _ = make_inputs(H, B, D, E, dt, 1.0, seed=B + E, with_do=False)
    xd, w1d, w2d = (t.cuda() for t in (x, w1, w2))
    ref = emulate.emu_fwd(x, w1, w2, act, dt, round_out=False)
    for nb in {0, n}:
        ws = torch.full((nb // 4,), float("nan"), device="cuda") if nb else None
        s = _fwd(L, xd, w1d, w2d, act, code | _lib.FMLP_OUT_F32, torch.float32, ws, nb, fill_nan=True)
        assert torch.isfinite(s).all()
        # fp32 sums of the same rounded h up to its rounding ties (the bar of the other forward tests)
        assert _normrel(s.cpu(), ref) <= 1e-4
        o = _fwd(L, xd, w1d, w2d, act, code, dt, ws, nb, fill_nan=True)
        assert torch.equal(o, s.to(dt))
        assert torch.equal(o, _fwd(L, xd, w1d, w2d, act, code, dt, ws, nb))
    if n and E % 8 == 0:  # a workspace too small for every part: fmlp_fwd's bits
        ws = torch.empty(n - 16, dtype=torch.uint8, device="cuda")
        assert torch.equal(_fwd(L, xd, w1d, w2d, act, code, dt, ws, n - 16), _fwd(L, xd, w1d, w2d, act, code, dt))


@pytest.mark.parametrize("D,E", [(128, 96), (128, 2016), (256, 96), (256, 2016)])
def test_small_grid_infinite_rows(D, E):
    # an infinite x saturates the sigmoid: chunks that a part does not have must not turn it into NaN
    H, B, dt = 2, 40, torch.bfloat16
    L = _lib.lib()
    x, w1, w2, _ = make_inputs(H, B, D, E, dt, 1.0, seed=5, with_do=False)
    w1[w1 == 0] = 0.125  # inf * 0 is the oracle's NaN
    x[:, 3, 7] = float("inf")
    x[:, 20, 0] = float("-inf")
    n = L.fmlp_fwd_workspace_bytes(H, B, D, E, _DT[dt])
    ws = torch.empty(n, dtype=torch.uint8, device="cuda") if n else None
    print(f"[fwd-small] infinite rows D={D} E={E} ws={n}", flush=True)
    s = _fwd(L, x.cuda(), w1.cuda(), w2.cuda(), "sigmoid", _DT[dt] | _lib.FMLP_OUT_F32, torch.float32, ws, n)
    ref = emulate.emu_fwd(x, w1, w2, "sigmoid", dt, round_out=False)
    assert torch.isfinite(ref).all()
    assert _normrel(s.cpu(), ref) <= 1e-4
