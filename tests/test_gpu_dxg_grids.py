"""The dX GEMM over the stored dZ on both sides of the line between its two kernels (small grids in
64-row workgroups, larger ones in 256-row blocks), at the edges of rows, chunks and E parts, from a
workspace that starts as NaN: dX against the recompute form's (fp32 sums in another order)."""
import pytest
import torch

from flashmlp_amd import _lib
from oracle.inputs import make_inputs
from test_gpu_odd_e import _DT, _bwd, _rel

pytestmark = pytest.mark.gpu

CASES = [
    # H, B, D, E: small grids (one row, one chunk, fewer chunks than E parts, ragged rows and chunks)
    (1, 1, 128, 8), (2, 63, 64, 32), (3, 65, 128, 96), (1, 129, 64, 136), (2, 300, 128, 1000), (1, 4097, 64, 264),
    (8, 4096, 64, 128),  # exactly two rounds of 64-row workgroups on 256 CUs
    # larger grids: one past the line, ragged rows, odd block counts
    (9, 4096, 64, 128), (140, 300, 128, 264), (600, 33, 64, 48), (70, 520, 128, 40),
]


@pytest.mark.parametrize("H,B,D,E", CASES)
@pytest.mark.parametrize("dt,act", [(torch.bfloat16, "silu"), (torch.float16, "sigmoid")], ids=["bf16", "fp16"])
def test_dx_from_stored_dz(H, B, D, E, dt, act):
    print(f"[dxg] H={H} B={B} D={D} E={E} {dt} act='{act}'", flush=True)
    L = _lib.lib()
    code = _DT[dt] | _lib.FMLP_BWD_STORE_DZ
    assert L.fmlp_bwd_stores_dz(H, B, D, E, code, _lib.ACT_CODES[act]) == 1
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=B + E))
    f32 = _lib.FMLP_OUT_F32
    n = L.fmlp_bwd_workspace_bytes(H, B, D, E, code | f32)
    nr = L.fmlp_bwd_workspace_bytes(H, B, D, E, _DT[dt] | f32 | _lib.FMLP_BWD_RECOMPUTE)
    sums = _bwd(x, w1, w2, do, act, _lib.FMLP_BWD_STORE_DZ | f32, n, torch.float32)
    rec = _bwd(x, w1, w2, do, act, _lib.FMLP_BWD_RECOMPUTE | f32, nr, torch.float32)
    assert all(torch.isfinite(t).all() for t in sums)
    assert _rel(sums[0], rec[0]) <= 1e-6  # the same dZ bits, E / 2 additions in another order
    io = _bwd(x, w1, w2, do, act, _lib.FMLP_BWD_STORE_DZ, n, dt)
    for name, a, s in zip(("dx", "dw1", "dw2"), io, sums):
        assert torch.equal(a, s.to(dt)), name
    again = _bwd(x, w1, w2, do, act, _lib.FMLP_BWD_STORE_DZ, n, dt)
    for a, b in zip(io, again):
        assert torch.equal(a, b)
