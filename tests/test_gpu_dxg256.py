"""The stored-dZ form at D = 256 (dw256_kernel storing dZ, dxg256_kernel): the same bits as the
recomputing programs in every output, from a workspace that starts as NaN, at the edges of the
128-row tiles, the 256-row dZ blocks, the chunks of E and a B split."""
import pytest
import torch

from flashmlp_amd import _lib
from oracle.inputs import make_inputs
from test_gpu_odd_e import _DT, _bwd

pytestmark = pytest.mark.gpu

CASES = [(2, 1, 8), (3, 127, 136), (2, 128, 96), (1, 129, 45), (5, 300, 264), (2, 2100, 1000), (9, 513, 32)]


@pytest.mark.parametrize("H,B,E", CASES)
@pytest.mark.parametrize("dt,act", [(torch.bfloat16, "silu"), (torch.float16, "leaky_relu"), (torch.float16, "sigmoid"),
                                    (torch.bfloat16, "")], ids=["bf16-silu", "fp16-leaky", "fp16-sigmoid", "bf16-linear"])
def test_same_bits_as_the_recompute_form(H, B, E, dt, act):
    print(f"[dxg256] H={H} B={B} E={E} {dt} act='{act}'", flush=True)
    L = _lib.lib()
    D, code = 256, _DT[dt]
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=B + E))
    assert L.fmlp_bwd_stores_dz(H, B, D, E, code, _lib.ACT_CODES[act]) == 1
    assert L.fmlp_bwd_stores_dz(H, B, D, E, code | _lib.FMLP_BWD_RECOMPUTE, _lib.ACT_CODES[act]) == 0
    need = H * -(-E // 128) * 128 * -(-B // 256) * 256 * 2
    for mode in (0, _lib.FMLP_DW_HILO):
        for out in (_lib.FMLP_OUT_F32, 0):
            f = mode | out
            odt = torch.float32 if out else dt
            n = L.fmlp_bwd_workspace_bytes(H, B, D, E, code | f)
            nr = L.fmlp_bwd_workspace_bytes(H, B, D, E, code | f | _lib.FMLP_BWD_RECOMPUTE)
            assert n >= need and nr <= n
            stored = _bwd(x, w1, w2, do, act, f, n, odt)
            rec = _bwd(x, w1, w2, do, act, f | _lib.FMLP_BWD_RECOMPUTE, nr, odt)
            for name, a, b in zip(("dx", "dw1", "dw2"), stored, rec):
                assert torch.isfinite(a).all() and torch.equal(a, b), (name, hex(f))
    # a workspace that holds no dZ (E % 8 != 0: W1's padded copy alone): the recompute form
    n = (H * D * -(-E // 8) * 8 * 2 + 255) // 256 * 256 if E % 8 else 0
    for a, b in zip(_bwd(x, w1, w2, do, act, 0, n, dt), _bwd(x, w1, w2, do, act, _lib.FMLP_BWD_RECOMPUTE, n, dt)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("H,B,E", [(1, 33, 2048), (1, 1000, 2048), (3, 129, 1500), (2, 300, 1355)])
@pytest.mark.parametrize("dt,act", [(torch.bfloat16, "silu"), (torch.float16, "sigmoid")], ids=["bf16", "fp16"])
def test_tiles_split_over_e(H, B, E, dt, act):
    # grids that leave the chip idle: the recompute form's sums in another order, also from a
    # workspace too short for every part
    print(f"[dxg256-split] H={H} B={B} E={E} {dt} act='{act}'", flush=True)
    L = _lib.lib()
    D, code = 256, _DT[dt]
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=B + E))
    f = _lib.FMLP_OUT_F32
    n = L.fmlp_bwd_workspace_bytes(H, B, D, E, code | f)
    sums = _bwd(x, w1, w2, do, act, f, n, torch.float32)
    rec = _bwd(x, w1, w2, do, act, f | _lib.FMLP_BWD_RECOMPUTE, n, torch.float32)
    assert all(torch.isfinite(t).all() for t in sums)
    assert not torch.equal(sums[0], rec[0]), "the case must split its tiles"
    assert ((sums[0] - rec[0]).norm() / rec[0].norm()).item() <= 1e-6  # the same dZ bits, E / 2 additions regrouped
    assert torch.equal(sums[1], rec[1]) and torch.equal(sums[2], rec[2])
    for flags in (0, _lib.FMLP_DW_HILO):  # dX does not depend on the dW mode; repeats agree
        nf = L.fmlp_bwd_workspace_bytes(H, B, D, E, code | flags)
        assert torch.equal(_bwd(x, w1, w2, do, act, flags, nf, dt)[0], sums[0].to(dt))
    short = _bwd(x, w1, w2, do, act, f, n - 16, torch.float32)  # whole tiles
    assert ((short[0] - rec[0]).norm() / rec[0].norm()).item() <= 1e-6


@pytest.mark.parametrize("H,B,E", [(1, 33, 2048), (2, 300, 1355)])
def test_a_workspace_too_short_for_every_part_takes_whole_tiles(H, B, E):
    # dX has the split's bits or the recompute form's, nothing between them
    L = _lib.lib()
    D, dt, act = 256, torch.bfloat16, "silu"
    x, w1, w2, do = (t.cuda() for t in make_inputs(H, B, D, E, dt, seed=B + E))
    f = _lib.FMLP_OUT_F32
    n = L.fmlp_bwd_workspace_bytes(H, B, D, E, _DT[dt] | f)
    rec = _bwd(x, w1, w2, do, act, f | _lib.FMLP_BWD_RECOMPUTE, n, torch.float32)
    assert not torch.equal(_bwd(x, w1, w2, do, act, f, n, torch.float32)[0], rec[0]), "the case must split its tiles"
    for short in (n - 16, n - H * -(-B // 128) * 128 * 256 * 4):  # one part of each tile less
        print(f"[dxg256-short] H={H} B={B} E={E} workspace {short} of {n}", flush=True)
        assert torch.equal(_bwd(x, w1, w2, do, act, f, short, torch.float32)[0], rec[0])
