"""The work a program has this framework do, as cases that can be timed and checked.

A case is one call pattern through the public entry points: a forward alone
(``flashmlp_fwd``), a forward and its backward (``flashmlp_fwd`` + ``flashmlp_bwd``), or the
``FlashMLP`` module under autograd with an input per head or one input shared by every head.
``listed()`` holds the representative ones, ``draw(rng)`` gives further ones of the same ranges.

Sizes: H heads, B rows, D hidden columns, E intermediate columns; u = H B D E. Inputs follow
the distributions of the repository's configurations: X ~ N(0, 1) (N(0, 4) where ``x_std`` is 2),
W1 ~ N(0, 1/D), W2 ~ N(0, 1/E), dO ~ N(0, 1).
"""
import math

import torch

from flashmlp_amd import FlashMLP, flashmlp_bwd, flashmlp_fwd

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_BYTES = {"fp16": 2, "bf16": 2, "fp32": 4}


def _case(kind, dtype, act, H, B, D, E, x_std=1.0, accurate_dw=False, name=None):
    c = {"kind": kind, "dtype": dtype, "act": act, "H": H, "B": B, "D": D, "E": E, "x_std": x_std,
         "accurate_dw": accurate_dw}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one small inference request: a few tens of rows, all latency
        _case("fwd", "bf16", "silu", 8, 33, 64, 512, name="infer_tiny"),
        # a small training step, one round of short tiles (an fp16 configuration of the benchmark)
        _case("step", "fp16", "silu", 12, 1024, 64, 768, name="step_small"),
        # the module under autograd at a middle size, as a training loop calls it
        _case("module", "bf16", "silu", 16, 2048, 64, 1024, name="module_mid"),
        # one activation matrix through every head (2-D input, mean over heads), with the
        # weight gradients' accuracy mode on
        _case("shared", "bf16", "silu", 16, 4096, 128, 512, accurate_dw=True, name="module_shared"),
        # a middle-sized training step with a piecewise linear activation
        _case("step", "bf16", "leaky_relu", 16, 8192, 128, 512, name="step_leaky"),
        # the training-scale step the headline metric is quoted on
        _case("step", "bf16", "silu", 32, 16384, 128, 1024, name="step_large"),
        # long-batch inference, forward only
        _case("fwd", "fp16", "sigmoid", 8, 65536, 64, 2048, name="infer_long"),
        # rows one past a tile multiple, saturated sigmoid
        _case("step", "fp16", "sigmoid", 8, 4097, 64, 2048, x_std=2.0, name="step_ragged"),
        # full precision training (the reference's fp32 configuration)
        _case("step", "fp32", "silu", 12, 1024, 64, 768, name="step_fp32"),
        # wide heads
        _case("step", "bf16", "silu", 8, 4096, 256, 1024, name="step_wide"),
        # narrow heads
        _case("step", "bf16", "silu", 32, 4096, 32, 512, name="step_narrow"),
        # an intermediate size that is no multiple of anything (2/3 of 1024), ragged rows
        _case("step", "bf16", "silu", 16, 4095, 128, 683, name="step_odd"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# The largest work a drawn case may have, in units of u = H B D E: the largest listed case's for
# 16-bit tuned sizes, less where the listed cases of that type and alignment are smaller.
_U_MAX = 32 * 16384 * 128 * 1024
_U_ODD = 16 * 4095 * 128 * 683
_U_FP32 = 12 * 1024 * 64 * 768


def draw(rng):
    """One more case: sizes over the whole range of the listed ones, odd ones among them."""
    while True:
        kind = rng.choice(["fwd", "step", "step", "step", "module", "shared"])
        dtype = rng.choice(["fp16", "bf16", "bf16", "bf16", "fp32"])
        act = rng.choice(["silu", "silu", "leaky_relu", "sigmoid", ""])
        H = _log_int(rng, 1, 32)
        B = _log_int(rng, 16, 65536 if kind == "fwd" else 16384)
        D = rng.choice([16, 32, 64, 64, 128, 128, 256])
        E = _log_int(rng, 64, 2048)
        if rng.random() < 0.7:
            E = max(64, E // 64 * 64)
        if rng.random() < 0.5:
            B = max(16, B // 64 * 64)
        x_std = 2.0 if act == "sigmoid" else 1.0
        accurate = kind != "fwd" and dtype != "fp32" and D <= 128 and rng.random() < 0.2
        u = H * B * D * E
        cap = _U_FP32 if dtype == "fp32" else _U_ODD if (E % 8 or D < 64 or accurate) else _U_MAX
        if u <= cap and u >= 1 << 19:
            return _case(kind, dtype, act, H, B, D, E, x_std=x_std, accurate_dw=accurate)


def _inputs(case, seed):
    """x, w1, w2 and the gradient of the output, made on the GPU from the seed alone."""
    H, B, D, E = case["H"], case["B"], case["D"], case["E"]
    dt = _DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(shape, std):
        return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std).to(dt)

    rows = (B, D) if case["kind"] == "shared" else (H, B, D)
    x = normal(rows, case["x_std"])
    w1 = normal((H, D, E), 1.0 / math.sqrt(D))
    w2 = normal((H, E, D), 1.0 / math.sqrt(E))
    dout = normal(rows, 1.0) if case["kind"] != "fwd" else None
    return x, w1, w2, dout


def prepare(case, seed):
    x, w1, w2, dout = _inputs(case, seed)
    state = {"kind": case["kind"], "act": case["act"], "accurate_dw": case["accurate_dw"], "x": x, "w1": w1,
             "w2": w2, "dout": dout}
    if case["kind"] in ("module", "shared"):
        m = FlashMLP(case["H"], case["D"], case["E"], activation=case["act"], dtype=_DTYPES[case["dtype"]],
                     device="cuda", accurate_dw=case["accurate_dw"])
        with torch.no_grad():
            m.w1.copy_(w1)
            m.w2.copy_(w2)
        state["module"] = m
        state["x"] = x.requires_grad_(True)
        del state["w1"], state["w2"]
    return state


def run(state):
    x, dout = state["x"], state["dout"]
    if state["kind"] in ("module", "shared"):
        m = state["module"]
        o = m(x)
        dx, dw1, dw2 = torch.autograd.grad(o, (x, m.w1, m.w2), dout)
        return o.detach(), dx, dw1, dw2
    w1, w2, act = state["w1"], state["w2"], state["act"]
    o = flashmlp_fwd(x, w1, w2, act)
    if state["kind"] == "fwd":
        return (o,)
    dx, dw1, dw2 = flashmlp_bwd(x, w1, w2, dout, act, accurate_dw=state["accurate_dw"])
    return o, dx, dw1, dw2


def work(case):
    """Forward 4u (X W1 and h W2); backward 10u (Z again, dO W2^T, and the three gradients'
    products dX, dW1, dW2: the backward call is given no Z). Every tensor of the calls moves once;
    a shared input and its gradients are (B, D)."""
    H, B, D, E = case["H"], case["B"], case["D"], case["E"]
    s = _BYTES[case["dtype"]]
    u = H * B * D * E
    rows = (1 if case["kind"] == "shared" else H) * B * D * s
    weights = 2 * H * D * E * s
    if case["kind"] == "fwd":
        return {"bytes": 2 * rows + weights, "flops": 4 * u}
    # forward: x, weights -> o; backward: x, weights, dout -> dx, two weight gradients
    return {"bytes": 2 * rows + weights + 3 * rows + 2 * weights, "flops": 14 * u}


def tolerance(case):
    # relative error of the outputs against 64-bit arithmetic: about 2.4e-3 for bf16, 3e-4 for
    # fp16 (the io type's rounding of h, dZ and the results) and 3e-7 for fp32 sums; about four
    # times that for another correct order of the same operations
    return {"fp16": {"rel": 1.5e-3}, "bf16": {"rel": 1.2e-2}, "fp32": {"rel": 1.5e-6}}[case["dtype"]]


def _act64(name, z):
    """act(z) and act'(z) in 64 bits."""
    if name == "silu":
        s = torch.sigmoid(z)
        return z * s, s * (1 + z * (1 - s))
    if name == "leaky_relu":
        p = z > 0
        return torch.where(p, z, 0.01 * z), torch.where(p, torch.ones_like(z), torch.full_like(z, 0.01))
    if name == "sigmoid":
        s = torch.sigmoid(z)
        return s, s * (1 - s)
    return z, torch.ones_like(z)


def exact(case, seed):
    """The same outputs in 64 bits, one head at a time with plain torch matrix products."""
    x, w1, w2, dout = _inputs(case, seed)
    H, shared = case["H"], case["kind"] == "shared"
    o, dx, dw1, dw2 = [], [], [], []
    for h in range(H):
        xh = (x if shared else x[h]).double()
        a, b = w1[h].double(), w2[h].double()
        act, dact = _act64(case["act"], xh @ a)
        o.append(act @ b)
        if dout is None:
            continue
        g = dout.double() / H if shared else dout[h].double()
        dz = (g @ b.t().contiguous()) * dact
        dx.append(dz @ a.t().contiguous())
        dw1.append(xh.t().contiguous() @ dz)
        dw2.append(act.t().contiguous() @ g)
    if shared:
        return torch.stack(o).mean(0), torch.stack(dx).sum(0), torch.stack(dw1), torch.stack(dw2)
    if dout is None:
        return (torch.stack(o),)
    return torch.stack(o), torch.stack(dx), torch.stack(dw1), torch.stack(dw2)
