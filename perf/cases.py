"""The calls a program of this framework makes, with sizes, inputs and a float64 statement of their results.

Four kinds of call, over the state counts (8, 16, 32, 64) and storage types (fp32, fp16, bf16) that the
kernels are built for:
  step   SelectiveScanCuda.step: one token of a decode loop
  infer  SelectiveScanCuda.forward_with_state without gradients: prefill, a chunk of a stream, a short call
  train  SelectiveScanCuda / FusedSelectiveScan forward and backward through autograd
  scan   parallel_scan_fn, forward alone or forward and backward, over (B, D, L, N) or (B, L, C)
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mamba-windows-cuda_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from mamba_windows_cuda import FusedSelectiveScan, SelectiveScanCuda, parallel_scan_fn, workloads  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
DEV = "cuda"


def _ssm(name, kind, B, L, D, N=16, dtype="f16", gated=False, state=False, level=0):
    """gated: delta' = softplus(delta + delta_bias) and out * silu(z), as a Mamba block applies them around the
    scan. state: a carried state comes in (and, in training, a gradient of the one that goes out)."""
    c = {"kind": kind, "B": B, "L": L, "D": D, "N": N, "dtype": dtype, "gated": gated, "state": state, "level": level}
    return {"name": name, **c} if name else c


def _scan(name, shape, dtype="f32", backward=False):
    c = {"kind": "scan", "B": shape[0], "D": shape[1] if len(shape) == 4 else 0, "L": shape[-2], "C": shape[-1],
         "dtype": dtype, "backward": backward}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one token for a handful of users: the launch and the host path are all there is
        _ssm("step_b8", "step", 8, 1, 1536, gated=True),
        # one token for a full serving batch: the state's round trip through memory
        _ssm("step_b1024", "step", 1024, 1, 1536),
        # the smallest scan of the reference's own benchmark, a single short sequence in fp32
        _ssm("infer_short", "infer", 1, 1024, 256, dtype="f32"),
        # the prompt of one user through a Mamba-130M layer, all transforms fused
        _ssm("prefill_b1", "infer", 1, 2048, 1536, dtype="bf16", gated=True),
        # one chunk of a long fp32 sequence that is streamed with a carried state
        _ssm("stream_chunk", "infer", 1, 4096, 2048, dtype="f32", state=True),
        # the training step of a Mamba-130M layer (the benchmark's own workload)
        _ssm("train_130m", "train", 8, 2048, 1536),
        # the same layer as a block calls it: bias, softplus and gate fused, bf16
        _ssm("train_130m_gated", "train", 8, 2048, 1536, dtype="bf16", gated=True),
        # a Mamba-2.8B layer, whose activations are recomputed rather than kept
        _ssm("train_2p8b_recompute", "train", 4, 4096, 5120, level=1),
        # ragged sizes in fp32 with the state carried across segments of a sequence, both ways
        _ssm("train_ragged", "train", 3, 1001, 777, dtype="f32", state=True),
        # the largest state count
        _ssm("train_n64", "train", 2, 2048, 1536, N=64),
        # the standalone scan over wide rows (inference): the largest call
        _scan("scan_rows", (4, 65536, 1024)),
        # the standalone scan over (batch, channel, step, state) with its gradient: the reference's own layout
        _scan("scan_states_train", (2, 1536, 1024, 16), backward=True),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "infer", "infer", "train", "train", "train", "scan", "scan"])
    dtype = rng.choice(["f32", "f16", "f16", "bf16"])
    if kind == "scan":
        if rng.random() < 0.5:
            shape = (rng.randint(1, 4), _spread(rng, 16, 1536), _spread(rng, 64, 2048), rng.choice([8, 16, 16, 32, 64]))
        else:
            shape = (rng.randint(1, 4), _spread(rng, 256, 32768), _spread(rng, 16, 1024))
        return _scan(None, shape, dtype, rng.random() < 0.5)
    N = rng.choice([8, 16, 16, 16, 16, 32, 64])
    gated, state = rng.random() < 0.5, rng.random() < 0.5
    D = rng.choice([_spread(rng, 64, 5120), 64 * rng.randint(1, 80)])
    if kind == "step":
        return _ssm(None, "step", _spread(rng, 1, 1024), 1, min(D, 2560), N, dtype, gated, True)
    B = _spread(rng, 1, 8)
    L = rng.choice([_spread(rng, 64, 4096), 128 * rng.randint(1, 32)])
    while B * L * D * N > 4 * 4096 * 5120 * 4:  # a quarter of the largest listed step
        B, L = max(1, B // 2), max(64, L * 3 // 4)
    return _ssm(None, kind, B, L, D, N, dtype, gated, state, rng.choice([0, 0, 1]) if kind == "train" else 0)


def _ssm_tensors(case, seed):
    """What the layer holds before the call. delta is what the scan sees (uniform in 1e-3..1e-1) or, with the
    transforms, the projection that softplus turns into it."""
    dt = DTYPES[case["dtype"]]
    B, L, D = case["B"], case["L"], case["D"]
    x = workloads.ssm_inputs(B, L, D, dtype=dt, nstate=case["N"], seed=seed, device=DEV, gen_device=DEV,
                             h_prev=True, dout=case["kind"] == "train")
    g = torch.Generator(device=DEV).manual_seed(seed + 1)
    if case["gated"]:
        x["delta"] = (torch.randn(B, L, D, generator=g, device=DEV) - 4.0).to(dt)
        x["bias"] = (0.5 * torch.randn(D, generator=g, device=DEV)).to(dt)
        x["z"] = torch.randn(B, L, D, generator=g, device=DEV).to(dt)
    if case["kind"] == "train" and case["state"]:
        x["dh_last"] = torch.randn(B, D, case["N"], generator=g, device=DEV).to(dt)
    if case["kind"] != "step" and not case["state"]:
        del x["h_prev"]
    if case["kind"] == "step":
        for k in ("u", "delta", "B", "C", "z"):
            if k in x:
                x[k] = x[k][:, 0].contiguous()
    return x


def _scan_tensors(case, seed):
    shape = (case["B"], case["D"], case["L"], case["C"]) if case["D"] else (case["B"], case["L"], case["C"])
    a, b = workloads.pscan_inputs(shape, dtype=DTYPES[case["dtype"]], seed=seed, device=DEV, gen_device=DEV)
    x = {"a": a, "b": b}
    if case["backward"]:
        g = torch.Generator(device=DEV).manual_seed(seed + 1)
        x["dout"] = torch.randn(shape, generator=g, device=DEV).to(a.dtype)
    return x


_LEAVES = ("u", "delta", "A", "B", "C", "D", "h_prev", "z", "bias")


def prepare(case, seed):
    if case["kind"] == "scan":
        x = _scan_tensors(case, seed)
        if case["backward"]:
            x["a"].requires_grad_(True)
            x["b"].requires_grad_(True)
        return {"case": case, "x": x}
    x = _ssm_tensors(case, seed)
    state = {"case": case, "x": x}
    if case["kind"] == "train":
        for k in _LEAVES:
            if k in x:
                x[k].requires_grad_(True)
    if case["kind"] == "train" and not case["gated"]:
        state["module"] = FusedSelectiveScan(checkpoint_lvl=case["level"])
    else:
        state["module"] = SelectiveScanCuda(checkpoint_lvl=case["level"])
    if case["kind"] == "step":  # a decode loop alternates between two state buffers that it keeps
        state["h_next"] = torch.empty_like(x["h_prev"])
    return state


def run(state):
    case, x = state["case"], state["x"]
    if case["kind"] == "scan":
        if not case["backward"]:
            with torch.no_grad():
                return parallel_scan_fn(x["a"], x["b"])
        x["a"].grad = x["b"].grad = None
        h = parallel_scan_fn(x["a"], x["b"])
        h.backward(x["dout"])
        return h.detach(), x["a"].grad, x["b"].grad
    m = state["module"]
    args = (x["u"], x["delta"], x["A"], x["B"], x["C"], x["D"])
    kw = dict(z=x["z"], delta_bias=x["bias"], delta_softplus=True) if case["gated"] else {}
    if case["kind"] == "step":
        with torch.no_grad():
            return m.step(*args, x["h_prev"], out_state=state["h_next"], **kw)
    if case["kind"] == "infer":
        with torch.no_grad():
            return m.forward_with_state(*args, x.get("h_prev"), **kw)
    leaves = [x[k] for k in _LEAVES if k in x]
    for t in leaves:
        t.grad = None
    if case["state"]:
        out, h_last = m.forward_with_state(*args, x["h_prev"], **kw)
        torch.autograd.backward((out, h_last), (x["dout"], x["dh_last"]))
        return (out.detach(), h_last.detach(), *[t.grad for t in leaves])
    out = m(*args, **kw)
    torch.autograd.backward(out, x["dout"])
    return (out.detach(), *[t.grad for t in leaves])


def work(case):
    s = 4 if case["dtype"] == "f32" else 2
    if case["kind"] == "scan":
        n = case["B"] * max(case["D"], 1) * case["L"] * case["C"]
        return {"bytes": s * n * (6 if case["backward"] else 3), "flops": n * (5 if case["backward"] else 2)}
    B, L, D, N = case["B"], case["L"], case["D"], case["N"]
    bld, bln, bdn = B * L * D, B * L * N, B * D * N
    state = case["state"] or case["kind"] == "step"
    if case["kind"] != "train":
        # u, delta, out and perhaps z; B, C; A, D and perhaps the bias; h_prev and h_last
        n = bld * (3 + case["gated"]) + 2 * bln + D * N + D * (1 + case["gated"]) + bdn * (1 + state)
        # decay (product and exponential), state (product, multiply-add), output (multiply-add)
        return {"bytes": s * n, "flops": 7 * bld * N}
    # the inputs and dout once, the output and the gradients once
    n = bld * (6 + 2 * case["gated"]) + 4 * bln + 2 * D * N + 2 * D * (1 + case["gated"]) + bdn * 4 * case["state"]
    # the forward's, then the adjoint state (3), its sums over n (5), over channels (4) and over time (4)
    return {"bytes": s * n, "flops": 23 * bld * N}


# About four times the largest error against float64 over the outputs of these calls on MI355X (fp32: 3.8e-6 in
# the gradient of A, fp16: 2.9e-4, bf16: 2.3e-3; the 16-bit ones are the rounding of the stored result).
_TOL = {"f32": 1.5e-5, "f16": 1.2e-3, "bf16": 9e-3}


def tolerance(case):
    return {"rel": _TOL[case["dtype"]]}


def _f64(x):
    return {k: v.detach().double() for k, v in x.items()}


def _exact_scan(case, seed):
    x = _f64(_scan_tensors(case, seed))
    a, b = x["a"], x["b"]
    L = case["L"]
    h = torch.empty_like(b)
    s = h[..., 0, :] = b[..., 0, :]
    for t in range(1, L):
        s = torch.addcmul(b[..., t, :], a[..., t, :], s, out=h[..., t, :])
    if not case["backward"]:
        return h
    dx = torch.empty_like(b)
    g = dx[..., L - 1, :] = x["dout"][..., L - 1, :]
    for t in range(L - 2, -1, -1):
        g = torch.addcmul(x["dout"][..., t, :], a[..., t + 1, :], g, out=dx[..., t, :])
    da = torch.zeros_like(a)
    torch.mul(dx[..., 1:, :], h[..., :-1, :], out=da[..., 1:, :])
    return h, da, dx


def exact(case, seed):
    if case["kind"] == "scan":
        return _exact_scan(case, seed)
    x = _f64(_ssm_tensors(case, seed))
    step = case["kind"] == "step"
    if step:
        for k in ("u", "delta", "B", "C", "z"):
            if k in x:
                x[k] = x[k].unsqueeze(1)
    u, A, Bm, Cm, Dv = x["u"], x["A"], x["B"], x["C"], x["D"]
    raw = x["delta"]
    dl = raw
    if case["gated"]:
        raw = raw + x["bias"]
        dl = torch.nn.functional.softplus(raw)
    B, L, D = u.shape
    h0 = x["h_prev"] if "h_prev" in x else u.new_zeros(B, D, case["N"])
    train = case["kind"] == "train"
    hs = u.new_empty(L, B, D, case["N"]) if train else None
    y = torch.empty_like(u)
    h = h0
    decay = lambda t: torch.exp((dl[:, t, :, None] * A).clamp_(-88.0, 88.0))
    for t in range(L):
        h = decay(t) * h + (dl[:, t] * u[:, t])[:, :, None] * Bm[:, t, None, :]
        y[:, t] = (h * Cm[:, t, None, :]).sum(-1)
        if train:
            hs[t] = h
    y += u * Dv
    sig = torch.sigmoid(x["z"]) if case["gated"] else None
    out = y * x["z"] * sig if case["gated"] else y
    if step:
        return out[:, 0], h
    if not train:
        return out, h
    dout = x["dout"]
    grads = {}
    if case["gated"]:
        grads["z"] = dout * y * sig * (1 + x["z"] * (1 - sig))
        dout = dout * x["z"] * sig
    du, dd = dout * Dv, torch.empty_like(dl)
    dB, dC, dA = torch.empty_like(Bm), torch.empty_like(Cm), torch.zeros_like(h0)
    g = x["dh_last"] if case["state"] else torch.zeros_like(h0)
    for t in range(L - 1, -1, -1):
        g = g + dout[:, t, :, None] * Cm[:, t, None, :]
        dC[:, t] = (dout[:, t, :, None] * hs[t]).sum(1)
        dB[:, t] = (g * (dl[:, t] * u[:, t])[:, :, None]).sum(1)
        s1 = (g * Bm[:, t, None, :]).sum(-1)
        g = g * decay(t)
        s = g * (hs[t - 1] if t else h0)
        du[:, t] += dl[:, t] * s1
        dd[:, t] = (A * s).sum(-1) + u[:, t] * s1
        dA += dl[:, t, :, None] * s
    if case["gated"]:
        dd = dd * torch.sigmoid(raw)
        grads["bias"] = dd.sum((0, 1))
    grads.update(u=du, delta=dd, A=dA.sum(0), B=dB, C=dC, D=(dout * u).sum((0, 1)), h_prev=g)
    head = (out, h) if case["state"] else (out,)
    return (*head, *[grads[k] for k in _LEAVES if k in x])
