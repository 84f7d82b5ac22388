"""The measurements behind the cost model of small grids in csrc/capi.hip, and its fit.

    python3 profiles/plan_model.py measure OUT.jsonl    # one GPU: times every plan of the shapes below
    python3 profiles/plan_model.py fit DATA.jsonl       # no GPU: prints kFwdCost and kBwdCost

plan_sweep.jsonl holds, per shape (B, L, D, N), storage type and direction, [states per lane, segments, chunks per
segment, carry split, us per call] of every plan: the least of three or four runs of ten calls, back to back behind a
matrix product, with the plans of a shape in random order. Its first lines are the workgroups per CU that the
runtime's occupancy query gives the main and the carry kernel of each instance; write new ones after a change of
their registers.
"""
import json
import math
import os
import random
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CUS = 256
LANES = {8: (1, 2), 16: (1, 2), 32: (2, 4), 64: (4,)}  # states per lane that are planned, by state count
SEGMENTS = (1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 40, 48)
FIXED = [(1, 1024, 256, 16), (2, 1000, 100, 16), (2, 777, 333, 16), (6, 400, 300, 32), (2, 2048, 512, 16),
         (5, 100, 2000, 16), (1, 2048, 1536, 16), (1, 4096, 2048, 16), (3, 1001, 777, 16), (2, 2048, 1536, 64),
         (8, 2048, 192, 16), (8, 2048, 384, 16), (4, 2268, 530, 8), (1, 64, 2560, 16), (2, 200, 64, 64),
         (1, 256, 64, 16)]


def ceil_div(a, b):
    return -(-a // b)


def groups(D, N, spl):
    return ceil_div(D, 256 * spl // N)


def shapes(count, seed, fixed):
    """`fixed`, then random shapes of fewer than 1.5 workgroups a CU."""
    rng, out = random.Random(seed), list(fixed)
    while len(out) < count:
        N = rng.choice([16, 16, 16, 8, 32, 64])
        B, L, D = int(round(8 ** rng.random())), int(64 * 64 ** rng.random()), int(64 * 80 ** rng.random())
        D = max(64, D // 64 * 64) if rng.random() < 0.4 else D
        L = max(64, L // 128 * 128) if rng.random() < 0.3 else L
        if min(B * groups(D, N, s) for s in LANES[N]) < 384:
            out.append((B, L, D, N))
    return out


def plans(shape, bwd):
    """{(states per lane, segments, chunks per segment, carry split): the overrides that force it}"""
    _, L, _, N = shape
    nck, out = ceil_div(L, 16), {}
    for spl in LANES[N]:
        for n in SEGMENTS:
            for f in (1, 2, 4) if n > 1 else (1,):
                cps = ceil_div(ceil_div(nck, n), f) * f
                nseg = ceil_div(nck, cps)
                if n == 1 or (nseg > 1 and cps > 1):
                    out.setdefault((spl, nseg, cps, f), {"MWC_SPL": spl, "MWC_NSEG": n, "MWC_CFOLD": f})
    return out


def measure(path, few=None):
    sys.path.insert(0, os.path.join(os.path.dirname(HERE), "mamba-windows-cuda_amd"))
    import torch

    from mamba_windows_cuda import ops, workloads

    with open(os.path.join(HERE, "plan_sweep.jsonl")) as f:
        caps = [line for line in f if "fwd_caps" in line]
    busy = torch.randn(4096, 4096, device="cuda", dtype=torch.float16)
    with open(path, "w") as out:
        out.writelines(caps)
        todo = shapes(84, 20, FIXED) + shapes(200, 77, [(1, 64, 2560, 16), (4, 64, 5000, 16)])
        for i, shape in enumerate(todo[:few]):
            B, L, D, N = shape
            dt = ("f16", "bf16", "f16", "f32")[i % 4]
            x = workloads.ssm_inputs(B, L, D, nstate=N, seed=i, device="cuda", gen_device="cuda", dout=True,
                                     dtype={"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[dt])
            args = [x[k] for k in ("u", "delta", "A", "B", "C", "D")]
            ckpt = ops.ssm_forward(*args, want_ckpt=True)[2]
            calls = (lambda: ops.ssm_forward(*args, want_ckpt=True),
                     lambda: ops.ssm_backward(*args, x["dout"], ckpt))
            for bwd, call in enumerate(calls):
                best = {}
                for rnd in range(3):
                    items = list(plans(shape, bwd).items())
                    random.Random(rnd).shuffle(items)
                    for plan, env in items:
                        os.environ.update({k: str(v) for k, v in env.items()})
                        call()
                        torch.mm(busy, busy)  # the host runs ahead of the GPU by this
                        torch.mm(busy, busy)
                        torch.mm(busy, busy)
                        t0, t1 = torch.cuda.Event(True), torch.cuda.Event(True)
                        t0.record()
                        for _ in range(10):
                            call()
                        t1.record()
                        t1.synchronize()
                        best[plan] = min(t0.elapsed_time(t1) * 100, best.get(plan, math.inf))
                us = [[*p, round(t, 1)] for p, t in best.items()]
                out.write(json.dumps({"shape": shape, "dtype": dt, "bwd": bwd, "us": us}, separators=(",", ":")) + "\n")
            print(i, shape, dt, flush=True)


# Parameters, as in the C++ tables: fold and launch; per states per lane the prologues of the main and of the carry
# pass and the two rates' ratios from one wave count to the next; a chunk's time per (N, states per lane) in both
# passes; the finishing kernel's three costs; what each further workgroup of a CU adds to the prologues. The bounds
# of the ratios keep q / rate[q] from falling and rate[q] at q or less.
PAIRS = [(n, s) for n in LANES for s in LANES[n]]
LOW = ([0.02, 0.5] + [1, 0.3, 1, 0.85, 0.85, 0.85, 1, 0.85, 0.85, 0.85] * 3 + [0.2, 0.05] * 7 + [0.01, 0.05, 0.02] +
       [0] * 6)
HIGH = [0.6, 8] + [15, 12, 2, 1.5, 4 / 3, 1.5, 2, 1.5, 4 / 3, 1.5] * 3 + [8, 3] * 7 + [0.3, 3, 2] + [2] * 6
START = [0.13, 2.5] + [5, 3, 1.5, 1.25, 1.1, 1.1, 1.3, 1.15, 1.1, 1.1] * 3 + [1, 0.4] * 7 + [0.08, 0.5, 0.2] + [0.2] * 6


def tables(x):
    import numpy as np

    x = np.asarray(x)
    spl = x[2:32].reshape(3, 10)
    return {"fold": x[0], "launch": x[1], "main": spl[:, 0], "carry": spl[:, 1], "rate": np.cumprod(spl[:, 2:6], 1),
            "crate": np.cumprod(spl[:, 6:], 1), "chunk": x[32:46].reshape(7, 2), "fin": x[46:49],
            "main_more": x[49:52], "carry_more": x[52:]}


def model(points, caps, bwd):
    """points: [(shape, plan)]; returns the function from tables() to their modelled times."""
    import numpy as np

    rows = [(*s, *p, *caps[s[3], p[0]][bwd], p[0].bit_length() - 1, PAIRS.index((s[3], p[0]))) for s, p in points]
    B, L, D, N, spl, nseg, cps, f, cap_main, cap_carry, si, pair = np.array(rows, dtype=np.int64).T
    nck, ng = -(-L // 16), -(-D // (256 * spl // N))
    ncar = np.where(nseg < 2, 0, -(-(nck - cps) * f // cps) if bwd else (nseg - 1) * f)

    def grid(wgs, cap):  # full rounds, and workgroups per CU of the last one
        full = wgs // CUS // cap
        return full, -(-wgs // CUS) - full * cap, cap

    main_grid, carry_grid = grid(B * ng * nseg, cap_main), grid(B * ng * ncar, cap_carry)

    def pass_us(grid, chunks, chunk, prologue, more, rate):
        r = np.ones((3, 9))
        r[:, 2:5], r[:, 5], r[:, 6:] = rate[:, :3], rate[:, 2:].mean(1), rate[:, 3:]
        full, q, cap = grid
        one = lambda n: chunks * chunk * n / r[si, np.minimum(n, 8)] + prologue[si] + more[si] * (n - 1)
        return full * one(cap) + np.where(q > 0, one(q), 0.0)

    def times(t):
        us = pass_us(main_grid, cps, t["chunk"][pair, 0], t["main"], t["main_more"], t["rate"])
        carry = pass_us(carry_grid, cps // f, t["chunk"][pair, 1], t["carry"], t["carry_more"], t["crate"])
        us = us + np.where(nseg > 1, t["launch"] + t["fold"] * (ncar if bwd else (nseg - 1) * f) + carry, 0.0)
        if bwd:
            fin = t["fin"]
            us = us + np.maximum(fin[0] * ng, fin[1] * -(-nseg * B // 32)) + fin[2] * 8e-6 * B * ng * L * N
        return us

    return times


def fit(path):
    import numpy as np
    from scipy.optimize import least_squares

    lines = [json.loads(line) for line in open(path)]
    caps = {(r["states"], r["per_lane"]): (r["fwd_caps"], r["bwd_caps"]) for r in lines if "states" in r}
    for bwd, name in enumerate(("kFwdCost", "kBwdCost")):
        points, logs, weights, firsts = [], [], [], []
        for r in (r for r in lines if r.get("bwd") == bwd):
            least = min(u[4] for u in r["us"])
            firsts.append(len(points))
            for u in r["us"]:  # the plans near the fastest one count most, every shape alike
                points.append((r["shape"], u[:4]))
                logs.append(math.log(u[4]))
                weights.append(max(math.exp(-1.5 * (u[4] / least - 1)), 0.05) / math.sqrt(len(r["us"])))
        logs, weights, times = np.array(logs), np.array(weights), model(points, caps, bwd)
        x = least_squares(lambda x: weights * (np.log(times(tables(x))) - logs), START, bounds=(LOW, HIGH),
                          loss="soft_l1", f_scale=0.02, max_nfev=300).x
        t = tables(x)
        us = times(t)
        lost = [math.exp(logs[a + int(np.argmin(us[a:b]))] - logs[a:b].min())
                for a, b in zip(firsts, firsts[1:] + [len(points)])]
        print(f"// {len(points)} plans of {len(firsts)} shapes; the modelled choice is "
              f"{100 * (np.exp(np.mean(np.log(lost))) - 1):.1f}% above the fastest plan, {max(lost):.2f}x at worst")
        num = lambda v: f"{v:.2f}"
        many = lambda v: ", ".join(map(num, v))
        fin = t["fin"] if bwd else (0, 0, 0)
        print(f"constexpr CostModel {name} = {{\n    {t['fold']:.3f}, {num(t['launch'])},")
        print(f"    {fin[0]:.3f}, {many(fin[1:])},")
        print("    {" + ",\n     ".join(
            f"{{{many([t[k][i] for k in ('main', 'main_more', 'carry', 'carry_more')])}, "
            f"{{{many(t['rate'][i])}}}, {{{many(t['crate'][i])}}}}}" for i in range(3)) + "},")
        print("    {" + ",\n     ".join("{" + ", ".join(
            "{" + many(t["chunk"][PAIRS.index((n, s))]) + "}" if s in LANES[n] else "{0, 0}" for s in (1, 2, 4)) + "}"
            for n in LANES) + "}};", flush=True)


if __name__ == "__main__":
    {"measure": measure, "fit": fit}[sys.argv[1]](sys.argv[2])
