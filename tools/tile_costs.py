"""The costs of the decode GEMM tiles that tile_cost() in csrc/ql_gemm.hip is made of: time random calls on every tile and number of slices,
fit the costs, and time the calls whose plan they change.

    python tools/tile_costs.py collect calls.csv --seconds 240          # GPU: random shapes, 1 to 256 rows, over 2048 k
    python tools/tile_costs.py fit profiles/tile_costs_calls.csv        # CPU (scipy): the numbers of tile_cost(), and how far off they are
    python tools/tile_costs.py compare --plans p.json out.csv           # GPU: two plans of each call, p.json: [[form, N, K, type, [[rows, a, b]]]]

The fit leaves out every second call; what it chooses there is compared with the plan that the call had."""
import argparse
import csv
import json
import math
import os
import random
import sys
import time

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TILES = [(1, 1, 8, 4), (1, 1, 8, 8), (1, 2, 4, 8), (1, 2, 4, 4), (2, 2, 4, 8), (2, 4, 2, 4)]
FORMS = [(*t, s) for t in TILES for s in range(1, 9)]
HEAD = ["activations", "weights", "columns", "k", "rows", "plan", "us"]


def gpu():
    os.environ["QLINEAR_NO_PLANS"] = "1"
    sys.path.insert(0, os.path.join(ROOT, "nano-vllm-hw3_amd"))
    sys.path.insert(0, os.path.join(ROOT, "tools"))
    import bench_kernels as BK
    import torch
    from nanovllm import _qlinear as Q
    from nanovllm.utils import quantization as NQ
    Q.workspace.reserve("cuda", 256 << 20)
    lib, dtypes = Q.load(), {"int8": torch.int8, "fp8": torch.float8_e4m3fn}

    def timer(N, K, weights, kind):
        """us of a call on weights from memory: (rows, tile and slices or None) -> us"""
        w = torch.randn(N, K, device="cuda").mul_(K ** -0.5).bfloat16()
        mods = [NQ.QLinear(dtypes[weights], w, None, weight_only=kind == "bf16").tile() for _ in range(max(4, min(200, int(600e6 // (N * K)) + 1)))]
        inputs = {}

        def us(M, form=None):
            if M not in inputs:
                x = torch.randn(M, K, device="cuda").bfloat16()
                inputs[M] = (x,) if kind == "bf16" else NQ.per_row_quant(x, dtypes[weights])
            x = inputs[M]
            fn = (lambda i: mods[i](*x)) if kind == "bf16" else (lambda i: mods[i].forward_quantized(*x))
            lib.ql_gemm_force_config(*(form or (0, 0, 0, 0, 0)))
            try:
                return BK.time_fn(fn, len(mods), len(mods))
            finally:
                lib.ql_gemm_force_config(0, 0, 0, 0, 0)
        return us

    def plan(M, N, K, weights, kind):
        return Q.plan_query(Q.QL_PLAN_W8A8 if kind != "bf16" else 0, M, N, K, Q.dtype_code(dtypes[weights]))
    return timer, plan


def slices(form, K):
    """The slices that a call asked for in `form` has."""
    chunks = -(-K // (32 * form[2] * form[3]))
    return -(-chunks // -(-chunks // form[4])) if form[4] <= chunks else 0


def collect(path, seconds, seed):
    timer, plan = gpu()
    rng, end = random.Random(seed), time.time() + seconds
    with open(path, "w", newline="") as f:
        out = csv.writer(f)
        out.writerow(HEAD + [" ".join(map(str, c)) for c in FORMS])
        while time.time() < end:
            if rng.random() < 0.5:
                N, K = rng.choice([1024, 2560, 3072, 4096, 5120, 6144]), rng.choice([2560, 3072, 4096, 9728, 12288])
            else:
                N = int(math.exp(rng.uniform(math.log(512), math.log(12288)))) // 32 * 32
                K = int(math.exp(rng.uniform(math.log(2112), math.log(16384)))) // 64 * 64
            for kind in ("bf16", "8 bits"):
                for weights in ("int8", "fp8"):
                    us = timer(N, K, weights, kind)
                    for M in sorted({rng.choice([33, 48, 64, 96, 128]), rng.randint(33, 256), int(math.exp(rng.uniform(0, math.log(32))))}):
                        p = plan(M, N, K, weights, kind)
                        if p[1] == 8:
                            continue
                        row = [kind, weights, N, K, M, " ".join(map(str, p)), round(us(M), 2)]
                        for c in FORMS:
                            tiles = -(-M // (32 * c[0])) * -(-N // (32 * c[1]))
                            runs = slices(c, K) == c[4] and not (M <= 32 and c[0] > 1) and (c[4] == 1 or tiles * c[4] <= 1100)
                            row.append(round(us(M, c), 2) if runs else "")
                        out.writerow(row)
            print(N, K, flush=True)


def read(path):
    with open(path, newline="") as f:
        for r in csv.DictReader(f):
            times = {c: float(r[" ".join(map(str, c))]) for c in FORMS if r[" ".join(map(str, c))]}
            yield dict(kind=r["activations"], weights=r["weights"], N=int(r["columns"]), K=int(r["k"]), M=int(r["rows"]),
                       plan=tuple(map(int, r["plan"].split())), us=float(r["us"]), times=times)


def features(call, form):
    mt, wn, wk, cp, s = form
    rows, kb = -(-call["M"] // (32 * mt)), 32 * cp * wk
    chunks = -(-call["K"] // kb)
    return (min(call["K"], -(-chunks // s) * kb) / 1000, rows * -(-call["N"] // (32 * wn)) * s / 256, -(-call["M"] // 32) / (rows * mt), s,
            call["N"] * call["K"] * 1e-6)


def cost(c, feature):
    import numpy as np
    k, load, full, s, weights = feature
    start, sl, slice_, group, kk, k_full, q, way = c
    return (start + sl * (s > 1) + slice_ * (s - 1) + way * weights +
            (group + (kk + k_full * full) * k) * ((1 - q) * np.maximum(1, load) + q * np.ceil(load)))


def fit(path):
    import numpy as np
    from scipy.optimize import least_squares
    calls = list(read(path))
    groups = {"int8": ("bf16", ("int8",)), "fp8": ("bf16", ("fp8",)), "8-bit activations": ("8 bits", ("int8", "fp8"))}
    for name, (kind, weights) in groups.items():
        mine = [(i, c) for i, c in enumerate(calls) if c["kind"] == kind and c["weights"] in weights]
        found = {}
        print(name)
        for tile in TILES:
            got = [(features(c, f), t) for i, c in mine if i % 2 == 0 for f, t in c["times"].items() if f[:4] == tile]
            x, y = np.array([g[0] for g in got]).T, np.array([g[1] for g in got])
            best = min((least_squares(lambda v: np.log(np.maximum(cost(v, x), .5)) - np.log(y), v0, loss="soft_l1", f_scale=.1,
                                      bounds=([0] * 8, [12, 8, 3, 8, 20, 20, 1, 1]))
                        for v0 in ([3, 1, .3, 1, 2, 1, .5, .02], [2, 2, .1, .5, 4, 2, .2, .05])), key=lambda r: r.cost)
            found[tile] = best.x
            print("   ", tile, [round(float(v), 3) for v in best.x], f"{len(y)} times, off by {np.sqrt(np.mean(best.fun ** 2)):.3f} (rms of the logarithm)")
        gain = []
        for i, c in mine:
            if i % 2 and c["times"] and c["plan"][:4] in found:
                line = 0.86 if c["M"] <= 32 else 0.9 if c["M"] <= 64 else 0.88
                price = {f: cost(found[f[:4]], features(c, f)) for f in c["times"]}
                f = min(price, key=price.get)
                if price[f] < line * cost(found[c["plan"][:4]], features(c, c["plan"])):
                    gain.append(c["times"][f] / c["us"])
        print(f"    {len(gain)} calls change: {math.exp(np.mean(np.log(gain))):.3f} of the time, {sum(g > 1.04 for g in gain)} slower by more than 4 %")


def compare(plans, path):
    timer, _ = gpu()
    with open(plans) as f:
        shapes = json.load(f)
    with open(path, "w", newline="") as f:
        out = csv.writer(f)
        out.writerow(HEAD[:5] + ["rules", "us", "costs", "us", "ratio"])
        for n, (form, N, K, weights, calls) in enumerate(shapes):
            kind = "8 bits" if form else "bf16"
            us = timer(N, K, weights, kind)
            for M, old, new in calls:
                a, b = (min(t) for t in zip(*((us(M, tuple(old)), us(M, tuple(new))) for _ in range(2))))
                out.writerow([kind, weights, N, K, M, " ".join(map(str, old)), round(a, 2), " ".join(map(str, new)), round(b, 2), round(b / a, 3)])
            if n % 100 == 0:
                print(n, flush=True)


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("what", choices=["collect", "fit", "compare"])
    ap.add_argument("file")
    ap.add_argument("--seconds", type=float, default=240)
    ap.add_argument("--seed", type=int, default=1)
    ap.add_argument("--plans", default="")
    args = ap.parse_args()
    if args.what == "collect":
        collect(args.file, args.seconds, args.seed)
    elif args.what == "fit":
        fit(args.file)
    else:
        compare(args.plans, args.file)
