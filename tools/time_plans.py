"""Time entries of the plan table beside what the rules take in their place: the product alone (autotune_plans.py times o_proj and down_proj together with
the norm behind them), over more copies of the weights than the memory-side cache holds, in one hipGraph, int8 and fp8 weights, at the
first, middle and last row count of each entry.

    python tools/time_plans.py                                     # the entries marked "timed": "alone", up to 256 rows
    python tools/time_plans.py --shape 4096x4096 --form 8          # every entry of a shape and form
    python tools/time_plans.py --out new.json                      # the table with the marked entries' times of this run
"""
import argparse
import json
import math
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "nano-vllm-hw3_amd"))
sys.path.insert(0, os.path.join(ROOT, "tools"))
import torch  # noqa: E402
from nanovllm import _qlinear as Q  # noqa: E402
from nanovllm.utils import quantization as NQ  # noqa: E402
import bench_kernels as BK  # noqa: E402


def modules(form, N, K, dtype):
    w = torch.randn(N, K, device="cuda").mul_(K ** -0.5).bfloat16()
    made = []
    for _ in range(max(4, min(200, int(600e6 // (N * K)) + 1))):
        m = NQ.QLinear(dtype, w, None, weight_only=not form & Q.QL_PLAN_W8A8)
        if form & Q.QL_PLAN_SILU:
            m.enable_silu_mul()
        made.append(m.tile())
    return made


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--shape", default="")
    ap.add_argument("--form", type=int, default=-1)
    ap.add_argument("--runs", type=int, default=3)
    ap.add_argument("--out", default="")
    args = ap.parse_args()
    with open(Q.PLAN_TABLE) as f:
        doc = json.load(f)
    plain = (0, Q.QL_PLAN_SILU, Q.QL_PLAN_W8A8, Q.QL_PLAN_SILU | Q.QL_PLAN_W8A8)
    if args.shape:
        shape = tuple(int(v) for v in args.shape.split("x"))
        chosen = [e for e in doc["plans"] if (e["N"], e["K"]) == shape and (args.form < 0 or e["form"] == args.form) and e["form"] in plain]
    else:
        chosen = [e for e in doc["plans"] if e.get("timed") == "alone"]
    chosen = [e for e in chosen if e["m_hi"] <= 256 and e["split"] > 0]
    lib = Q.load()
    lib.ql_gemm_plan_clear()
    Q.workspace.reserve("cuda", 256 << 20)
    for form, N, K in sorted({(e["form"], e["N"], e["K"]) for e in chosen}):
        times = {}
        for dtype in (torch.int8, torch.float8_e4m3fn):
            mods = modules(form, N, K, dtype)
            for i, e in enumerate(chosen):
                if (e["form"], e["N"], e["K"]) != (form, N, K):
                    continue
                for M in sorted({e["m_lo"], (e["m_lo"] + e["m_hi"]) // 2, e["m_hi"]}):
                    x = torch.randn(M, K, device="cuda").bfloat16()
                    if form & Q.QL_PLAN_W8A8:
                        q = NQ.per_row_quant(x, dtype)
                        fn = lambda j: mods[j].forward_quantized(*q)  # noqa: E731
                    else:
                        fn = lambda j: mods[j](x)  # noqa: E731
                    us = [1e9, 1e9]
                    for _ in range(args.runs):
                        for k, config in enumerate(((0, 0, 0, 0, 0), (*e["tile"], e["split"]))):
                            lib.ql_gemm_force_config(*config)
                            try:
                                us[k] = min(us[k], BK.time_fn(fn, len(mods), len(mods)))
                            finally:
                                lib.ql_gemm_force_config(0, 0, 0, 0, 0)
                    times.setdefault(i, []).append(us)
                    rule = Q.plan_query(form, M, N, K, Q.dtype_code(dtype))
                    print(f"form {form} {N} x {K}, {M} rows, {str(dtype)[6:]}: rules {rule} {us[0]:.2f} us, entry {e['tile']} in {e['split']} {us[1]:.2f} "
                          f"({us[1] / us[0]:.3f})", flush=True)
            del mods
        for i, us in times.items():
            rules, entry = (math.exp(sum(math.log(u[k]) for u in us) / len(us)) for k in range(2))
            e = chosen[i]
            print(f"== form {form} {N} x {K}, rows {e['m_lo']}..{e['m_hi']}: {entry / rules:.3f}", flush=True)
            if e.get("timed") == "alone":
                e["us"], e["heuristic_us"] = round(entry, 2), round(rules, 2)
    if args.out:
        with open(args.out, "w") as f:
            f.write('{"device": %s,\n "plans": [\n' % json.dumps(doc["device"]))
            f.write(",\n".join("  " + json.dumps(p) for p in doc["plans"]))
            f.write("\n ]}\n")


if __name__ == "__main__":
    main()
