"""Where the constants of csrc/plan.h come from: times of its tile forms with cold weights, and their fit.

On the device, the launches under a kernel trace, then the times out of the trace:
    rocprofv3 --kernel-trace --output-format csv -d DIR -o t -- python tools/plan_fit.py launch
    python tools/plan_fit.py collect DIR/t_kernel_trace.csv > sweep.csv
Anywhere, the fit of each form's c, a, b and lo beside plan.h's, and how far the rule's choice is from the best one measured:
    python tools/plan_fit.py fit sweep.csv            (the committed times: profiles/gemm_plan_sweep.csv.gz)"""
import csv
import gzip
import os
import re
import statistics
import sys

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "multimodal-financial-analysis-tool-using-paligemma_amd")

# columns, K, gate and up: the layers of PaliGemma-3B and of the layered decoders' "1b", "2b" and "7b"
LAYERS = [(3456, 1152, 0), (1152, 1152, 0), (4304, 1152, 0), (1152, 4304, 0), (2048, 1152, 0), (1152, 640, 0), (2560, 2048, 0),
          (2048, 2048, 0), (16384, 2048, 1), (2048, 16384, 0), (4096, 1024, 0), (96, 2048, 0), (2048, 64, 0), (1024, 2048, 0),
          (3072, 1024, 0), (1024, 1024, 0), (4096, 1024, 1), (1024, 4096, 0), (8192, 2048, 0), (160, 4096, 0), (4096, 128, 0),
          (2048, 4096, 0), (6144, 2048, 0), (16384, 4096, 0), (4096, 8192, 0), (14336, 4096, 1), (4096, 14336, 0)]
ROWS = [32, 64, 96, 129, 160, 192, 224, 256, 288, 320, 384, 450, 512, 576, 640, 768, 900, 1024, 1056, 1280, 1540, 2048, 2304, 3000,
        4096, 4608]
REPS = 3
SLABS = 64 << 20  # the op's scratch


def read_price(M, N, split):  # csrc/gemm_plan.hip
    return max(0.0, 1e-6 * M * N * split - 2.0) * min(1.0, M / 700) if split > 1 else 0.0


# what follows a product, the forms that its rule leaves out, and the price of its slabs
RULES = [("layered decoders", ("R288w", "W288n", "W64x64", "W128x64"), lambda M, N, s: 1e-6 * M * N * (s - 1)),
         ("prefill, a norm follows", (), read_price),
         ("prefill, its own epilogue", (), lambda M, N, s: read_price(M, N, s) + (4.6 if s > 1 else 0.0))]


def forms():
    """plan.h's forms: name -> (cfg, bm, bn, per_cu, whole_k, c, a, b, lo)"""
    src = open(os.path.join(PKG, "csrc", "plan.h")).read()
    cfg = {n: int(v) for n, v in re.findall(r"^ +(\w+) = (\d+),", src, re.M)}
    rows = re.findall(r"\{(\w+), (\d+), (\d+), (\d+), (true|false), ([\d.]+)f, ([\d.]+)f, ([\d.]+)f, ([\d.]+)f\}", src)
    return {r[0]: (cfg[r[0]], int(r[1]), int(r[2]), int(r[3]), r[4] == "true", *map(float, r[5:])) for r in rows}


def rounds(f, M, N, nkt, split, dual, lo):
    bm, bn, per_cu = f[1], f[2] // (2 if dual else 1), f[3]
    per = -(-nkt // split)
    t = -(-M // bm) * -(-N // bn) * -(-nkt // per)
    full, rest = divmod(t, 256 * per_cu)
    return full + (lo + (1 - lo) * rest / (256 * per_cu) if rest else 0), per


def predicted(f, M, N, K, split, dual):
    r, per = rounds(f, M, N, -(-K // 64), split, dual, f[8])
    return f[5] + r * (f[6] + f[7] * per)


def launches():
    """(form, M, N, K, dual, split): the unsliced forms predicted within three times the least, slices within 1.6 times"""
    out, F = [], forms()
    for N, K, dual in LAYERS:
        nkt = -(-K // 64)
        for M in ROWS:
            may = []
            for name, f in F.items():
                if (f[4] and K % 64) or (dual and name == "W288n"):
                    continue
                for s in range(1, 9):
                    if s > 1 and (dual or nkt // s < 4 or -(-nkt // -(-nkt // s)) != s or s * M * N * 4 > SLABS):
                        continue
                    may.append((predicted(f, M, N, K, s, dual), name, s))
            least = min(may)[0]
            out += [(n, M, N, K, dual, s) for us, n, s in may if us <= least * (3.0 if s == 1 else 1.6)]
    return out


def launch():
    import torch
    for p in (REPO, PKG):
        sys.path.insert(0, p)
    from oracle import weights as W
    from pgmi import Engine, _native as N_
    e = Engine(W.small_config(1, 1, 1024), max_batch=1, max_seq=320, max_kv=512)
    e.fill_synthetic(1, W.init_policy)
    e.prepare()
    g = torch.Generator("cuda").manual_seed(1)
    A = torch.randn(max(ROWS) * 16384, device="cuda", generator=g).bfloat16()
    weights = torch.empty(1 << 30, dtype=torch.bfloat16, device="cuda")  # 2 GB: a launch's own part is cold when its turn comes again
    for i in range(0, weights.numel(), 1 << 26):
        weights[i:i + (1 << 26)] = (torch.randn(1 << 26, device="cuda", generator=g) * 0.02).bfloat16()
    out = torch.empty(max(ROWS) * 16384, dtype=torch.bfloat16, device="cuda")
    s, at, F = torch.cuda.current_stream().cuda_stream, 0, forms()
    todo = launches()
    print(len(todo), "plans", flush=True)
    for i, (name, M, N, K, dual, split) in enumerate(todo):
        n = N * K * (2 if dual else 1)
        N_.check(e.lib.pgmi_tune_gemm(F[name][0], split))
        for _ in range(REPS):
            at = at if at + n <= weights.numel() else 0
            N_.check(e.lib.pgmi_op_gemm(e.ctx, A.data_ptr(), weights.data_ptr() + 2 * at, M, N, K, 7 if dual else 0, None, None,
                                        out.data_ptr(), s))
            at += (n + 127) // 128 * 128
        if i % 500 == 0:
            torch.cuda.synchronize()
            print(i, flush=True)
    torch.cuda.synchronize()
    N_.check(e.lib.pgmi_tune_gemm(-1, 0))


def collect(trace):
    rows = [(int(r["Start_Timestamp"]), int(r["End_Timestamp"])) for r in csv.DictReader(open(trace))
            if "k_gemm_" in r["Kernel_Name"]]
    rows.sort()
    todo = launches()
    extra = len(rows) - REPS * len(todo)  # (none: the engine launches no product by itself)
    assert extra == 0, extra
    print("form,M,N,K,dual,split,us")
    for i, t in enumerate(todo):
        us = statistics.median((b - a) / 1e3 for a, b in rows[REPS * i:REPS * i + REPS])
        print(",".join(map(str, t)) + ",%.2f" % us)


def fit(path):
    import numpy as np
    F, data = forms(), []
    for r in csv.DictReader(gzip.open(path, "rt") if path.endswith(".gz") else open(path)):
        data.append((r["form"], *(int(r[k]) for k in ("M", "N", "K", "dual", "split")), float(r["us"])))
    print(len(data), "times")
    fits = {}
    for name, f in F.items():
        pts = [d for d in data if d[0] == name]
        us, best = np.array([d[6] for d in pts]), None
        for lo in np.arange(0.0, 1.001, 0.01):
            R = [rounds(f, d[1], d[2], -(-d[3] // 64), d[5], d[4], lo) for d in pts]
            X = np.array([[1.0, r, r * per] for r, per in R]) / us[:, None]
            k, *_ = np.linalg.lstsq(X, np.ones(len(us)), rcond=None)
            err = np.abs(X @ k - 1).mean()
            if best is None or err < best[0]:
                best = (err, *k, lo)
        now = np.mean([abs(predicted(f, *d[1:4], d[5], d[4]) / d[6] - 1) for d in pts])
        fits[name] = (*f[:5], *best[1:])
        print(f"{name:9s} {len(pts):5d}  plan.h c {f[5]:6.2f} a {f[6]:6.2f} b {f[7]:.3f} lo {f[8]:.2f}: off by {now:6.1%}   "
              f"fitted c {best[1]:6.2f} a {best[2]:6.2f} b {best[3]:.3f} lo {best[4]:.2f}: {best[0]:6.1%}")
    for what, skip, price in RULES:
        shapes = {}
        for d in data:
            if d[0] not in skip:
                shapes.setdefault(d[1:5], []).append(d)
        for whose, P in (("plan.h", F), ("fitted", fits)):
            loss = []
            for v in shapes.values():
                took = min(v, key=lambda d: predicted(P[d[0]], *d[1:4], d[5], d[4]) + price(*d[1:3], d[5]))
                loss.append((took[6] + price(*took[1:3], took[5])) / min(d[6] + price(*d[1:3], d[5]) for d in v) - 1)
            loss.sort()
            print(f"{what}, {whose}: {len(loss)} shapes, the choice is {statistics.mean(loss):.1%} slower than the best measured, "
                  f"{statistics.mean(loss[-(len(loss) // 10):]):.1%} over the worst tenth, {loss[-1]:.0%} at worst")


if __name__ == "__main__":
    {"launch": launch, "collect": collect, "fit": fit}[sys.argv[1]](*sys.argv[2:])
