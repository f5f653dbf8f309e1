"""Short-batch GEMM sweep: achieved HBM bandwidth of the M<=16 streaming kernel, the skinny kernel and every tile and K split of
the M<=512 kernel per (shape, M), timed inside captured hipGraphs over rotating weight copies, so that W never comes from
the 256 MB cache; the library beside them runs outside a graph.

    PYTHONPATH=. python benchmarks/stream_gemm_sweep.py [--full] [--model]

``--model``: the M<=512 kernel alone, its K-split slabs left unreduced, against the time that ``hip.mid_choose`` reckons with.
"""
import argparse
import sys

import torch
import torch.nn.functional as F

from vllm_distributed_amd.ops import hip

hip.load()
DEV = "cuda"
SHAPES = {  # name: (N, K)
    "70b.qkv": (10240, 8192), "70b.o": (8192, 8192), "70b.gate_up": (57344, 8192), "70b.down": (8192, 28672),
    "70b.lm_head": (128256, 8192),
    "8b.qkv": (6144, 4096), "8b.o": (4096, 4096), "8b.gate_up": (28672, 4096), "8b.down": (4096, 14336),
    "70b/tp8.qkv": (1280, 8192), "70b/tp8.o": (8192, 1024), "70b/tp8.gate_up": (7168, 8192),
    "70b/tp8.down": (8192, 3584),
    "8b.lm_head": (128256, 4096), "32k.lm_head": (32000, 4096), "2048": (2048, 2048), "3072": (3072, 3072), "6144": (6144, 6144),
    "4608x3072": (4608, 3072), "18432x3072": (18432, 3072), "2816x2048": (2816, 2048),
}


def timed(fn, copies, reps=3):
    """us per call: a graph of len(copies) calls, each on its own weight copy."""
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        for w in copies[:2]:
            fn(w)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            for w in copies:
                fn(w)
        g.replay()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        best = 1e9
        for _ in range(reps):
            e0.record()
            g.replay()
            e1.record()
            torch.cuda.synchronize()
            best = min(best, e0.elapsed_time(e1) * 1e3 / len(copies))
    return best


def eager(fn, copies, reps=3):
    """us per call, launched from Python: a library GEMM may bring memory-set nodes into a graph."""
    best = 1e9
    for _ in range(reps + 1):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        e0.record()
        for w in copies:
            fn(w)
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) * 1e3 / len(copies))
    return best


def model_check(names, ms, pad):
    """Measured and reckoned time of every tile and split, and what the choice loses against the best of them."""
    errs, losses = [], []
    for name in names:
        n, k = SHAPES[name]
        copies = [torch.randn(n, k + pad, device=DEV).mul_(0.02).bfloat16()[:, :k] for _ in range(max(2, min(16, (900 << 20) // (n * k * 2) + 1)))]
        for m in ms:
            x = torch.randn(m, k, device=DEV).bfloat16()
            best = {}
            for bm, bn in hip._MID_TILES:
                if bm < min(m, 256) or (bm > 64 and bm >= 4 * m):
                    continue
                for ks in hip._MID_KSPLITS:
                    if ks > 1 and k // 64 // ks < (4 if ks <= 8 else 8) or ks * m * n * 4 > 1 << 30:
                        break
                    t = timed(lambda w: hip.mid_gemm(x, w, bm=bm, bn=bn, ksplit=ks, partials=ks > 1), copies)
                    best[(bm, bn, ks)] = t
                    reckoned = hip._mid_estimate(m, n, k, bm, bn, ks, False)
                    slabs = ks * m * n * 4 * 0.2e-6 if ks > 1 else 0.0        # (their reading is the next kernel's)
                    errs.append(abs(reckoned - slabs - t) / t)
            choice = hip.mid_choose(m, n, k, False)
            least = min(best, key=best.get)
            losses.append(best[choice] / best[least])
            print(f"{name:14s} {n:6d} x {k:5d} M={m:3d} chosen {choice} {best[choice]:7.1f} us {n * k * 2 / best[choice] / 1e6:5.2f} TB/s  "
                  f"least {least} {best[least]:7.1f}", flush=True)
        del copies
        torch.cuda.empty_cache()
    print(f"{len(errs)} timings of {len(names)} shapes: the model is {100 * sum(errs) / len(errs):.1f} % off in the mean; the choice is "
          f"{100 * (sum(losses) / len(losses) - 1):.1f} % above the least in the mean, {100 * (max(losses) - 1):.0f} % at most")


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--full", action="store_true")
    ap.add_argument("--shapes", type=str, default="")
    ap.add_argument("--ms", type=str, default="1,8,16")
    ap.add_argument("--model", action="store_true")
    ap.add_argument("--pad", type=int, default=0, help="row padding of W in elements (W is a [:, :K] view)")
    args = ap.parse_args()
    names = [s for s in args.shapes.split(",") if s] or list(SHAPES)
    if args.model:
        return model_check(names, [int(v) for v in args.ms.split(",")], args.pad)
    for name in names:
        n, k = SHAPES[name]
        nbytes = n * k * 2
        ncopies = max(2, min(12, (600 << 20) // nbytes + 1))
        copies = []
        for _ in range(ncopies):
            buf = torch.empty(n, k + args.pad, device=DEV, dtype=torch.bfloat16)
            buf[:, :k] = (torch.randn(n, k, device=DEV) * 0.02).to(torch.bfloat16)
            copies.append(buf[:, :k])
        for m in [int(v) for v in args.ms.split(",")]:
            x = torch.randn(m, k, device=DEV).to(torch.bfloat16)
            ref = F.linear(x.float(), copies[0].float())
            res = {}
            res["lib (eager)"] = eager(lambda w: F.linear(x, w), copies)
            if m <= 128 and hip.skinny_supported(x, copies[0]):
                res["skinny"] = timed(lambda w: hip.skinny_gemm(x, w), copies)
            cfgs = [(None, None, None, False)]
            if m > 16:
                cfgs = []
            if args.full and m <= 16:
                cfgs = [(ntw, ks, d, nt) for ntw in (1, 2) for ks in (1, 2, 4, 8) for d in (2, 3, 4)
                        for nt in (False, True) if ks <= k // 128 // 4]
            best = None
            for ntw, ks, d, nt in cfgs:
                got = hip.stream_gemm(x, copies[0], ntw=ntw, ksplit=ks, depth=d, nt=nt)
                err = (got.float() - ref).abs().max().item()
                assert err < 0.05 * max(1.0, ref.abs().max().item()), (name, m, ntw, ks, d, nt, err)
                t = timed(lambda w: hip.stream_gemm(x, w, ntw=ntw, ksplit=ks, depth=d, nt=nt), copies)
                if best is None or t < best[0]:
                    best = (t, ntw, ks, d, nt)
                if args.full:
                    print(f"    {name} M={m} ntw={ntw} ks={ks} d={d} nt={int(nt)}: {t:7.1f} us "
                          f"{nbytes / t / 1e6:5.2f} TB/s", flush=True)
            if best is not None:
                res["stream"] = best[0]
            mbest = None
            if hip.mid_supported(x, copies[0]):
                mcfgs = [(None, None, None)]
                if args.full:
                    mcfgs = [(bm, bn, ks) for bm, bn in hip._MID_TILES for ks in hip._MID_KSPLITS
                             if (bm >= min(m, 256) or (bm == 128 and m > 128)) and ks <= k // 64]
                for bm, bn, ks in mcfgs:
                    got = hip.mid_gemm(x, copies[0], bm=bm, bn=bn, ksplit=ks)
                    err = (got.float() - ref).abs().max().item()
                    assert err < 0.05 * max(1.0, ref.abs().max().item()), (name, m, bm, bn, ks, err)
                    t = timed(lambda w: hip.mid_gemm(x, w, bm=bm, bn=bn, ksplit=ks), copies)
                    if mbest is None or t < mbest[0]:
                        mbest = (t, bm, bn, ks)
                    if args.full:
                        print(f"    {name} M={m} bm={bm} bn={bn} ks={ks}: {t:7.1f} us {nbytes / t / 1e6:5.2f} TB/s "
                              f"{2 * m * n * k / t / 1e6:6.0f} TF", flush=True)
                res["mid"] = mbest[0]
            line = f"{name:16s} N={n:6d} K={k:5d} M={m:2d} | " + " | ".join(
                f"{kk} {v:7.1f} us {nbytes / v / 1e6:5.2f} TB/s" for kk, v in res.items())
            if args.full and best is not None:
                line += f" | best ntw={best[1]} ks={best[2]} d={best[3]} nt={int(best[4])}"
            elif best is not None:
                line += f" | cfg {hip.stream_choose(n, k)}"
            if mbest is not None:
                line += f" | mid cfg {mbest[1:] if args.full else hip.mid_choose(m, n, k)}"
            print(line, flush=True)
        del copies
        torch.cuda.empty_cache()


if __name__ == "__main__":
    sys.exit(main())
