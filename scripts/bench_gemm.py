"""Micro-benchmark: decode projection GEMMs on the llama3.2-3B shapes — hipBLASLt
against gemm_rows, gemm_skinny and gemm_tile, timed as the tuner times them
(captured, weights cycled past the 256 MB Infinity Cache, as in-situ decode
streams them).

Usage: python scripts/bench_gemm.py [M] [--splitk-sweep]
The sweep times every tiling of gemm_tile that the tuner tries.
"""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import torch
import torch.nn.functional as F
from gridllm_amd.ops import autotune, hip_ops


def main():
    dev = "cuda:0"
    args = [a for a in sys.argv[1:] if not a.startswith("-")]
    M = int(args[0]) if args else 256
    sweep = "--splitk-sweep" in sys.argv
    shapes = [("qkv", 3072, 5120), ("o", 3072, 3072),
              ("gateup", 3072, 16384), ("down", 8192, 3072),
              ("lm_head", 3072, 128256)]
    print(f"M={M}")
    total = {}
    for name, K, N in shapes:
        x = (torch.randn(M, K, device=dev) * 0.1).to(torch.bfloat16)
        ws = autotune._weights(N, K, dev)
        ref = x.float() @ ws[0].float().t()
        scale = ref.abs().max().item()
        gb = N * K * 2 / 1e9

        def bench(what, fn):
            err = (fn(ws[0]).float() - ref).abs().max().item()
            us = autotune._time_fn(fn, ws) * 1e6
            ok = "OK" if err < 0.02 * scale + 1e-6 else f"FAIL({err:.3f})"
            return us, f"{what} {us:7.1f}us ({gb / us * 1e3:5.2f} TB/s) {ok}"
        kinds = {"blas": lambda w: F.linear(x, w)}
        if hip_ops.gemm_rows_supported(x, ws[0]):
            kinds["rows"] = lambda w: hip_ops.gemm_rows(x, w)
        if hip_ops.gemm_skinny_supported(M, N, K):
            kinds["skinny"] = lambda w: hip_ops.gemm_skinny(x, w)
        tilings = hip_ops.gemm_tilings(M, N, K)
        rule = hip_ops.gemm_tiling(M, N, K)
        if rule:
            kinds["tile"] = lambda w: hip_ops.gemm_tile(x, w, *rule)
        line = f"{name:8s} K={K:6d} N={N:6d} W={gb * 1000:7.1f}MB "
        for kind, fn in kinds.items():
            us, text = bench(kind, fn)
            line += f" {text} "
            total[kind] = total.get(kind, 0.0) + us
        print(line, flush=True)
        best = None
        for t in tilings if sweep else ():
            us, text = bench("rows={} cols={} splitk={}".format(*t),
                             lambda w: hip_ops.gemm_tile(x, w, *t))
            print(f"    {name} tile {text}", flush=True)
            best = us if best is None else min(best, us)
        if best:
            total["best tile"] = total.get("best tile", 0.0) + best
    print("layer-sum:", {k: round(v, 1) for k, v in total.items()})


if __name__ == "__main__":
    main()
