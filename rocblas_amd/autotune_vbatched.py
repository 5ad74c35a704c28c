"""Autotuner of the variable-size batched solve (rocblas_amd_{s,d}trsm_vbatched).

Sweeps ``panel_groups`` per size bucket of k (<= 64, <= 128, <= 256, larger;
the last bucket is timed on k in [257, --mhi]) -- how many work items an
instance is split into (each solves a strided share of its pieces of 16 or 32 vectors)
-- each bucket timed on a seeded synthetic workload of its own sizes (default:
4096 instances, n uniform in [1, 64], side left, lower, no transpose; A with
diagonal U[1, 2] and off-diagonal U[-1, 1] / m, B uniform in [-1, 1]), then
the whole workload (m log-uniform in [8, 512]) with the winners, and writes
them as ``vbatched_tuning.hpp``.  The values are set through
rocblas_amd_vbatched_set_bucket_tuning, so no rebuild is needed per
candidate; rebuild the library after the header is written to make the
winners the built-in defaults.

    python -m rocblas_amd.autotune_vbatched [--out PATH] [--batch N] [--reps R] [--mhi K]
"""
import argparse
import os
import sys
import time

import torch

import rocblas_amd as rb
from rocblas_amd import workloads

HEADER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc", "vbatched_tuning.hpp")

PANEL_GROUPS = [1, 2, 4, 8]


def time_config(h, w, reps):
    s = torch.cuda.current_stream()
    best = float("inf")
    for r in range(reps + 1):
        w["dB"].copy_(w["dB0"])
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        e0.record(s)
        rb.check(workloads.call_vbatched(h, w), "vbatched")
        e1.record(s)
        torch.cuda.synchronize()
        if r:
            best = min(best, e0.elapsed_time(e1) * 1e-3)
    return best


def buckets(mhi):
    """k ranges of the tuning table's buckets (the last one up to mhi)."""
    return [(8, 64), (65, 128), (129, 256), (257, mhi)]


def write_header(path, groups, note):
    with open(path, "w") as f:
        f.write(f"""// vbatched_tuning.hpp -- size-bucket table of the variable-size batched solve.
// Generated by rocblas_amd/autotune_vbatched.py ({note}).
#pragma once

namespace rbamd
{{
// work items per instance of the panel kernel (each a strided share of the
// instance's pieces of 16 or 32 vectors), by size bucket of k: <= 64, <= 128, <= 256,
// larger
constexpr int kVbPanelBuckets                  = 4;
constexpr int kVbPanelGroups[kVbPanelBuckets] = {{{", ".join(str(g) for g in groups)}}};
}} // namespace rbamd
""")


def main(argv=None):
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--out", default=HEADER)
    ap.add_argument("--batch", type=int, default=4096)
    ap.add_argument("--reps", type=int, default=5)
    ap.add_argument("--seed", type=int, default=0)
    ap.add_argument("--mhi", type=int, default=512)
    args = ap.parse_args(argv)
    assert torch.cuda.is_available(), "the autotuner runs on the GPU"
    L = rb.lib()
    h = rb.Handle()
    rb.check(h.set_stream(torch.cuda.current_stream().cuda_stream))
    L.rocblas_amd_vbatched_set_tuning(0)
    # 1. each size bucket of the panel kernel on its own workload
    best_groups = []
    log = []
    try:
        for b, (lo, hi) in enumerate(buckets(args.mhi)):
            w = workloads.variable_batch(h, args.batch, lo, hi, 1, 64, args.seed)
            res = []
            for groups in PANEL_GROUPS:
                rb.check(L.rocblas_amd_vbatched_set_bucket_tuning(b, groups), "set_bucket_tuning")
                t = time_config(h, w, args.reps)
                res.append((t, groups))
                print(f"bucket k in [{lo},{hi}]: panel_groups={groups}: {t * 1e6:9.1f} us "
                      f"{w['flops'] / t / 1e12:6.2f} TFLOP/s", flush=True)
            L.rocblas_amd_vbatched_set_bucket_tuning(b, 0)
            t, g = min(res)
            best_groups.append(g)
            log.append(f"k<={hi}: {g} ({t * 1e6:.0f} us)")
            del w
            torch.cuda.empty_cache()
        # 2. the whole workload with the winners against one split for all buckets
        w = workloads.variable_batch(h, args.batch, 8, min(args.mhi, 512), 1, 64, args.seed)
        for b, g in enumerate(best_groups):
            L.rocblas_amd_vbatched_set_bucket_tuning(b, g)
        t_best = time_config(h, w, args.reps)
        L.rocblas_amd_vbatched_set_tuning(1)
        t_one = time_config(h, w, args.reps)
        print(f"whole workload: per-bucket {t_best * 1e6:.1f} us, one item per instance "
              f"{t_one * 1e6:.1f} us", flush=True)
    finally:
        L.rocblas_amd_vbatched_set_tuning(0)
    name = torch.cuda.get_device_name(0)
    write_header(args.out, best_groups,
                 f"{name}; per bucket, {args.batch} instances each, n uniform [1,64]: "
                 + "; ".join(log) + f"; whole workload m log-uniform [8,512]: "
                 f"{t_best * 1e6:.0f} us")
    print("wrote", args.out)
    h.close()
    return 0


if __name__ == "__main__":
    sys.exit(main())
