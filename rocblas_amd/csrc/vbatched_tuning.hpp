// vbatched_tuning.hpp -- size-bucket table of the variable-size batched solve.
// Generated by rocblas_amd/autotune_vbatched.py with the panel solve that the
// present one replaces, 16 vectors at a time (per bucket, 4096 instances each,
// n uniform [1,64]: k<=64: 1 (141 us); k<=128: 1 (301 us); k<=256: 8 (641 us);
// k<=512: 8 (1602 us); whole workload m log-uniform [8,512]: 520 us) and kept:
// the whole workload takes 309 us with it now.
#pragma once

namespace rbamd
{
// work items per instance of the panel kernel (each a strided share of the
// instance's pieces of 16 or 32 vectors), by size bucket of k: <= 64, <= 128,
// <= 256, larger
constexpr int kVbPanelBuckets                  = 4;
constexpr int kVbPanelGroups[kVbPanelBuckets] = {1, 1, 8, 8};
} // namespace rbamd
