// gemm_tile.hpp -- launch interface of the any-alignment dense GEMM (gemm_tile.hip).
#pragma once

#include "device_common.hpp"

namespace rbamd
{
// Whether the product can run there: dense operands, K > 0, leading
// dimensions up to 2^21.
template <typename T>
bool gemm_tile_eligible(const GemmArgsT<T, T, T>& a);

// Whether it loads 16 bytes per lane: aligned operands and leading dimensions,
// whole K steps (else 4 bytes).
template <typename T>
bool gemm_tile_vec16(const GemmArgsT<T, T, T>& a);

// tile: 128 (128 x 128, whole K steps of 128 bytes), 64 (64 x 64) or, FP64 only, 32 (32 x 64)
template <typename T>
rocblas_status launch_gemm_tile(rocblas_handle h, const GemmArgsT<T, T, T>& a, int tile);
} // namespace rbamd
