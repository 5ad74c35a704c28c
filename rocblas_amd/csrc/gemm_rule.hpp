// gemm_rule.hpp -- which dense products run on the LDS-load tiles of
// gemm_tile.hip (host only, no HIP headers).
#pragma once

#include <cstdint>

namespace rbamd
{
// Whether they take less time than the register-staged kernels, for a product
// below the 128 x 128 kernels' range: `size` bytes per element, `vec16`: 16-byte
// loads (else 4-byte ones), `cold`: a solve's update, whose operands the launch
// before has just written, `tiles64`: 64 x 64 tiles over the batch.
//
// With 16-byte loads always.  Measured on 256 CUs, LDS-load / register-staged
// time of C := A B + C, plain, A transposed, B transposed, operands from memory:
//   FP32: 16 tiles K = 64 0.95 0.95 0.85, K = 1024 0.70 0.84 0.58; 100 tiles K = 64
//     0.91 0.91 0.85; 256 tiles K = 256 0.57 0.58 0.49
//   FP64: 16 tiles K = 64 0.86 0.90 0.84; 132 tiles K = 64 0.92 0.96 0.91
// (the same operands again and again, in L2: FP32 16 tiles K = 256 1.13 1.12 0.97,
// 64 tiles K = 1024 1.07 1.10 0.87, 132 tiles 0.98 at most).
//
// 4-byte loads need more work to hide their issue, and the register-staged 32 x
// 32 tiles spread a small product over more workgroups:
//   FP64, from memory: 16 tiles K = 64 1.26, K = 1024 1.08 1.12 1.01; 182 tiles
//     1.08 1.12 1.15; 256 tiles 0.94 1.04 0.96; 376 tiles 0.94 0.99 1.01
//   FP32, from memory / from L2: 64 tiles K = 64 1.27 / 1.40, K = 256 1.08 1.01
//     0.96 / 1.45 1.28 1.27, K = 1024 0.97 0.90 0.86 / 1.45 1.32 1.28, K = 4096
//     0.94 0.88 0.82 either way; 128 tiles K = 1024 0.97 / 0.97; 256 tiles K = 64
//     0.84 0.76 0.74 / 0.93 0.83 0.82.  In solves (us, on / off): 520 x 1024, K = 320
//     40.7 / 35.0; 700 x 3072, K = 384 52.8 / 61.1; 2048 x 256 147 / 159
inline bool gemm_tile_pays(int size, bool vec16, bool cold, bool transA, bool transB,
                           int64_t tiles64, int K, int64_t cus)
{
    if(vec16 || tiles64 >= 3 * cus / 2)
        return true;
    if(size == 8)
        return tiles64 >= cus && !(transA && !transB);
    return tiles64 >= cus || K >= (cold ? 384 : 4096) || (2 * tiles64 >= cus && K >= 1024);
}

// Whether the 128 x 128 LDS-DMA kernel is faster than 64 x 64 tiles with 4-byte
// loads where both can run (aligned operands, K no multiple of 128 bytes):
// where its tiles fill the CUs once, or nearly twice.  Measured, us, DMA / 64 x
// 64, FP64: 2048 x 2048 x 1032 (256 tiles) 172 / 181, 1000 x 5000 x 3000 (320)
// 750 / 652, 2048 x 3072 x 2048 (384) 525 / 502; FP32 2048 x 2048 x 48 16.7 /
// 19.1; from two tiles per CU on the 64 x 64 tiles lose (FP64 2048 x 4096 x
// 2048 66.7 / 51.3 TF/s).
inline bool gemm_dma_beats_4byte(int64_t tiles128, int64_t cus)
{
    return (tiles128 >= cus && 16 * tiles128 <= 17 * cus) || 4 * tiles128 >= 7 * cus;
}
} // namespace rbamd
