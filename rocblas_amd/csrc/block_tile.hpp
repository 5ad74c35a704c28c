// block_tile.hpp -- 64-row block products through LDS tiles (residual.hip).
#pragma once

#include "panel_trsm.hpp"

namespace rbamd
{
namespace panel
{
constexpr int PNB  = 64;       // rows per block
constexpr int PLDA = PNB + 1;  // LDS row stride of a staged tile
constexpr int PLDY = PNC + 1;  // LDS row stride of the solved panel
constexpr int PEPT = PNB * PNB / PNT; // tile elements per thread
constexpr int MCH  = 2;        // MFMA accumulator chains of a tile update

// One 64 x 64 tile's update of a block's accumulators, sum_k L[row][k] y[k][v]
// on MFMA: lrow = the tile in LDS at (16 w + lane % 16, lane / 16), ycol = the
// solved block in LDS at (lane / 16, lane % 16) with row stride PLDY.  Each
// half of the fragments is read before its first product; the products
// alternate over MCH accumulator chains (fold_acc sums them).
template <typename T>
__device__ __forceinline__ void mfma_tile(typename Mfma<T>::acc_t (&acc)[MCH], const T* lrow,
                                          const T* ycol)
{
    constexpr int HALF = PNB / 8;
#pragma unroll
    for(int h = 0; h < 2; ++h)
    {
        T af[HALF], yf[HALF];
#pragma unroll
        for(int k = 0; k < HALF; ++k)
        {
            af[k] = lrow[4 * (h * HALF + k)];
            yf[k] = ycol[4 * (h * HALF + k) * PLDY];
        }
#pragma unroll
        for(int k = 0; k < HALF; ++k)
            acc[k % MCH] = Mfma<T>::run(af[k], yf[k], acc[k % MCH]);
    }
}

template <typename T>
__device__ __forceinline__ T fold_acc(const typename Mfma<T>::acc_t (&acc)[MCH], int r)
{
    static_assert(MCH == 2 || MCH == 4, "two or four chains");
    if constexpr(MCH == 2)
        return acc[0][r] + acc[1][r];
    else
        return (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]);
}
} // namespace panel
} // namespace rbamd
