// block_tile.hpp -- 64-row block arithmetic through LDS tiles, shared by the
// chained solve (chain_trsm.hip) and the residual kernel (residual.hip).
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

// Fused substitution: Ln holds -L of the diagonal block with
// its diagonal and upper part zero, rd[r] = 1 / L_ii of this lane's rows
// i = g + 16 r.  Step J: the owner lane (g == J % 16) holds
// x_J = c_J * rd_J in register q = J / 16, and each update is one
// v_fmac_{f64,f32}_dpp broadcasting x_J from that lane:
// c[r] += x_J * (-L[g + 16 r][J]).  Rows <= J are unchanged (their entries of
// Ln are zero), so after the last step row i still holds c_i and
// y_i = c_i * rd_i, which is x_i exactly as the step that owned row i computed it.
// Registers r < q hold rows above J only, which are final: step J updates
// (and loads the column entries of) registers q..3 alone.
//
// The inline-assembly updates are scheduling barriers, so the LDS reads of
// column J are issued by hand FUSED_AHEAD steps early, into a ring of
// FUSED_AHEAD + 1 register quadruples.
constexpr int FUSED_AHEAD = 4;
constexpr int FUSED_RING  = FUSED_AHEAD + 1;

template <typename T, int J>
__device__ __forceinline__ void fused_load(T (&l)[4], const T* Ln, int g)
{
#pragma unroll
    for(int r = J / 16; r < 4; ++r)
        l[r] = Ln[(g + 16 * r) * PLDA + J];
}

template <typename T, int J>
struct FusedSolve
{
    static __device__ __forceinline__ void run(T (&c)[4], const T (&rd)[4], const T* Ln, int g,
                                               int nrows, T (&lb)[FUSED_RING][4])
    {
        if constexpr(J < PNB)
        {
            // rows past the block's last real row hold c = 0: their steps
            // would add exact zeros (uniform branch)
            if(J >= nrows)
                return;
            if constexpr(J + FUSED_AHEAD < PNB)
                fused_load<T, J + FUSED_AHEAD>(lb[(J + FUSED_AHEAD) % FUSED_RING], Ln, g);
            constexpr int q  = J / 16;
            constexpr int jl = J % 16;
            const T       x  = c[q] * rd[q];
            T(&l)[4]         = lb[J % FUSED_RING];
            // x was written just before the step's first update; the solve's
            // very first update also covers a possible EXEC write
            fmac_bcast<jl, J == 0 ? 5 : 2>(c[q], x, l[q]);
            if constexpr(q < 1)
                fmac_bcast<jl, 0>(c[1], x, l[1]);
            if constexpr(q < 2)
                fmac_bcast<jl, 0>(c[2], x, l[2]);
            if constexpr(q < 3)
                fmac_bcast<jl, 0>(c[3], x, l[3]);
            FusedSolve<T, J + 1>::run(c, rd, Ln, g, nrows, lb);
        }
    }
};

// nrows: real rows of the block (steps nrows..63 are skipped)
template <typename T>
__device__ __forceinline__ void fused_solve(T (&c)[4], const T (&rd)[4], const T* Ln, int g,
                                            int nrows)
{
    T lb[FUSED_RING][4];
    fused_load<T, 0>(lb[0], Ln, g);
    fused_load<T, 1>(lb[1], Ln, g);
    fused_load<T, 2>(lb[2], Ln, g);
    fused_load<T, 3>(lb[3], Ln, g);
    static_assert(FUSED_AHEAD == 4, "prologue loads FUSED_AHEAD columns");
    FusedSolve<T, 0>::run(c, rd, Ln, g, nrows, lb);
}

// One 64 x 64 tile's update of a block's accumulators, sum_k L[row][k] y[k][v]
// on MFMA: lrow = the tile in LDS at (16 w + lane % 16, lane / 16), ycol = the
// solved block in LDS at (lane / 16, lane % 16) with row stride PLDY.  Each
// half of the fragments is read before its first product; the products
// alternate over MCH accumulator chains (fold_acc sums them).  The chained and panel solves both
// accumulate through this function, so they round identically.
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
