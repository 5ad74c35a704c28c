// small_trsm.hpp -- the k <= 32 triangular-solve kernel (instantiated per KMAX
// in small_k*.hip).
//
// Every side/uplo/trans case is reduced to forward substitution L y = c on a
// canonical lower triangle, one right-hand-side vector per lane:
//   side L:  op(A) X = alpha B, vectors = columns of B, M = op(A)
//   side R:  X op(A) = alpha B <=> op(A)^T X^T = alpha B^T, vectors = rows of B,
//            M = op(A)^T
//   M[i][j] = TA ? A[j][i] : A[i][j];  when M is upper triangular (REV) the
//   canonical index i is the real index KMAX-1-i, so L[i][j] = M[KMAX-1-i][KMAX-1-j].
// The matrix is embedded in a KMAX x KMAX triangle: entries outside the K x K
// problem are 0 (1 on the diagonal) and right-hand-side entries outside it are
// 0, so padded rows never change real rows -- and because the reversal is
// relative to KMAX, every offset in the substitution is a compile-time
// constant for each (UPPER, TA) variant.
//
// A wavefront serves four slots (instances) of 16 vectors each, also where an
// instance has fewer vectors.  Packing more, narrower slots with the triangles
// in LDS measured slower up to 20000 instances (FP64, side L: order 32 with 8
// vectors 102 us against 40, order 8 with one vector 11.8 against 5.9; one
// instance of order 32 with 8 vectors 17.4 against 8.6) and from order 12 on
// (200000 of order 12 with 4 vectors 0.53 of the time).  Only several 100000
// instances of order 8 or less with one to four vectors take longer this way,
// by up to 11% (FP64, order 4, 3 vectors: 28.9 us against 27.9) or 17% (FP32,
// order 2, 2 vectors: 23.6 against 20.2), others of them less (0.81 at best): not
// worth a second kernel.  Four wavefronts per workgroup change nothing there.
// Every global load of a wavefront is issued before the first wait.
//
// Pair order: within a KMAX x KMAX triangle, column c and column KMAX-1-c
// together hold exactly KMAX+1 entries, so entry t lies in pair t / (KMAX+1)
// -- constant divisions, no search -- and consecutive t walk down a column.
#pragma once

#include "device_common.hpp"

namespace rbamd
{

// offset of stored entry (p, q) of a KMAX triangle in pair order
template <int KMAX, bool UPPER>
__host__ __device__ constexpr int pair_off(int p, int q)
{
    const bool first = q < KMAX / 2;
    const int  c     = first ? q : KMAX - 1 - q;
    if(!UPPER) // column c: rows c..KMAX-1; column KMAX-1-c: rows KMAX-1-c..KMAX-1
        return c * (KMAX + 1) + (first ? p - q : (KMAX - c) + (p - q));
    else // column c: rows 0..c; column KMAX-1-c: rows 0..KMAX-1-c
        return c * (KMAX + 1) + (first ? p : (c + 1) + p);
}

// inverse of pair_off: entry t -> (p, q)
template <int KMAX, bool UPPER>
__host__ __device__ inline void pair_decode(int t, int& p, int& q)
{
    const int c = t / (KMAX + 1);
    const int o = t % (KMAX + 1);
    if(!UPPER)
    {
        const bool first = o < KMAX - c;
        q                = first ? c : KMAX - 1 - c;
        p                = first ? c + o : q + (o - (KMAX - c));
    }
    else
    {
        const bool first = o <= c;
        q                = first ? c : KMAX - 1 - c;
        p                = first ? o : o - (c + 1);
    }
}

// pair-order offset of canonical L[i][j]
template <int KMAX, bool UPPER, bool TA>
__host__ __device__ constexpr int lofs(int i, int j)
{
    constexpr bool REV = UPPER != TA;
    const int      mi  = REV ? KMAX - 1 - i : i;
    const int      mj  = REV ? KMAX - 1 - j : j;
    return TA ? pair_off<KMAX, UPPER>(mj, mi) : pair_off<KMAX, UPPER>(mi, mj);
}

// ---------------------------------------------------------------------------
// The kernel (KMAX <= 32; slots of 16 vectors, four slots per wavefront):
// each 16-lane row holds its slot's triangle in registers -- entry t of the
// pair order in lane t % 16, register t / 16, stored negated -- and every
// update c[i] -= L[i][j] x_j is a single v_fmac_{f64,f32}_dpp whose first
// operand is broadcast from the owning lane of the row (row_newbcast), so the
// substitution reads no LDS and spends no separate broadcast instruction.
// Lane n also holds the reciprocal diagonal entries n + 16 d.  An instance
// with more than 16 vectors occupies several slots, each loading the
// triangle (the duplicate loads are the same addresses in one instruction).
//
// Slot bookkeeping is wave-uniform: slot s is unit unit0 + blockIdx.x * 4 + s, and
// its instance pointers and first vector are read into scalar registers.
// Side L loads B coalesced down the columns -- load step s covers
// 64 / KMAX whole columns of one slot -- so every address is a per-lane
// constant plus a uniform base.  FULL launches (K == KMAX, every slot holds
// 16 vectors) carry no masks at all.
// ---------------------------------------------------------------------------

template <typename T, int KMAX>
using DppTri = T[(KMAX * (KMAX + 1) / 2 + 15) / 16];

// column J of the substitution: c[I] -= L[I][J] x for I = J+1 .. KMAX-1
template <typename T, int KMAX, bool UPPER, bool TA, int J, int I>
struct DppColumn
{
    static __device__ __forceinline__ void run(T (&c)[KMAX], const DppTri<T, KMAX>& Lr, T x)
    {
        if constexpr(I < KMAX)
        {
            constexpr int t = lofs<KMAX, UPPER, TA>(I, J);
            // x was written just before the column's first update; the very
            // first update of the solve also covers a possible EXEC write
            constexpr int W = I == J + 1 ? (J == 0 ? 5 : 2) : 0;
            fmac_bcast<t % 16, W>(c[I], Lr[t / 16], x);
            DppColumn<T, KMAX, UPPER, TA, J, I + 1>::run(c, Lr, x);
        }
    }
};

template <typename T, int KMAX, bool UPPER, bool TA, int J>
struct DppSolve
{
    static __device__ __forceinline__ void run(T (&c)[KMAX], const DppTri<T, KMAX>& Lr,
                                               const T (&Dr)[(KMAX + 15) / 16])
    {
        if constexpr(J < KMAX)
        {
            // lane n holds the reciprocal of the stored diagonal entry n + 16 d,
            // i.e. of real index n + 16 d; canonical J is real index JR
            constexpr int JR = (UPPER != TA) ? KMAX - 1 - J : J;
            const T       x  = c[J] * row_bcast_ordered<JR % 16>(Dr[JR / 16]);
            c[J]             = x;
            DppColumn<T, KMAX, UPPER, TA, J, J + 1>::run(c, Lr, x);
            DppSolve<T, KMAX, UPPER, TA, J + 1>::run(c, Lr, Dr);
        }
    }
};

template <typename T, int KMAX, bool UPPER, bool TA, bool COLS, bool FULL>
__global__ void __launch_bounds__(WAVE) small_trsm_dpp_kernel(const SmallArgs<T> a)
{
    static_assert(KMAX <= 32 && WAVE % KMAX == 0, "register-resident triangles up to 32");
    constexpr bool REV = UPPER != TA;
    constexpr int  TRI = KMAX * (KMAX + 1) / 2;
    constexpr int  NR  = (TRI + 15) / 16;
    constexpr int  ND  = (KMAX + 15) / 16;
    constexpr int  VP  = DPP_VP;
    constexpr int  G   = DPP_G;
    // side L: one load step covers SPS whole columns; STEPS steps per slot
    constexpr int SPS   = WAVE / KMAX;
    constexpr int STEPS = VP / SPS;

    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* const RB = reinterpret_cast<T*>(smem_raw); // side-L staging, 64 x bs_stride
    __shared__ const T* slotA[G];
    __shared__ T*       slotB[G];
    __shared__ int      slotV0[G];

    const unsigned lane = threadIdx.x;
    const unsigned n    = lane & 15;
    const unsigned g    = lane >> 4;
    const int      K    = FULL ? KMAX : a.K;
    const bool     unit = a.flags & SF_UNIT;
    const int      lda  = a.lda;
    const int      ldb  = a.ldb;
    const int      bs   = a.bs_stride;
    const int      nvec = a.nvec;

    const T alpha = a.alpha_dev ? *a.alpha_dev : a.alpha_host;

    if(lane < G)
    {
        const int64_t u = a.unit0 + int64_t(blockIdx.x) * G + lane;
        if(u < a.units)
        {
            const int64_t inst = a.chunks == 1 ? u : u / a.chunks;
            slotA[lane]        = a.A.get(inst);
            slotB[lane]        = a.B.get(inst);
            slotV0[lane]       = int(u - inst * a.chunks) * VP;
        }
        else
        {
            slotA[lane]  = nullptr;
            slotB[lane]  = nullptr;
            slotV0[lane] = 0;
        }
    }
    __syncthreads();

    // this lane's slot (row g) and vector
    const T*   myA   = slotA[g];
    T* const   myB   = slotB[g];
    const int  vec   = slotV0[g] + int(n);
    const bool valid = FULL || (myB != nullptr && vec < nvec);

    if(alpha == T(0))
    {
        if(valid)
            for(int i = 0; i < K; ++i)
                gstore(myB + (COLS ? (i + int64_t(vec) * ldb) : (vec + int64_t(i) * ldb)), T(0));
        return;
    }

    // Out-of-range lanes load from a valid address (slot 0 always exists) and
    // discard the value, so no load sits behind a branch.
    const T* const safeA = uniform_ptr(slotA[0]);
    T* const       safeB = uniform_ptr(slotB[0]);

    // ---- 1a. right-hand sides ----
    T c[KMAX];
    T bv[COLS ? KMAX : 1];
    // side L: lane = (vq, rl) loads row rl of column vq + SPS * s of its step
    const unsigned rl      = lane % KMAX;
    const unsigned vq      = lane / KMAX;
    const int64_t  laneoff = int64_t(rl) + int64_t(vq) * ldb;
    if constexpr(COLS)
    {
#pragma unroll
        for(int s = 0; s < KMAX; ++s)
        {
            const int slot = s / STEPS;
            const int k    = s % STEPS;
            T* const  sB   = uniform_ptr(slotB[slot]);
            const int sv   = uniform_int(slotV0[slot]) + SPS * k;
            const T*  p    = sB + (int64_t(sv) * ldb + laneoff);
            if constexpr(FULL)
                bv[s] = gload(p);
            else
            {
                const bool ok = sB != nullptr && int(rl) < K && sv + int(vq) < nvec;
                const T    x  = gload(ok ? p : safeB);
                bv[s]         = ok ? x : T(0);
            }
        }
    }
    else
    {
        const T* rowB = valid ? myB + vec : safeB;
#pragma unroll
        for(int i = 0; i < KMAX; ++i)
        {
            const int r = REV ? KMAX - 1 - i : i;
            if constexpr(FULL)
                c[i] = gload(rowB + int64_t(r) * ldb);
            else
            {
                const bool ok = valid && r < K;
                const T    x  = gload(ok ? rowB + int64_t(r) * ldb : safeB);
                c[i]          = ok ? x : T(0);
            }
        }
    }

    // ---- 1b. this lane's share of the triangle (negated) and of the diagonal ----
    DppTri<T, KMAX> Lr;
    const T* const  rowA   = FULL || myA ? myA : safeA;
    const bool      slotok = FULL || myA != nullptr;
#pragma unroll
    for(int r = 0; r < NR; ++r)
    {
        const unsigned t = n + 16 * r;
        int            p, q;
        pair_decode<KMAX, UPPER>(int(t < TRI ? t : 0), p, q);
        bool ok = p != q;
        if(TRI % 16 != 0 && r == NR - 1)
            ok = ok && t < TRI;
        if constexpr(!FULL)
            ok = ok && slotok && p < K && q < K;
        const T x = gload(ok ? rowA + (p + int64_t(q) * lda) : rowA);
        Lr[r]     = ok ? -x : T(0);
    }
    T Dr[ND];
#pragma unroll
    for(int d = 0; d < ND; ++d)
    {
        const int  j  = n + 16 * d;
        const bool ok = slotok && j < K && !unit;
        const T    x  = gload(rowA + (ok ? j + int64_t(j) * lda : 0));
        Dr[d]         = ok ? T(1) / x : T(1);
    }

    // ---- 1c. side L: stage the columns so lane v can read column v ----
    if constexpr(COLS)
    {
        const unsigned rr = REV ? KMAX - 1 - rl : rl;
#pragma unroll
        for(int s = 0; s < KMAX; ++s)
            RB[(vq + SPS * s) * bs + rr] = bv[s];
        __syncthreads();
#pragma unroll
        for(int i = 0; i < KMAX; ++i)
            c[i] = RB[lane * bs + i];
    }
    if(a.flags & SF_SCALE)
    {
#pragma unroll
        for(int i = 0; i < KMAX; ++i)
            c[i] *= alpha;
    }

    // ---- 2. forward substitution, one DPP multiply-add per update ----
    // Every operand the DPP instructions read is final here (an empty asm
    // that redefines it), so the compiler cannot sink the last VALU
    // instruction producing one of them (a negation, a select, the alpha
    // scaling) in front of its first DPP reader, where the required wait
    // states would be missing.  The first update of the solve pads five.
#pragma unroll
    for(int r = 0; r < NR; ++r)
        asm volatile("" : "+v"(Lr[r]));
#pragma unroll
    for(int d = 0; d < ND; ++d)
        asm volatile("" : "+v"(Dr[d]));
#pragma unroll
    for(int i = 0; i < KMAX; ++i)
        asm volatile("" : "+v"(c[i]));
    DppSolve<T, KMAX, UPPER, TA, 0>::run(c, Lr, Dr);

    // ---- 3. store ----
    if constexpr(COLS)
    {
#pragma unroll
        for(int i = 0; i < KMAX; ++i)
            RB[lane * bs + i] = c[i];
        __syncthreads();
        const unsigned rr = REV ? KMAX - 1 - rl : rl;
#pragma unroll
        for(int s = 0; s < KMAX; ++s)
        {
            const int slot = s / STEPS;
            const int k    = s % STEPS;
            T* const  sB   = uniform_ptr(slotB[slot]);
            const int sv   = uniform_int(slotV0[slot]) + SPS * k;
            const T   y    = RB[(vq + SPS * s) * bs + rr];
            T* const  p    = sB + (int64_t(sv) * ldb + laneoff);
            if constexpr(FULL)
                gstore(p, y);
            else if(sB != nullptr && int(rl) < K && sv + int(vq) < nvec)
                gstore(p, y);
        }
    }
    else if(valid)
    {
        T* const rowB = myB + vec;
#pragma unroll
        for(int i = 0; i < KMAX; ++i)
        {
            const int r = REV ? KMAX - 1 - i : i;
            if(FULL || r < K)
                gstore(rowB + int64_t(r) * ldb, c[i]);
        }
    }
}

template <typename T, int KMAX, bool UPPER, bool TA, bool COLS>
static void launch_dpp(rocblas_handle h, const SmallArgs<T>& a, dim3 grid, size_t lds)
{
    if(a.flags & SF_FULL)
        hipLaunchKernelGGL((small_trsm_dpp_kernel<T, KMAX, UPPER, TA, COLS, true>), grid,
                           dim3(WAVE), lds, h->stream, a);
    else
        hipLaunchKernelGGL((small_trsm_dpp_kernel<T, KMAX, UPPER, TA, COLS, false>), grid,
                           dim3(WAVE), lds, h->stream, a);
}

template <typename T, int KMAX, bool UPPER, bool TA>
static rocblas_status launch_small_side(rocblas_handle h, const SmallArgs<T>& a, dim3 grid,
                                        size_t lds)
{
    if(a.flags & SF_COLS)
        launch_dpp<T, KMAX, UPPER, TA, true>(h, a, grid, lds);
    else
        launch_dpp<T, KMAX, UPPER, TA, false>(h, a, grid, lds);
    return launch_status();
}

template <typename T, int KMAX>
rocblas_status launch_small_kmax(rocblas_handle h, const SmallArgs<T>& a, dim3 grid, size_t lds)
{
    const bool upper = a.flags & SF_UPPER;
    const bool ta    = a.flags & SF_TA;
    if(!upper && !ta)
        return launch_small_side<T, KMAX, false, false>(h, a, grid, lds);
    if(!upper && ta)
        return launch_small_side<T, KMAX, false, true>(h, a, grid, lds);
    if(upper && !ta)
        return launch_small_side<T, KMAX, true, false>(h, a, grid, lds);
    return launch_small_side<T, KMAX, true, true>(h, a, grid, lds);
}

} // namespace rbamd

#define RBAMD_INSTANTIATE_SMALL(KMAX)                                                     \
    namespace rbamd                                                                       \
    {                                                                                     \
    template rocblas_status launch_small_kmax<float, KMAX>(rocblas_handle,                \
                                                           const SmallArgs<float>&, dim3, \
                                                           size_t);                       \
    template rocblas_status launch_small_kmax<double, KMAX>(rocblas_handle,               \
                                                            const SmallArgs<double>&,     \
                                                            dim3, size_t);                \
    }
