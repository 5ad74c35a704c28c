// panel_trsm.hpp -- the panel solve shared by the single-launch k <= 512
// path (panel_trsm.hip), the persistent variable-size batch (vbatched.hip), the
// chained solve (chain_trsm.hip) and the inverses of trtri (trtri_panel.hip).
//
// PanelSolver<T, NT, NVG> solves 16 * NVG right-hand-side vectors of one
// instance with all four wavefronts of a workgroup.  Canonical form as in
// small_trsm.hpp: forward substitution L y = c on the canonical lower triangle
// (side L: vectors are columns of B, M = op(A); side R: vectors are rows of B,
// M = op(A)^T; SF_REV reverses the index).
//
// The triangle is cut into 16-row sub-blocks; wavefront w owns the sub-blocks
// t = w (mod 4) of a super-block of up to 64 NT rows and keeps their updates
// in registers, as MFMA accumulators, until each is solved (right-looking):
//
//   for e = 0, 1, ...:  s_t -= L_te y_e   for every own t > e   (MFMA)
//   own t:              y_t = L_tt^{-1} (scale b_t + s_t)       (DPP substitution)
//
// Each entry of L feeds exactly one wavefront, so L goes from memory straight
// to the MFMA operand registers: no LDS staging and no workgroup barrier in
// the loop.  The solved sub-blocks are the only shared data: the owner writes
// -y_t into a ring of LDS slots in operand order and raises a counter, and
// the others poll that counter, so a wavefront waits only for what it needs --
// the owner of the next sub-block applies y_{t-1} to that sub-block first,
// solves and publishes it, and only then updates its other sub-blocks.
//
// MFMA operands: the product is formed as Y^T L^T, so the accumulator of a
// sub-block is [vector][row]: lane l holds row l % 16, and register r a
// vector of the 16-lane group l / 16.  That is the layout the substitution
// wants: every 16-lane row of the wavefront holds the 16 rows of four vectors
// (one per register), a step's solved values are broadcast from lane J by the
// DPP multiply-add itself (row_newbcast), and the four registers are four
// independent chains that hide each other's latency.  K slot q of product kk is
// column 4 q + kk of L, so a lane's four values of y are contiguous in LDS.
//
// Bound: the chain of sub-blocks, about 1600 cycles per 16 rows (FP64, 16
// vectors): 60 DPP multiply-adds (540), publishing through LDS (310),
// noticing it (280), four dependent MFMAs (360) -- until, with many
// sub-blocks left, the matrix cores are: 256 cycles per sub-block product.
// Measured on MI355X against the solve this replaces (64-row blocks staged
// through LDS, left-looking, workgroup barriers): FP64 256 instances
// 200 x 64 79 -> 26 us, 512 x 512 on 6001 vectors 113 -> 57 us, one 512 x 256
// solve 59 (chained over workgroups) -> 35 us.
#pragma once

#include "device_common.hpp"

namespace rbamd
{
namespace panel
{
constexpr int PNC   = 16;  // vectors per vector group, rows per sub-block
constexpr int PNT   = 256; // threads
// LDS slots of solved sub-blocks.  The owner of t writes its slot after it has
// read y_{t-1}; each publisher in that chain had finished reading everything up
// to two sub-blocks before its own, and every other wavefront with sub-blocks
// left published one of the last three, so none still reads t - 5 or earlier.
constexpr int PRING = 8;

// Row pitch (elements) of a solved sub-block in LDS, [vector][row]: a lane
// reads four consecutive rows of a vector as 16-byte words, conflict-free.
template <typename T>
constexpr int ypitch()
{
    return sizeof(T) == 8 ? 18 : 20;
}

// LDS bytes of one workgroup: the ring, a diagonal block with its reciprocal
// diagonal per wavefront, and the published-sub-block counter
template <typename T, int NVG>
constexpr size_t lds_bytes()
{
    return sizeof(T) * PNC * (size_t(PRING) * NVG * ypitch<T>() + 4 * (ypitch<T>() + 1)) + 16;
}

// One substitution step for the vectors a 16-lane row holds, one per register
// r < NR: c_r += c_r[lane J] * l, with l = -L[g][J] / L[J][J] below the
// diagonal and 0 elsewhere.  A register is read through DPP at least two wait
// states after the previous step wrote it (the other registers' updates, or
// padding); the padding of step 0 covers whatever came before.
template <int J, int NR>
__device__ __forceinline__ void solve_step(double (&c)[4], double l)
{
    if constexpr(NR == 4 && J == 0)
        asm volatile("s_nop 4\n\t"
                     "v_fmac_f64_dpp %0, %0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f64_dpp %1, %1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f64_dpp %2, %2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f64_dpp %3, %3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3])
                     : "v"(l), "n"(J));
    else if constexpr(NR == 4)
        asm volatile("v_fmac_f64_dpp %0, %0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f64_dpp %1, %1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f64_dpp %2, %2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f64_dpp %3, %3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3])
                     : "v"(l), "n"(J));
    if constexpr(NR == 2 && J == 0)
        asm volatile("s_nop 4\n\t"
                     "v_fmac_f64_dpp %0, %0, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f64_dpp %1, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0]), "+v"(c[1])
                     : "v"(l), "n"(J));
    else if constexpr(NR == 2)
        asm volatile("s_nop 0\n\t"
                     "v_fmac_f64_dpp %0, %0, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f64_dpp %1, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0]), "+v"(c[1])
                     : "v"(l), "n"(J));
    if constexpr(NR == 1 && J == 0)
        asm volatile("s_nop 4\n\t"
                     "v_fmac_f64_dpp %0, %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0])
                     : "v"(l), "n"(J));
    else if constexpr(NR == 1)
        asm volatile("s_nop 1\n\t"
                     "v_fmac_f64_dpp %0, %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0])
                     : "v"(l), "n"(J));
}
template <int J, int NR>
__device__ __forceinline__ void solve_step(float (&c)[4], float l)
{
    if constexpr(NR == 4 && J == 0)
        asm volatile("s_nop 4\n\t"
                     "v_fmac_f32_dpp %0, %0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f32_dpp %1, %1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f32_dpp %2, %2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f32_dpp %3, %3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3])
                     : "v"(l), "n"(J));
    else if constexpr(NR == 4)
        asm volatile("v_fmac_f32_dpp %0, %0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f32_dpp %1, %1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f32_dpp %2, %2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f32_dpp %3, %3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3])
                     : "v"(l), "n"(J));
    if constexpr(NR == 2 && J == 0)
        asm volatile("s_nop 4\n\t"
                     "v_fmac_f32_dpp %0, %0, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f32_dpp %1, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0]), "+v"(c[1])
                     : "v"(l), "n"(J));
    else if constexpr(NR == 2)
        asm volatile("s_nop 0\n\t"
                     "v_fmac_f32_dpp %0, %0, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                     "v_fmac_f32_dpp %1, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0]), "+v"(c[1])
                     : "v"(l), "n"(J));
    if constexpr(NR == 1 && J == 0)
        asm volatile("s_nop 4\n\t"
                     "v_fmac_f32_dpp %0, %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0])
                     : "v"(l), "n"(J));
    else if constexpr(NR == 1)
        asm volatile("s_nop 1\n\t"
                     "v_fmac_f32_dpp %0, %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf bound_ctrl:1"
                     : "+v"(c[0])
                     : "v"(l), "n"(J));
}

template <typename T, int NVG, int NR, int J>
struct SolveSteps
{
    static __device__ __forceinline__ void run(T (&c)[NVG][4], const T (&l)[PNC - 1])
    {
        if constexpr(J < PNC - 1) // row 15 has no rows below
        {
#pragma unroll
            for(int v = 0; v < NVG; ++v)
                solve_step<J, NR>(c[v], l[J]);
            SolveSteps<T, NVG, NR, J + 1>::run(c, l);
        }
    }
};

// Range in which a scaled entry -L[i][J] / L[J][J] stands for the division of
// the step's value: finite, and not so small that bits of a non-zero entry
// are lost.
__device__ __forceinline__ bool scaled_ok(double l, double s)
{
    return (__builtin_fabs(s) <= 0x1p+1000) & ((__builtin_fabs(s) >= 0x1p-1000) | (l == 0.0));
}
__device__ __forceinline__ bool scaled_ok(float l, float s)
{
    return (__builtin_fabsf(s) <= 0x1p+120f) & ((__builtin_fabsf(s) >= 0x1p-120f) | (l == 0.0f));
}

// an infinity or NaN
__device__ __forceinline__ bool not_finite(double x)
{
    return __builtin_amdgcn_class(x, 0x207);
}
__device__ __forceinline__ bool not_finite(float x)
{
    return __builtin_amdgcn_classf(x, 0x207);
}

// Bounds of the LDS waits.  Every wait ends by itself (all wavefronts of a
// workgroup are resident, and the owner of the first unpublished sub-block
// waits for published ones only); the poll limit turns a mistake into a
// reported error instead of a hang: the wait raises the handle's error word
// and goes on.  `bias` (0 in normal launches) makes every target unreachable.
struct PanelWait
{
    unsigned* err;
    int       spin_limit;
    int       bias;
};

inline PanelWait panel_wait(rocblas_handle h)
{
    return h->chain_debug_timeout ? PanelWait{h->async_error, 64, 1 << 30}
                                  : PanelWait{h->async_error, 1 << 20, 0};
}

// Register r of 16-lane group q is row mfma_row(q, r) of the MFMA result.
template <typename T>
__device__ __forceinline__ int mfma_row(int q, int r)
{
    return Mfma<T>::row(q << 4, r);
}

// Four contiguous elements at any element-aligned address
template <typename T>
__device__ __forceinline__ void load4(T (&x)[4], const T* p)
{
    typedef T v4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    const v4  v = *(const __attribute__((address_space(1))) v4*)(p);
#pragma unroll
    for(int r = 0; r < 4; ++r)
        x[r] = v[r];
}
// Agent-scope accesses: written through to, and read from, the point where the
// XCDs' L2 caches agree
template <typename T>
__device__ __forceinline__ T coherent_load(const T* p)
{
    return __hip_atomic_load(const_cast<__attribute__((address_space(1))) T*>(
                                 (const __attribute__((address_space(1))) T*)(p)),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void coherent_store(T* p, T x)
{
    __hip_atomic_store((__attribute__((address_space(1))) T*)(p), x, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T>
__device__ __forceinline__ void store4(T* p, const T (&x)[4])
{
    typedef T v4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    *(__attribute__((address_space(1))) v4*)(p) = v4{x[0], x[1], x[2], x[3]};
}

// Rows i0..i1 - 1 of nv (16 or 32) vectors of B from v0 := 0 (alpha == 0; A is
// not referenced)
template <typename T>
__device__ void panel_zero(T* Bp, int i0, int i1, int nvec, int ldb, int flags, int v0, int nv)
{
    const int vend = min(v0 + nv, nvec);
    int       tid  = threadIdx.x;
    asm volatile("" : "+v"(tid)); // (nothing of this is kept in registers beside a solve)
    if(flags & SF_COLS)
    {
        for(int v = v0 + tid / WAVE; v < vend; v += PNT / WAVE)
            for(int i = i0 + tid % WAVE; i < i1; i += WAVE)
                gstore(Bp + (int64_t(i) + int64_t(v) * ldb), T(0));
    }
    else
    {
        const int lg = nv > PNC ? 5 : 4;
        const int v  = v0 + (tid & (nv - 1));
        for(int i = i0 + (tid >> lg); v < vend && i < i1; i += PNT >> lg)
            gstore(Bp + (int64_t(v) + int64_t(i) * ldb), T(0));
    }
}

// How a triangle of more than 64 NT rows is walked.
enum PanelMode
{
    PM_SINGLE, // it has at most 64 NT rows: one super-block
    PM_MULTI,  // this workgroup solves its super-blocks one after another
    PM_CHAIN,  // each super-block has a workgroup of its own (chain_trsm.hip)
    PM_INVERSE // one super-block whose right-hand side is the unit vectors 0..15
               // of canonical order (trtri_panel.hip): B is only written
};

// Flags of a panel of the chained solve, in device memory: word w counts the
// sub-blocks of wavefront w (t % 4 == w, over all super-blocks) whose solution
// is in B, word 4 the workgroups that have finished.
constexpr int CHAIN_WORDS = 8;

// NR: registers (vectors per 16-lane row) in use, 4 NR vectors of the group
// KC: the columns of canonical L are contiguous in memory (op(A) transposed on
// the left, plain on the right), so a lane's four operand entries are one load
template <typename T, int NT, int NVG, PanelMode MODE, int NR, bool KC>
struct PanelSolver
{
    using acc_t             = typename Mfma<T>::acc_t;
    static constexpr int YP = ypitch<T>();
    static constexpr int YV = PNC * YP;  // elements of one vector group in a slot
    static constexpr int YS = NVG * YV;  // elements of one slot
    // FP32 holds four adjacent vectors per lane (4 q + r): where they are rows
    // of B, one 16-byte access instead of four (20000 instances of 48 rows and
    // 128 vectors 540 -> 364 us).  FP64 holds q + 4 r.
    static constexpr bool WIDE = sizeof(T) == 4;

    // instance: canonical L(i, j) at Ab[i rs + j cs], right-hand side (row i,
    // vector v) at Bb[i br + v bv]
    const T* Ab;
    T*       Bb;
    int      rs, cs, br, bv;
    int      K, nsub, nvec, v0;
    bool     unit;
    bool     full_rows; // the vectors are rows of B and all 16 NVG of them exist
    bool     turned;    // PM_INVERSE: the result goes below the diagonal only, transposed
    T        scale;
    // wavefront and lane
    int     w, g, q;
    int64_t lq; // 4 q columns
    // operand kk is column 4 q + (kk ^ kx) of L: 3 where the columns run
    // backwards in memory (KC, reversed), so that the load stays one ascending
    // access; bk: the matching step between rows of B
    int kx, bk;
    // LDS
    T*        Y;
    T*        D; // this wavefront's diagonal block and reciprocal diagonal
    int*      done;
    int       seen;
    PanelWait pw;
    unsigned* link;  // PM_CHAIN: the panel's flags
    int       avail; // PM_CHAIN: sub-blocks known to be in B

    // state: -sum of L y so far, L operands in flight; of the next sub-block to
    // solve the right-hand sides and the diagonal block
    acc_t C[NT][NVG];
    T     Lf[NT][4];
    T     bq[NVG][4];
    T     Dr[4];       // the diagonal block as loaded
    T     dg;          // and this lane's diagonal entry, then its reciprocal
    int   sb; // first sub-block of the super-block
    int   e;  // next solved sub-block to apply

    __device__ __forceinline__ int tile(int mine, int act) const
    {
        return sb + w + 4 * (mine - act);
    }

    // One address register pair, stepped from load to load: a set of
    // addresses computed ahead would need more registers than the operands.
    static __device__ __forceinline__ void pin(const T*& p)
    {
        asm volatile("" : "+v"(p));
    }

    // Vector of a group in register r of 16-lane group q: the result layout's
    // order, except where only NR registers are used, which then hold the
    // first 4 NR vectors in both types.
    static __device__ __forceinline__ int group_vec(int q_, int r)
    {
        return NR == 4 ? mfma_row<T>(q_, r) : q_ + 4 * r;
    }
    // the same for an MFMA row (lane index l % 16 of the y operand)
    static __device__ __forceinline__ int row_vec(int row)
    {
        return NR == 4 || sizeof(T) == 8 ? row : (row >> 2) + 4 * (row & 3);
    }

    // operand registers of L(t, ev): row 16 t + g, columns 16 ev + 4 q + kk.
    // Rows past K - 1 (last sub-block) read row K - 1; they feed only rows
    // that are never stored.  ev < t, so every column is below K.
    __device__ __forceinline__ void load_l(T (&f)[4], int t, int ev)
    {
        const int row = min(PNC * t + g, K - 1);
        const T*  p   = Ab + int64_t(PNC * ev) * cs + (int64_t(row) * rs + lq);
        if constexpr(KC)
            load4(f, p);
        else
        {
#pragma unroll
            for(int kk = 0; kk < 4; ++kk)
            {
                f[kk] = gload(p);
                p += cs;
                pin(p);
            }
        }
    }

    // raw diagonal block of sub-block t: row 16 t + g, columns 16 t + 4 q + kk,
    // and the row's diagonal entry (indices past K - 1 read K - 1 instead)
    __device__ __forceinline__ void load_diag(int t)
    {
        const int row = min(PNC * t + g, K - 1);
        const T*  p   = Ab + int64_t(row) * rs;
        dg            = gload(p + int64_t(row) * cs);
#pragma unroll
        for(int kk = 0; kk < 4; ++kk)
            Dr[kk] = gload(p + int64_t(min(PNC * t + 4 * q + kk, K - 1)) * cs);
    }

    // Diagonal block of sub-block t: its reciprocal diagonal, and its columns
    // below the diagonal scaled by it (0 elsewhere, and in rows past K - 1,
    // whose entries may lie outside the triangle), row g in every lane of
    // column g.  Each lane scales the four entries it loaded, and a wavefront's
    // own 16 x 16 corner of LDS spreads the rows (a wavefront's LDS accesses
    // execute in order).  False if an entry leaves the range (a nearly
    // singular or badly scaled block): solve() then takes the unscaled form.
    // Pinned, so that all of it is done before the wait for the last update.
    __device__ __forceinline__ bool prep_diag(T (&Ld)[PNC - 1], int t)
    {
        constexpr int PER = 16 / int(sizeof(T));
        typedef T     word __attribute__((ext_vector_type(PER)));
        const int     below = PNC * t + g < K ? g : 0;
        T* const      rd    = D + PNC * YP;
        dg                  = unit ? T(1) : T(1) / dg;
        rd[g]               = dg;
        asm volatile("" ::: "memory");
        bool ok = true;
        T    s[4];
#pragma unroll
        for(int kk = 0; kk < 4; ++kk)
        {
            const bool low = 4 * q + kk < below;
            const T    x   = low ? -Dr[kk] : T(0);
            s[kk]          = x * rd[4 * q + kk];
            ok             = ok & (!low | scaled_ok(x, s[kk]));
            s[kk]          = low ? s[kk] : T(0);
        }
        T* const dw = D + g * YP;
#pragma unroll
        for(int k0 = 0; k0 < 4; k0 += PER)
        {
            word x;
#pragma unroll
            for(int i = 0; i < PER; ++i)
                x[i] = s[k0 + i];
            *reinterpret_cast<word*>(dw + 4 * q + k0) = x;
        }
        const bool all = __builtin_amdgcn_ballot_w64(!ok) == 0;
        asm volatile("" ::: "memory");
#pragma unroll
        for(int j = 0; j < PNC; j += PER)
        {
            const word x = *reinterpret_cast<const word*>(dw + j);
#pragma unroll
            for(int i = 0; i < PER; ++i)
                if(j + i < PNC - 1)
                    Ld[j + i] = x[i];
        }
#pragma unroll
        for(int j = 0; j < PNC - 1; ++j)
            asm volatile("" : "+v"(Ld[j]));
        return all;
    }

    // right-hand sides of sub-block t
    __device__ __forceinline__ void load_rhs(int t)
    {
        load_rhs(t, br, bv);
    }
    __device__ __forceinline__ void load_rhs(int t, int br, int bv)
    {
        if constexpr(MODE == PM_INVERSE)
        {
#pragma unroll
            for(int r = 0; r < NR; ++r)
                bq[0][r] = PNC * t + g == group_vec(q, r) ? T(1) : T(0);
            return;
        }
        const T* p = Bb + int64_t(min(PNC * t + g, K - 1)) * br;
        if(WIDE && NR == 4 && MODE != PM_CHAIN && full_rows)
        {
#pragma unroll
            for(int v = 0; v < NVG; ++v)
                load4(bq[v], p + (v0 + PNC * v + 4 * q));
        }
        else
        {
#pragma unroll
            for(int v = 0; v < NVG; ++v)
#pragma unroll
                for(int r = 0; r < NR; ++r)
                    bq[v][r] = gload(p + int64_t(min(v0 + PNC * v + group_vec(q, r), nvec - 1)) * bv);
        }
    }

    // y of sub-block ev of an earlier super-block, read back from B (negated)
    __device__ __forceinline__ void load_y(T (&y)[NVG][4], int ev)
    {
#pragma unroll
        for(int v = 0; v < NVG; ++v)
        {
            const T* p = Bb + int64_t(min(v0 + PNC * v + row_vec(g), nvec - 1)) * bv
                         + int64_t(PNC * ev + 4 * q + kx) * br;
#pragma unroll
            for(int kk = 0; kk < 4; ++kk)
                y[v][kk] = MODE == PM_CHAIN ? coherent_load(p + int64_t(kk) * bk)
                                            : gload(p + int64_t(kk) * bk);
        }
    }

    // y of sub-block ev, once it is published.  Each poll reads the counter
    // and then the slot: a wavefront's LDS reads execute in order, so when the
    // counter says the slot is written, the values read after it are the
    // published ones (otherwise they are read again).
    __device__ __forceinline__ void wait_y(T (&yf)[NVG][4], int ev)
    {
        // 16-byte words (every term of the address is a multiple of one)
        constexpr int PER = 16 / int(sizeof(T));
        typedef T     word __attribute__((ext_vector_type(PER)));
        const T*      p    = Y + (ev % PRING) * YS + g * YP + 4 * q;
        const int     need = ev + 1 + pw.bias;
        for(int it = 0;; ++it)
        {
            int n = seen;
            if(n < need)
                n = __hip_atomic_load(done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            asm volatile("" ::: "memory"); // the slot is read after the counter
#pragma unroll
            for(int v = 0; v < NVG; ++v)
#pragma unroll
                for(int k0 = 0; k0 < 4; k0 += PER)
                {
                    const word x = *reinterpret_cast<const word*>(p + v * YV + k0);
#pragma unroll
                    for(int i = 0; i < PER; ++i)
                        yf[v][k0 + i] = x[i];
                }
            seen = __builtin_amdgcn_readfirstlane(n);
            if(seen >= need)
                break;
            if(it >= pw.spin_limit)
            {
                if(pw.err)
                    __hip_atomic_store(pw.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                seen = 0x7fffffff;
                break;
            }
            asm volatile("" ::: "memory");
        }
    }

    // c_t += (-y)^T L^T
    template <int I>
    __device__ __forceinline__ void apply(const T (&yf)[NVG][4])
    {
#pragma unroll
        for(int kk = 0; kk < 4; ++kk)
#pragma unroll
            for(int v = 0; v < NVG; ++v)
                C[I][v] = Mfma<T>::run(yf[v][kk], Lf[I][kk], C[I][v]);
    }

    // apply the current y to own tiles I..NT-1 and load their next operands
    // (tile I is sub-block t, the others follow 4 apart)
    template <int I>
    __device__ __forceinline__ void apply_from(const T (&yf)[NVG][4], int t)
    {
        if constexpr(I < NT)
        {
            apply<I>(yf);
            load_l(Lf[I], t, e + 1);
            apply_from<I + 1>(yf, t + 4);
        }
    }

    // The unscaled substitution: x_J = c_J / L_JJ first, then c_i -= L_iJ x_J for
    // the rows below only, column by column from memory.  For blocks that
    // prep_diag() refuses, and for what is not finite after the scaled steps:
    // those multiply the rows from J up by 0, which an infinity turns into NaN
    // there too.
    __device__ __forceinline__ void solve_unscaled(T (&c)[NVG][4], int t)
    {
        // (opaque: what this seldom taken path computes is not to be kept in
        // registers outside it)
        int rs_ = rs, cs_ = cs, K_ = K, t_ = t;
        asm volatile("" : "+s"(rs_), "+s"(cs_), "+s"(K_), "+s"(t_));
        const int below = PNC * t_ + g < K_ ? g : 0;
        const T*  p     = Ab + int64_t(min(PNC * t_ + g, K_ - 1)) * rs_ + int64_t(PNC * t_) * cs_;
        for(int j = 0; j < PNC - 1 && PNC * t_ + j < K_; ++j)
        {
            const T x = gload(p);
            p += cs_;
#pragma unroll
            for(int v = 0; v < NVG; ++v)
#pragma unroll
                for(int r = 0; r < NR; ++r)
                {
                    const T    y   = __shfl(c[v][r] * dg, 16 * q + j, WAVE);
                    const bool use = j < below && !above_unit(t, j, r);
                    c[v][r]        = use ? fma(y, -x, c[v][r]) : c[v][r];
                }
        }
    }

    // PM_INVERSE: row j of sub-block t is above the 1 of the unit vector in
    // register r, so the inverse has a zero there (a zero pivot makes 0 / 0 of it)
    __device__ __forceinline__ bool above_unit(int t, int j, int r) const
    {
        return MODE == PM_INVERSE && t == 0 && j < group_vec(q, r);
    }

    // c by dg or -dg: y_t from the eliminated right-hand sides.  Two products
    // rather than a product and a negation, which takes two instructions in
    // FP64; only the negated one, for the LDS slot, is on the chain.
    __device__ __forceinline__ void scale_y(T (&y)[NVG][4], const T (&c)[NVG][4], T by, int t) const
    {
#pragma unroll
        for(int v = 0; v < NVG; ++v)
#pragma unroll
            for(int r = 0; r < NR; ++r)
                y[v][r] = c[v][r] * by;
        if constexpr(MODE == PM_INVERSE)
            if(t == 0)
            {
#pragma unroll
                for(int r = 0; r < NR; ++r)
                    y[0][r] = above_unit(t, g, r) ? T(0) : y[0][r];
            }
    }
    // -y_t into its LDS slot
    __device__ __forceinline__ void write_y(const T (&y)[NVG][4], int t) const
    {
        T* p = Y + (t % PRING) * YS + (g ^ kx);
#pragma unroll
        for(int v = 0; v < NVG; ++v)
#pragma unroll
            for(int r = 0; r < NR; ++r)
                p[v * YV + mfma_row<T>(q, r) * YP] = y[v][r];
    }

    // own sub-block t (tile I) is final: solve, publish, store
    template <int I>
    __device__ __forceinline__ void solve(const T (&Ld)[PNC - 1], int t, bool scaled)
    {
        // the accumulated sums join the right-hand sides only here, so their
        // roundings are of the sums' own size (and the MFMA results are first
        // read by instructions the compiler pads for: it does not look into
        // inline assembly)
        T c[NVG][4];
#pragma unroll
        for(int v = 0; v < NVG; ++v)
#pragma unroll
            for(int r = 0; r < NR; ++r)
                c[v][r] = fma(scale, bq[v][r], C[I][v][r]);
        if(scaled)
            SolveSteps<T, NVG, NR, 0>::run(c, Ld);
        // A value that is not finite when its step reads it leaves none of its
        // vector finite.  The checks run beside the LDS writes, where they cost
        // the chain nothing (512 x 256 35.4 -> 35.5 us; in front of the writes
        // 36.5), and up to 5% where many short solves fill the vector units (FP64
        // 2000 instances 65 x 130 125 -> 130 us).
        T y[NVG][4];
        T ndg = -dg;
        asm volatile("" : "+v"(ndg)); // (not folded into negations)
        scale_y(y, c, ndg, t);
        write_y(y, t);
        uint64_t again = scaled ? 0 : 1;
#pragma unroll
        for(int v = 0; v < NVG; ++v)
#pragma unroll
            for(int r = 0; r < NR; ++r)
                again |= __builtin_amdgcn_ballot_w64(not_finite(y[v][r]));
        // the slot is written before the counter says so
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if(__builtin_expect(again != 0, 0))
        {
            T d[NVG][4];
            // (the right-hand sides are not kept during the steps; opaque as in
            // solve_unscaled)
            int br_ = br, bv_ = bv;
            asm volatile("" : "+s"(br_), "+s"(bv_));
            load_rhs(t, br_, bv_);
#pragma unroll
            for(int v = 0; v < NVG; ++v)
#pragma unroll
                for(int r = 0; r < NR; ++r)
                    d[v][r] = fma(scale, bq[v][r], C[I][v][r]);
            solve_unscaled(d, t);
            // finite results keep their bits whatever their neighbours hold
#pragma unroll
            for(int v = 0; v < NVG; ++v)
#pragma unroll
                for(int r = 0; r < NR; ++r)
                    c[v][r] = scaled && !not_finite(y[v][r]) ? c[v][r] : d[v][r];
            scale_y(y, c, ndg, t);
            write_y(y, t);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        __hip_atomic_store(done, t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        scale_y(c, c, dg, t);
        // (opaque, so the addresses are not kept in registers all along)
        int qs = q;
        asm volatile("" : "+v"(qs));
        const int row = PNC * t + g;
        T*        b   = Bb + int64_t(row) * br;
        if(WIDE && NR == 4 && MODE != PM_CHAIN && full_rows)
        {
            if(row < K)
            {
#pragma unroll
                for(int v = 0; v < NVG; ++v)
                    store4(b + (v0 + PNC * v + 4 * qs), c[v]);
            }
            return;
        }
#pragma unroll
        for(int v = 0; v < NVG; ++v)
#pragma unroll
            for(int r = 0; r < NR; ++r)
            {
                const int vec = v0 + PNC * v + group_vec(qs, r);
                if(row < K && vec < nvec && (MODE != PM_INVERSE || !turned || row > vec))
                {
                    if constexpr(MODE == PM_CHAIN)
                        coherent_store(b + int64_t(vec) * bv, c[v][r]);
                    else
                        gstore(b + int64_t(vec) * bv, c[v][r]);
                }
            }
    }

    // Own tiles are C[NT - mine]..C[NT - 1].  Tile I is the first one not yet
    // solved (if this wavefront has so many): bring it up to date, solve it,
    // go on with the others.
    template <int I>
    __device__ __forceinline__ void segments(int mine)
    {
        if constexpr(I < NT)
        {
            if(mine >= NT - I)
            {
                const int t = sb + w + 4 * (mine - (NT - I));
                T         yf[NVG][4];
                T         Ld[PNC - 1];
                for(; e < t - 1; ++e)
                {
                    wait_y(yf, e);
                    apply_from<I>(yf, t);
                }
                const bool scaled = prep_diag(Ld, t);
                if(t > sb)
                {
                    wait_y(yf, e); // e == t - 1
                    apply<I>(yf);
                }
                solve<I>(Ld, t, scaled);
                if(I + 1 < NT)
                {
                    load_diag(t + 4);
                    load_rhs(t + 4);
                    if(t > sb)
                    {
                        apply_from<I + 1>(yf, t + 4);
                        ++e;
                    }
                }
                if constexpr(MODE == PM_CHAIN)
                    raise(t);
            }
            segments<I + 1>(mine);
        }
    }

    __device__ __forceinline__ void clear(int i)
    {
#pragma unroll
        for(int v = 0; v < NVG; ++v)
            C[i][v] = acc_t{0, 0, 0, 0};
#pragma unroll
        for(int kk = 0; kk < 4; ++kk)
            Lf[i][kk] = T(0);
    }

    // a super-block in which this wavefront owns `mine` sub-blocks
    __device__ __forceinline__ void super_block(int mine)
    {
        const int t0 = sb + w;
        dg = T(0);
#pragma unroll
        for(int kk = 0; kk < 4; ++kk)
            Dr[kk] = T(0);
#pragma unroll
        for(int v = 0; v < NVG; ++v)
#pragma unroll
            for(int r = 0; r < 4; ++r)
                bq[v][r] = T(0);
        if(mine > 0)
        {
            load_diag(t0);
            load_rhs(t0);
        }
#pragma unroll
        for(int i = 0; i < NT; ++i)
        {
            clear(i); // (nothing is carried over from an earlier solve)
            if(mine >= NT - i)
            {
                const int t = t0 + 4 * (mine - (NT - i));
                if(t > 0)
                    load_l(Lf[i], t, 0);
            }
        }
        e = 0;
        if(MODE == PM_CHAIN && sb > 0)
            early_chain(mine);
        if(MODE == PM_MULTI && sb > 0)
        {
            // the earlier super-blocks' solution, without a chain
            T yf[NVG][4], yn[NVG][4];
            load_y(yn, 0);
            for(; e < sb; ++e)
            {
#pragma unroll
                for(int v = 0; v < NVG; ++v)
#pragma unroll
                    for(int kk = 0; kk < 4; ++kk)
                        yf[v][kk] = -yn[v][kk];
                load_y(yn, min(e + 1, sb - 1));
                early<0>(yf, mine);
            }
        }
        // (no load of the loops above is in flight from here on: else the
        // compiler waits for it, and with it for the operands loaded later,
        // wherever one of its registers is used again)
        if(MODE == PM_CHAIN || MODE == PM_MULTI)
            __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
        segments<0>(mine);
    }

    // y_t is in B: this wavefront's stores are complete (they are write-through),
    // then its flag says so
    __device__ __forceinline__ void raise(int t)
    {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __hip_atomic_store(link + w, unsigned(t / 4 + 1), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }

    // Sub-blocks 0..count - 1 are in B once flag i has passed those of wavefront i
    __device__ __forceinline__ unsigned read_flags() const
    {
        return __hip_atomic_load(link + (g & 3), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ int count_of(unsigned f) const
    {
        const int n  = int(4 * f) + (g & 3);
        const int n0 = __builtin_amdgcn_readlane(n, 0), n1 = __builtin_amdgcn_readlane(n, 1);
        const int n2 = __builtin_amdgcn_readlane(n, 2), n3 = __builtin_amdgcn_readlane(n, 3);
        return min(min(n0, n1), min(n2, n3));
    }
    __device__ __forceinline__ void wait_avail(int ev)
    {
        const int need = ev + pw.bias;
        for(int it = 0; avail <= need; ++it)
        {
            avail = count_of(read_flags());
            if(it >= pw.spin_limit && avail <= need)
            {
                if(pw.err)
                    __hip_atomic_store(pw.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                avail = 0x7fffffff;
            }
        }
        asm volatile("" ::: "memory"); // B is read after the flags
    }

    // The earlier super-blocks' solution as their workgroups publish it: y of
    // the next sub-block is in flight during the products of one wherever it
    // is known to be there, and the flags are read beside the products where
    // it is not.
    __device__ __forceinline__ void early_chain(int mine)
    {
        T    yf[NVG][4], yn[NVG][4];
        bool have = false;
        for(; e < sb; ++e)
        {
            if(!have)
            {
                wait_avail(e);
                load_y(yn, e);
            }
#pragma unroll
            for(int v = 0; v < NVG; ++v)
#pragma unroll
                for(int kk = 0; kk < 4; ++kk)
                    yf[v][kk] = -yn[v][kk];
            have = e + 1 < sb && avail > e + 1 + pw.bias;
            if(have)
            {
                load_y(yn, e + 1);
                early<0>(yf, mine);
            }
            else
            {
                const unsigned f = read_flags();
                early<0>(yf, mine);
                avail = max(avail, count_of(f));
            }
        }
    }

    // one sub-block of an earlier super-block, applied to every own tile
    template <int I>
    __device__ __forceinline__ void early(const T (&yf)[NVG][4], int mine)
    {
        if constexpr(I < NT)
        {
            if(mine >= NT - I)
            {
                const int t = sb + w + 4 * (mine - (NT - I));
                apply<I>(yf);
                if(e + 1 < t)
                    load_l(Lf[I], t, e + 1);
            }
            early<I + 1>(yf, mine);
        }
    }

    __device__ __forceinline__ void run(const T* Ap, T* Bp, int K_, int nvec_, int lda, int ldb,
                                        int flags, T scale_, int v0_, unsigned char* smem,
                                        PanelWait pw_, unsigned* link_ = nullptr, int sb_ = 0)
    {
        const bool tA   = flags & SF_TA;
        const bool rev  = flags & SF_REV;
        const bool cols = flags & SF_COLS;
        const int  lane = threadIdx.x & (WAVE - 1);
        K               = K_;
        nsub            = (K + PNC - 1) / PNC;
        nvec            = nvec_;
        v0              = v0_;
        unit            = flags & SF_UNIT;
        full_rows       = !cols && v0 + PNC * NVG <= nvec;
        scale           = scale_;
        w               = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
        g               = lane & 15;
        q               = lane >> 4;
        const int s     = rev ? -1 : 1;
        rs              = s * (tA ? lda : 1);
        cs              = s * (tA ? 1 : lda);
        br              = s * (cols ? 1 : ldb);
        bv              = cols ? ldb : 1;
        kx              = KC && rev ? 3 : 0;
        bk              = kx ? -br : br;
        lq              = int64_t(4 * q + kx) * cs;
        Ab              = Ap + (rev ? int64_t(K - 1) * (int64_t(lda) + 1) : 0);
        Bb              = Bp + (rev ? int64_t(K - 1) * (cols ? 1 : ldb) : 0);
        if constexpr(MODE == PM_INVERSE)
        {
            Bb     = Bp + (rev ? int64_t(K - 1) * (int64_t(ldb) + 1) : 0);
            turned = flags & SF_TRANSPOSED;
            bv     = s * (turned ? 1 : ldb); // the columns of the inverse are reversed with its rows
            br     = s * (turned ? ldb : 1);
        }
        Y               = reinterpret_cast<T*>(smem);
        D               = Y + PRING * YS + w * PNC * (YP + 1);
        done            = reinterpret_cast<int*>(Y + PRING * YS + 4 * PNC * (YP + 1));
        pw              = pw_;
        seen            = 0;
        if(threadIdx.x == 0)
            *done = sb_;
        __syncthreads();
        if constexpr(MODE == PM_CHAIN)
        {
            link  = link_;
            avail = 0;
            sb    = sb_;
            seen  = sb; // the counter starts where this super-block does
            super_block((min(4 * NT, nsub - sb) - w + 3) / 4);
        }
        else if constexpr(MODE == PM_SINGLE || MODE == PM_INVERSE)
        {
            sb = 0;
            super_block((nsub - w + 3) / 4);
        }
        else
            for(sb = 0; sb < nsub; sb += 4 * NT)
            {
                // the earlier super-blocks' stores to B are visible, the ring is free
                if(sb > 0)
                    __syncthreads();
                super_block((min(4 * NT, nsub - sb) - w + 3) / 4);
            }
        __syncthreads(); // LDS reuse by the caller's next panel
    }
};

// One panel, by the storage order of its triangle.
template <typename T, int NT, int NVG, PanelMode MODE, int NR = 4, typename... Rest>
__device__ __forceinline__ void panel_solve(const T* Ap, T* Bp, int K, int nvec, int lda, int ldb,
                                            int flags, T scale, int v0, unsigned char* smem,
                                            PanelWait pw, Rest... rest)
{
    if(flags & SF_TA)
    {
        PanelSolver<T, NT, NVG, MODE, NR, true> s;
        s.run(Ap, Bp, K, nvec, lda, ldb, flags, scale, v0, smem, pw, rest...);
    }
    else
    {
        PanelSolver<T, NT, NVG, MODE, NR, false> s;
        s.run(Ap, Bp, K, nvec, lda, ldb, flags, scale, v0, smem, pw, rest...);
    }
}
} // namespace panel
} // namespace rbamd
