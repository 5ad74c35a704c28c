// gemm_tile.hip -- dense GEMM for operands of any alignment and for products
// with few 128 x 128 tiles: C := alpha * op(A) * op(B) + beta * C.
//
// The operand tiles go straight into LDS (global_load_lds), 16 bytes per lane
// where the operands are aligned, else 4 -- then neither the addresses nor the
// leading dimensions need more than the element's own alignment, which the
// trailing updates of a solve of odd order or odd leading dimension lack.  A
// load needs one 32-bit lane offset, fixed over K, and a scalar base.
//
// An operand tile (x = row of op(A) or column of op(B), BX of them, by BK k;
// BK is 128 bytes: 16 doubles or 32 floats) takes one of two LDS layouts, by
// which index is contiguous in memory:
//   x contiguous (A, or B transposed): BK rows (k) of BX elements, element x
//            at x ^ 16 (k % 2) (FP64) or x ^ 16 (k % 4) (FP32);
//   k contiguous (B, or A transposed): BX rows (x) of 128 bytes, element k
//            of row x at k ^ (16 / size) (x / 2 % 8).
// Both put the elements one fragment read touches in distinct banks, and keep
// 16-byte words whole; a load lane fetches the element its place holds.
// Rows / columns past M / N are read clamped and feed only parts of C that are
// not stored; k past K (last step) is read clamped and cleared in LDS in both
// operands.
//
// Bound: the matrix cores, less what the tile quantisation leaves idle; with
// 4-byte loads the load issue (about 28 cycles per load and CU: 16 loads
// against the 1024 cycles of products of a 64 x 64 step).  Measured on MI355X
// against the register-staged kernels (us): FP64 1024 x 2048 x 1024 104 -> 78,
// 256 x 2048 x 256 12.7 -> 9.7; unaligned 4096^3 FP64 2277 -> 2035 (67.5
// TF/s), FP32 1304 -> 1042 (132 TF/s); FP32 1465 x 2999 x 1536 246 -> 169.
#include "device_common.hpp"
#include "gemm_tile.hpp"

namespace rbamd
{
namespace
{
// One load of VEC (4 or 16) bytes per lane from base + off into 64 VEC
// contiguous LDS bytes at dst (M0), as inline assembly so that the compiler's
// wait-count pass does not make every later LDS read wait for it (it cannot
// tell the stages apart); the kernel's explicit waits order it.  One wait
// state separates the M0 write from the load.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm" // m0 is reserved; the clobber is still honoured
template <int VEC>
__device__ __forceinline__ void dma(const void* base, unsigned off, uint32_t lds)
{
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds);
    if constexpr(VEC == 16)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                     :
                     : "v"(off), "s"(base), "s"(dst)
                     : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                     :
                     : "v"(off), "s"(base), "s"(dst)
                     : "memory", "m0");
}
#pragma clang diagnostic pop

// wait until at most N of this wavefront's vector-memory loads are in flight
// (gfx9 s_waitcnt encoding: vmcnt is split over bits 3:0 and 15:14)
template <int N>
__device__ __forceinline__ void wait_loads()
{
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// workgroup barrier that leaves the loads in flight alone
__device__ __forceinline__ void barrier_lds()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// byte address of an LDS array
template <typename T>
__device__ __forceinline__ uint32_t lds_addr(const T* p)
{
    return uint32_t(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) T*)(p)));
}

template <typename T, int BX, bool XC, int VEC>
struct TileOperand
{
    static constexpr int SZ  = int(sizeof(T));
    static constexpr int BK  = 128 / SZ;
    static constexpr int ELS = BX * BK;
    static constexpr int PER = BX * 128 / (64 * VEC) / 4; // load instructions per wavefront per tile
    static_assert(PER >= 1, "every wavefront loads");

    // element (k, x) of a stage
    static __device__ __forceinline__ int at(int k, int x)
    {
        if constexpr(XC)
            return k * BX + (x ^ (16 * (k & (SZ == 8 ? 1 : 3))));
        else
            return x * BK + (k ^ ((16 / SZ) * ((x >> 1) & 7)));
    }

    // this lane's byte offset from the tile's first element (k0, x0) in load
    // instruction g of wavefront w, for k below kleft
    static __device__ __forceinline__ unsigned lane_off(int w, int g, int lane, int x0, int X,
                                                        int ld, int kleft)
    {
        const int pos = ((w * PER + g) * 64 + lane) * VEC; // byte in the stage
        int       k, x;
        if constexpr(XC)
        {
            k = pos / (BX * SZ);
            x = (pos % (BX * SZ)) / SZ ^ (16 * (k & (SZ == 8 ? 1 : 3)));
        }
        else
        {
            x = pos / 128;
            k = (pos % 128) / SZ ^ ((16 / SZ) * ((x >> 1) & 7));
        }
        // (a 16-byte load holds 16 / SZ elements along the contiguous index)
        x = min(x0 + x, XC && VEC == 16 ? X - 16 / SZ : X - 1) - x0;
        k = min(k, kleft - 1);
        return unsigned(XC ? k : x) * unsigned(ld) * SZ + unsigned(XC ? x : k) * SZ + pos % SZ;
    }
};

template <typename T, int BM, int BN, int NS, int VEC, bool TAIL, int OPA, int OPB>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
    gemm_tile_kernel(const GemmArgsT<T, T, T> a)
{
    using acc_t         = typename Mfma<T>::acc_t;
    using OA            = TileOperand<T, BM, OPA == 0, VEC>;
    using OB            = TileOperand<T, BN, OPB == 1, VEC>;
    constexpr int SZ    = int(sizeof(T));
    constexpr int BK    = OA::BK;
    constexpr int LOADS = OA::PER + OB::PER;
    constexpr int TM    = BM / 32; // 16 x 16 MFMA tiles per wavefront (2 x 2 wavefronts)
    constexpr int TN    = BN / 32;
    // C is read ahead, beside the first K steps, where the registers allow
    constexpr bool AHEAD = TM * TN <= 4;
    static_assert((NS - 2) * LOADS < 64, "vmcnt");
    __shared__ __align__(16) T As[NS][OA::ELS];
    __shared__ __align__(16) T Bs[NS][OB::ELS];

    if(a.skip_if_zero && *a.skip_if_zero == T(0))
        return;

    const int tid  = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int w    = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int wm   = w % 2;
    const int wn   = w / 2;

    // contiguous runs of tiles per XCD, grouped by eight row panels
    const int total = a.tiles_m * a.tiles_n;
    int       bid   = blockIdx.x;
    {
        const int q = total / 8, r = total % 8;
        const int x = bid % 8, l = bid / 8;
        bid         = x * q + min(x, r) + l;
    }
    constexpr int GROUP = 8;
    const int     grp   = bid / (GROUP * a.tiles_n);
    const int     fm    = grp * GROUP;
    const int     gsz   = min(a.tiles_m - fm, GROUP);
    const int     m0    = (fm + (bid % gsz)) * BM;
    const int     n0    = ((bid % (GROUP * a.tiles_n)) / gsz) * BN;
    const int     ksteps = (a.K + BK - 1) / BK;
    const int     ktail  = a.K - (ksteps - 1) * BK; // k of the last step, 1..BK

    const uint32_t la = lds_addr(&As[0][0]), lb = lds_addr(&Bs[0][0]);
    unsigned       oa[OA::PER], ob[OB::PER];
#pragma unroll
    for(int g = 0; g < OA::PER; ++g)
        oa[g] = OA::lane_off(w, g, lane, m0, a.M, a.lda, BK);
#pragma unroll
    for(int g = 0; g < OB::PER; ++g)
        ob[g] = OB::lane_off(w, g, lane, n0, a.N, a.ldb, BK);

    for(int b = blockIdx.y; b < a.batch; b += gridDim.y)
    {
        const T* Ap
            = uniform_ptr(a.A.get(b) + (OPA == 0 ? int64_t(m0) : int64_t(m0) * a.lda));
        const T* Bp
            = uniform_ptr(a.B.get(b) + (OPB == 1 ? int64_t(n0) : int64_t(n0) * a.ldb));
        T* Cp = a.C.get(b);

        // steps past the last one re-read the last one into a stage nobody
        // reads any more, so every step waits the same way
        auto issue = [&](int kt, int st) {
            const int  k0   = min(kt, ksteps - 1) * BK;
            const bool tail = TAIL && a.K - k0 < BK;
            const T*   pa   = Ap + (OPA == 0 ? int64_t(k0) * a.lda : int64_t(k0));
            const T*   pb   = Bp + (OPB == 1 ? int64_t(k0) * a.ldb : int64_t(k0));
#pragma unroll
            for(int g = 0; g < OA::PER; ++g)
                dma<VEC>(pa, tail ? OA::lane_off(w, g, lane, m0, a.M, a.lda, a.K - k0) : oa[g],
                         la + st * OA::ELS * SZ + (w * OA::PER + g) * 64 * VEC);
#pragma unroll
            for(int g = 0; g < OB::PER; ++g)
                dma<VEC>(pb, tail ? OB::lane_off(w, g, lane, n0, a.N, a.ldb, a.K - k0) : ob[g],
                         lb + st * OB::ELS * SZ + (w * OB::PER + g) * 64 * VEC);
        };
        // the last step's stage cleared past K
        auto clear_tail = [&](int st) {
            for(int e = tid; e < (BK - ktail) * BM; e += 256)
                As[st][OA::at(ktail + e / BM, e % BM)] = T(0);
            for(int e = tid; e < (BK - ktail) * BN; e += 256)
                Bs[st][OB::at(ktail + e / BN, e % BN)] = T(0);
        };

        acc_t acc[TM][TN];
#pragma unroll
        for(int i = 0; i < TM; ++i)
#pragma unroll
            for(int j = 0; j < TN; ++j)
                acc[i][j] = acc_t{0, 0, 0, 0};

        // lane holds row lane % 16 and columns Mfma<T>::row(lane, r) of each tile
        const int row0 = m0 + wm * (BM / 2) + (lane & 15);
        const int col0 = n0 + wn * (BN / 2);
        T         cv[AHEAD ? TM : 1][AHEAD ? TN : 1][4];
        if constexpr(AHEAD)
        {
            if(a.beta != T(0) && ksteps > 0)
            {
#pragma unroll
                for(int i = 0; i < TM; ++i)
#pragma unroll
                    for(int j = 0; j < TN; ++j)
#pragma unroll
                        for(int r = 0; r < 4; ++r)
                        {
                            const int row = min(row0 + i * 16, a.M - 1);
                            const int col = min(col0 + j * 16 + Mfma<T>::row(lane, r), a.N - 1);
                            cv[i][j][r]   = gload(Cp + (row + int64_t(col) * a.ldc));
                        }
            }
        }

        auto compute = [&](int st) {
            const T* as = As[st];
            const T* bs = Bs[st];
#pragma unroll
            for(int k4 = 0; k4 < BK / 4; ++k4)
            {
                const int kr = k4 * 4 + lane / 16;
                T         af[TM], bf[TN];
#pragma unroll
                for(int i = 0; i < TM; ++i)
                    af[i] = as[OA::at(kr, wm * (BM / 2) + i * 16 + (lane & 15))];
#pragma unroll
                for(int j = 0; j < TN; ++j)
                    bf[j] = bs[OB::at(kr, wn * (BN / 2) + j * 16 + (lane & 15))];
                // operands swapped: a lane's results run down a column of C
#pragma unroll
                for(int i = 0; i < TM; ++i)
#pragma unroll
                    for(int j = 0; j < TN; ++j)
                        acc[i][j] = Mfma<T>::run(bf[j], af[i], acc[i][j]);
            }
        };
        // steps kt .. kt + NS - 2 are in flight; waiting down to NS - 2 of
        // them retires step kt, the barrier publishes it and frees the stage
        // that step kt + NS - 1 goes to
        auto step = [&](int kt, int st) {
            wait_loads<(NS - 2) * LOADS>();
            barrier_lds();
            issue(kt + NS - 1, (st + NS - 1) % NS);
            if(TAIL && kt == ksteps - 1 && ktail < BK)
            {
                clear_tail(st);
                barrier_lds();
            }
            compute(st);
        };
        if(ksteps > 0)
        {
#pragma unroll
            for(int t = 0; t < NS - 1; ++t)
                issue(t, t);
            for(int kt = 0; kt < ksteps; kt += NS)
            {
#pragma unroll
                for(int t = 0; t < NS; ++t)
                    if(t == 0 || kt + t < ksteps)
                        step(kt + t, t);
            }
            wait_loads<0>(); // the steps past the end
        }

#pragma unroll
        for(int i = 0; i < TM; ++i)
#pragma unroll
            for(int j = 0; j < TN; ++j)
#pragma unroll
                for(int r = 0; r < 4; ++r)
                {
                    const int row = row0 + i * 16;
                    const int col = col0 + j * 16 + Mfma<T>::row(lane, r);
                    if(row < a.M && col < a.N)
                    {
                        T* cp = Cp + (row + int64_t(col) * a.ldc);
                        T  v  = a.alpha * acc[i][j][r];
                        if(a.beta != T(0))
                        {
                            if constexpr(AHEAD)
                                v = fma(a.beta, cv[i][j][r], v);
                            else
                                v = fma(a.beta, gload(cp), v);
                        }
                        gstore(cp, v);
                    }
                }
        __syncthreads(); // LDS reuse by the next instance
    }
}

// TAIL: K need not be a multiple of BK
template <typename T, int BM, int BN, int NS, int VEC, bool TAIL>
rocblas_status launch_tile(rocblas_handle h, GemmArgsT<T, T, T> a)
{
    a.tiles_m        = (a.M + BM - 1) / BM;
    a.tiles_n        = (a.N + BN - 1) / BN;
    const int64_t nt = int64_t(a.tiles_m) * a.tiles_n;
    if(nt > int64_t(0x7fffffff))
        return rocblas_status_invalid_size;
    const dim3 grid(unsigned(nt), grid_batch(a.batch)), block(256);
    if(a.opA == 0 && a.opB == 0)
        hipLaunchKernelGGL((gemm_tile_kernel<T, BM, BN, NS, VEC, TAIL, 0, 0>), grid, block, 0,
                           h->stream, a);
    else if(a.opA == 1 && a.opB == 0)
        hipLaunchKernelGGL((gemm_tile_kernel<T, BM, BN, NS, VEC, TAIL, 1, 0>), grid, block, 0,
                           h->stream, a);
    else if(a.opA == 0)
        hipLaunchKernelGGL((gemm_tile_kernel<T, BM, BN, NS, VEC, TAIL, 0, 1>), grid, block, 0,
                           h->stream, a);
    else
        hipLaunchKernelGGL((gemm_tile_kernel<T, BM, BN, NS, VEC, TAIL, 1, 1>), grid, block, 0,
                           h->stream, a);
    return launch_status();
}

} // namespace

// 16-byte loads: aligned operands and leading dimensions, whole K steps, and a
// whole number of 16-byte words along an x-contiguous operand
template <typename T>
bool gemm_tile_vec16(const GemmArgsT<T, T, T>& a)
{
    constexpr int E    = 16 / int(sizeof(T));
    auto          al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    return a.K % (128 / int(sizeof(T))) == 0 && a.lda % E == 0 && a.ldb % E == 0
           && (a.opA == 1 || a.M % E == 0) && (a.opB == 0 || a.N % E == 0) && !a.A.arr && !a.B.arr
           && al16(a.A.base + a.A.offset) && al16(a.B.base + a.B.offset) && a.A.stride % E == 0
           && a.B.stride % E == 0;
}
template <typename T>
bool gemm_tile_eligible(const GemmArgsT<T, T, T>& a)
{
    // a lane's offset inside a tile is 32 bits: 128 rows of a k-contiguous operand
    return !a.tri && a.K > 0 && a.lda <= (1 << 21) && a.ldb <= (1 << 21);
}

template <typename T>
rocblas_status launch_gemm_tile(rocblas_handle h, const GemmArgsT<T, T, T>& a, int tile)
{
    if(tile >= 128)
        return launch_tile<T, 128, 128, 2, 4, false>(h, a);
    const bool vec = gemm_tile_vec16(a);
    if constexpr(sizeof(T) == 8)
    {
        if(tile < 64)
            return vec ? launch_tile<T, 32, 64, 4, 16, false>(h, a)
                       : launch_tile<T, 32, 64, 4, 4, true>(h, a);
    }
    return vec ? launch_tile<T, 64, 64, 4, 16, false>(h, a)
               : launch_tile<T, 64, 64, 4, 4, true>(h, a);
}

template bool gemm_tile_vec16(const GemmArgsT<float, float, float>&);
template bool gemm_tile_vec16(const GemmArgsT<double, double, double>&);
template bool gemm_tile_eligible(const GemmArgsT<float, float, float>&);
template bool gemm_tile_eligible(const GemmArgsT<double, double, double>&);
template rocblas_status launch_gemm_tile(rocblas_handle, const GemmArgsT<float, float, float>&,
                                         int);
template rocblas_status launch_gemm_tile(rocblas_handle, const GemmArgsT<double, double, double>&,
                                         int);

} // namespace rbamd
