// trtri_panel.hip -- inverses of the diagonal blocks (order up to
// kTrtriPanelNB) of a batch of triangles with the panel solve.
//
// A workgroup computes 16 columns of one block's inverse, L X = I, from the
// unit vectors (nothing is read from invA): columns [16 p, 16 p + 16) are zero
// above row 16 p, so it solves the trailing triangle from there on and writes
// the rows above, in the block, as zeros.  The blocks of every instance and all
// their panels are one launch.
//
// In place: pointer arrays that differ may hold the same matrices, and strided
// batches of different base and stride may meet in an instance (strided calls of
// one base, and pointer arrays that are the same array, read a copy of A).  The
// panels of such a block read columns that others solve, so they leave A's
// triangle alone and write their results below the diagonal transposed into
// the opposite triangle, which nobody reads; a second launch moves them over.
// It does nothing for other matrices, whose pointer-array calls it costs 2 to 3
// us (FP64, one instance of order 33 4.0 -> 7.0, of order 512 33.7 -> 35.7).
// Solving the panels of a block in order in one workgroup instead took 473 us
// for one instance of order 512 in place, against 69 this way.
//
// Bound: the panel solve's chain of sub-blocks.  It replaces inverses of order
// 32 joined by doubling products of 32 to 256 rows, two launches per level.
// Measured on MI355X, FP64, us: n = 64 22 -> 4.8, 256 48 -> 13.5, 512 72 -> 34,
// 1024 121 -> 83; 500 instances of order 200 303 -> 95.
#include "launch_slices.hpp"
#include "panel_trsm.hpp"
#include "trtri_kernels.hpp"

namespace rbamd
{
namespace
{
template <typename T, int NT>
__global__ void __launch_bounds__(panel::PNT) __attribute__((amdgpu_waves_per_eu(2)))
    trtri_panel_kernel(const TrtriDiagArgs<T> a, int panels, int64_t unit0, panel::PanelWait pw)
{
    __shared__ __align__(16) unsigned char smem[panel::lds_bytes<T, 1>()];
    const int     nblk = (a.n + a.nb - 1) / a.nb;
    const int64_t u    = unit0 + blockIdx.x;
    const int     p    = int(u % panels);
    const int     blk  = int(u / panels % nblk);
    const int64_t inst = u / panels / nblk;
    const int     r0   = blk * a.nb;
    const int     j0   = p * panel::PNC;
    const int     K    = min(a.nb, a.n - r0); // order of the block
    if(j0 >= K)
        return;
    const int kt = K - j0; // order of the trailing triangle
    // canonical trailing triangle: rows and columns j0.. (lower), or the
    // leading ones in memory (upper, reversed)
    const int64_t d  = r0 + (a.upper ? 0 : j0);
    const T*      A0 = a.A.get(inst);
    const T*      Ap = A0 + d * (int64_t(a.lda) + 1);
    T*            Xp = a.X.get(inst);
    T*            Xd = Xp + d * (int64_t(a.ldx) + 1);
    const int     nv = min(panel::PNC, kt);
    const bool    in_place = A0 == Xp;

    // canonical rows above the trailing triangle: real rows r0.. (lower) or
    // past it (upper), of the columns solved here
    const int zr = r0 + (a.upper ? kt : 0);
    const int zc = r0 + (a.upper ? kt - nv : j0);
    for(int e = threadIdx.x; !in_place && e < j0 * nv; e += panel::PNT)
        gstore(Xp + (zr + e % j0 + int64_t(zc + e / j0) * a.ldx), T(0));

    panel::PanelSolver<T, NT, 1, panel::PM_INVERSE, 4, false> s;
    s.run(Ap, Xd, kt, nv, a.lda, a.ldx,
          SF_COLS | (a.upper ? SF_UPPER | SF_REV : 0) | (a.unit ? SF_UNIT : 0)
              | (in_place ? SF_TRANSPOSED : 0),
          T(1), 0, smem, pw);
}

// In-place blocks: the inverse's entries off the diagonal move from the
// opposite triangle to their own, which is cleared, and the diagonal, still
// A's, is inverted.  A workgroup takes TS rows and columns of one block, tile
// by tile away from the diagonal.
constexpr int TS = 32;

template <typename T>
__global__ void __launch_bounds__(256) trtri_turn_kernel(const TrtriDiagArgs<T> a, int strips,
                                                         int64_t unit0)
{
    __shared__ T  tile[TS][TS + 1];
    const int     nblk = (a.n + a.nb - 1) / a.nb;
    const int64_t u    = unit0 + blockIdx.x;
    const int     s    = int(u % strips) * TS;
    const int     r0   = int(u / strips % nblk) * a.nb;
    const int64_t inst = u / strips / nblk;
    const int     K    = min(a.nb, a.n - r0);
    T*            X    = a.X.get(inst);
    if(s >= K || a.A.get(inst) != X)
        return;
    X += int64_t(r0) * (int64_t(a.ldx) + 1);
    const int x = threadIdx.x % TS, y = threadIdx.x / TS;
    for(int t = s; t < K; t += TS)
    {
        // the tile as written: rows s.. and columns t.. above the diagonal
        // (lower triangle), rows t.. and columns s.. below it (upper)
        const int fr = a.upper ? t : s, fc = a.upper ? s : t;
        for(int j = y; j < TS; j += 256 / TS)
            if(fr + x < K && fc + j < K)
            {
                T* p       = X + (fr + x) + int64_t(fc + j) * a.ldx;
                tile[j][x] = *p;
                if(t > s)
                    *p = T(0);
            }
        __syncthreads();
        for(int j = y; j < TS; j += 256 / TS)
            if(fc + x < K && fr + j < K)
            {
                T* p = X + (fc + x) + int64_t(fr + j) * a.ldx;
                if(t > s)
                    *p = tile[x][j];
                else // the diagonal tile
                {
                    const bool own = a.upper ? x < j : x > j;
                    *p = x == j ? (a.unit ? T(1) : T(1) / tile[j][x]) : own ? tile[x][j] : T(0);
                }
            }
        __syncthreads();
    }
}
} // namespace

// Whether an instance's A can be its X: pointer arrays are device data; strided
// batches that differ in base and stride meet in at most one instance.
template <typename T>
static bool may_be_in_place(const TrtriDiagArgs<T>& a)
{
    if(a.A.arr || a.X.arr)
        return a.A.arr && a.X.arr;
    const int64_t bytes = int64_t(reinterpret_cast<intptr_t>(a.X.base + a.X.offset)
                                  - reinterpret_cast<intptr_t>(a.A.base + a.A.offset));
    const int64_t step  = (a.A.stride - a.X.stride) * int64_t(sizeof(T));
    return step ? bytes % step == 0 && bytes / step >= 0 && bytes / step < a.batch : bytes == 0;
}

template <typename T>
rocblas_status trtri_panel_launch(rocblas_handle h, const TrtriDiagArgs<T>& a)
{
    if(a.nb > kTrtriPanelNB)
        return rocblas_status_internal_error;
    DeviceGuard   g(h->device);
    const int     nblk   = (a.n + a.nb - 1) / a.nb;
    const int     panels = (std::min(a.n, a.nb) + panel::PNC - 1) / panel::PNC;
    const int64_t units  = int64_t(a.batch) * nblk * panels;
    const auto    pw     = panel::panel_wait(h);
    for_launch_slices(units, panel::PNT, [&](int64_t u, unsigned count) {
        const dim3 grid(count);
        if(std::min(a.n, a.nb) <= 256)
            hipLaunchKernelGGL((trtri_panel_kernel<T, 4>), grid, dim3(panel::PNT), 0, h->stream, a,
                               panels, u, pw);
        else
            hipLaunchKernelGGL((trtri_panel_kernel<T, 8>), grid, dim3(panel::PNT), 0, h->stream, a,
                               panels, u, pw);
    });
    if(!may_be_in_place(a))
        return launch_status();
    const int     strips = (std::min(a.n, a.nb) + TS - 1) / TS;
    const int64_t turns  = int64_t(a.batch) * nblk * strips;
    for_launch_slices(turns, 256, [&](int64_t u, unsigned count) {
        hipLaunchKernelGGL(trtri_turn_kernel<T>, dim3(count), dim3(256), 0, h->stream, a, strips, u);
    });
    return launch_status();
}

template rocblas_status trtri_panel_launch<float>(rocblas_handle, const TrtriDiagArgs<float>&);
template rocblas_status trtri_panel_launch<double>(rocblas_handle, const TrtriDiagArgs<double>&);

} // namespace rbamd
