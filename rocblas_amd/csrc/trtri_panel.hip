// trtri_panel.hip -- inverses of the diagonal blocks (order up to
// kTrtriPanelNB) of a batch of triangles with the panel solve.
//
// A workgroup computes 16 columns of one block's inverse, L X = I, from the
// unit vectors (nothing is read from invA): columns [16 p, 16 p + 16) are zero
// above row 16 p, so it solves the trailing triangle from there on and writes
// the rows above, in the block, as zeros.  The blocks of every instance and all
// their panels are one launch.
//
// Bound: the panel solve's chain of sub-blocks.  It replaces inverses of order
// 32 joined by doubling products of 32 to 256 rows, two launches per level.
// Measured on MI355X, FP64, us: n = 64 22 -> 4.8, 256 48 -> 13.5, 512 72 -> 34,
// 1024 121 -> 83; 500 instances of order 200 303 -> 95.
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
    const T*      Ap = a.A.get(inst) + d * (int64_t(a.lda) + 1);
    T*            Xp = a.X.get(inst);
    T*            Xd = Xp + d * (int64_t(a.ldx) + 1);
    const int     nv = min(panel::PNC, kt);

    // canonical rows above the trailing triangle: real rows r0.. (lower) or
    // past it (upper), of the columns solved here
    const int zr = r0 + (a.upper ? kt : 0);
    const int zc = r0 + (a.upper ? kt - nv : j0);
    for(int e = threadIdx.x; e < j0 * nv; e += panel::PNT)
        gstore(Xp + (zr + e % j0 + int64_t(zc + e / j0) * a.ldx), T(0));

    panel::PanelSolver<T, NT, 1, panel::PM_INVERSE, 4, false> s;
    s.run(Ap, Xd, kt, nv, a.lda, a.ldx,
          SF_COLS | (a.upper ? SF_UPPER | SF_REV : 0) | (a.unit ? SF_UNIT : 0), T(1), 0, smem, pw);
}
} // namespace

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
    for(int64_t u = 0; u < units; u += 1 << 30)
    {
        const dim3 grid(unsigned(std::min<int64_t>(units - u, 1 << 30)));
        if(std::min(a.n, a.nb) <= 256)
            hipLaunchKernelGGL((trtri_panel_kernel<T, 4>), grid, dim3(panel::PNT), 0, h->stream, a,
                               panels, u, pw);
        else
            hipLaunchKernelGGL((trtri_panel_kernel<T, 8>), grid, dim3(panel::PNT), 0, h->stream, a,
                               panels, u, pw);
    }
    return launch_status();
}

template rocblas_status trtri_panel_launch<float>(rocblas_handle, const TrtriDiagArgs<float>&);
template rocblas_status trtri_panel_launch<double>(rocblas_handle, const TrtriDiagArgs<double>&);

} // namespace rbamd
