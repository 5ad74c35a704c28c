// panel_trsm.hip -- single-launch solve for 32 < k <= 512: one workgroup per 16
// or 32 right-hand-side vectors of one instance (panel_trsm.hpp).  Workgroups
// are independent, so a whole k <= 512 solve is one launch (2^23 workgroups at
// a time) with no inter-workgroup communication.
#include "launch_slices.hpp"
#include "panel_trsm.hpp"

namespace rbamd
{
namespace
{
// Work units (an instance's vectors [v0, v0 + 16 NVG)) are numbered instance
// by instance, and consecutive runs of them go to one XCD: the units that
// share a triangle read it through one L2.
template <typename T, int NT, int NVG>
__device__ __forceinline__ void panel_unit(const SmallArgs<T>& a, panel::PanelWait pw,
                                           unsigned char* smem)
{
    const T        alpha = a.alpha_dev ? *a.alpha_dev : a.alpha_host;
    const T        scale = (a.flags & SF_SCALE) ? alpha : T(1);
    const unsigned qn = gridDim.x / 8, rn = gridDim.x % 8;
    const unsigned x = blockIdx.x % 8, l = blockIdx.x / 8;
    const int64_t  unit = a.unit0 + (x * qn + min(x, rn) + l);
    const int64_t  b    = unit / a.chunks;
    const int      v0   = int(unit - b * a.chunks) * panel::PNC * NVG;
    T*             Bp   = a.B.get(b);
    if(alpha == T(0))
        panel::panel_zero<T>(Bp, 0, a.K, a.nvec, a.ldb, a.flags, v0, panel::PNC * NVG);
    else
    {
        panel::panel_solve<T, NT, NVG, panel::PM_SINGLE>(
            a.A.get(b), Bp, a.K, a.nvec, a.lda, a.ldb, a.flags, scale, v0, smem, pw);
    }
}

// 256 < k <= 512, 16 vectors
template <typename T>
__global__ void __launch_bounds__(panel::PNT) 
    panel_trsm_kernel(const SmallArgs<T> a, panel::PanelWait pw)
{
    __shared__ __align__(16) unsigned char smem[panel::lds_bytes<T, 1>()];
    panel_unit<T, 8, 1>(a, pw, smem);
}

// 256 < k <= 512, 32 vectors
template <typename T>
__global__ void __launch_bounds__(panel::PNT) __attribute__((amdgpu_waves_per_eu(1)))
    panel_pair_kernel(const SmallArgs<T> a, panel::PanelWait pw)
{
    __shared__ __align__(16) unsigned char smem[panel::lds_bytes<T, 2>()];
    panel_unit<T, 8, 2>(a, pw, smem);
}

// k <= 256, 16 NVG vectors
template <typename T, int NVG>
__global__ void __launch_bounds__(panel::PNT)
    __attribute__((amdgpu_waves_per_eu(2)))
    panel_short_kernel(const SmallArgs<T> a, panel::PanelWait pw)
{
    __shared__ __align__(16) unsigned char smem[panel::lds_bytes<T, NVG>()];
    panel_unit<T, 4, NVG>(a, pw, smem);
}
} // namespace

template <typename T>
bool panel_fits(rocblas_handle, int K)
{
    return K <= kPanelMaxK;
}

template <typename T>
rocblas_status launch_panel(rocblas_handle h, const SmallArgs<T>& a, int batch)
{
    if(!panel_fits<T>(h, a.K))
        return rocblas_status_internal_error;
    // 32 vectors per workgroup halve the traffic of L and the operand loads per
    // product, but also the workgroups; from two 16-vector workgroups per CU
    // on the chip stays full either way.  Measured, 16 / 32 (/ 64) vectors: 256
    // instances 200 x 64 (1024 groups) 32.5 / 27.9 / 30.8 us; 2048 vectors in
    // 256-row leaves (128 groups) 348 / 391 / 489 us for the whole 2048^2 solve.
    const int64_t groups = (a.nvec + panel::PNC - 1) / panel::PNC;
    const int     nvg    = groups > 1 && groups * batch >= 2 * int64_t(h->num_cus) ? 2 : 1;
    SmallArgs<T> s = a;
    s.chunks       = (a.nvec + panel::PNC * nvg - 1) / (panel::PNC * nvg);
    const int64_t          units = int64_t(batch) * s.chunks;
    const panel::PanelWait pw    = panel::panel_wait(h);
    s.units                      = units;
    for_launch_slices(units, panel::PNT, [&](int64_t first, unsigned count) {
        const dim3 grid(count);
        s.unit0 = first;
        if(a.K > 256 && nvg == 1)
            hipLaunchKernelGGL(panel_trsm_kernel<T>, grid, dim3(panel::PNT), 0, h->stream, s, pw);
        else if(a.K > 256)
            hipLaunchKernelGGL(panel_pair_kernel<T>, grid, dim3(panel::PNT), 0, h->stream, s, pw);
        else if(nvg == 1)
            hipLaunchKernelGGL((panel_short_kernel<T, 1>), grid, dim3(panel::PNT), 0, h->stream, s,
                               pw);
        else
            hipLaunchKernelGGL((panel_short_kernel<T, 2>), grid, dim3(panel::PNT), 0, h->stream, s,
                               pw);
    });
    return launch_status();
}

template rocblas_status launch_panel<float>(rocblas_handle, const SmallArgs<float>&, int);
template rocblas_status launch_panel<double>(rocblas_handle, const SmallArgs<double>&, int);
template bool panel_fits<float>(rocblas_handle, int);
template bool panel_fits<double>(rocblas_handle, int);

} // namespace rbamd
