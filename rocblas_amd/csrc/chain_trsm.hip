// chain_trsm.hip -- single-launch solve of one instance whose triangle is long
// and whose right-hand side is narrow: one workgroup per (super-block of
// 128 or 256 rows, panel of 16 vectors).
//
// Each workgroup runs the panel solve (panel_trsm.hpp) on its super-block: it
// applies the solution of the super-blocks above as their workgroups publish
// it, sub-block by sub-block, then solves its own with the chain inside the
// workgroup, so only one hand-over in 8 or 16 goes through memory.
// The solution is published through B itself: agent-scope (write-through)
// stores, a wait for them, then the wavefront's flag; readers poll the flags
// and read B with agent-scope loads.  No cache is written back or invalidated
// as a whole.
//
// Ordering: workgroup (p, S) has linear index S * P + p and only waits for
// smaller linear indices, which are dispatched first, so the chain cannot
// deadlock.  Every wait is bounded: one that runs out raises the handle's
// error word (host-visible memory, read by the next call on the handle and by
// rocblas_amd_get_async_status) and proceeds, so every wave reaches its exit.
//
// The last workgroup of a panel to finish clears the panel's flags (every
// other one has counted itself after its last access to them), so they are
// zero after every launch -- after a wait that gave up, too -- and a graph
// replay starts from zero.
//
// Bound: the chain of sub-blocks, as the panel solve's, and about 4 us per
// hand-over.  Measured on MI355X against 64-row blocks, each a workgroup that
// released and acquired whole caches per hand-over (FP64, us): 4096 x 8 376 ->
// 283, 4096 x 128 615 -> 347, 8192 x 64 1243 -> 704, 1024 x 256 133 -> 82,
// 2048 x 512 340 -> 180, 16384 x 8 2056 -> 1400.
#include "panel_trsm.hpp"

namespace rbamd
{
namespace
{
using namespace panel;

// NT: 16-row sub-blocks per wavefront, 64 NT rows per super-block
template <typename T, int NT, int NR>
__device__ __forceinline__ void chain_unit(const SmallArgs<T>& a, unsigned* flags, int P, int R,
                                           PanelWait pw, unsigned char* smem)
{
    const int S  = blockIdx.x / P;
    const int p  = blockIdx.x % P;
    const int v0 = p * PNC;
    T* const  Bp = a.B.get(0);

    const T alpha = a.alpha_dev ? *a.alpha_dev : a.alpha_host;
    const T scale = (a.flags & SF_SCALE) ? alpha : T(1);
    if(alpha == T(0))
    {
        // B := 0 (nobody waits: alpha is uniform); every workgroup its rows
        const int r0 = S * 64 * NT;
        panel_zero<T>(Bp, r0, min(r0 + 64 * NT, a.K), a.nvec, a.ldb, a.flags, v0, PNC);
        return;
    }
    unsigned* const link = flags + p * CHAIN_WORDS;
    panel_solve<T, NT, 1, PM_CHAIN, NR>(a.A.get(0), Bp, a.K, a.nvec, a.lda, a.ldb, a.flags, scale,
                                        v0, smem, pw, link, S * 4 * NT);
    // every wavefront's flag is written before this workgroup counts itself
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if(threadIdx.x == 0)
    {
        const unsigned old
            = __hip_atomic_fetch_add(link + 4, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if(old == unsigned(R - 1))
        {
#pragma unroll
            for(int i = 0; i < 5; ++i)
                __hip_atomic_store(link + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(PNT) __attribute__((amdgpu_waves_per_eu(2)))
    chain_trsm_kernel(const SmallArgs<T> a, unsigned* flags, int P, int R, PanelWait pw)
{
    __shared__ __align__(16) unsigned char smem[lds_bytes<T, 1>()];
    chain_unit<T, 4, 4>(a, flags, P, R, pw, smem);
}

// 128-row super-blocks: half the products per wavefront between two solved
// sub-blocks.  NR < 4, at most 4 NR vectors: fewer registers to solve and hand
// on.
template <typename T, int NR>
__global__ void __launch_bounds__(PNT) __attribute__((amdgpu_waves_per_eu(2)))
    chain_short_kernel(const SmallArgs<T> a, unsigned* flags, int P, int R, PanelWait pw)
{
    __shared__ __align__(16) unsigned char smem[lds_bytes<T, 1>()];
    chain_unit<T, 2, NR>(a, flags, P, R, pw, smem);
}
} // namespace

template <typename T>
bool chain_fits(rocblas_handle h, int K, int nvec, int batch)
{
    // Each super-block streams its own rows of the triangle once per panel, so
    // the traffic grows with P while the recursion's does not: the chain takes
    // small grids and triangles long relative to the panel count.
    const int64_t R = (K + 63) / 64, P = (nvec + PNC - 1) / PNC, cus = h->num_cus;
    return h->chain_flags != nullptr && batch == 1 && K > kPanelMaxK && P <= kChainMaxPanels
           && (R * P <= 2 * cus || (P <= R && R * P <= 8 * cus));
}

template <typename T>
rocblas_status launch_chain(rocblas_handle h, const SmallArgs<T>& a)
{
    if(!chain_fits<T>(h, a.K, a.nvec, 1))
        return rocblas_status_internal_error;
    // 128-row super-blocks while each workgroup has a CU to itself, else
    // 256-row ones, of which there are half as many.  Measured, FP64, 128 /
    // 256 rows: 4096 x 8 283 / 327 us, 4096 x 128 (256 workgroups of 128 rows)
    // 347 / 364; 4096 x 256 (512) 415 / 368, 8192 x 256 1059 / 911.
    const int       P = (a.nvec + PNC - 1) / PNC;
    const int64_t   R2 = (int64_t(a.K) + 127) / 128, R4 = (int64_t(a.K) + 255) / 256;
    const bool      two = R2 * P <= h->num_cus;
    const int       R   = int(two ? R2 : R4);
    const dim3      grid(unsigned(R * P)), block(PNT);
    const PanelWait pw    = panel_wait(h);
    unsigned* const flags = static_cast<unsigned*>(h->chain_flags);
    if(!two)
        hipLaunchKernelGGL(chain_trsm_kernel<T>, grid, block, 0, h->stream, a, flags, P, R, pw);
    else if(a.nvec <= 4)
        hipLaunchKernelGGL((chain_short_kernel<T, 1>), grid, block, 0, h->stream, a, flags, P, R,
                           pw);
    else if(a.nvec <= 8)
        hipLaunchKernelGGL((chain_short_kernel<T, 2>), grid, block, 0, h->stream, a, flags, P, R,
                           pw);
    else
        hipLaunchKernelGGL((chain_short_kernel<T, 4>), grid, block, 0, h->stream, a, flags, P, R,
                           pw);
    return launch_status();
}

template bool           chain_fits<float>(rocblas_handle, int, int, int);
template bool           chain_fits<double>(rocblas_handle, int, int, int);
template rocblas_status launch_chain<float>(rocblas_handle, const SmallArgs<float>&);
template rocblas_status launch_chain<double>(rocblas_handle, const SmallArgs<double>&);

} // namespace rbamd
