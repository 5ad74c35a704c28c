// launch_slices.hpp -- one-dimensional launches of any number of workgroups
// (host only, no HIP headers).
#pragma once

#include <algorithm>
#include <cstdint>

namespace rbamd
{
// A launch has fewer than 2^32 threads along x (the limit hipLaunchKernel
// documents for gridDim * blockDim), so more workgroups than that take several
// launches.  The slice is a power of two: which XCD a workgroup goes to does not
// change with its slice.
constexpr int64_t launch_slice(int threads)
{
    int64_t n = 1;
    while(2 * n * threads < (int64_t(1) << 32))
        n *= 2;
    return n;
}
static_assert(launch_slice(256) == 1 << 23 && launch_slice(64) == 1 << 25, "below 2^32 threads");

// launch(first, count) for consecutive slices of `blocks` workgroups
template <typename F>
void for_launch_slices(int64_t blocks, int threads, F&& launch)
{
    const int64_t slice = launch_slice(threads);
    for(int64_t first = 0; first < blocks; first += slice)
        launch(first, unsigned(std::min(blocks - first, slice)));
}
} // namespace rbamd
