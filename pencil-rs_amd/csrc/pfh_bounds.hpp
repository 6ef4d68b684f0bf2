// Bounds of a launch: HIP refuses gridDim.x * blockDim.x of 2^32 and more. Work
// that needs more runs as several launches.
#pragma once

#include <cstddef>
#include <cstdint>

#include "pfh_kernels.hpp"

namespace pfh {

constexpr int64_t kMaxLaunchThreads = ((int64_t)1 << 32) - 1;
constexpr int64_t kMaxBlocks256 = (int64_t)1 << 24; // one more than workgroups of 256 may have

// Device scratch of the allocation-free entry point (pfh_noalloc.hip).
constexpr size_t kNoallocBytes = (size_t)128 << 20;

// Elementwise kernels: elements of a workgroup and of one launch.
constexpr int kElementsPerBlock = 256 * 8;
constexpr int64_t kElementsPerLaunch = (kMaxBlocks256 - 1) * kElementsPerBlock;

// k_scale_axes: threads along a row of nx elements, rows of a thread, and
// workgroups over the rows.
constexpr int kScaleRows = 4;
inline int scale_axes_cols(int64_t nx)
{
    int cols = 1;
    while (cols < 256 && cols < nx) cols *= 2;
    return cols;
}
inline int64_t scale_axes_blocks(int64_t rows, int64_t nx)
{
    const int64_t per = (int64_t)(256 / scale_axes_cols(nx)) * kScaleRows;
    return (rows + per - 1) / per;
}

// Calls fn(part, first element) for parts of s that one launch holds (the
// kernel also divides row indexes in 32 bits): halves of the extras, then of the
// slowest axis that has any.
template <typename Fn>
void scale_axes_parts(const ScaleAxesArgs &s, int64_t first, Fn &&fn)
{
    const int64_t nx = s.mext[s.nd - 1], rows = s.len * s.extra / nx;
    if (rows <= INT32_MAX && scale_axes_blocks(rows, nx) < kMaxBlocks256) {
        fn(s, first);
        return;
    }
    ScaleAxesArgs lo = s, hi = s;
    if (s.extra > 1) {
        lo.extra = s.extra / 2;
        hi.extra = s.extra - lo.extra;
    } else {
        int p = 0;
        while (s.mext[p] == 1) ++p; // rows > 1: some axis before the last
        lo.mext[p] = s.mext[p] / 2;
        hi.mext[p] = s.mext[p] - lo.mext[p];
        hi.foff[p] += lo.mext[p];
        lo.len = s.len / s.mext[p] * lo.mext[p];
        hi.len = s.len - lo.len;
    }
    scale_axes_parts(lo, first, fn);
    scale_axes_parts(hi, first + lo.len * lo.extra, fn);
}

} // namespace pfh
