// Compile-time line plans: the radix sequence, the threads per line and the
// LDS layout of k_line_plan (pfh_line.hip), shared with the host planner.
#pragma once

#include "pfh_stage.hpp"

namespace pfh {

// Butterflies of radix R a thread holds in one pass (em values per thread).
__host__ __device__ constexpr int line_plan_mb(int em, int R) { return em / R > 0 ? em / R : 1; }

__host__ __device__ constexpr int line_plan_need(int m, int em, int R)
{
    return (m / R + line_plan_mb(em, R) - 1) / line_plan_mb(em, R);
}

// Threads per line: the fewest that cover every pass's butterflies. Any
// number, not a power of two: the 385-point line of a DST-I takes 39 threads,
// of which the radix 5 / 7 / 11 passes keep 99 / 71 / 90% busy (64 threads:
// 60 / 86 / 55%).
__host__ __device__ constexpr int line_plan_tpl(int r0, int r1, int r2, int em)
{
    const int m = r0 * r1 * (r2 ? r2 : 1);
    int t = line_plan_need(m, em, r0);
    if (line_plan_need(m, em, r1) > t) t = line_plan_need(m, em, r1);
    if (r2 && line_plan_need(m, em, r2) > t) t = line_plan_need(m, em, r2);
    return t;
}

// A plan whose values per thread are below its largest radix is a variant for
// the real-to-real modes (k_line_plan KIND 2) and the f64 half-complex ones: about
// twice the threads per line. Their loads, pre- and post-processing set the pace,
// and 5 to 8 threads a line leave few wavefronts on a CU (f64 DCT-I of 129 points
// in a 192 x 160 x 129 channel, forward + inverse 128 -> 120 us; 256 x 384 x 240 f32
// R2R 335 -> 326 us).
__host__ __device__ constexpr bool line_plan_real_only(int r0, int r1, int r2, int em)
{
    return em < r0 || em < r1 || em < r2;
}

// LDS stride of a line (complex values, odd): between passes the line is kept
// as m / r0 rows of r0 values at the odd row stride r0 | 1, before the first
// and after the last pass as m (+ 1) values in natural order.
__host__ __device__ constexpr int line_plan_stride(int r0, int r1, int r2)
{
    const int m = r0 * r1 * (r2 ? r2 : 1);
    const int rows = m / r0 * (r0 | 1);
    return (rows > m + 1 ? rows : m + 1) | 1;
}

// Longest FFT length of the real-to-real modes' plans (other than DHT).
constexpr int kLinePlanRealMax = 512;

// Convolution lengths of k_line_blue, among the line plans' lengths: steps of
// at most 20% from 160 on (its FFT lengths m are 79 to kBlueMax).
__host__ __device__ constexpr bool blue_length(int M)
{
    return M == 160 || M == 180 || M == 196 || M == 210 || M == 225 || M == 240 || M == 256 || M == 288 || M == 320 ||
           M == 360 || M == 400 || M == 450 || M == 512 || M == 600 || M == 700 || M == 800 || M == 900 || M == 1024;
}
constexpr int kBlueMax = 512;

// Most threads of a workgroup of k_line_plan.
constexpr int kLinePlanThreads = 512;

} // namespace pfh
