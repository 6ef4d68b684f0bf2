// Device pointwise operations on pencil arrays: the pieces a pseudo-spectral
// step needs between transforms. They follow the reference's pointwise and
// grid helpers (crates/pencil-array/src/pointwise.rs:40-598, a closure over
// co-located elements; grid.rs:20-120, per-axis coordinate arrays seen in the
// pencil's memory order) and its l2 reduction (collectives.rs:519-560), as
// memory-bound element kernels.
#include <hip/hip_runtime.h>

#include "pfh_bounds.hpp"
#include "pfh_kernels.hpp"

namespace pfh {

namespace {

constexpr int kBlock = 256;

// data[e][memory index] *= prod_a f_a[i_a]: rows of the fastest memory
// position, its factor times the slower positions' (that order of products,
// f holds the per-axis factors concatenated in logical axis order; complex
// factors: (re, im) pairs, e.g. i k_a for a spectral derivative). Bound by HBM
// (one read and one write): cols threads along a row and kRows rows a thread
// keep the row's index arithmetic off the elements and their loads in flight.
// 256^3 f32 half spectrum (67 MB) on MI355X: 41 us with one element and its
// 64-bit divisions a thread, 30 us so.
constexpr int kRows = kScaleRows;
template <typename T, int C, bool CF>
__global__ __launch_bounds__(kBlock) void k_scale_axes(ScaleAxesArgs s, T *data, const T *f, uint32_t rows, int cols,
                                                       int csh)
{
    const int x = threadIdx.x & (cols - 1), y = threadIdx.x >> csh;
    const uint32_t per = (uint32_t)kBlock >> csh;
    const uint32_t r0 = blockIdx.x * (per * kRows) + (uint32_t)y;
    const int last = s.nd - 1;
    const int64_t nx = s.mext[last];
    const T *fx = f + s.foff[last] * (CF ? 2 : 1);
    for (int64_t i = (int64_t)blockIdx.y * cols + x; i < nx; i += (int64_t)gridDim.y * cols) {
        T v[kRows][C];
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            const uint32_t r = r0 + (uint32_t)k * per;
            if (r < rows) {
#pragma unroll
                for (int c = 0; c < C; ++c) v[k][c] = data[((int64_t)r * nx + i) * C + c];
            }
        }
        const T xr = fx[CF ? 2 * i : i], xi = CF ? fx[2 * i + 1] : (T)0;
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            const uint32_t r = r0 + (uint32_t)k * per;
            if (r >= rows) continue;
            T wr = xr, wi = xi;
            uint32_t q = r;
#pragma unroll
            for (int p = 6; p >= 0; --p) {
                if (p < last) {
                    const uint32_t d = fastdiv(q, s.dmag[p], s.dsh[p]);
                    const int64_t idx = s.foff[p] + (int64_t)(q - d * (uint32_t)s.mext[p]);
                    q = d;
                    if (CF) {
                        const T fr = f[2 * idx], fi = f[2 * idx + 1];
                        const T t = wr * fr - wi * fi;
                        wi = wr * fi + wi * fr;
                        wr = t;
                    } else {
                        wr *= f[idx];
                    }
                }
            }
            T *o = data + ((int64_t)r * nx + i) * C;
            if (CF) {
                o[0] = v[k][0] * wr - v[k][C - 1] * wi;
                o[C - 1] = v[k][0] * wi + v[k][C - 1] * wr;
            } else {
#pragma unroll
                for (int c = 0; c < C; ++c) o[c] = v[k][c] * wr;
            }
        }
    }
}

// Elementwise kernels: kUnroll elements a thread, all loads issued first.
// 256^3 f32 on MI355X, one element a thread before: quadratic step (134 MB) 32
// -> 22 us, its adjoint (201 MB) 52 -> 36 us.
constexpr int kUnroll = kElementsPerBlock / kBlock;
unsigned chunks_for(int64_t n)
{
    return (unsigned)((n + (int64_t)kBlock * kUnroll - 1) / ((int64_t)kBlock * kUnroll));
}

// u = w + a w^2 (a pointwise quadratic step)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_quadratic(const T *w, T *u, int64_t n, T a)
{
    const int64_t b = (int64_t)blockIdx.x * (kBlock * kUnroll) + threadIdx.x;
    T v[kUnroll];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k)
        if (b + k * kBlock < n) v[k] = w[b + k * kBlock];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k)
        if (b + k * kBlock < n) u[b + k * kBlock] = fma(a * v[k], v[k], v[k]);
}

// out = g (1 + 2 a w): the transpose of the quadratic step's derivative
template <typename T>
__global__ __launch_bounds__(kBlock) void k_quadratic_adjoint(const T *w, const T *g, T *out, int64_t n, T a)
{
    const int64_t b = (int64_t)blockIdx.x * (kBlock * kUnroll) + threadIdx.x;
    T v[kUnroll], h[kUnroll];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k)
        if (b + k * kBlock < n) {
            v[k] = w[b + k * kBlock];
            h[k] = g[b + k * kBlock];
        }
#pragma unroll
    for (int k = 0; k < kUnroll; ++k)
        if (b + k * kBlock < n) out[b + k * kBlock] = h[k] * ((T)1 + (T)2 * a * v[k]);
}

__device__ __forceinline__ double block_sum(double v, double *sh)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) r += sh[k];
    return r;
}

// Deterministic sum of squares: a fixed grid of partial sums (each block a
// fixed chunk), then one block adds the partials in order.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_sumsq_partial(const T *x, int64_t n, double *partial)
{
    __shared__ double sh[kBlock / 64];
    const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
    const int64_t b = (int64_t)blockIdx.x * chunk;
    const int64_t e = b + chunk < n ? b + chunk : n;
    double acc = 0.0;
    for (int64_t i = b + threadIdx.x; i < e; i += blockDim.x) {
        const double v = (double)x[i];
        acc += v * v;
    }
    const double r = block_sum(acc, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = r;
}

__global__ __launch_bounds__(kBlock) void k_sumsq_final(const double *partial, int nparts, double *result)
{
    __shared__ double sh[kBlock / 64];
    double acc = 0.0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) acc += partial[i];
    const double r = block_sum(acc, sh);
    if (threadIdx.x == 0) *result = r;
}

} // namespace

template <typename T>
hipError_t launch_scale_axes(const ScaleAxesArgs &s0, void *data, const void *factors, hipStream_t st)
{
    if (s0.len * s0.extra <= 0) return hipSuccess;
    hipError_t err = hipSuccess;
    scale_axes_parts(s0, 0, [&](const ScaleAxesArgs &part, int64_t first) {
        if (err != hipSuccess) return;
        ScaleAxesArgs s = part;
        const int64_t nx = s.mext[s.nd - 1], rows = s.len * s.extra / nx;
        for (int p = 0; p + 1 < s.nd; ++p) {
            const FastDiv d = make_fastdiv((uint32_t)s.mext[p]);
            s.dmag[p] = d.mag;
            s.dsh[p] = d.sh;
        }
        const int cols = scale_axes_cols(nx);
        int csh = 0;
        while ((1 << csh) < cols) ++csh;
        int64_t gy = (nx + cols - 1) / cols;
        if (gy > 64) gy = 64;
        const dim3 grid((unsigned)scale_axes_blocks(rows, nx), (unsigned)gy);
        T *d = static_cast<T *>(data) + first * (s.complex_data ? 2 : 1);
        const T *f = static_cast<const T *>(factors);
        if (s.complex_factors)
            hipLaunchKernelGGL((k_scale_axes<T, 2, true>), grid, dim3(kBlock), 0, st, s, d, f, (uint32_t)rows, cols, csh);
        else if (s.complex_data)
            hipLaunchKernelGGL((k_scale_axes<T, 2, false>), grid, dim3(kBlock), 0, st, s, d, f, (uint32_t)rows, cols, csh);
        else
            hipLaunchKernelGGL((k_scale_axes<T, 1, false>), grid, dim3(kBlock), 0, st, s, d, f, (uint32_t)rows, cols, csh);
        err = hipGetLastError();
    });
    return err;
}
template hipError_t launch_scale_axes<float>(const ScaleAxesArgs &, void *, const void *, hipStream_t);
template hipError_t launch_scale_axes<double>(const ScaleAxesArgs &, void *, const void *, hipStream_t);

template <typename T>
hipError_t launch_quadratic(const void *w, void *u, int64_t n, double a, hipStream_t st)
{
    for (int64_t i = 0; i < n; i += kElementsPerLaunch) {
        const int64_t m = n - i < kElementsPerLaunch ? n - i : kElementsPerLaunch;
        hipLaunchKernelGGL(k_quadratic<T>, dim3(chunks_for(m)), dim3(kBlock), 0, st, static_cast<const T *>(w) + i,
                           static_cast<T *>(u) + i, m, (T)a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
template hipError_t launch_quadratic<float>(const void *, void *, int64_t, double, hipStream_t);
template hipError_t launch_quadratic<double>(const void *, void *, int64_t, double, hipStream_t);

template <typename T>
hipError_t launch_quadratic_adjoint(const void *w, const void *g, void *out, int64_t n, double a, hipStream_t st)
{
    for (int64_t i = 0; i < n; i += kElementsPerLaunch) {
        const int64_t m = n - i < kElementsPerLaunch ? n - i : kElementsPerLaunch;
        hipLaunchKernelGGL(k_quadratic_adjoint<T>, dim3(chunks_for(m)), dim3(kBlock), 0, st,
                           static_cast<const T *>(w) + i, static_cast<const T *>(g) + i, static_cast<T *>(out) + i, m,
                           (T)a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
template hipError_t launch_quadratic_adjoint<float>(const void *, const void *, void *, int64_t, double, hipStream_t);
template hipError_t launch_quadratic_adjoint<double>(const void *, const void *, void *, int64_t, double,
                                                     hipStream_t);

template <typename T>
hipError_t launch_sum_squares(const void *x, int64_t n, double *partial, int nparts, double *result, hipStream_t st)
{
    if (nparts < 1 || nparts > kSumSquaresParts) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_sumsq_partial<T>, dim3((unsigned)nparts), dim3(kBlock), 0, st, static_cast<const T *>(x),
                       n, partial);
    hipLaunchKernelGGL(k_sumsq_final, dim3(1), dim3(kBlock), 0, st, partial, nparts, result);
    return hipGetLastError();
}
template hipError_t launch_sum_squares<float>(const void *, int64_t, double *, int, double *, hipStream_t);
template hipError_t launch_sum_squares<double>(const void *, int64_t, double *, int, double *, hipStream_t);

} // namespace pfh
