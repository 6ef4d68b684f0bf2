// Bit-exact layout copies: LocalTransposePlan / AllToAllvTransposePlan at one
// rank and the identity stages of routes.
//
// A copy moves points (stride ss_p in the source, ds_p in the destination)
// of lines (ss_l, ds_l) over any further digits. Two shapes cover the layouts
// whose fastest axes both have extent above one:
//  - the source's and the destination's fastest axes differ: tiles of TL x TP
//    elements go through LDS, read along the source's fastest axis and
//    written along the destination's, 64-element runs on both sides (16-byte
//    elements: 32), 16 (4) loads in flight a thread;
//  - they are the same: rows, moved in 16-byte pieces where lengths, strides
//    and addresses allow.
// Each is taken where it beats the callers' own kernels (pfh_copy.hpp); both are
// bound by HBM. 256 x 384 x 240 complex f32, z,y,x -> x,z,y (189 MB
// each way) on MI355X: 74 us; the line kernel's copy stage, which held whole
// lines on one wave per workgroup in LDS, took 154 us.
#include <hip/hip_runtime.h>

#include "pfh_bounds.hpp"
#include "pfh_copy.hpp"
#include "pfh_kernels.hpp"

namespace pfh {

namespace {

struct CopyArgs {
    const void *src;
    void *dst;
    const int *gate;   // if non-null and *gate != 0 nothing is written
    int64_t n, e0;     // points, lines of the tile digit
    int64_t ss_p, ds_p, ss_l, ds_l;
    int64_t tiles_p, tiles_l;
    int nd;            // further digits, fastest first
    uint32_t ext[kMaxDigits + 4];
    uint32_t dmag[kMaxDigits + 4];
    int dsh[kMaxDigits + 4];
    int64_t is[kMaxDigits + 4], os[kMaxDigits + 4];
};
constexpr int kCopyDigits = kMaxDigits + 4;

struct alignas(8) W16 {
    uint64_t a, b;
};

__device__ __forceinline__ void copy_offsets(const CopyArgs &a, uint32_t x, int64_t &so, int64_t &dof)
{
    so = dof = 0;
#pragma unroll
    for (int d = 0; d < kCopyDigits; ++d) {
        if (d < a.nd) {
            const uint32_t q = fastdiv(x, a.dmag[d], a.dsh[d]);
            const uint32_t r = x - q * a.ext[d];
            so += (int64_t)r * a.is[d];
            dof += (int64_t)r * a.os[d];
            x = q;
        }
    }
}

// ss_l == 1 and ds_p == 1; grid.x = tiles over points x lines x digits
template <typename W, int TILE>
__global__ __launch_bounds__(256) void k_copy_tile(const CopyArgs a)
{
    __shared__ W sh[TILE][TILE + 1];
    if (a.gate != nullptr && *a.gate != 0) return;
    constexpr int ROWS = 256 / TILE, K = TILE / ROWS;
    const uint32_t b = blockIdx.x;
    const uint32_t tl = b % (uint32_t)a.tiles_l, r = b / (uint32_t)a.tiles_l;
    const uint32_t tp = r % (uint32_t)a.tiles_p, rest = r / (uint32_t)a.tiles_p;
    int64_t so, dof;
    copy_offsets(a, rest, so, dof);
    const int x = threadIdx.x % TILE, y = threadIdx.x / TILE;
    const int64_t p0 = (int64_t)tp * TILE, l0 = (int64_t)tl * TILE;
    const W *src = static_cast<const W *>(a.src) + so;
    W *dst = static_cast<W *>(a.dst) + dof;
    W v[K];
    const int64_t l = l0 + x;
    if (l < a.e0) {
        const W *s = src + l + (p0 + y) * a.ss_p;
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (p0 + y + k * ROWS < a.n) v[k] = s[(int64_t)(k * ROWS) * a.ss_p];
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (p0 + y + k * ROWS < a.n) sh[y + k * ROWS][x] = v[k];
    }
    __syncthreads();
    const int64_t p = p0 + x;
    if (p < a.n) {
        W *d = dst + p + (l0 + y) * a.ds_l;
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (l0 + y + k * ROWS < a.e0) d[(int64_t)(k * ROWS) * a.ds_l] = sh[x][y + k * ROWS];
    }
}

// rows (ss_p == ds_p == 1): cols threads along a row, 256 / cols rows at a
// time, kCopyRows such groups per workgroup; grid.y = pieces of 256 points
constexpr int kRows = kCopyRows;
template <typename W>
__global__ __launch_bounds__(256) void k_copy_rows(const CopyArgs a, uint32_t rows, int cols, int csh)
{
    if (a.gate != nullptr && *a.gate != 0) return;
    const int x = threadIdx.x & (cols - 1), y = threadIdx.x >> csh;
    const uint32_t per = 256u >> csh;
    const uint32_t r0 = blockIdx.x * (per * kRows) + (uint32_t)y;
    for (int64_t p = (int64_t)blockIdx.y * cols + x; p < a.n; p += (int64_t)gridDim.y * cols) {
        W v[kRows];
        int64_t dof[kRows];
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            const uint32_t r = r0 + (uint32_t)k * per;
            if (r < rows) {
                int64_t so;
                copy_offsets(a, r, so, dof[k]);
                v[k] = static_cast<const W *>(a.src)[so + p];
            }
        }
#pragma unroll
        for (int k = 0; k < kRows; ++k)
            if (r0 + (uint32_t)k * per < rows) static_cast<W *>(a.dst)[dof[k] + p] = v[k];
    }
}

template <typename W>
hipError_t run_tile(CopyArgs &a, int64_t rest, hipStream_t s, bool &done)
{
    constexpr int TILE = copy_tile((int)sizeof(W));
    a.tiles_p = (a.n + TILE - 1) / TILE;
    a.tiles_l = (a.e0 + TILE - 1) / TILE;
    const int64_t grid = copy_tile_blocks((int)sizeof(W), a.n, a.e0, rest);
    if (grid >= kMaxBlocks256) return hipSuccess; // left to the caller's kernel
    done = true;
    hipLaunchKernelGGL((k_copy_tile<W, TILE>), dim3((unsigned)grid), dim3(256), 0, s, a);
    return hipGetLastError();
}

template <typename W>
hipError_t run_rows(const CopyArgs &a, int64_t rows, hipStream_t s)
{
    const int cols = copy_row_cols(a.n);
    int csh = 0;
    while ((1 << csh) < cols) ++csh;
    int64_t gy = (a.n + cols - 1) / cols;
    if (gy > 64) gy = 64;
    hipLaunchKernelGGL(k_copy_rows<W>, dim3((unsigned)copy_row_blocks(rows, a.n), (unsigned)gy), dim3(256), 0, s, a,
                       (uint32_t)rows, cols, csh);
    return hipGetLastError();
}

} // namespace

// Copies the axes of c; done stays false (nothing launched) where neither
// shape applies or pays (pfh_copy.hpp). Axes of extent 1 may be listed. src and dst do not overlap
// unless they are the same array in the same layout.
hipError_t launch_copy_axes(const CopyAxes &c, const void *src, void *dst, int word, const int *gate, hipStream_t s,
                            bool &done)
{
    done = false;
    CopyArgs a{};
    a.src = src;
    a.dst = dst;
    a.gate = gate;
    int ip = -1, il = -1; // axes of unit stride: destination's, source's
    int64_t total = 1;
    for (int i = 0; i < c.nd; ++i) {
        total *= c.ext[i];
        if (c.ext[i] <= 1) continue;
        if (c.os[i] == 1) ip = i;
        if (c.is[i] == 1) il = i;
    }
    if (ip < 0 || il < 0 || total <= 0) return hipSuccess;
    int64_t rest = 1;
    // further digits, by destination stride
    int order[16], no = 0;
    for (int i = 0; i < c.nd; ++i)
        if (c.ext[i] > 1 && i != ip && i != il) order[no++] = i;
    for (int i = 1; i < no; ++i)
        for (int j = i; j > 0 && c.os[order[j]] < c.os[order[j - 1]]; --j) {
            const int t = order[j];
            order[j] = order[j - 1];
            order[j - 1] = t;
        }
    if (no > kCopyDigits) return hipSuccess;
    for (int i = 0; i < no; ++i) {
        const int d = order[i];
        if (c.ext[d] > INT32_MAX) return hipSuccess;
        const FastDiv f = make_fastdiv((uint32_t)c.ext[d]);
        a.ext[i] = (uint32_t)c.ext[d];
        a.dmag[i] = f.mag;
        a.dsh[i] = f.sh;
        a.is[i] = c.is[d];
        a.os[i] = c.os[d];
        rest *= c.ext[d];
    }
    a.nd = no;
    if (rest > INT32_MAX) return hipSuccess;
    a.n = c.ext[ip];
    a.ss_p = c.is[ip];
    a.ds_p = 1;
    if (ip != il) {
        a.e0 = c.ext[il];
        a.ss_l = 1;
        a.ds_l = c.os[il];
        if (!copy_tile_pays(word, a.n, a.e0)) return hipSuccess;
        switch (word) {
        case 1: return run_tile<uint8_t>(a, rest, s, done);
        case 2: return run_tile<uint16_t>(a, rest, s, done);
        case 4: return run_tile<uint32_t>(a, rest, s, done);
        case 8: return run_tile<uint64_t>(a, rest, s, done);
        case 16: return run_tile<W16>(a, rest, s, done);
        default: return hipSuccess;
        }
    }
    // rows: the widest word that lengths, strides and addresses are multiples of
    a.ss_l = a.ds_l = 0;
    a.e0 = 1;
    const int word0 = word;
    while (word < 16) {
        bool even = a.n % 2 == 0 && reinterpret_cast<uintptr_t>(src) % (2 * (size_t)word) == 0 &&
                    reinterpret_cast<uintptr_t>(dst) % (2 * (size_t)word) == 0;
        for (int i = 0; i < no; ++i) even = even && a.is[i] % 2 == 0 && a.os[i] % 2 == 0;
        if (!even) break;
        word *= 2;
        a.n /= 2;
        for (int i = 0; i < no; ++i) {
            a.is[i] /= 2;
            a.os[i] /= 2;
        }
    }
    if (!copy_rows_pay(word0, c.ext[ip], a.n) || copy_row_blocks(rest, a.n) >= kMaxBlocks256) return hipSuccess;
    done = true;
    switch (word) {
    case 1: return run_rows<uint8_t>(a, rest, s);
    case 2: return run_rows<uint16_t>(a, rest, s);
    case 4: return run_rows<uint32_t>(a, rest, s);
    case 8: return run_rows<uint64_t>(a, rest, s);
    case 16: return run_rows<W16>(a, rest, s);
    default: done = false; return hipSuccess;
    }
}

} // namespace pfh
