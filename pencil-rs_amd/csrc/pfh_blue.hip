// k_line_blue: stages whose FFT length m has no line plan and a prime factor of
// 79 and more (blue_pays in pfh_api.cpp), as Bluestein's chirp convolution inside
// one workgroup.
//
// With c_j = exp(-i pi j^2 / m) and b_t = exp(+i pi t^2 / m),
//   Z_k = c_k sum_j (x_j c_j) b_{k-j},
// a cyclic convolution of a planned length M >= 2m - 1: the line is padded in
// LDS, transformed, multiplied by FFT_M(b) / M, transformed back (by
// conjugation) and multiplied by c_k, so a stage still reads and writes global
// memory once. It costs two FFTs of about 2.1 m points, some 270 lane
// instructions per complex value in f32; the generic kernel's O(p^2) pass for
// a prime factor p costs 8 p and its own index arithmetic. MI355X, 2^21 points
// of f32 / f64 C2C lines, generic and here: n = 97 192 / 215 -> 18 / 30 us.
// Every mode of the line kernels runs here, its pre-processing placing the
// length-m FFT input in natural order in LDS.
// Compiled once per precision and kind (PFH_LINE_F64, PFH_LINE_KIND).
#include "pfh_line_dev.hpp"

#ifndef PFH_LINE_KIND
#define PFH_LINE_KIND 0
#endif

namespace pfh {

// KIND 0: C2C; 1: all real modes. a.xvalid_in = m, a.xtab_in = c (m entries),
// a.xtab_out = FFT_M(b) / M.
template <typename T, int R0, int R1, int R2, int EM, int KIND>
__global__ __launch_bounds__(kLinePlanThreads) void k_line_blue(const StageArgs<T> a)
{
    using P = LinePlan<T, R0, R1, R2, EM>;
    using V = typename P::V;
    constexpr int M = P::M, TPL = P::TPL, RL = P::RL;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    V *tws = reinterpret_cast<V *>(smem_raw);
    V *data = tws + a.twn;
    if (a.gate != nullptr && *a.gate != 0) return;
    const int tid = threadIdx.x, lt = a.lt, m = a.xvalid_in;
    const uint32_t tile0 = tile_of_block(a, blockIdx.x) * (uint32_t)lt;
    const uint32_t nlines = (uint32_t)a.nlines;
    if (tile0 >= nlines) return;
    const int lsh = __builtin_ctz((unsigned)lt);
    const int rl = (int)((unsigned)tid / (unsigned)TPL), rt = tid - rl * TPL;
    const int cl = tid & (lt - 1), ct = tid >> lsh;
    const int il = a.in_col ? cl : rl, it = a.in_col ? ct : rt;
    const int ol = a.out_col ? cl : rl, ot = a.out_col ? ct : rt;
    V *iln = data + il * a.ls;
    V *oln = data + ol * a.ls;
    uint32_t iline = tile0 + (uint32_t)il < nlines ? tile0 + (uint32_t)il : nlines - 1;
    uint32_t oline = tile0 + (uint32_t)ol;
    const bool store = oline < nlines;
    const void *src = a.src;
    void *dst = a.dst;
    if (a.g.nd == 1) { // offsets relative to the tile, as in k_line_plan
        src = static_cast<const char *>(src) + (int64_t)tile0 * a.g.is[0] * (complex_in(a.mode) ? 2 : 1) * (int64_t)sizeof(T);
        dst = static_cast<char *>(dst) + (int64_t)tile0 * a.g.os[0] * (complex_out(a.mode) ? 2 : 1) * (int64_t)sizeof(T);
        iline -= tile0;
        oline -= tile0;
    }
    const V *twg = reinterpret_cast<const V *>(a.tw);
    for (int i = tid; i < a.twn; i += (int)blockDim.x) tws[i] = twg[i];
    const V *tw1 = tws + a.twoff[1];
    const V *twl = tws + a.twoff[R2 ? 2 : 1];
    const bool cj = (a.flags & F_CONJ_IN) != 0;
    const V *chirp = reinterpret_cast<const V *>(a.xtab_in);
    const V *bhat = reinterpret_cast<const V *>(a.xtab_out);
    const bool odd = (a.n & 1) != 0;
    constexpr int N0 = P::template rounds<R0>(), NB0 = M / R0;
    constexpr int NL = P::template rounds<RL>(), NB = M / RL;

    cpx<T> v[N0][R0];
    if constexpr (KIND == 0) {
        const uint32_t st = (uint32_t)a.ips * (uint32_t)(2 * sizeof(T));
        const uint32_t off = line_offset<false>(a.g, iline, 2 * sizeof(T)) + (uint32_t)it * st;
#pragma unroll
        for (int b = 0; b < N0; ++b) {
            const int j = it + TPL * b;
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                v[b][r] = mk((T)0, (T)0);
                // (indexes from M / 2 + 1 on are padding for every m)
                if (r * NB0 <= M / 2 && P::template has<R0>(b, j) && j + r * NB0 < m)
                    v[b][r] = gread<cpx<T>>(src, off + (uint32_t)(b * TPL + r * NB0) * st);
            }
        }
#pragma unroll
        for (int b = 0; b < N0; ++b) {
            const int j = it + TPL * b;
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                if (r * NB0 <= M / 2 && P::template has<R0>(b, j) && j + r * NB0 < m) {
                    if (cj) v[b][r].y = -v[b][r].y;
                    v[b][r] = cmul(v[b][r], get<T>(chirp + j + r * NB0));
                }
            }
        }
    } else {
        __syncthreads(); // the tables
        if (a.mode == M_C2R) {
            const uint32_t st = (uint32_t)a.ips * (uint32_t)(2 * sizeof(T));
            const uint32_t off = line_offset<false>(a.g, iline, 2 * sizeof(T));
            const bool half = (a.flags & F_HERM_HALF) != 0;
#pragma unroll 2
            for (int q = it; q <= m / 2; q += TPL) {
                cpx<T> x = gread<cpx<T>>(src, off + (uint32_t)q * st), y = mk((T)0, (T)0);
                if (!odd) y = gread<cpx<T>>(src, off + (uint32_t)(m - q) * st);
                if (cj) {
                    x.y = -x.y;
                    y.y = -y.y;
                }
                if (q == 0) {
                    x.y = (T)0;
                    y.y = (T)0;
                } else if (half) {
                    x = scal(x, (T)0.5);
                    y = scal(y, (T)0.5);
                }
                if (odd) {
                    put<T>(iln + q, conjg(x));
                    if (q != 0) put<T>(iln + m - q, x);
                } else {
                    cpx<T> z0, z1;
                    merge_pair(x, y, get<T>(tws + a.pre0 + q), z0, z1);
                    put<T>(iln + q, z0);
                    if (q != 0 && 2 * q != m) put<T>(iln + m - q, z1);
                }
            }
        } else if (a.mode == M_R2C || a.mode == M_DHT) {
            const uint32_t s1 = (uint32_t)a.ips * (uint32_t)sizeof(T);
            const uint32_t off = line_offset<false>(a.g, iline, sizeof(T));
#pragma unroll 4
            for (int i = it; i < m; i += TPL) {
                if (odd) put<T>(iln + i, mk(gread<T>(src, off + (uint32_t)i * s1), (T)0));
                else put<T>(iln + i, mk(gread<T>(src, off + (uint32_t)(2 * i) * s1), gread<T>(src, off + (uint32_t)(2 * i + 1) * s1)));
            }
        } else {
            load_real<P, T>(a, src, iln, tws, line_offset<false>(a.g, iline, sizeof(T)), it);
        }
        __syncthreads();
        if (a.mode == M_DCT3) merge_dct3<P, T>(a, iln, tws, it, m);
        const bool pre = a.mode == M_DCT4;
#pragma unroll
        for (int b = 0; b < N0; ++b) {
            const int j = it + TPL * b;
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                v[b][r] = mk((T)0, (T)0);
                if (r * NB0 <= M / 2 && P::template has<R0>(b, j) && j + r * NB0 < m) {
                    cpx<T> z = get<T>(iln + j + r * NB0);
                    if (pre) z = cmul(z, get<T>(tws + a.pre0 + j + r * NB0));
                    v[b][r] = cmul(z, get<T>(chirp + j + r * NB0));
                }
            }
        }
        __syncthreads();
    }
    P::first_store(iln, it, v);
    P::mid(iln, tw1, it);
    {
        cpx<T> w[NL][RL];
        P::last(iln, twl, it, w);
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NL; ++b) {
            const int j = it + TPL * b;
            if (P::template has<RL>(b, j)) {
#pragma unroll
                for (int r = 0; r < RL; ++r) put<T>(iln + j + r * NB, conjg(cmul(w[b][r], get<T>(bhat + j + r * NB))));
            }
        }
        __syncthreads();
    }
    P::template first_lds<false>(oln, nullptr, ot);
    P::mid(oln, tw1, ot);
    cpx<T> w[NL][RL];
    P::last(oln, twl, ot, w);
    const T sc = a.scale;
    if constexpr (KIND == 0) {
        if (!store) return;
        const uint32_t st = (uint32_t)a.ops * (uint32_t)(2 * sizeof(T));
        const uint32_t off = line_offset<true>(a.g, oline, 2 * sizeof(T)) + (uint32_t)ot * st;
        const T sy = (a.flags & F_CONJ_OUT) ? -sc : sc;
#pragma unroll
        for (int b = 0; b < NL; ++b) {
            const int j = ot + TPL * b;
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                if (r * NB <= M / 2 && P::template has<RL>(b, j) && j + r * NB < m) {
                    const cpx<T> z = cmul(conjg(w[b][r]), get<T>(chirp + j + r * NB));
                    gwrite<cpx<T>>(dst, off + (uint32_t)(b * TPL + r * NB) * st, mk(z.x * sc, z.y * sy));
                }
            }
        }
    } else {
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NL; ++b) {
            const int j = ot + TPL * b;
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                if (r * NB <= M / 2 && P::template has<RL>(b, j) && j + r * NB < m)
                    put<T>(oln + j + r * NB, cmul(conjg(w[b][r]), get<T>(chirp + j + r * NB)));
            }
        }
        __syncthreads();
        if (!store) return;
        const uint32_t s1 = (uint32_t)a.ops * (uint32_t)sizeof(T);
        if (a.mode == M_R2C) {
            const uint32_t st = 2 * s1;
            const uint32_t off = line_offset<true>(a.g, oline, 2 * sizeof(T));
            const bool dbl = (a.flags & F_HERM_DOUBLE) != 0;
            if (odd) {
                const T inner = dbl ? sc * (T)2 : sc;
#pragma unroll 2
                for (int k = ot; k <= m / 2; k += TPL) {
                    const cpx<T> z = get<T>(oln + k);
                    gwrite<cpx<T>>(dst, off + (uint32_t)k * st, k == 0 ? mk(z.x * sc, (T)0) : scal(z, inner));
                }
            } else {
                const T hs = sc * (T)0.5, inner = dbl ? sc : hs;
#pragma unroll 2
                for (int q = ot; q <= m / 2; q += TPL) {
                    cpx<T> x0, x1;
                    split_pair(get<T>(oln + q), get<T>(oln + (q == 0 ? 0 : m - q)), get<T>(tws + a.post0 + q), x0, x1);
                    if (q == 0) {
                        gwrite<cpx<T>>(dst, off, mk(x0.x * hs, (T)0));
                        gwrite<cpx<T>>(dst, off + (uint32_t)m * st, mk(x1.x * hs, (T)0));
                    } else {
                        gwrite<cpx<T>>(dst, off + (uint32_t)q * st, scal(x0, inner));
                        if (2 * q != m) gwrite<cpx<T>>(dst, off + (uint32_t)(m - q) * st, scal(x1, inner));
                    }
                }
            }
        } else if (a.mode == M_C2R) {
            const uint32_t off = line_offset<true>(a.g, oline, sizeof(T));
#pragma unroll 2
            for (int k = ot; k < m; k += TPL) {
                const cpx<T> z = get<T>(oln + k);
                if (odd) {
                    gwrite<T>(dst, off + (uint32_t)k * s1, z.x * sc);
                } else {
                    gwrite<T>(dst, off + (uint32_t)(2 * k) * s1, z.x * sc);
                    gwrite<T>(dst, off + (uint32_t)(2 * k + 1) * s1, -z.y * sc);
                }
            }
        } else {
            const uint32_t off = line_offset<true>(a.g, oline, sizeof(T));
            if (a.mode == M_DHT) post_mode<P, T, true, M_DHT>(a, dst, oln, tws, off, s1, ot, m);
            else post_real<P, T, true>(a, dst, oln, tws, off, s1, ot, m);
        }
    }
}

namespace {

template <typename T, int R0, int R1, int R2, int EM, int KIND>
hipError_t launch_blue(const StageArgs<T> &a, int threads, size_t lds_bytes, int64_t grid, hipStream_t s)
{
    // the shapes the kernel assumes
    if (a.tpl != line_plan_tpl(R0, R1, R2, EM) || threads != a.lt * a.tpl || threads > kLinePlanThreads ||
        a.ls < line_plan_stride(R0, R1, R2) || ((a.in_col || a.out_col) && (a.lt & (a.lt - 1)) != 0) ||
        a.xvalid_in < 1 || 2 * a.xvalid_in - 1 > R0 * R1 * (R2 ? R2 : 1) || !a.xtab_in || !a.xtab_out)
        return hipErrorInvalidValue;
    static std::atomic<uint64_t> done{0};
    if (lds_bytes > 64 * 1024) {
        const hipError_t e = allow_lds(reinterpret_cast<const void *>(&k_line_blue<T, R0, R1, R2, EM, KIND>), done);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_line_blue<T, R0, R1, R2, EM, KIND>), dim3((unsigned)grid), dim3(threads), lds_bytes, s, a);
    return hipGetLastError();
}

} // namespace

#ifdef PFH_LINE_F64
using LineT = double;
#else
using LineT = float;
#endif

template <>
hipError_t launch_line_blue<LineT, PFH_LINE_KIND>(const StageArgs<LineT> &a, int r0, int r1, int r2, int em, int threads,
                                                  size_t lds_bytes, int64_t grid, hipStream_t s)
{
#define PFH_BLUE_CASE(TT, A, B, C, E)                                                                      \
    if constexpr (sizeof(TT) == sizeof(LineT) && blue_length((A) * (B) * ((C) ? (C) : 1)) &&               \
                  !line_plan_real_only(A, B, C, E))                                                        \
        if (r0 == A && r1 == B && r2 == C && em == E)                                                      \
            return launch_blue<LineT, A, B, C, E, PFH_LINE_KIND>(a, threads, lds_bytes, grid, s);
    PFH_FAST_ROUTE_PLANS(PFH_BLUE_CASE)
#undef PFH_BLUE_CASE
    return hipErrorInvalidValue;
}

} // namespace pfh
