// k_line_plan: route stages whose FFT length has a compile-time radix plan.
//
// A workgroup transforms lt lines, TPL threads each; TPL and every LDS offset
// of the radix passes are compile-time constants. What bounds an f32 stage on
// this GPU is vector issue: without packed arithmetic the 256 CUs issue about
// 39 T lane instructions a second, 126 for each complex f32 value that a
// stage reads and writes at 5 TB/s (63 for a real one), so the kernel is laid
// out to spend few instructions outside the butterflies:
//  - between passes a line is kept as rows of R0 values at an odd row stride,
//    so all R values of a butterfly lie at constant offsets from one address
//    (one address per butterfly, no padding arithmetic per value);
//  - global accesses are a uniform base plus a 32-bit byte offset per lane,
//    advanced by a uniform step (arrays of 4 GiB and more run on k_line_fast
//    or the generic kernel);
//  - real transforms handle the spectrum in pairs X_q, X_{m-q}: one twiddle
//    product gives both, and their two (DCT-IV), three or four real outputs;
//  - composite radices (6, 9, 10, 12, 14, 15, 16) keep lengths up to 256 at
//    two passes, one LDS exchange.
// Measured per launch on MI355X, before (generic kernel, or k_line_fast with
// run-time threads per line) and after: 180 x 225 x 200 x 3 f32 R2C, 97 MB in
// and out, 147 / 159 / 176 -> 51 / 44 / 48 us; 256 x 384 x 240 f32, 94 MB in
// and out, DST-I 124 -> 75 us, DCT-II / III 71 / 78 -> 55 us, DCT-IV 75 -> 51
// us; f64 DCT-I of 129 points 41 -> 27 us (32 MB), FFT of 192 points 24 -> 15
// us.
// This file is compiled once per precision and kind (PFH_LINE_F64,
// PFH_LINE_KIND) so that the parts build in parallel.
#include <hip/hip_runtime.h>

#include <atomic>

#include "pfh_kernels.hpp"
#include "pfh_line.hpp"

#ifndef PFH_LINE_KIND
#define PFH_LINE_KIND 0
#endif

namespace pfh {

namespace {

template <typename T>
struct Vec2;
template <>
struct Vec2<float> {
    typedef float type __attribute__((ext_vector_type(2)));
};
template <>
struct Vec2<double> {
    typedef double type __attribute__((ext_vector_type(2)));
};

template <typename T>
__device__ __forceinline__ cpx<T> get(const typename Vec2<T>::type *p)
{
    const typename Vec2<T>::type v = *p;
    return mk(v.x, v.y);
}
template <typename T>
__device__ __forceinline__ void put(typename Vec2<T>::type *p, cpx<T> v)
{
    typename Vec2<T>::type w;
    w.x = v.x;
    w.y = v.y;
    *p = w;
}

// global accesses: uniform base + 32-bit byte offset
template <typename V>
__device__ __forceinline__ V gread(const void *base, uint32_t off)
{
    return *reinterpret_cast<const V *>(static_cast<const char *>(base) + off);
}
template <typename V>
__device__ __forceinline__ void gwrite(void *base, uint32_t off, V v)
{
    *reinterpret_cast<V *>(static_cast<char *>(base) + off) = v;
}

// Coordinate of line digit xdig of a line (pieces of long lines).
__device__ __forceinline__ uint32_t line_digit(const LineGeom &g, uint32_t line, int xdig)
{
    uint32_t x = line, c = 0;
#pragma unroll
    for (int d = 0; d < kMaxDigits; ++d) {
        if (d < g.nd) {
            const uint32_t q = fastdiv(x, g.dmag[d], g.dsh[d]);
            if (d == xdig) c = x - q * (uint32_t)g.ext[d];
            x = q;
        }
    }
    return c;
}

__device__ __forceinline__ bool complex_in(int mode) { return mode == M_C2C || mode == M_C2R; }
__device__ __forceinline__ bool complex_out(int mode) { return mode == M_C2C || mode == M_R2C; }

// Byte offset of a line's first element (32 bits: the planner sends larger
// arrays elsewhere).
template <bool OUT>
__device__ __forceinline__ uint32_t line_offset(const LineGeom &g, uint32_t line, uint32_t eb)
{
    uint32_t off = 0, x = line;
#pragma unroll
    for (int d = 0; d < kMaxDigits; ++d) {
        if (d < g.nd) {
            const uint32_t st = (uint32_t)(OUT ? g.os[d] : g.is[d]) * eb;
            if (d + 1 < g.nd) {
                const uint32_t q = fastdiv(x, g.dmag[d], g.dsh[d]);
                off += (x - q * (uint32_t)g.ext[d]) * st;
                x = q;
            } else {
                off += x * st;
            }
        }
    }
    return off;
}

template <typename T, int R0, int R1, int R2, int EM>
struct LinePlan {
    using V = typename Vec2<T>::type;
    static constexpr int M = R0 * R1 * (R2 ? R2 : 1);
    static constexpr int RL = R2 ? R2 : R1;
    static constexpr int RP = R0 | 1;
    static constexpr int TPL = line_plan_tpl(R0, R1, R2, EM);

    // every thread's butterflies b = 0 .. MB - 1 of a radix-R pass: j = t +
    // TPL b; the last round may be partial
    template <int R>
    static constexpr int rounds()
    {
        return (M / R + TPL - 1) / TPL;
    }
    template <int R>
    __device__ static __forceinline__ bool has(int b, int j)
    {
        return TPL * (b + 1) <= M / R || j < M / R;
    }

    // first pass: values in registers -> rows of R0
    template <int N>
    __device__ static __forceinline__ void first_store(V *ln, int t, cpx<T> (&v)[N][R0])
    {
#pragma unroll
        for (int b = 0; b < N; ++b) {
            const int j = t + TPL * b;
            if (has<R0>(b, j)) {
                Dft<T, R0>::run(v[b]);
                V *p = ln + j * RP;
#pragma unroll
                for (int r = 0; r < R0; ++r) put<T>(p + r, v[b][r]);
            }
        }
        __syncthreads();
    }

    // first pass of a line in natural order in LDS (times pre[j] when PRE)
    template <bool PRE>
    __device__ static __forceinline__ void first_lds(V *ln, const V *pre, int t)
    {
        constexpr int N = rounds<R0>(), NB = M / R0;
        cpx<T> v[N][R0];
#pragma unroll
        for (int b = 0; b < N; ++b) {
            const int j = t + TPL * b;
            if (has<R0>(b, j)) {
#pragma unroll
                for (int r = 0; r < R0; ++r) {
                    v[b][r] = get<T>(ln + j + r * NB);
                    if (PRE) v[b][r] = cmul(v[b][r], get<T>(pre + j + r * NB));
                }
            }
        }
        __syncthreads();
        first_store(ln, t, v);
    }

    // middle pass (three-pass plans): rows -> rows
    __device__ static __forceinline__ void mid(V *ln, const V *twp, int t)
    {
        if constexpr (R2 != 0) {
            constexpr int N = rounds<R1>(), NB = M / R1;
            cpx<T> v[N][R1];
#pragma unroll
            for (int b = 0; b < N; ++b) {
                const int j = t + TPL * b;
                if (has<R1>(b, j)) {
                    const int q = (int)((uint32_t)j / (uint32_t)R0), k = j - q * R0;
                    const V *p = ln + j + q * (RP - R0);
                    const V *w = twp + k * (R1 - 1);
#pragma unroll
                    for (int r = 0; r < R1; ++r) v[b][r] = get<T>(p + r * (NB / R0) * RP);
#pragma unroll
                    for (int r = 1; r < R1; ++r) v[b][r] = cmul(v[b][r], get<T>(w + r - 1));
                    Dft<T, R1>::run(v[b]);
                }
            }
            __syncthreads();
#pragma unroll
            for (int b = 0; b < N; ++b) {
                const int j = t + TPL * b;
                if (has<R1>(b, j)) {
                    const int q = (int)((uint32_t)j / (uint32_t)R0), k = j - q * R0;
                    V *p = ln + q * (R1 * RP) + k;
#pragma unroll
                    for (int r = 0; r < R1; ++r) put<T>(p + r * RP, v[b][r]);
                }
            }
            __syncthreads();
        }
    }

    // last pass into registers: v[b][r] is output j + r M / RL
    template <int N>
    __device__ static __forceinline__ void last(const V *ln, const V *twp, int t, cpx<T> (&v)[N][RL])
    {
        constexpr int NB = M / RL;
#pragma unroll
        for (int b = 0; b < N; ++b) {
            const int j = t + TPL * b;
            if (has<RL>(b, j)) {
                const int q = R2 ? (int)((uint32_t)j / (uint32_t)R0) : 0;
                const V *p = ln + j + q * (RP - R0);
                const V *w = twp + j * (RL - 1);
#pragma unroll
                for (int r = 0; r < RL; ++r) v[b][r] = get<T>(p + r * (NB / R0) * RP);
#pragma unroll
                for (int r = 1; r < RL; ++r) v[b][r] = cmul(v[b][r], get<T>(w + r - 1));
                Dft<T, RL>::run(v[b]);
            }
        }
    }

    // last pass, natural order back into the LDS line
    __device__ static __forceinline__ void last_lds(V *ln, const V *twp, int t)
    {
        constexpr int N = rounds<RL>(), NB = M / RL;
        cpx<T> v[N][RL];
        last(ln, twp, t, v);
        __syncthreads();
#pragma unroll
        for (int b = 0; b < N; ++b) {
            const int j = t + TPL * b;
            if (has<RL>(b, j)) {
#pragma unroll
                for (int r = 0; r < RL; ++r) put<T>(ln + j + r * NB, v[b][r]);
            }
        }
        __syncthreads();
    }
};

// The spectrum pair of a real line from its half-length transform: with A =
// Z_q, B = conj Z_{m-q} and w = exp(-i pi q / m), x0 = 2 X_q and x1 = 2
// X_{m-q}. q = 0 gives X_0 and X_m (imaginary parts exactly zero).
template <typename T>
__device__ __forceinline__ void split_pair(cpx<T> zq, cpx<T> zm, cpx<T> w, cpx<T> &x0, cpx<T> &x1)
{
    const cpx<T> B = conjg(zm);
    const cpx<T> E = zq + B, P = mul_mi(cmul(w, zq - B));
    x0 = E + P;
    x1 = conjg(E - P);
}

// Its transpose: the conjugated half-length inputs z_q, z_{m-q} of a positive
// sign real transform from X_q, X_{m-q} and w = exp(+i pi q / m).
template <typename T>
__device__ __forceinline__ void merge_pair(cpx<T> xq, cpx<T> xm, cpx<T> w, cpx<T> &z0, cpx<T> &z1)
{
    const cpx<T> B = conjg(xm);
    const cpx<T> E = xq + B, P = mul_pi(cmul(w, xq - B));
    z0 = conjg(E + P);
    z1 = E - P;
}

// Real output k of an R2R line: reversal, alternating sign, end weights and
// scale (FLAGS: any of the first three is asked for).
template <typename T, bool FLAGS>
struct Emit {
    const StageArgs<T> &a;
    void *dst;
    uint32_t off, step;
    T sc;
    __device__ __forceinline__ void operator()(int k, T y) const
    {
        if constexpr (FLAGS) {
            if (a.flags & F_POST_REV) k = a.n - 1 - k;
            if ((a.flags & F_POST_ALT) && (k & 1)) y = -y;
            if (a.flags & F_WEIGHTS) {
                if (k == 0) y = y * a.postw0;
                if (k == a.n - 1) y = y * a.postw1;
            }
        }
        gwrite<T>(dst, off + (uint32_t)k * step, y * sc);
    }
};

constexpr int kPostFlags = F_POST_REV | F_POST_ALT | F_WEIGHTS;

// Post-processing of the R2R modes: pairs (or points) q = t, t + TPL, ... of
// the transformed line Z (natural order).
template <typename P, typename T, bool FLAGS, int mode>
__device__ __forceinline__ void post_mode(const StageArgs<T> &a, void *dst, const typename P::V *Z, const typename P::V *tws,
                                          uint32_t off, uint32_t step, int t)
{
    constexpr int M = P::M, TPL = P::TPL;
    const Emit<T, FLAGS> emit{a, dst, off, step, a.scale};
    const int n = a.n;
    const T two = (T)2;
    if constexpr (mode == M_DCT2 || mode == M_DHT || mode == M_DCT1 || mode == M_DST1) {
        const typename P::V *w = tws + a.post0;
        const typename P::V *u = tws + a.post1;
        const T half = (T)0.5;
#pragma unroll 2
        for (int q = t; q <= M / 2; q += TPL) {
            const cpx<T> zq = get<T>(Z + q), zm = get<T>(Z + (q == 0 ? 0 : M - q));
            cpx<T> x0, x1;
            split_pair(zq, zm, get<T>(w + q), x0, x1);
            const bool self = 2 * q == M;
            if constexpr (mode == M_DCT2) {
                // y_k = 2 Re(u_k X_k), y_{n-k} = -2 Im(u_k X_k), n = 2 M
                const cpx<T> c0 = cmul(get<T>(u + q), x0), c1 = cmul(get<T>(u + M - q), x1);
                emit(q, c0.x);
                if (q != 0) emit(n - q, -c0.y);
                if (!self) {
                    emit(M - q, c1.x);
                    if (q != 0) emit(M + q, -c1.y);
                }
            } else if constexpr (mode == M_DHT) {
                x0 = scal(x0, half);
                x1 = scal(x1, half);
                emit(q, x0.x - x0.y);
                if (q != 0) emit(n - q, x0.x + x0.y);
                if (!self) {
                    emit(M - q, x1.x - x1.y);
                    if (q != 0) emit(M + q, x1.x + x1.y);
                }
            } else if constexpr (mode == M_DCT1) {
                emit(q, x0.x * half);
                if (!self) emit(M - q, x1.x * half);
            } else {
                if (q != 0) {
                    emit(q - 1, -x0.y * half);
                    if (!self) emit(M - q - 1, -x1.y * half);
                }
            }
        }
    } else if constexpr (mode == M_DCT3) {
        // reals r_i of conj(Z): output 2 i (i < M) or 2 (n - 1 - i) + 1
#pragma unroll 2
        for (int c = t; c < M; c += TPL) {
            const cpx<T> z = get<T>(Z + c);
            const int i = 2 * c;
            emit(i < M ? 2 * i : 2 * (n - 1 - i) + 1, z.x);
            emit(i + 1 < M ? 2 * i + 2 : 2 * (n - 2 - i) + 1, -z.y);
        }
    } else if constexpr (mode == M_DCT4) {
        const typename P::V *w = tws + a.post0;
#pragma unroll 2
        for (int q = t; q < M; q += TPL) {
            const cpx<T> c = cmul(get<T>(Z + q), get<T>(w + q));
            emit(2 * q, two * c.x);
            emit(n - 1 - 2 * q, -two * c.y);
        }
    } else if constexpr (mode == M_DCT2_ODD || mode == M_DCT4_ODD) {
        const typename P::V *w = tws + a.post0;
#pragma unroll 2
        for (int k = t; k < n; k += TPL) emit(k, two * cmul(get<T>(w + k), get<T>(Z + k)).x);
    } else if constexpr (mode == M_DCT3_ODD) {
#pragma unroll 2
        for (int i = t; i < n; i += TPL) emit(2 * i < n ? 2 * i : 2 * (n - 1 - i) + 1, two * get<T>(Z + i).x);
    } else { // M_DHT_ODD
#pragma unroll 2
        for (int k = t; k < n; k += TPL) {
            const cpx<T> z = get<T>(Z + k);
            emit(k, z.x - z.y);
        }
    }
}

template <typename P, typename T, bool FLAGS>
__device__ __forceinline__ void post_real(const StageArgs<T> &a, void *dst, const typename P::V *Z, const typename P::V *tws,
                                          uint32_t off, uint32_t step, int t)
{
    switch (a.mode) {
    case M_DCT1: return post_mode<P, T, FLAGS, M_DCT1>(a, dst, Z, tws, off, step, t);
    case M_DST1: return post_mode<P, T, FLAGS, M_DST1>(a, dst, Z, tws, off, step, t);
    case M_DCT2: return post_mode<P, T, FLAGS, M_DCT2>(a, dst, Z, tws, off, step, t);
    case M_DCT3: return post_mode<P, T, FLAGS, M_DCT3>(a, dst, Z, tws, off, step, t);
    case M_DCT4: return post_mode<P, T, FLAGS, M_DCT4>(a, dst, Z, tws, off, step, t);
    case M_DCT2_ODD: return post_mode<P, T, FLAGS, M_DCT2_ODD>(a, dst, Z, tws, off, step, t);
    case M_DCT3_ODD: return post_mode<P, T, FLAGS, M_DCT3_ODD>(a, dst, Z, tws, off, step, t);
    case M_DCT4_ODD: return post_mode<P, T, FLAGS, M_DCT4_ODD>(a, dst, Z, tws, off, step, t);
    default: return post_mode<P, T, FLAGS, M_DHT_ODD>(a, dst, Z, tws, off, step, t);
    }
}


// Raw real points 2 i and 2 i + 1 (v0, v1; the second absent past the end of
// an odd line) into the FFT input of an R2R mode, after the alternating sign
// and the end weights on raw points and the reversal. Every mode's input is a
// signed permutation of the line plus zeros, times a factor per point in the
// odd-length cosine modes (tws + pre0); DCT-III's raw line stays in natural
// order for merge_dct3.
template <typename T, int MODE>
__device__ __forceinline__ void scatter_pair(const StageArgs<T> &a, typename Vec2<T>::type *ln,
                                             const typename Vec2<T>::type *tws, int i, T v0, T v1)
{
    const int n = a.n;
    T *lr = reinterpret_cast<T *>(ln);
    int p0 = 2 * i, p1 = 2 * i + 1;
    const bool second = p1 < n;
    if (a.flags & (F_PRE_REV | F_PRE_ALT | F_WEIGHTS)) {
        if (a.flags & F_PRE_ALT) v1 = -v1;
        if (a.flags & F_WEIGHTS) {
            if (p0 == 0) v0 = v0 * a.prew0;
            if (p0 == n - 1) v0 = v0 * a.prew1;
            if (p1 == n - 1) v1 = v1 * a.prew1;
        }
        if (a.flags & F_PRE_REV) {
            p0 = n - 1 - p0;
            p1 = n - 1 - p1;
        }
    }
    auto one = [&](int p, T v) {
        if constexpr (MODE == M_DCT2) { // even points forward, odd points backward
            lr[(p & 1) ? n - 1 - (p >> 1) : (p >> 1)] = v;
        } else if constexpr (MODE == M_DCT4) { // z_j = (x_2j, x_{n-1-2j})
            lr[(p & 1) ? n - p : p] = v;
        } else if constexpr (MODE == M_DST1) { // odd extension, o_0 = o_{n+1} = 0
            lr[p + 1] = v;
            lr[2 * n + 1 - p] = -v;
        } else if constexpr (MODE == M_DCT1) { // even extension
            lr[p] = v;
            if (p != 0 && p != n - 1) lr[2 * (n - 1) - p] = v;
        } else if constexpr (MODE == M_DCT2_ODD) {
            put<T>(ln + ((p & 1) ? n - 1 - (p >> 1) : (p >> 1)), mk(v, (T)0));
        } else if constexpr (MODE == M_DHT_ODD) {
            put<T>(ln + p, mk(v, (T)0));
        } else if constexpr (MODE == M_DCT3_ODD) {
            put<T>(ln + p, scal(get<T>(tws + a.pre0 + p), p == 0 ? v * (T)0.5 : v));
        } else if constexpr (MODE == M_DCT4_ODD) {
            put<T>(ln + p, scal(get<T>(tws + a.pre0 + p), v));
            put<T>(ln + n + p, mk((T)0, (T)0));
        } else { // M_DCT3
            lr[p] = v;
        }
    };
    one(p0, v0);
    if (second) one(p1, v1);
}

// The raw real line of an R2R stage from global memory to its FFT-input
// slots: point pairs i = t, t + TPL, ...
template <typename P, typename T, int MODE>
__device__ __forceinline__ void load_mode(const StageArgs<T> &a, const void *src, typename P::V *ln,
                                          const typename P::V *tws, uint32_t off, int t)
{
    constexpr int TPL = P::TPL, U = 4;
    const uint32_t s1 = (uint32_t)a.ips * (uint32_t)sizeof(T);
    const int np = (a.n + 1) >> 1;
    if (MODE == M_DST1 && t == 0) {
        reinterpret_cast<T *>(ln)[0] = (T)0;
        reinterpret_cast<T *>(ln)[a.n + 1] = (T)0;
    }
#pragma unroll 1
    for (int base = t; base < np; base += TPL * U) {
        cpx<T> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = base + TPL * u;
            const uint32_t o = off + (uint32_t)(2 * i) * s1;
            if (2 * i + 1 < a.n) {
                if (a.ips == 1) v[u] = gread<cpx<T>>(src, o);
                else v[u] = mk(gread<T>(src, o), gread<T>(src, o + s1));
            } else if (i < np) {
                v[u] = mk(gread<T>(src, o), (T)0);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = base + TPL * u;
            if (i < np) scatter_pair<T, MODE>(a, ln, tws, i, v[u].x, v[u].y);
        }
    }
}

template <typename P, typename T>
__device__ __forceinline__ void load_real(const StageArgs<T> &a, const void *src, typename P::V *ln,
                                          const typename P::V *tws, uint32_t off, int t)
{
    switch (a.mode) {
    case M_DCT1: return load_mode<P, T, M_DCT1>(a, src, ln, tws, off, t);
    case M_DST1: return load_mode<P, T, M_DST1>(a, src, ln, tws, off, t);
    case M_DCT2: return load_mode<P, T, M_DCT2>(a, src, ln, tws, off, t);
    case M_DCT3: return load_mode<P, T, M_DCT3>(a, src, ln, tws, off, t);
    case M_DCT4: return load_mode<P, T, M_DCT4>(a, src, ln, tws, off, t);
    case M_DCT2_ODD: return load_mode<P, T, M_DCT2_ODD>(a, src, ln, tws, off, t);
    case M_DCT3_ODD: return load_mode<P, T, M_DCT3_ODD>(a, src, ln, tws, off, t);
    case M_DCT4_ODD: return load_mode<P, T, M_DCT4_ODD>(a, src, ln, tws, off, t);
    default: return load_mode<P, T, M_DHT_ODD>(a, src, ln, tws, off, t);
    }
}

// DCT-III: the raw line y (natural order, n = 2 M reals) -> the conjugated
// half-length input. V_k = exp(i pi k / 2n) (y_k - i y_{n-k}) is the half
// spectrum of the reordered output.
template <typename P, typename T>
__device__ __forceinline__ void merge_dct3(const StageArgs<T> &a, typename P::V *ln, const typename P::V *tws, int t)
{
    constexpr int M = P::M, TPL = P::TPL, N = (M / 2 + 1 + TPL - 1) / TPL;
    const T *lr = reinterpret_cast<const T *>(ln);
    cpx<T> z0[N], z1[N];
#pragma unroll
    for (int b = 0; b < N; ++b) {
        const int q = t + TPL * b;
        if (q <= M / 2) {
            const T yq = lr[q], ym = lr[M - q];
            const T yn = q == 0 ? (T)0 : -lr[2 * M - q], yp = -lr[M + q];
            cpx<T> Va = cmul(get<T>(tws + a.pre0 + q), mk(yq, yn));
            cpx<T> Vb = cmul(get<T>(tws + a.pre0 + M - q), mk(ym, yp));
            if (q == 0) {
                Va.y = (T)0;
                Vb.y = (T)0;
            }
            merge_pair(Va, Vb, get<T>(tws + a.pre1 + q), z0[b], z1[b]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < N; ++b) {
        const int q = t + TPL * b;
        if (q <= M / 2) {
            put<T>(ln + q, z0[b]);
            if (q != 0 && 2 * q != M) put<T>(ln + M - q, z1[b]);
        }
    }
    __syncthreads();
}

} // namespace

// KIND 0: C2C lines; 1: R2C / C2R / DHT lines of even length (the half-length
// transform of real pairs); 2: the other real-to-real modes; 3: C2C pieces of
// long lines (load and store factors, zero padding, crop, split twiddles).
// Lines past the end of the last tile repeat the last line's loads and store
// nothing.
template <typename T, int R0, int R1, int R2, int EM, int KIND>
__global__ __launch_bounds__(kLinePlanThreads) void k_line_plan(const StageArgs<T> a)
{
    using P = LinePlan<T, R0, R1, R2, EM>;
    using V = typename P::V;
    constexpr int M = P::M, TPL = P::TPL, RL = P::RL;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    V *tws = reinterpret_cast<V *>(smem_raw);
    V *data = tws + a.twn;
    if (a.gate != nullptr && *a.gate != 0) return;
    const int tid = threadIdx.x;
    const int lt = a.lt;
    const uint32_t tile0 = (uint32_t)blockIdx.x * (uint32_t)lt;
    const uint32_t nlines = (uint32_t)a.nlines;
    // column side: consecutive lanes on consecutive lines (lt is a power of
    // two); row side: consecutive lanes along a line
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
    if (a.g.nd == 1) {
        // one line digit (local plans, whose batch is only known at the
        // call): offsets relative to the tile, so arrays may exceed 4 GiB
        src = static_cast<const char *>(src) + (int64_t)tile0 * a.g.is[0] * (complex_in(a.mode) ? 2 : 1) * (int64_t)sizeof(T);
        dst = static_cast<char *>(dst) + (int64_t)tile0 * a.g.os[0] * (complex_out(a.mode) ? 2 : 1) * (int64_t)sizeof(T);
        iline -= tile0;
        oline -= tile0;
    }
    const V *twg = reinterpret_cast<const V *>(a.tw);
    auto stage_tables = [&]() {
        for (int i = tid; i < a.twn; i += (int)blockDim.x) tws[i] = twg[i];
    };
    const V *tw1 = tws + a.twoff[1];
    const V *twl = tws + a.twoff[R2 ? 2 : 1];
    const bool cj = (a.flags & F_CONJ_IN) != 0;

    // pieces of long lines: coordinates of the line digit that the factors and
    // full indexes run over (iline, oline may be relative to the tile)
    uint32_t idco = 0, odco = 0;
    if constexpr (KIND == 3) {
        if (a.xdig >= 0) {
            const uint32_t last = nlines - 1;
            idco = line_digit(a.g, tile0 + (uint32_t)il < nlines ? tile0 + (uint32_t)il : last, a.xdig);
            odco = line_digit(a.g, tile0 + (uint32_t)ol < nlines ? tile0 + (uint32_t)ol : last, a.xdig);
        }
    }
    if constexpr (KIND == 3) {
        constexpr int N0 = P::template rounds<R0>(), NB0 = M / R0;
        cpx<T> v[N0][R0];
        const uint32_t st = (uint32_t)a.ips * (uint32_t)(2 * sizeof(T));
        const uint32_t off = line_offset<false>(a.g, iline, 2 * sizeof(T)) + (uint32_t)it * st;
        const bool pad = (a.flags & F_XIN) != 0;
        const uint32_t fmul = (uint32_t)a.xmul_in, f0 = idco + (uint32_t)it * fmul, fend = (uint32_t)a.xvalid_in;
#pragma unroll
        for (int b = 0; b < N0; ++b) {
            if (P::template has<R0>(b, it + TPL * b)) {
#pragma unroll
                for (int r = 0; r < R0; ++r) {
                    const uint32_t p = (uint32_t)(b * TPL + r * NB0);
                    v[b][r] = mk((T)0, (T)0);
                    if (!pad || f0 + p * fmul < fend) v[b][r] = gread<cpx<T>>(src, off + p * st);
                }
            }
        }
        stage_tables();
        if (cj) {
#pragma unroll
            for (int b = 0; b < N0; ++b)
#pragma unroll
                for (int r = 0; r < R0; ++r) v[b][r].y = -v[b][r].y;
        }
        if (pad && a.xtab_in != nullptr) {
#pragma unroll
            for (int b = 0; b < N0; ++b) {
                if (P::template has<R0>(b, it + TPL * b)) {
#pragma unroll
                    for (int r = 0; r < R0; ++r) {
                        const uint32_t f = f0 + (uint32_t)(b * TPL + r * NB0) * fmul;
                        if (f < fend) v[b][r] = cmul(v[b][r], gread<cpx<T>>(a.xtab_in, f * (uint32_t)(2 * sizeof(T))));
                    }
                }
            }
        }
        P::first_store(iln, it, v);
        P::mid(iln, tw1, it);
    } else if constexpr (KIND == 0) {
        constexpr int N0 = P::template rounds<R0>(), NB0 = M / R0;
        cpx<T> v[N0][R0];
        const uint32_t st = (uint32_t)a.ips * (uint32_t)(2 * sizeof(T));
        const uint32_t off = line_offset<false>(a.g, iline, 2 * sizeof(T)) + (uint32_t)it * st;
#pragma unroll
        for (int b = 0; b < N0; ++b) {
            if (P::template has<R0>(b, it + TPL * b)) {
#pragma unroll
                for (int r = 0; r < R0; ++r) v[b][r] = gread<cpx<T>>(src, off + (uint32_t)(b * TPL + r * NB0) * st);
            }
        }
        stage_tables();
        if (cj) {
#pragma unroll
            for (int b = 0; b < N0; ++b)
#pragma unroll
                for (int r = 0; r < R0; ++r) v[b][r].y = -v[b][r].y;
        }
        P::first_store(iln, it, v);
        P::mid(iln, tw1, it);
    } else if constexpr (KIND == 1) {
        if (a.mode == M_C2R) {
            constexpr int N = (M / 2 + 1 + TPL - 1) / TPL;
            cpx<T> x[N], y[N];
            const uint32_t st = (uint32_t)a.ips * (uint32_t)(2 * sizeof(T));
            const uint32_t off = line_offset<false>(a.g, iline, 2 * sizeof(T));
#pragma unroll
            for (int b = 0; b < N; ++b) {
                const int q = it + TPL * b;
                if (q <= M / 2) {
                    x[b] = gread<cpx<T>>(src, off + (uint32_t)q * st);
                    y[b] = gread<cpx<T>>(src, off + (uint32_t)(M - q) * st);
                }
            }
            stage_tables();
            __syncthreads();
            const bool half = (a.flags & F_HERM_HALF) != 0;
#pragma unroll
            for (int b = 0; b < N; ++b) {
                const int q = it + TPL * b;
                if (q <= M / 2) {
                    if (cj) {
                        x[b].y = -x[b].y;
                        y[b].y = -y[b].y;
                    }
                    if (q == 0) { // X_0 and X_M: imaginary parts dropped
                        x[b].y = (T)0;
                        y[b].y = (T)0;
                    } else if (half) { // adjoint weights on interior bins
                        x[b] = scal(x[b], (T)0.5);
                        y[b] = scal(y[b], (T)0.5);
                    }
                    cpx<T> z0, z1;
                    merge_pair(x[b], y[b], get<T>(tws + a.pre0 + q), z0, z1);
                    put<T>(iln + q, z0);
                    if (q != 0 && 2 * q != M) put<T>(iln + M - q, z1);
                }
            }
            __syncthreads();
            P::template first_lds<false>(iln, nullptr, it);
        } else {
            // R2C / DHT: real pairs as the half-length complex input
            constexpr int N0 = P::template rounds<R0>(), NB0 = M / R0;
            cpx<T> v[N0][R0];
            const uint32_t s1 = (uint32_t)a.ips * (uint32_t)sizeof(T), st = 2 * s1;
            const uint32_t off = line_offset<false>(a.g, iline, sizeof(T)) + (uint32_t)it * st;
            if (a.ips == 1) {
#pragma unroll
                for (int b = 0; b < N0; ++b) {
                    if (P::template has<R0>(b, it + TPL * b)) {
#pragma unroll
                        for (int r = 0; r < R0; ++r)
                            v[b][r] = gread<cpx<T>>(src, off + (uint32_t)((b * TPL + r * NB0) * 2 * sizeof(T)));
                    }
                }
            } else {
#pragma unroll
                for (int b = 0; b < N0; ++b) {
                    if (P::template has<R0>(b, it + TPL * b)) {
#pragma unroll
                        for (int r = 0; r < R0; ++r) {
                            const uint32_t o = off + (uint32_t)(b * TPL + r * NB0) * st;
                            v[b][r] = mk(gread<T>(src, o), gread<T>(src, o + s1));
                        }
                    }
                }
            }
            stage_tables();
            P::first_store(iln, it, v);
        }
        P::mid(iln, tw1, it);
    } else {
        // real-to-real modes: raw lines scattered to their FFT-input slots
        const bool pre_tab = a.mode == M_DCT3_ODD || a.mode == M_DCT4_ODD;
        if (pre_tab) {
            stage_tables();
            __syncthreads();
        }
        load_real<P, T>(a, src, iln, tws, line_offset<false>(a.g, iline, sizeof(T)), it);
        if (!pre_tab) stage_tables();
        __syncthreads();
        if (a.mode == M_DCT3) merge_dct3<P, T>(a, iln, tws, it);
        if (a.mode == M_DCT4) P::template first_lds<true>(iln, tws + a.pre0, it);
        else P::template first_lds<false>(iln, nullptr, it);
        P::mid(iln, tw1, it);
    }

    const T sc = a.scale;
    if constexpr (KIND == 3) {
        constexpr int NL = P::template rounds<RL>(), NB = M / RL;
        if (!store) return;
        cpx<T> v[NL][RL];
        P::last(oln, twl, ot, v);
        const uint32_t st = (uint32_t)a.ops * (uint32_t)(2 * sizeof(T));
        const uint32_t off = line_offset<true>(a.g, oline, 2 * sizeof(T)) + (uint32_t)ot * st;
        if (a.flags & F_XTW) {
            // exp(-2 pi i d k / (m n2)), k = j + r NB: neighbouring lines d read
            // neighbouring table entries
            const uint32_t n2 = (uint32_t)(a.xtw_m / M), lo = (1u << a.xtw_bsh) - 1u;
            const V *hi = reinterpret_cast<const V *>(a.xtw) + lo + 1;
#pragma unroll
            for (int b = 0; b < NL; ++b) {
                const int j = ot + TPL * b;
                if (P::template has<RL>(b, j)) {
                    if (a.xtw_full) {
                        const uint32_t w0 = ((uint32_t)j * n2 + odco) * (uint32_t)(2 * sizeof(T));
#pragma unroll
                        for (int r = 0; r < RL; ++r)
                            v[b][r] = cmul(v[b][r], gread<cpx<T>>(a.xtwr, w0 + (uint32_t)(r * NB) * n2 * (uint32_t)(2 * sizeof(T))));
                    } else {
                        const uint32_t q = odco * (uint32_t)j;
                        const cpx<T> w = cmul(get<T>(reinterpret_cast<const V *>(a.xtw) + (q & lo)), get<T>(hi + (q >> a.xtw_bsh)));
                        v[b][0] = cmul(v[b][0], w);
#pragma unroll
                        for (int r = 1; r < RL; ++r)
                            v[b][r] = cmul(v[b][r], cmul(w, gread<cpx<T>>(a.xtwr, ((uint32_t)r * n2 + odco) * (uint32_t)(2 * sizeof(T)))));
                    }
                }
            }
        }
        const T sy = (a.flags & F_CONJ_OUT) ? -sc : sc;
        const bool crop = (a.flags & F_XOUT) != 0;
        const uint32_t fmul = (uint32_t)a.xmul_out, f0 = odco + (uint32_t)ot * fmul, fend = (uint32_t)a.xvalid_out;
#pragma unroll
        for (int b = 0; b < NL; ++b) {
            if (P::template has<RL>(b, ot + TPL * b)) {
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const uint32_t p = (uint32_t)(b * TPL + r * NB), f = f0 + p * fmul;
                    cpx<T> w = mk(v[b][r].x * sc, v[b][r].y * sy);
                    if (crop) {
                        if (f >= fend) continue;
                        if (a.xtab_out != nullptr) w = cmul(w, gread<cpx<T>>(a.xtab_out, f * (uint32_t)(2 * sizeof(T))));
                    }
                    gwrite<cpx<T>>(dst, off + p * st, w);
                }
            }
        }
    } else if constexpr (KIND == 0) {
        constexpr int NL = P::template rounds<RL>(), NB = M / RL;
        if (!store) return;
        cpx<T> v[NL][RL];
        P::last(oln, twl, ot, v);
        const uint32_t st = (uint32_t)a.ops * (uint32_t)(2 * sizeof(T));
        const uint32_t off = line_offset<true>(a.g, oline, 2 * sizeof(T)) + (uint32_t)ot * st;
        const T sy = (a.flags & F_CONJ_OUT) ? -sc : sc;
#pragma unroll
        for (int b = 0; b < NL; ++b) {
            if (P::template has<RL>(b, ot + TPL * b)) {
#pragma unroll
                for (int r = 0; r < RL; ++r)
                    gwrite<cpx<T>>(dst, off + (uint32_t)(b * TPL + r * NB) * st, mk(v[b][r].x * sc, v[b][r].y * sy));
            }
        }
    } else if constexpr (KIND == 1) {
        if (a.mode == M_C2R) {
            constexpr int NL = P::template rounds<RL>(), NB = M / RL;
            if (!store) return;
            cpx<T> v[NL][RL];
            P::last(oln, twl, ot, v);
            const uint32_t s1 = (uint32_t)a.ops * (uint32_t)sizeof(T), st = 2 * s1;
            const uint32_t off = line_offset<true>(a.g, oline, sizeof(T)) + (uint32_t)ot * st;
#pragma unroll
            for (int b = 0; b < NL; ++b) {
                if (P::template has<RL>(b, ot + TPL * b)) {
#pragma unroll
                    for (int r = 0; r < RL; ++r) {
                        const uint32_t o = off + (uint32_t)(b * TPL + r * NB) * st;
                        const cpx<T> w = mk(v[b][r].x * sc, -v[b][r].y * sc);
                        if (a.ops == 1) {
                            gwrite<cpx<T>>(dst, o, w);
                        } else {
                            gwrite<T>(dst, o, w.x);
                            gwrite<T>(dst, o + s1, w.y);
                        }
                    }
                }
            }
        } else {
            P::last_lds(oln, twl, ot);
            if (!store) return;
            if (a.mode == M_R2C) {
                const uint32_t st = (uint32_t)a.ops * (uint32_t)(2 * sizeof(T));
                const uint32_t off = line_offset<true>(a.g, oline, 2 * sizeof(T));
                const V *w = tws + a.post0;
                const T hs = sc * (T)0.5;
                const T inner = (a.flags & F_HERM_DOUBLE) ? sc : hs; // adjoint weights: interior bins doubled
#pragma unroll 2
                for (int q = ot; q <= M / 2; q += TPL) {
                    cpx<T> x0, x1;
                    split_pair(get<T>(oln + q), get<T>(oln + (q == 0 ? 0 : M - q)), get<T>(w + q), x0, x1);
                    if (q == 0) { // DC and Nyquist are exactly real
                        gwrite<cpx<T>>(dst, off, mk(x0.x * hs, (T)0));
                        gwrite<cpx<T>>(dst, off + (uint32_t)M * st, mk(x1.x * hs, (T)0));
                    } else {
                        gwrite<cpx<T>>(dst, off + (uint32_t)q * st, scal(x0, inner));
                        if (2 * q != M) gwrite<cpx<T>>(dst, off + (uint32_t)(M - q) * st, scal(x1, inner));
                    }
                }
            } else {
                const uint32_t st = (uint32_t)a.ops * (uint32_t)sizeof(T);
                post_mode<P, T, false, M_DHT>(a, dst, oln, tws, line_offset<true>(a.g, oline, sizeof(T)), st, ot);
            }
        }
    } else {
        P::last_lds(oln, twl, ot);
        if (!store) return;
        const uint32_t st = (uint32_t)a.ops * (uint32_t)sizeof(T);
        const uint32_t off = line_offset<true>(a.g, oline, sizeof(T));
        if (a.flags & kPostFlags) post_real<P, T, true>(a, dst, oln, tws, off, st, ot);
        else post_real<P, T, false>(a, dst, oln, tws, off, st, ot);
    }
}

namespace {

// Raises a kernel's dynamic LDS limit on this device, once per kernel and
// device (bit d of `done`; devices above 63 set it on every launch).
hipError_t allow_lds(const void *f, std::atomic<uint64_t> &done)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = dev < 64 ? 1ull << dev : 0;
    if (done.load(std::memory_order_relaxed) & bit) return hipSuccess;
    e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_relaxed);
    return e;
}

template <typename T, int R0, int R1, int R2, int EM, int KIND>
hipError_t launch_one(const StageArgs<T> &a, int threads, size_t lds_bytes, int64_t grid, hipStream_t s)
{
    // the shapes the kernel assumes
    if (a.tpl != line_plan_tpl(R0, R1, R2, EM) || threads != a.lt * a.tpl || threads > kLinePlanThreads ||
        a.ls < line_plan_stride(R0, R1, R2) || ((a.in_col || a.out_col) && (a.lt & (a.lt - 1)) != 0))
        return hipErrorInvalidValue;
    static std::atomic<uint64_t> done{0};
    if (lds_bytes > 64 * 1024) {
        const hipError_t e = allow_lds(reinterpret_cast<const void *>(&k_line_plan<T, R0, R1, R2, EM, KIND>), done);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_line_plan<T, R0, R1, R2, EM, KIND>), dim3((unsigned)grid), dim3(threads), lds_bytes, s, a);
    return hipGetLastError();
}

} // namespace

#ifdef PFH_LINE_F64
using LineT = double;
#else
using LineT = float;
#endif

template <>
hipError_t launch_line_plan<LineT, PFH_LINE_KIND>(const StageArgs<LineT> &a, int r0, int r1, int r2, int em, int threads,
                                                  size_t lds_bytes, int64_t grid, hipStream_t s)
{
#define PFH_LINE_CASE(TT, A, B, C, E)                                                                      \
    if constexpr (sizeof(TT) == sizeof(LineT) &&                                                           \
                  (PFH_LINE_KIND != 2 || (A) * (B) * ((C) ? (C) : 1) <= kLinePlanRealMax))                 \
        if (r0 == A && r1 == B && r2 == C && em == E)                                                      \
            return launch_one<LineT, A, B, C, E, PFH_LINE_KIND>(a, threads, lds_bytes, grid, s);
    PFH_FAST_ROUTE_PLANS(PFH_LINE_CASE)
#undef PFH_LINE_CASE
    return hipErrorInvalidValue;
}

} // namespace pfh
