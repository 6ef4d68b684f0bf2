// Device code shared by the compile-time line kernels (pfh_line.hip,
// pfh_blue.hip): the radix passes of a line plan in LDS, and the pre- and
// post-processing of real lines around a complex FFT of length m.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>

#include "pfh_kernels.hpp"
#include "pfh_line.hpp"

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

// Post-processing of the real-output modes around an FFT of length M: pairs (or points) q = t, t + TPL, ... of
// the transformed line Z (natural order).
template <typename P, typename T, bool FLAGS, int mode>
__device__ __forceinline__ void post_mode(const StageArgs<T> &a, void *dst, const typename P::V *Z, const typename P::V *tws,
                                          uint32_t off, uint32_t step, int t, const int M)
{
    constexpr int TPL = P::TPL;
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
                                          uint32_t off, uint32_t step, int t, const int M)
{
    switch (a.mode) {
    case M_DCT1: return post_mode<P, T, FLAGS, M_DCT1>(a, dst, Z, tws, off, step, t, M);
    case M_DST1: return post_mode<P, T, FLAGS, M_DST1>(a, dst, Z, tws, off, step, t, M);
    case M_DCT2: return post_mode<P, T, FLAGS, M_DCT2>(a, dst, Z, tws, off, step, t, M);
    case M_DCT3: return post_mode<P, T, FLAGS, M_DCT3>(a, dst, Z, tws, off, step, t, M);
    case M_DCT4: return post_mode<P, T, FLAGS, M_DCT4>(a, dst, Z, tws, off, step, t, M);
    case M_DCT2_ODD: return post_mode<P, T, FLAGS, M_DCT2_ODD>(a, dst, Z, tws, off, step, t, M);
    case M_DCT3_ODD: return post_mode<P, T, FLAGS, M_DCT3_ODD>(a, dst, Z, tws, off, step, t, M);
    case M_DCT4_ODD: return post_mode<P, T, FLAGS, M_DCT4_ODD>(a, dst, Z, tws, off, step, t, M);
    default: return post_mode<P, T, FLAGS, M_DHT_ODD>(a, dst, Z, tws, off, step, t, M);
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
    // (4 pairs in flight: the whole line's 16 at once took 3-6% longer, the
    // registers cost more than the latency)
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
__device__ __forceinline__ void merge_dct3(const StageArgs<T> &a, typename P::V *ln, const typename P::V *tws, int t,
                                           const int M)
{
    constexpr int TPL = P::TPL, N = (P::M / 2 + 1 + TPL - 1) / TPL; // M <= P::M
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

// Raises a kernel's dynamic LDS limit on this device, once per kernel and
// device (bit d of `done`; devices above 63 set it on every launch).
inline hipError_t allow_lds(const void *f, std::atomic<uint64_t> &done)
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

} // namespace

} // namespace pfh
