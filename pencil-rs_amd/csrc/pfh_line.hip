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
//  - composite radices (6, 9, 10, 12, 14, 15, 16) keep most lengths up to 256 at
//    two passes, one LDS exchange.
// Measured per launch on MI355X, before (generic kernel, or k_line_fast with
// run-time threads per line) and after: 180 x 225 x 200 x 3 f32 R2C, 97 MB in
// and out, 147 / 159 / 176 -> 48 / 37 / 35 us; 256 x 384 x 240 f32, 94 MB in
// and out, DST-I 124 -> 75 us, DCT-II / III 71 / 78 -> 49 us, DCT-IV 75 -> 57
// us; f64 DCT-I of 129 points 41 -> 26 us (32 MB), FFT of 192 points 24 -> 15
// us.
// This file is compiled once per precision and kind (PFH_LINE_F64,
// PFH_LINE_KIND) so that the parts build in parallel.
#include "pfh_line_dev.hpp"

#ifndef PFH_LINE_KIND
#define PFH_LINE_KIND 0
#endif

namespace pfh {

// KIND 0: C2C lines; 1: R2C / C2R / DHT lines of even length (the half-length
// transform of real pairs) and R2C / C2R lines of odd length n = M (the complex
// transform of the real line, half of its outputs or inputs); 2: the other real-to-real modes; 3: C2C pieces of
// long lines (load and store factors, zero padding, crop, split twiddles); 4: the
// middle of a split Bluestein convolution: rows k1 of N2 = M values, FFT, times
// the transformed chirp (xtab_out, [k1][k2]), conjugate, FFT, times the split's
// twiddles (xtwr, [k1][q2]), in place; 5: KIND 0 with outputs times per-axis
// factors; 6: C2R (KIND 1) with outputs y + quad y^2. The two fold a pointwise
// pass over the array into the store: 256^3 f32 on MI355X, 67 MB read and written
// by each, 30 us for the factors, 22 us for the quadratic step (the 20-step
// gradient 13.2 -> 11.2 ms).
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
    const uint32_t tile0 = tile_of_block(a, blockIdx.x) * (uint32_t)lt;
    const uint32_t nlines = (uint32_t)a.nlines;
    if (tile0 >= nlines) return;
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
    if constexpr (KIND == 3 || KIND == 4) {
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
    } else if constexpr (KIND == 0 || KIND == 4 || KIND == 5) {
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
    } else if constexpr (KIND == 1 || KIND == 6) {
        const bool odd = (M & 1) && a.n == M;
        if (odd && a.mode == M_C2R) {
            if constexpr ((M & 1) != 0) {
                // X_j and its conjugate at n - j, conjugated for the positive sign
                constexpr int N = (M / 2 + 1 + TPL - 1) / TPL;
                cpx<T> x[N];
                const uint32_t st = (uint32_t)a.ips * (uint32_t)(2 * sizeof(T));
                const uint32_t off = line_offset<false>(a.g, iline, 2 * sizeof(T));
#pragma unroll
                for (int b = 0; b < N; ++b) {
                    const int q = it + TPL * b;
                    if (q <= M / 2) x[b] = gread<cpx<T>>(src, off + (uint32_t)q * st);
                }
                stage_tables();
                const bool half = (a.flags & F_HERM_HALF) != 0;
#pragma unroll
                for (int b = 0; b < N; ++b) {
                    const int q = it + TPL * b;
                    if (q <= M / 2) {
                        if (cj) x[b].y = -x[b].y;
                        if (q == 0) x[b].y = (T)0;
                        else if (half) x[b] = scal(x[b], (T)0.5);
                        put<T>(iln + q, conjg(x[b]));
                        if (q != 0) put<T>(iln + M - q, x[b]);
                    }
                }
                __syncthreads();
                P::template first_lds<false>(iln, nullptr, it);
            }
        } else if (odd) {
            if constexpr ((M & 1) != 0) {
                constexpr int N0 = P::template rounds<R0>(), NB0 = M / R0;
                cpx<T> v[N0][R0];
                const uint32_t st = (uint32_t)a.ips * (uint32_t)sizeof(T);
                const uint32_t off = line_offset<false>(a.g, iline, sizeof(T)) + (uint32_t)it * st;
#pragma unroll
                for (int b = 0; b < N0; ++b) {
                    if (P::template has<R0>(b, it + TPL * b)) {
#pragma unroll
                        for (int r = 0; r < R0; ++r)
                            v[b][r] = mk(gread<T>(src, off + (uint32_t)(b * TPL + r * NB0) * st), (T)0);
                    }
                }
                stage_tables();
                P::first_store(iln, it, v);
            }
        } else if (a.mode == M_C2R) {
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
        if (a.mode == M_DCT3) merge_dct3<P, T>(a, iln, tws, it, M);
        if (a.mode == M_DCT4) P::template first_lds<true>(iln, tws + a.pre0, it);
        else P::template first_lds<false>(iln, nullptr, it);
        P::mid(iln, tw1, it);
    }

    const T sc = a.scale;
    if constexpr (KIND == 4) {
        constexpr int NL = P::template rounds<RL>(), NB = M / RL;
        cpx<T> v[NL][RL];
        P::last(iln, twl, it, v);
        __syncthreads();
        const V *bh = reinterpret_cast<const V *>(a.xtab_out) + idco * (uint32_t)M;
        const V *tw = reinterpret_cast<const V *>(a.xtwr) + odco * (uint32_t)M;
#pragma unroll
        for (int b = 0; b < NL; ++b) {
            const int j = it + TPL * b;
            if (P::template has<RL>(b, j)) {
#pragma unroll
                for (int r = 0; r < RL; ++r) put<T>(iln + j + r * NB, conjg(cmul(v[b][r], get<T>(bh + j + r * NB))));
            }
        }
        __syncthreads();
        P::template first_lds<false>(iln, nullptr, it);
        P::mid(iln, tw1, it);
        P::last(oln, twl, ot, v);
        if (!store) return;
        const uint32_t st = (uint32_t)a.ops * (uint32_t)(2 * sizeof(T));
        const uint32_t off = line_offset<true>(a.g, oline, 2 * sizeof(T)) + (uint32_t)ot * st;
#pragma unroll
        for (int b = 0; b < NL; ++b) {
            const int j = ot + TPL * b;
            if (P::template has<RL>(b, j)) {
#pragma unroll
                for (int r = 0; r < RL; ++r)
                    gwrite<cpx<T>>(dst, off + (uint32_t)(b * TPL + r * NB) * st, cmul(v[b][r], get<T>(tw + j + r * NB)));
            }
        }
    } else if constexpr (KIND == 3) {
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
                        const V *two = reinterpret_cast<const V *>(a.xtw);
#pragma unroll
                        for (int r = 0; r < RL; ++r) {
                            const uint32_t q = odco * (uint32_t)(j + r * NB);
                            v[b][r] = cmul(v[b][r], cmul(get<T>(two + (q & lo)), get<T>(hi + (q >> a.xtw_bsh))));
                        }
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
    } else if constexpr (KIND == 5) {
        // the factors multiplied as scale_axes does, in the order of the
        // output's strides (q: the digits' by rank, the first sfac_pre of them
        // before the point's), so that both give the same bits
        constexpr int NL = P::template rounds<RL>(), NB = M / RL;
        if (!store) return;
        cpx<T> v[NL][RL];
        P::last(oln, twl, ot, v);
        T q[kMaxDigits];
#pragma unroll
        for (int r = 0; r < kMaxDigits; ++r) q[r] = (T)1;
        uint32_t x = tile0 + (uint32_t)ol;
#pragma unroll
        for (int d = 0; d < kMaxDigits; ++d) {
            if (d < a.g.nd) {
                const uint32_t y = fastdiv(x, a.g.dmag[d], a.g.dsh[d]);
                if (a.sfac_dig[d] >= 0) {
                    const T f = a.sfac[(uint32_t)a.sfac_dig[d] + x - y * (uint32_t)a.g.ext[d]];
#pragma unroll
                    for (int r = 0; r < kMaxDigits; ++r)
                        if (a.sfac_rank[d] == r) q[r] = f;
                }
                x = y;
            }
        }
        T pre = (T)1;
#pragma unroll
        for (int r = 0; r < kMaxDigits; ++r) {
            if (r < a.sfac_pre) {
                pre *= q[r];
                q[r] = (T)1;
            }
        }
        const uint32_t st = (uint32_t)a.ops * (uint32_t)(2 * sizeof(T));
        const uint32_t off = line_offset<true>(a.g, oline, 2 * sizeof(T)) + (uint32_t)ot * st;
        const T *fp = a.sfac + a.sfac_pt + ot;
        const T sy = (a.flags & F_CONJ_OUT) ? -sc : sc;
#pragma unroll
        for (int b = 0; b < NL; ++b) {
            if (P::template has<RL>(b, ot + TPL * b)) {
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    T f = pre * fp[b * TPL + r * NB];
#pragma unroll
                    for (int d = 0; d < kMaxDigits; ++d)
                        if (d < a.g.nd) f *= q[d];
                    gwrite<cpx<T>>(dst, off + (uint32_t)(b * TPL + r * NB) * st, mk(v[b][r].x * sc * f, v[b][r].y * sy * f));
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
    } else if constexpr (KIND == 1 || KIND == 6) {
        auto fin = [&](T y) {
            y = y * sc;
            // (one fused multiply-add of the rounded y, as k_quadratic computes it)
            if constexpr (KIND == 6) y = fma(a.quad * y, y, y);
            return y;
        };
        if ((M & 1) && a.n == M) {
            if constexpr ((M & 1) != 0) {
                constexpr int NL = P::template rounds<RL>(), NB = M / RL;
                if (!store) return;
                cpx<T> v[NL][RL];
                P::last(oln, twl, ot, v);
                if (a.mode == M_C2R) {
                    const uint32_t st = (uint32_t)a.ops * (uint32_t)sizeof(T);
                    const uint32_t off = line_offset<true>(a.g, oline, sizeof(T)) + (uint32_t)ot * st;
#pragma unroll
                    for (int b = 0; b < NL; ++b) {
                        if (P::template has<RL>(b, ot + TPL * b)) {
#pragma unroll
                            for (int r = 0; r < RL; ++r)
                                gwrite<T>(dst, off + (uint32_t)(b * TPL + r * NB) * st, fin(v[b][r].x));
                        }
                    }
                } else {
                    const uint32_t st = (uint32_t)a.ops * (uint32_t)(2 * sizeof(T));
                    const uint32_t off = line_offset<true>(a.g, oline, 2 * sizeof(T));
                    const T inner = (a.flags & F_HERM_DOUBLE) ? sc * (T)2 : sc; // adjoint weights
#pragma unroll
                    for (int b = 0; b < NL; ++b) {
                        const int j = ot + TPL * b;
                        if (P::template has<RL>(b, j)) {
#pragma unroll
                            for (int r = 0; r < RL; ++r) {
                                const int k = j + r * NB;
                                if (r * NB <= M / 2 && k <= M / 2)
                                    gwrite<cpx<T>>(dst, off + (uint32_t)k * st,
                                                   k == 0 ? mk(v[b][r].x * sc, (T)0) : scal(v[b][r], inner));
                            }
                        }
                    }
                }
            }
        } else if (a.mode == M_C2R) {
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
                        const cpx<T> w = mk(fin(v[b][r].x), fin(-v[b][r].y));
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
                post_mode<P, T, false, M_DHT>(a, dst, oln, tws, line_offset<true>(a.g, oline, sizeof(T)), st, ot, M);
            }
        }
    } else {
        P::last_lds(oln, twl, ot);
        if (!store) return;
        const uint32_t st = (uint32_t)a.ops * (uint32_t)sizeof(T);
        const uint32_t off = line_offset<true>(a.g, oline, sizeof(T));
        if (a.flags & kPostFlags) post_real<P, T, true>(a, dst, oln, tws, off, st, ot, M);
        else post_real<P, T, false>(a, dst, oln, tws, off, st, ot, M);
    }
}

namespace {

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
                  (PFH_LINE_KIND == 2   ? (A) * (B) * ((C) ? (C) : 1) <= kLinePlanRealMax                 \
                   : (PFH_LINE_KIND == 1 || PFH_LINE_KIND == 6) && sizeof(TT) == 8 ? true                \
                                        : !line_plan_real_only(A, B, C, E)))                            \
        if (r0 == A && r1 == B && r2 == C && em == E)                                                      \
            return launch_one<LineT, A, B, C, E, PFH_LINE_KIND>(a, threads, lds_bytes, grid, s);
    PFH_FAST_ROUTE_PLANS(PFH_LINE_CASE)
#undef PFH_LINE_CASE
    return hipErrorInvalidValue;
}

} // namespace pfh
