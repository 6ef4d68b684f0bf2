// Launch description of one line stage: a batch of 1D lines, each read from
// one layout, transformed, and written to another layout. The layout change
// is how a route transition (the reference's pack / exchange / unpack,
// crates/pencil-array/src/transpose.rs:1107-1315, or a LocalTransposePlan
// permutation, local_transpose.rs:87-132) is fused into a stage.
#pragma once

#include <cstdint>

#include "pfh_math.hpp"

namespace pfh {

constexpr int kMaxPasses = 12;
constexpr int kMaxDigits = 5;
// Complex values a thread holds in registers during one radix pass: 16 for
// f32, 8 for f64 (same register footprint).
template <typename T>
struct Regs {
    // generic kernel: 8 values per thread and pass (f32 and f64)
    static constexpr int emax = 8;
    static constexpr int unroll = sizeof(T) == 4 ? 16 : 8; // fast kernels: loads / stores in flight per chunk
#ifndef PFH_GUNROLL_F32
#define PFH_GUNROLL_F32 4
#endif
#ifndef PFH_GUNROLL_F64
#define PFH_GUNROLL_F64 4
#endif
    // generic kernel: loads / stores per unrolled chunk
    static constexpr int gunroll = sizeof(T) == 4 ? PFH_GUNROLL_F32 : PFH_GUNROLL_F64;
    static constexpr int max_radix = sizeof(T) == 4 ? 32 : 8;
};
constexpr int kEmax = 8;         // generic kernel values per thread and pass
// Generic kernel budgets. The instantiation with the odd-prime passes gives
// the radix 5 and 7 passes 3 and 2 butterflies per thread and, in f32, the
// radix 11 / 13 passes 2 and the pre-processing 16 values per thread, so a
// line of 5 x 7 x 11 points takes 32 threads (f32) or 64 (f64) instead of 128; f64
// keeps the smaller budgets, whose registers would spill.
constexpr int generic_pre_e(bool wide, bool f32) { return (wide && f32) ? 16 : kEmax; }

constexpr int generic_mb(int R, bool wide, bool f32)
{
    if (wide && R == 5) return 3;
    if (wide && R == 7) return 2;
    if (wide && f32 && (R == 11 || R == 13)) return 2;
    return kEmax / R > 0 ? kEmax / R : 1;
}
constexpr int kMaxThreadsWide = 512; // generic kernel with the odd-prime passes
constexpr int kMaxThreads = 1024;

// Per-line transform applied by a stage (see pfh_kernels.hip for the math).
enum StageMode : int {
    M_COPY_C = 0,  // identity on complex values (layout change only)
    M_COPY_R,      // identity on real values
    M_C2C,         // complex FFT of length n
    M_R2C,         // real n (even) -> n/2+1 complex via the n/2 complex FFT
    M_R2C_ODD,     // real n (odd) -> (n+1)/2 complex via the n complex FFT
    M_C2R,         // n/2+1 complex -> real n (even), positive sign
    M_C2R_ODD,     // (n+1)/2 complex -> real n (odd)
    M_DCT2,        // REDFT10, n even (Makhoul reorder + n/2 complex FFT)
    M_DCT2_ODD,    // REDFT10, n odd (n complex FFT)
    M_DCT3,        // REDFT01, n even (transpose of M_DCT2)
    M_DCT3_ODD,    // REDFT01, n odd
    M_DCT4,        // REDFT11, n even (n/2 complex FFT, pre/post twiddle)
    M_DCT4_ODD,    // REDFT11, n odd (2n complex FFT of the twiddled line)
    M_DCT1,        // REDFT00 (even extension, n-1 complex FFT)
    M_DST1,        // RODFT00 (odd extension, n+1 complex FFT)
    M_DHT,         // Hartley, n even (n/2 complex FFT)
    M_DHT_ODD,     // Hartley, n odd (n complex FFT)
    M_COUNT
};

enum StageFlags : int {
    F_CONJ_IN = 1,      // conjugate on load (positive-sign C2C)
    F_CONJ_OUT = 2,     // conjugate on store
    F_PRE_REV = 4,      // read x[n-1-j] (DST-III / DST-IV from DCT-III / DCT-IV)
    F_PRE_ALT = 8,      // read (-1)^j x[j] (DST-II from DCT-II)
    F_POST_REV = 16,    // write y[k] = t[n-1-k]
    F_POST_ALT = 32,    // write y[k] = (-1)^k t[k]
    F_HERM_DOUBLE = 64, // R2C adjoint weights: x2 on interior bins, Im := 0 at DC/Nyquist
    F_HERM_HALF = 128,  // C2R adjoint weights: x1/2 on interior bins
    F_WEIGHTS = 256,    // apply pre/post edge weights (R2R adjoints)
    F_DIRECT_FIRST = 1024, // first radix pass reads global memory into registers
    F_DIRECT_LAST = 2048,  // last radix pass writes global memory from registers (C2C)
    F_NT = 4096,           // stage arrays exceed the last-level cache: non-temporal loads and stores
    // Pieces of a long line (generic kernel, complex lines; see StageArgs::x*):
    F_XIN = 8192,   // points whose full index reaches xvalid_in load as zero; xtab_in factor on load
    F_XOUT = 16384, // points whose full index reaches xvalid_out are not stored; xtab_out factor on store
    F_XTW = 32768,  // twiddle exp(-2 pi i d k / xtw_m) on the store of point k
    F_LINE_PLAN = 65536, // the stage runs on k_line_plan (its radices and em are a line plan)
    F_AXIS_SCALE = 524288, // outputs times the per-axis factors sfac
    F_QUADRATIC = 1048576, // real outputs y as y + quad y^2
    F_LINE_CONV = 262144, // with F_LINE_PLAN: the middle of a split Bluestein convolution (k_line_plan KIND 4)
    F_LINE_BLUE = 131072, // with F_LINE_PLAN: Bluestein inside k_line_blue (the plan's length M >= 2 m - 1)
};

struct LineGeom {
    int nd;                       // number of line digits
    int64_t ext[kMaxDigits];      // digit extents, digit 0 fastest
    int64_t is[kMaxDigits];       // input element stride of each digit
    int64_t os[kMaxDigits];       // output element stride of each digit
    uint32_t dmag[kMaxDigits];    // invariant-divisor constants of ext (make_fastdiv)
    int dsh[kMaxDigits];
};

// Exact quotient x / d for 0 <= x < 2^31 and an invariant 1 <= d < 2^31
// without a division: q = (x + mulhi(x, mag)) >> sh with sh = ceil(log2 d)
// and mag = floor(2^32 (2^sh - d) / d) + 1, the round-up method of
// Granlund and Montgomery (PLDI 1994, section 4). x + mulhi(x, mag) < 2^32
// because mag < 2^32 and x < 2^31.
struct FastDiv {
    uint32_t mag;
    int sh;
};

inline FastDiv make_fastdiv(uint32_t d)
{
    int sh = 0;
    while ((1ull << sh) < d) ++sh;
    FastDiv f;
    f.mag = (uint32_t)(((1ull << 32) * ((1ull << sh) - d)) / d + 1);
    f.sh = sh;
    return f;
}

__host__ __device__ __forceinline__ uint32_t fastdiv(uint32_t x, uint32_t mag, int sh)
{
    return (x + (uint32_t)(((uint64_t)x * mag) >> 32)) >> sh;
}

template <typename T>
struct StageArgs {
    const void *src;
    void *dst;
    const cpx<T> *tw;       // this stage's twiddle / pre / post tables
    const int *gate;        // if non-null and *gate != 0 the stage writes nothing
    int64_t nlines;
    int64_t ntiles;
    LineGeom g;
    int64_t ips, ops;       // point strides of the transform axis (elements)
    int mode, flags;
    int n;                  // logical line length
    int nin, nout;          // elements per line read / written
    int m;                  // complex FFT length (0: no FFT)
    int npass;
    int radix[kMaxPasses];
    int twoff[kMaxPasses];  // pass twiddle offsets (complex units) into tw
    uint32_t nsmag[kMaxPasses]; // make_fastdiv constants of each pass's Ns (product of the earlier radices)
    int nssh[kMaxPasses];
    int pre0, pre1, post0, post1; // table offsets into tw
    int twn;                // complex entries of tw staged into LDS
    int fem;                // values per thread and pass of the compile-time plan (0: generic kernel)
    int lt, tpl;            // lines per tile, threads per line
    int lc;                 // lines computed at a time (lc * tpl threads; lt is a multiple of lc)
    int ls;                 // LDS stride of one line (complex units)
    int in_col, out_col;    // column (lines adjacent in memory) access on load / store
    int xcd_per;            // consecutive tiles that go to one XCD (tile_of_block; 0: no grouping)
    T scale;
    T prew0, prew1, postw0, postw1;
    // Pieces of a long line (F_XIN / F_XOUT / F_XTW): a line too long for one
    // workgroup runs as several launches. d is the coordinate of line digit
    // xdig (0 when xdig < 0), and point p of a line stands for the index
    // p * xmul + d of the long line.
    const cpx<T> *xtab_in;  // factor of full index f on load (null: none)
    const cpx<T> *xtab_out; // factor of full index f on store (null: none)
    const cpx<T> *xtw;      // exp(-2 pi i q / xtw_m) = xtw[q mod 2^xtw_bsh] * xtw[2^xtw_bsh + (q >> xtw_bsh)]
    int xdig;
    int xmul_in, xmul_out;
    int xvalid_in, xvalid_out;
    int xtw_m, xtw_bsh;
    // k_line_plan: the split's twiddles in one table, exp(-2 pi i d k / xtw_m) at [k][d], d < n2 = xtw_m / m
    // (xtw_full; a longer split takes the two-level table)
    const cpx<T> *xtwr;
    int xtw_full;
    // Pointwise steps in the last stage's store (k_line_plan KIND 5 and 6).
    const T *sfac;          // per-axis factors (F_AXIS_SCALE): point k's at sfac_pt + k, digit d's at sfac_dig[d] + coordinate
    int sfac_pt, sfac_dig[kMaxDigits]; // (sfac_dig < 0: no factor)
    // the order of the products is launch_scale_axes': ascending output strides. Rank of each digit among the
    // digits, and how many of them come before the point
    int sfac_rank[kMaxDigits], sfac_pre;
    T quad;                 // y + quad y^2 (F_QUADRATIC)
};

// Tile of a workgroup: workgroup b runs on XCD b mod 8; with xcd_per = G > 0
// each XCD takes G consecutive tiles of every 8 G (the grid is a multiple of
// 8 G; tiles past the end do nothing).
template <typename T>
__host__ __device__ __forceinline__ uint32_t tile_of_block(const StageArgs<T> &a, uint32_t b)
{
    if (a.xcd_per <= 0) return b;
    const uint32_t G = (uint32_t)a.xcd_per, g = b / (8u * G), r = b - g * (8u * G);
    return (g * 8u + (r & 7u)) * G + (r >> 3);
}

// Pre- and post-processing of a long real line (k_long_prep / k_long_post,
// pfh_long.hip): the transform runs as a complex FFT of length m of the
// promoted line (real part, zero imaginary part, or the even / odd
// extension), whose input the prep kernel writes and whose output the post
// kernel reads, line-major (line l at l * m).
enum LongKind : int { LK_R2C = 0, LK_C2R, LK_DCT2, LK_DCT3, LK_DCT4, LK_DCT1, LK_DST1, LK_DHT };

template <typename T>
struct LongArgs {
    const void *src;
    void *dst;
    const cpx<T> *tab;   // plan tables (pre0 / post0 offsets)
    const int *gate;     // if non-null and *gate != 0 nothing is written
    int64_t nlines;
    LineGeom g;          // the stage's lines: is = input strides, os = output strides
    int64_t ips, ops;    // point strides of the stage's input / output
    int kind, flags;     // LongKind, stage flags (F_PRE_* / F_POST_* / F_WEIGHTS / F_HERM_*)
    int n;               // logical line length
    int m;               // promoted complex FFT length
    int nout;            // output points per line (post)
    int pre0, post0;     // table offsets
    T scale, prew0, prew1, postw0, postw1;
};

// Two route stages fused over whole planes (k_plane_batch): a plane of nc
// rows of nr contiguous elements is loaded into LDS, every row is
// transformed (first FFT axis, length nr), then every column (second axis,
// length nc), and the plane is written with the second axis contiguous
// (column c at c * nc). Planes of one item lie back to back (plane p at
// p * nr * nc in both arrays).
template <typename T>
struct PlaneArgs {
    const void *src;
    void *dst;
    const cpx<T> *tw_row;   // pass twiddles of the row FFT's plan (offsets twoff_row)
    const cpx<T> *tw_col;   // and of the column FFT's plan
    int64_t nplanes;
    int nr, nc;             // row length (first FFT), rows (second FFT length)
    int twn_row, twn_col;   // table entries staged into LDS
    int twoff_row[3], twoff_col[3];
    int rr[3], rem;         // compile-time plan of the rows (radices, values per thread)
    int cr[3], cem;         // and of the columns
    int tpl_r, tpl_c;       // threads per row / column line
    int rs;                 // LDS stride of a row (complex units, odd)
    int flags;              // F_CONJ_IN (rows' load), F_CONJ_OUT (columns' store)
    T scale;                // applied at the store
};

// Line plans {R0, R1, R2, EM}: the radix sequence and the values per thread
// and pass of the route stages that k_line_plan runs (pfh_line.hip): every
// length 2^a 3^b 5^c 7^d from 8 to 1024 that two or three radices of 2 to 10, 12,
// 14, 15 and 16 reach, and 385 = 5 x 7 x 11, the FFT of a DST-I line of 384 points,
// which has had a plan of its own from the start. The rule of the table, of
// all radix sequences and EM from the largest radix to 16 (8 below 64 points, so
// that a wave still covers long runs): the least sum over the passes of rounds x
// threads x (instructions of the radix-R butterfly + 14 R for the LDS exchange),
// idle lanes of partial rounds so included, times 1 + 0.002 EM, 1.03 above 32
// threads a line and 1.2 above 64; butterflies of 2 3 4 5 7 8 9 11 16 count 4 16 16 36
// 66 56 136 150 170 lane instructions, the composite ones B ops(A) + A ops(B). The
// variants with EM = R0 (line_plan_real_only) stand beside the plans of 65 to 128
// points that have at most 8 threads a line. tests/test_line_plan_table.py derives
// the table from this.
#define PFH_FAST_ROUTE_PLANS(X) \
    X(float, 2, 4, 0, 4)       \
    X(float, 3, 3, 0, 3)       \
    X(float, 2, 5, 0, 6)       \
    X(float, 2, 6, 0, 6)       \
    X(float, 2, 7, 0, 8)       \
    X(float, 3, 5, 0, 6)       \
    X(float, 4, 4, 0, 4)       \
    X(float, 3, 6, 0, 6)       \
    X(float, 4, 5, 0, 5)       \
    X(float, 3, 7, 0, 7)       \
    X(float, 4, 6, 0, 8)       \
    X(float, 5, 5, 0, 5)       \
    X(float, 3, 3, 3, 3)       \
    X(float, 4, 7, 0, 8)       \
    X(float, 5, 6, 0, 6)       \
    X(float, 4, 8, 0, 8)       \
    X(float, 5, 7, 0, 7)       \
    X(float, 6, 6, 0, 6)       \
    X(float, 5, 8, 0, 8)       \
    X(float, 6, 7, 0, 7)       \
    X(float, 3, 3, 5, 6)       \
    X(float, 6, 8, 0, 8)       \
    X(float, 7, 7, 0, 7)       \
    X(float, 2, 5, 5, 6)       \
    X(float, 3, 3, 6, 6)       \
    X(float, 7, 8, 0, 8)       \
    X(float, 2, 5, 6, 6)       \
    X(float, 3, 3, 7, 7)       \
    X(float, 8, 8, 0, 8)       \
    X(float, 5, 14, 0, 15)     \
    X(float, 6, 12, 0, 12)     \
    X(float, 5, 15, 0, 15)     \
    X(float, 8, 10, 0, 10)     \
    X(float, 9, 9, 0, 9)       \
    X(float, 7, 12, 0, 14)     \
    X(float, 9, 10, 0, 10)     \
    X(float, 8, 12, 0, 16)     \
    X(float, 7, 14, 0, 14)     \
    X(float, 10, 10, 0, 10)    \
    X(float, 7, 15, 0, 15)     \
    X(float, 9, 12, 0, 12)     \
    X(float, 8, 14, 0, 16)     \
    X(float, 8, 15, 0, 16)     \
    X(float, 5, 5, 5, 5)       \
    X(float, 3, 3, 14, 15)     \
    X(float, 8, 16, 0, 16)     \
    X(float, 3, 3, 15, 15)     \
    X(float, 10, 14, 0, 14)    \
    X(float, 12, 12, 0, 12)    \
    X(float, 3, 7, 7, 15)      \
    X(float, 10, 15, 0, 15)    \
    X(float, 10, 16, 0, 16)    \
    X(float, 2, 9, 9, 10)      \
    X(float, 12, 14, 0, 14)    \
    X(float, 5, 5, 7, 15)      \
    X(float, 12, 15, 0, 15)    \
    X(float, 3, 7, 9, 9)       \
    X(float, 12, 16, 0, 16)    \
    X(float, 14, 14, 0, 14)    \
    X(float, 2, 10, 10, 10)    \
    X(float, 14, 15, 0, 15)    \
    X(float, 3, 6, 12, 12)     \
    X(float, 14, 16, 0, 16)    \
    X(float, 15, 15, 0, 15)    \
    X(float, 15, 16, 0, 16)    \
    X(float, 3, 9, 9, 9)       \
    X(float, 5, 7, 7, 15)      \
    X(float, 5, 5, 10, 10)     \
    X(float, 3, 7, 12, 14)     \
    X(float, 16, 16, 0, 16)    \
    X(float, 3, 9, 10, 10)     \
    X(float, 4, 5, 14, 16)     \
    X(float, 2, 12, 12, 12)    \
    X(float, 3, 7, 14, 15)     \
    X(float, 4, 5, 15, 16)     \
    X(float, 3, 7, 15, 15)     \
    X(float, 5, 8, 8, 16)      \
    X(float, 3, 9, 12, 12)     \
    X(float, 4, 7, 12, 14)     \
    X(float, 7, 7, 7, 7)       \
    X(float, 5, 5, 14, 15)     \
    X(float, 3, 8, 15, 16)     \
    X(float, 5, 5, 15, 15)     \
    X(float, 3, 9, 14, 14)     \
    X(float, 3, 8, 16, 16)     \
    X(float, 5, 7, 11, 14)     \
    X(float, 2, 14, 14, 14)    \
    X(float, 4, 10, 10, 12)    \
    X(float, 5, 9, 9, 10)      \
    X(float, 2, 14, 15, 15)    \
    X(float, 3, 12, 12, 12)    \
    X(float, 7, 7, 9, 9)       \
    X(float, 2, 14, 16, 16)    \
    X(float, 2, 15, 15, 16)    \
    X(float, 4, 8, 15, 16)     \
    X(float, 6, 9, 9, 12)      \
    X(float, 5, 7, 14, 15)     \
    X(float, 5, 10, 10, 10)    \
    X(float, 6, 7, 12, 14)     \
    X(float, 8, 8, 8, 16)      \
    X(float, 5, 7, 15, 15)     \
    X(float, 3, 12, 15, 15)    \
    X(float, 5, 8, 14, 16)     \
    X(float, 7, 9, 9, 14)      \
    X(float, 4, 12, 12, 12)    \
    X(float, 3, 14, 14, 15)    \
    X(float, 5, 8, 15, 16)     \
    X(float, 3, 14, 15, 15)    \
    X(float, 5, 8, 16, 16)     \
    X(float, 8, 9, 9, 9)       \
    X(float, 4, 12, 14, 14)    \
    X(float, 3, 15, 15, 15)    \
    X(float, 7, 7, 14, 14)     \
    X(float, 7, 10, 10, 14)    \
    X(float, 3, 15, 16, 16)    \
    X(float, 9, 9, 9, 9)       \
    X(float, 7, 7, 15, 15)     \
    X(float, 5, 10, 15, 15)    \
    X(float, 7, 9, 12, 14)     \
    X(float, 3, 16, 16, 16)    \
    X(float, 4, 14, 14, 16)    \
    X(float, 8, 10, 10, 10)    \
    X(float, 9, 9, 10, 10)     \
    X(float, 4, 14, 15, 16)    \
    X(float, 6, 12, 12, 12)    \
    X(float, 7, 9, 14, 14)     \
    X(float, 8, 8, 14, 16)     \
    X(float, 4, 15, 15, 16)    \
    X(float, 7, 9, 15, 15)     \
    X(float, 8, 8, 15, 16)     \
    X(float, 9, 9, 12, 12)     \
    X(float, 5, 14, 14, 15)    \
    X(float, 10, 10, 10, 10)   \
    X(float, 7, 12, 12, 14)    \
    X(float, 8, 8, 16, 16)     \
    X(double, 2, 4, 0, 4)      \
    X(double, 3, 3, 0, 3)      \
    X(double, 2, 5, 0, 6)      \
    X(double, 2, 6, 0, 6)      \
    X(double, 2, 7, 0, 8)      \
    X(double, 3, 5, 0, 6)      \
    X(double, 4, 4, 0, 4)      \
    X(double, 3, 6, 0, 6)      \
    X(double, 4, 5, 0, 5)      \
    X(double, 3, 7, 0, 7)      \
    X(double, 4, 6, 0, 8)      \
    X(double, 5, 5, 0, 5)      \
    X(double, 3, 3, 3, 3)      \
    X(double, 4, 7, 0, 8)      \
    X(double, 5, 6, 0, 6)      \
    X(double, 4, 8, 0, 8)      \
    X(double, 5, 7, 0, 7)      \
    X(double, 6, 6, 0, 6)      \
    X(double, 5, 8, 0, 8)      \
    X(double, 6, 7, 0, 7)      \
    X(double, 3, 3, 5, 6)      \
    X(double, 6, 8, 0, 8)      \
    X(double, 7, 7, 0, 7)      \
    X(double, 2, 5, 5, 6)      \
    X(double, 3, 3, 6, 6)      \
    X(double, 7, 8, 0, 8)      \
    X(double, 2, 5, 6, 6)      \
    X(double, 3, 3, 7, 7)      \
    X(double, 8, 8, 0, 8)      \
    X(double, 5, 14, 0, 15)    \
    X(double, 6, 12, 0, 12)    \
    X(double, 5, 15, 0, 15)    \
    X(double, 8, 10, 0, 10)    \
    X(double, 9, 9, 0, 9)      \
    X(double, 7, 12, 0, 14)    \
    X(double, 9, 10, 0, 10)    \
    X(double, 8, 12, 0, 16)    \
    X(double, 7, 14, 0, 14)    \
    X(double, 10, 10, 0, 10)   \
    X(double, 7, 15, 0, 15)    \
    X(double, 9, 12, 0, 12)    \
    X(double, 8, 14, 0, 16)    \
    X(double, 8, 15, 0, 16)    \
    X(double, 5, 5, 5, 5)      \
    X(double, 3, 3, 14, 15)    \
    X(double, 8, 16, 0, 16)    \
    X(double, 3, 3, 15, 15)    \
    X(double, 10, 14, 0, 14)   \
    X(double, 12, 12, 0, 12)   \
    X(double, 3, 7, 7, 15)     \
    X(double, 10, 15, 0, 15)   \
    X(double, 10, 16, 0, 16)   \
    X(double, 2, 9, 9, 10)     \
    X(double, 12, 14, 0, 14)   \
    X(double, 5, 5, 7, 15)     \
    X(double, 12, 15, 0, 15)   \
    X(double, 3, 7, 9, 9)      \
    X(double, 12, 16, 0, 16)   \
    X(double, 14, 14, 0, 14)   \
    X(double, 2, 10, 10, 10)   \
    X(double, 14, 15, 0, 15)   \
    X(double, 3, 6, 12, 12)    \
    X(double, 14, 16, 0, 16)   \
    X(double, 15, 15, 0, 15)   \
    X(double, 15, 16, 0, 16)   \
    X(double, 3, 9, 9, 9)      \
    X(double, 5, 7, 7, 15)     \
    X(double, 5, 5, 10, 10)    \
    X(double, 3, 7, 12, 14)    \
    X(double, 16, 16, 0, 16)   \
    X(double, 3, 9, 10, 10)    \
    X(double, 4, 5, 14, 16)    \
    X(double, 2, 12, 12, 12)   \
    X(double, 3, 7, 14, 15)    \
    X(double, 4, 5, 15, 16)    \
    X(double, 3, 7, 15, 15)    \
    X(double, 5, 8, 8, 16)     \
    X(double, 3, 9, 12, 12)    \
    X(double, 4, 7, 12, 14)    \
    X(double, 7, 7, 7, 7)      \
    X(double, 5, 5, 14, 15)    \
    X(double, 3, 8, 15, 16)    \
    X(double, 5, 5, 15, 15)    \
    X(double, 3, 9, 14, 14)    \
    X(double, 3, 8, 16, 16)    \
    X(double, 5, 7, 11, 14)    \
    X(double, 2, 14, 14, 14)   \
    X(double, 4, 10, 10, 12)   \
    X(double, 5, 9, 9, 10)     \
    X(double, 2, 14, 15, 15)   \
    X(double, 3, 12, 12, 12)   \
    X(double, 7, 7, 9, 9)      \
    X(double, 2, 14, 16, 16)   \
    X(double, 2, 15, 15, 16)   \
    X(double, 4, 8, 15, 16)    \
    X(double, 6, 9, 9, 12)     \
    X(double, 5, 7, 14, 15)    \
    X(double, 5, 10, 10, 10)   \
    X(double, 6, 7, 12, 14)    \
    X(double, 8, 8, 8, 16)     \
    X(double, 5, 7, 15, 15)    \
    X(double, 3, 12, 15, 15)   \
    X(double, 5, 8, 14, 16)    \
    X(double, 7, 9, 9, 14)     \
    X(double, 4, 12, 12, 12)   \
    X(double, 3, 14, 14, 15)   \
    X(double, 5, 8, 15, 16)    \
    X(double, 3, 14, 15, 15)   \
    X(double, 5, 8, 16, 16)    \
    X(double, 8, 9, 9, 9)      \
    X(double, 4, 12, 14, 14)   \
    X(double, 3, 15, 15, 15)   \
    X(double, 7, 7, 14, 14)    \
    X(double, 7, 10, 10, 14)   \
    X(double, 3, 15, 16, 16)   \
    X(double, 9, 9, 9, 9)      \
    X(double, 7, 7, 15, 15)    \
    X(double, 5, 10, 15, 15)   \
    X(double, 7, 9, 12, 14)    \
    X(double, 3, 16, 16, 16)   \
    X(double, 4, 14, 14, 16)   \
    X(double, 8, 10, 10, 10)   \
    X(double, 9, 9, 10, 10)    \
    X(double, 4, 14, 15, 16)   \
    X(double, 6, 12, 12, 12)   \
    X(double, 7, 9, 14, 14)    \
    X(double, 8, 8, 14, 16)    \
    X(double, 4, 15, 15, 16)   \
    X(double, 7, 9, 15, 15)    \
    X(double, 8, 8, 15, 16)    \
    X(double, 9, 9, 12, 12)    \
    X(double, 5, 14, 14, 15)   \
    X(double, 10, 10, 10, 10)  \
    X(double, 7, 12, 12, 14)   \
    X(double, 8, 8, 16, 16)      \
    X(float, 6, 12, 0, 6)        \
    X(float, 5, 14, 0, 5)        \
    X(float, 5, 15, 0, 5)        \
    X(float, 7, 12, 0, 7)        \
    X(float, 8, 12, 0, 8)        \
    X(float, 7, 14, 0, 7)        \
    X(float, 7, 15, 0, 7)        \
    X(float, 8, 14, 0, 8)        \
    X(float, 8, 15, 0, 8)        \
    X(float, 8, 16, 0, 8)        \
    X(double, 6, 12, 0, 6)       \
    X(double, 5, 14, 0, 5)       \
    X(double, 5, 15, 0, 5)       \
    X(double, 7, 12, 0, 7)       \
    X(double, 8, 12, 0, 8)       \
    X(double, 7, 14, 0, 7)       \
    X(double, 7, 15, 0, 7)       \
    X(double, 8, 14, 0, 8)       \
    X(double, 8, 15, 0, 8)       \
    X(double, 8, 16, 0, 8)

// Plans of k_line_fast and the batched kernels: {R0, R1, R2, EM}.
#define PFH_FAST_PLANS(X)      \
    X(float, 8, 8, 0, 16)      \
    X(float, 8, 16, 0, 16)     \
    X(float, 16, 16, 0, 16)    \
    X(float, 16, 32, 0, 16)    \
    X(float, 16, 32, 0, 32)    \
    X(float, 8, 8, 8, 16)      \
    X(float, 32, 32, 0, 32)    \
    X(float, 16, 3, 0, 16)     \
    X(float, 4, 3, 5, 16)      \
    X(float, 16, 5, 0, 16)     \
    X(float, 4, 3, 7, 16)      \
    X(float, 8, 4, 3, 16)      \
    X(float, 16, 7, 0, 16)     \
    X(float, 8, 3, 5, 16)      \
    X(float, 8, 4, 5, 16)      \
    X(float, 16, 4, 3, 16)     \
    X(float, 16, 3, 5, 16)     \
    X(float, 16, 4, 5, 16)     \
    X(float, 16, 8, 3, 16)     \
    X(double, 8, 8, 0, 8)      \
    X(double, 4, 4, 8, 8)      \
    X(double, 4, 8, 8, 8)      \
    X(double, 8, 8, 8, 8)

// Threads of a plane-stage workgroup (the kernel's launch bound).
#ifndef PFH_PLANE_THREADS
#define PFH_PLANE_THREADS 1024
#endif
constexpr int kPlaneThreads = PFH_PLANE_THREADS;

// Compile-time plans the plane stage dispatches on (f32, 16 values per
// thread; lengths up to 384, longer lines do not leave room for a plane).
#define PFH_PLANE_PLANS(X)     \
    X(float, 8, 8, 0, 16)      \
    X(float, 8, 16, 0, 16)     \
    X(float, 16, 16, 0, 16)    \
    X(float, 16, 3, 0, 16)     \
    X(float, 4, 3, 5, 16)      \
    X(float, 16, 5, 0, 16)     \
    X(float, 4, 3, 7, 16)      \
    X(float, 8, 4, 3, 16)      \
    X(float, 16, 7, 0, 16)     \
    X(float, 8, 3, 5, 16)      \
    X(float, 8, 4, 5, 16)      \
    X(float, 16, 4, 3, 16)     \
    X(float, 16, 3, 5, 16)     \
    X(float, 16, 4, 5, 16)     \
    X(float, 16, 8, 3, 16)

} // namespace pfh
