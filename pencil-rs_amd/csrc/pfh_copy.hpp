// Which layout copies launch_copy_axes (pfh_copy.hip) takes from its callers' own
// kernels. Words of 1 and 2 bytes come from
// k_permute_words, wider ones from the line kernel's copy stage.
//
// Measured on MI355X over extents 2 to 2000 on both sides, 16 to 128 MiB each
// way, time with the caller's kernel over time here, worst and best of what each
// rule takes; what it leaves ran at 0.02 to 1.0 times the caller's speed but for a
// few shapes up to 1.4.
#pragma once

#include <cstdint>

namespace pfh {

constexpr int copy_tile(int word) { return word == 16 ? 32 : 64; }

// A tile costs the same however much of it lies inside the array, so tiles pay
// where a good part of them does. p: points (the destination's fastest axis), l:
// lines (the source's fastest axis).
//  - 1, 2 and 4 bytes from a fifth of the tile on (1.03 to 10): 64 x 12 elements of
//    2 bytes 0.84, 24 x 40 1.73; 2 x 64 0.34.
//  - 8 bytes from three eighths on (1.04 to 7), lines of 256 points and more, which
//    the line kernel holds in LDS a few at a time, from a fifth on: 16 x 64 0.95, 32 x
//    48 1.04, 256 x 16 1.31.
//  - 16 bytes, whole cache lines for the line kernel in a run of 8 lines, only
//    where that kernel is slow: from 768 points on (1000 x 16 1.21, 700 x 300 1.96;
//    256 x 256 0.59), or up to 6 of them, a few bytes a line (1.1 to 2; 8 x 64 0.99).
inline bool copy_tile_pays(int word, int64_t p, int64_t l)
{
    const int64_t t = copy_tile(word);
    const double used = (double)p * (double)l / ((double)((p + t - 1) / t * t) * (double)((l + t - 1) / t * t));
    if (word == 16) return (p >= 768 && used >= 0.4) || (p <= 6 && l >= 32);
    if (word == 8) return used >= 0.375 || (p >= 256 && used >= 0.2);
    return used >= 0.2;
}

// Workgroups of the tile kernel for `rest` planes of p x l elements.
inline int64_t copy_tile_blocks(int word, int64_t p, int64_t l, int64_t rest)
{
    const int64_t t = copy_tile(word);
    return ((p + t - 1) / t) * ((l + t - 1) / t) * rest;
}

// Threads along a row of nw words of the widest kind, and the rows of a
// workgroup of 256.
constexpr int kCopyRows = 8;
inline int copy_row_cols(int64_t nw)
{
    int cols = 1;
    while (cols < 256 && cols < nw) cols *= 2;
    return cols;
}
inline int64_t copy_row_blocks(int64_t rows, int64_t nw)
{
    const int64_t per = (int64_t)(256 / copy_row_cols(nw)) * kCopyRows;
    return (rows + per - 1) / per;
}

// Rows of n words, nw after widening: they pay where a row keeps its lanes
// busy and is long enough for the index arithmetic of its thread.
//  - 1 and 2 bytes: widened rows from 4 words on (1.04 to 8), odd ones where most
//    lanes are busy (7 1.08, 101 1.11; 5 0.85, 33 0.75).
//  - 4 bytes: widened rows from 16 words (64 bytes) on, odd ones from 32 on (1.08 to
//    9; 12 0.97, 17 0.86).
//  - 8 bytes: from 16 words on with most lanes busy, any from 64 on (1.0 to 5; 24
//    words, 12 of 16 lanes, 0.8).
//  - 16 bytes: from 96 on with most lanes busy (0.98 to 2.4; 64 0.81).
inline bool copy_rows_pay(int word, int64_t n, int64_t nw)
{
    const int64_t cols = copy_row_cols(nw);
    const double used = (double)nw / (double)((nw + cols - 1) / cols * cols);
    if (word <= 2) return n >= 4 && (nw < n || used >= 0.78);
    if (word == 4) return n >= 16 && (nw < n || n >= 32);
    if (word == 8) return n >= 16 && (n >= 64 || used >= 0.78);
    return n >= 96 && used >= 0.7;
}

} // namespace pfh
