// uvt_place.hpp -- which tile of a walk each workgroup runs (host and device).
//
// Workgroup i of a launch runs on XCD i % 8, and where all workgroups fit the
// GPU at once, i, i + cus, i + 2 cus, ... run on one compute unit (checked on
// the GPU: 1024 of 1024 workgroups, three launches).  A walk lays `inner`
// tiles of one depth after another, deepest first: tile b is outer row (or
// column) b / inner, inner tile b % inner.  Two permutations of it, both of
// which leave every workgroup as deep a tile as the plain order within a few
// positions:
//
// xcd_band: the inner tiles of every outer one go to the XCDs in runs: XCD 0's
// workgroups take the first, XCD 1's the next, and so on, so an XCD meets
// about the same inner tiles in every outer one and finds their panels in its
// L2.  Left as they come, the inner tiles of a count that is no multiple of 8
// wander over the XCDs, and each L2 holds the whole matrix.  With it (same
// bits): 6000 x 6000 3.11 -> 3.08 ms, 10000 x 4100 6.08 -> 6.01, 7777 x 7777
// 6.87 -> 6.78, 1900 x 2600 163 -> 159 us; counts that are a multiple of 8
// (4096^2, 32768 x 8192) within 0.3 %.  Both together in the BLAS forms: B =
// op(A) B with B 5000 x 1700 926 -> 730 us, 3000 x 2100 361 -> 337, B op(A)
// with B 3000 x 2048 241 -> 233, C 2500 x 2700 x 1000 237 -> 231.
//
// snake: of the workgroups that are resident at once, every second run of
// `cus` is turned round (by groups of 8, which keeps each on its XCD), so a
// compute unit's deep tiles meet shallow ones: 9000 x 500 (1128 tiles, 1024 of
// them resident) 718 -> 673 us, 2048 x 2048 167 -> 136 for the product, 4000 x
// 1000 275 -> 264 by turning a short last run too.
//
// All in 32 bits: a launch has fewer than 2^31 workgroups.
#pragma once

#include <stdint.h>

namespace uvt {

constexpr int kXcds = 8;  // MI355X

// The inner tile for position i of `count` whose first workgroup is `base`: a
// permutation of [0, count).
__host__ __device__ inline int xcd_band(int i, int base, int count)
{
    // XCD (base + i) % 8 has the positions i % 8, i % 8 + 8, ...; the count % 8
    // XCDs from base % 8 on (round the end) have one more than the rest
    const int first = base & (kXcds - 1), x = (first + i) & (kXcds - 1), each = count / kXcds;
    const int end = first + (count & (kXcds - 1));
    const int lo = (x < end ? x : end) - first, hi = x < end - kXcds ? x : end - kXcds;
    return x * each + (lo > 0 ? lo : 0) + (hi > 0 ? hi : 0) + i / kXcds;
}

// The tile for workgroup b of `total` (up to `blocks` resident on each of
// `cus` compute units): a permutation of [0, total) that is its own inverse.
__host__ __device__ inline int snake(int b, int total, int cus, int blocks)
{
    const int end = total < cus * blocks ? total : cus * blocks, run = (int)((unsigned)b / (unsigned)cus);
    if (b >= end || run % 2 == 0) return b;
    const int lo = run * cus, groups = (end - lo < cus ? end - lo : cus) / kXcds, g = (b - lo) / kXcds;
    return g < groups ? lo + (groups - 1 - g) * kXcds + (b - lo) % kXcds : b;
}

// The tile of a walk that workgroup b of `total` (below 2^31) runs.
struct WalkTile {
    int outer, inner;
};
__host__ __device__ inline WalkTile walk_tile(int b, int total, int inner, int cus, int blocks)
{
    const int t = snake(b, total, cus, blocks), outer = (int)((unsigned)t / (unsigned)inner);
    return WalkTile{outer, xcd_band(t - outer * inner, outer * inner, inner)};
}

// The place in a sequence of `count` tiles that workgroup b of a launch with
// 32 resident workgroups on each XCD runs, -1 for none (the launch is padded
// to a multiple of 256): an XCD takes runs of 32 tiles; every second round of
// runs goes the other way, as the sequence falls in depth (5000 x 1500 split
// products 507 us, 519 without), and the last, short round is shared evenly.
__host__ __device__ inline int run_place(int b, int count)
{
    const int x = b % kXcds, round = b / 256, i = b % 256 / kXcds, full = count / 256;
    if (round < full) return (round * kXcds + (round % 2 ? kXcds - 1 - x : x)) * 32 + i;
    const int rest = count % 256, lo = (x * rest + 7) / kXcds, hi = ((x + 1) * rest + 7) / kXcds;
    return lo + i < hi ? full * 256 + lo + i : -1;
}

}  // namespace uvt
