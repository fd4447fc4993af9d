// Host-only check of the placement of a walk's tiles (uvt_place.hpp; built
// and run by tests/test_place_host.py, no GPU): every tile is run by one
// workgroup, an outer row's inner tiles go to the XCDs in runs, and turning
// runs of workgroups round keeps each on its XCD; a sequence dealt out in runs
// gives every XCD as many tiles.
#include <stdio.h>

#include <vector>

#define __host__
#define __device__
#include "uvt_place.hpp"

using namespace uvt;

static int fails = 0;
#define CHECK(c, ...)                                          \
    do {                                                       \
        if (!(c) && ++fails <= 10) {                           \
            fprintf(stderr, "line %d: %s: ", __LINE__, #c);    \
            fprintf(stderr, __VA_ARGS__);                      \
            fprintf(stderr, "\n");                             \
        }                                                      \
    } while (0)

static void band(int base, int count)
{
    std::vector<int> xcd(count, -1);
    for (int i = 0; i < count; ++i) {
        const int t = xcd_band(i, base, count);
        CHECK(t >= 0 && t < count && xcd[t] < 0, "base %d count %d i %d: %d", base, count, i, t);
        if (t >= 0 && t < count) xcd[t] = (int)((base + i) % kXcds);
    }
    for (int t = 1; t < count; ++t)
        CHECK(xcd[t] >= xcd[t - 1], "base %d count %d: tile %d", base, count, t);
}

static void walk(int outer, int inner, int cus, int blocks)
{
    const int total = outer * inner, resident = cus * blocks;
    std::vector<char> seen(total, 0);
    for (int b = 0; b < total; ++b) {
        const int s = snake(b, total, cus, blocks);
        CHECK(s >= 0 && s < total && s % kXcds == b % kXcds && snake(s, total, cus, blocks) == b &&
                  s / cus == b / cus && (b < resident || s == b),
              "total %d cus %d blocks %d: %d -> %d", total, cus, blocks, b, s);
        const WalkTile w = walk_tile(b, total, inner, cus, blocks);
        const bool in = w.outer >= 0 && w.outer < outer && w.inner >= 0 && w.inner < inner;
        CHECK(in && w.outer == s / inner, "%d x %d, b %d", outer, inner, b);
        if (in) {
            char& v = seen[w.outer * inner + w.inner];
            CHECK(!v, "%d x %d: tile %d, %d twice", outer, inner, w.outer, w.inner);
            v = 1;
        }
    }
}

static void runs(int count)
{
    std::vector<int> xcd(count, -1);
    int none = 0, blocks = (count + 255) / 256 * 256, load[kXcds] = {0};
    for (int b = 0; b < blocks; ++b) {
        const int p = run_place(b, count);
        if (p < 0) {
            ++none;
            continue;
        }
        CHECK(p < count && xcd[p] < 0 && p / 256 == b / 256, "%d tiles, b %d: %d", count, b, p);
        if (p < count) xcd[p] = b % kXcds;
        ++load[b % kXcds];
    }
    CHECK(none == blocks - count, "%d tiles, %d workgroups without", count, none);
    for (int x = 0; x < kXcds; ++x)
        CHECK(load[x] == count / kXcds || load[x] == (count + kXcds - 1) / kXcds, "%d tiles, XCD %d: %d", count, x,
              load[x]);
    for (int p = 1; p < count; ++p)
        CHECK(p % 32 == 0 || p >= count / 256 * 256 || xcd[p] == xcd[p - 1], "%d tiles, place %d", count, p);
}

int main()
{
    for (int count = 1; count <= 1100; ++count) runs(count);
    for (int count = 1; count <= 70; ++count)
        for (int base = 0; base < 8; ++base) band(base, count);
    band(0x7FFFFFFF - 65535, 65535);
    for (int outer : {1, 2, 3, 16, 33, 141})
        for (int inner : {1, 2, 7, 8, 9, 31, 32, 47})
            for (int cus : {256, 304, 64, 8})
                for (int blocks : {1, 2, 3, 4}) walk(outer, inner, cus, blocks);
    if (fails) fprintf(stderr, "%d checks failed\n", fails);
    else printf("ok\n");
    return fails != 0;
}
