// Host-only check of a wave tile's operand (WaveIdx, uvt_panel.hpp; built and run
// by tests/test_wave_host.py, no GPU): for both layouts, one and two blocks and
// every count of rows, the 64 lanes' loads of a full panel stay inside the matrix
// as it is stored (a pair of an odd last row reaches one element past it,
// before the next one), their way through LDS keeps to its slot, aligned, and
// every fragment holds the element it stands for.
#include <stdio.h>

#include <initializer_list>
#include <vector>

#define __host__
#define __device__
#include "uvt_panel.hpp"

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

template <int F, bool KC>
static void operand(int nx, int k0, int kmax)
{
    using I = WaveIdx<F, KC>;
    const int ld = KC ? kmax : nx;  // the tightest the matrix can be stored
    std::vector<double> mem((size_t)nx * kmax);
    auto value = [](int x, int k) { return 1000.0 * x + k; };
    for (int x = 0; x < nx; ++x)
        for (int k = 0; k < kmax; ++k) mem[KC ? x * ld + k : k * ld + x] = value(x, k);
    const int slot = 16 * F * I::PITCH;
    std::vector<double> lds(slot, -1.0);
    double r[64][4 * F], v[64][F][4];
    for (int lane = 0; lane < 64; ++lane)
        for (int q = 0; q < I::LOADS; ++q) {
            const int x = I::load_x(q, lane, nx), k = k0 + I::load_k(q, lane);
            const int at = KC ? x * ld + k : k * ld + x, wide = KC || I::PAIR ? 2 : 1;
            CHECK(x >= 0 && x < nx && k >= k0 && k + (KC ? 1 : 0) < k0 + kTileK, "x %d k %d", x, k);
            for (int h = 0; h < wide; ++h) {
                const bool in = at + h >= 0 && at + h < (int)mem.size();
                CHECK(in, "F %d KC %d nx %d lane %d load %d: %d of %d", F, KC, nx, lane, q, at + h, (int)mem.size());
                r[lane][wide * q + h] = in ? mem[at + h] : -2.0;
            }
        }
    if (KC)
        for (int lane = 0; lane < 64; ++lane)
            for (int q = 0; q < I::LOADS; ++q) {
                const int at = I::lds_write(q, lane);
                CHECK(at >= 0 && at + 1 < slot && at % 2 == 0, "LDS %d", at);
                for (int h = 0; h < 2; ++h) lds[at + h] = r[lane][2 * q + h];
            }
    for (int lane = 0; lane < 64; ++lane)
        for (int f = 0; f < F; ++f) {
            for (int h = 0; KC && h < 2; ++h) {
                const int at = I::lds_read(f, h, lane);
                CHECK(at >= 0 && at + 1 < slot && at % 2 == 0, "LDS %d", at);
                for (int e = 0; e < 2; ++e) v[lane][f][2 * h + e] = lds[at + e];
            }
            for (int s = 0; !KC && s < 4; ++s) v[lane][f][s] = r[lane][I::PAIR ? 2 * s + f : s];
            const int x = I::row(f, lane);
            CHECK(x >= 0 && x < 16 * F, "row %d", x);
            for (int s = 0; s < 4 && x < nx; ++s)
                CHECK(v[lane][f][s] == value(x, k0 + 4 * (lane >> 4) + s), "F %d KC %d nx %d lane %d f %d s %d: %g", F,
                      KC, nx, lane, f, s, v[lane][f][s]);
        }
    // every row of the tile is some lane's
    std::vector<char> seen(16 * F, 0);
    for (int lane = 0; lane < 16; ++lane)
        for (int f = 0; f < F; ++f) seen[I::row(f, lane)]++;
    for (char c : seen) CHECK(c == 1, "row in %d lanes", c);
}

template <int F, bool KC>
static void shapes()
{
    for (int nx = 1; nx <= 16 * F; ++nx)
        for (int k0 : {0, 2, 16, 48})
            // the last full panel: an odd last row's pair stays off the last k row
            for (int more : {0, 5}) operand<F, KC>(nx, k0, k0 + kTileK + (!KC && (nx & 1) ? 1 : 0) + more);
    // 32-bit byte offsets wherever they are said to fit
    using I = WaveIdx<F, KC>;
    CHECK(I::fits(1 << 23), "fits");
    for (int64_t ld = 1; ld < (int64_t)1 << 27; ld += ld < (1 << 23) ? ld : 997)
        for (int lane = 0; lane < 64 && I::fits(ld); ++lane)
            for (int q = 0; q < I::LOADS; ++q) {
                const int64_t x = I::load_x(q, lane, 16 * F), k = I::load_k(q, lane);
                CHECK(8 * (KC ? x * ld + k : k * ld + x) + 16 <= (int64_t)1 << 32, "ld %lld", (long long)ld);
            }
}

int main()
{
    shapes<1, true>();
    shapes<1, false>();
    shapes<2, true>();
    shapes<2, false>();
    if (fails) fprintf(stderr, "%d checks failed\n", fails);
    else printf("ok\n");
    return fails != 0;
}
