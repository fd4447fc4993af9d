// Host-only check of what an FP64 tile reads (uvt_panel.hpp; built and run by
// tests/test_panel_host.py, no GPU).  For every operand shape of the tile
// kernels, tile widths, k ranges and triangles:
//   - a full panel reads only elements of the matrix (at most one past a row's
//     end, before the next row), inside [k_lo, k_hi) and, for the rows
//     (columns) the tile holds, strictly inside the triangle (unit: off its
//     diagonal); every pair of the panel is read once, in its own place;
//   - the full panels are one run [f0, f1) of the tile's panels, in the order
//     it runs them (f0 is 0 or 1, the diagonal comes last), and every
//     panel that could be one is, up to one beside the matrix's last k row;
//   - the other panels read each element at a place inside the matrix, the k
//     range's end and the triangle, and at its own place wherever that is one.
#include <stdio.h>

#include <initializer_list>

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

// One operand of X rows (columns), nx of them inside, of a matrix whose k runs
// to kmax; tri: the triangle GE / LE with the tile's first x at x0.
template <int X, int NT, bool KC, bool GE>
static void operand(int x0, int nx, int k_lo, int k_hi, int kmax, bool tri, bool unit)
{
    using I = PanelIdx<X, NT, KC>;
    const int64_t ld = KC ? kmax : x0 + nx;  // the tightest the matrix can be stored
    const int nk = panels(k_lo, k_hi);
    const bool odd = !KC && (nx & 1);
    const FullPanels fp = full_panels<GE>(k_lo, k_hi, tri, unit, x0, x0 + nx - 1, odd);
    CHECK(I::offsets_fit(ld), "%d", (int)ld);
    CHECK(fp.f1 <= nk && (fp.f0 == 0 || fp.f0 == 1), "%d %d of %d", fp.f0, fp.f1, nk);
    for (int p = 0; p < nk; ++p) {
        const int k0 = panel_k0<GE>(k_lo, nk, p);
        const bool full = p >= fp.f0 && p < fp.f1;
        bool could = k0 >= k_lo && k0 + kTileK <= k_hi - odd;
        if (tri && !GE) could = could && k0 + kTileK - 1 < x0 + (unit ? 0 : 1) - odd;
        if (tri && GE) could = could && k0 >= x0 + nx - 1 + (unit ? 1 : 0);
        CHECK(full == could, "X %d nx %d k [%d, %d) panel %d full %d", X, nx, k_lo, k_hi, p, full);
        CHECK(!full || I::inside(k0, k_lo, k_hi, nx, ld), "panel %d", p);
        static int seen[X * kTileK];
        for (int& s : seen) s = 0;
        for (int t = 0; t < NT; ++t)
            for (int q = 0; q < I::VEC; ++q) {
                const int v = t + q * NT;
                if (I::PART && v >= I::PIECES) break;
                CHECK(KC || (I::px(v) == I::px(t) && I::pk(v) == I::pk(t) + q * I::KSTEP), "piece %d", v);
                for (int h = 0; h < 2; ++h) {
                    const int xe = I::px(v) + (KC ? 0 : h), ke = k0 + I::pk(v) + (KC ? h : 0);
                    seen[xe * kTileK + ke - k0]++;
                    if (full) {
                        const int x = I::full_x(v, nx) + (KC ? 0 : h);
                        CHECK(x == xe || xe >= nx, "x %d for %d", x, xe);
                        const int64_t at = KC ? (int64_t)(x0 + x) * ld + ke : (int64_t)ke * ld + x0 + x;
                        const int64_t end = KC ? (int64_t)(x0 + nx - 1) * ld + kmax - 1
                                               : (int64_t)(kmax - 1) * ld + x0 + nx - 1;
                        CHECK(at >= 0 && at <= end, "X %d nx %d k %d x %d", X, nx, ke, x);
                        CHECK(ke >= k_lo && ke < k_hi, "k %d", ke);
                        if (tri && x < nx)
                            CHECK(GE ? ke >= x0 + x + (unit ? 1 : 0) : ke <= x0 + x - (unit ? 1 : 0), "k %d x %d", ke,
                                  x0 + x);
                    } else {
                        const int x = xe < nx ? xe : nx - 1, k = near_k<GE>(ke, x0 + x, k_hi, tri);
                        CHECK(k >= 0 && k < kmax, "k %d of %d", k, kmax);
                        CHECK(!tri || (GE ? k >= x0 + x : k <= x0 + x), "k %d x %d", k, x0 + x);
                        const bool own = ke < k_hi && (!tri || (GE ? ke >= x0 + x : ke <= x0 + x));
                        CHECK(!own || k == ke, "k %d for %d", k, ke);
                    }
                }
            }
        for (int s : seen) CHECK(s == 1, "element read %d times", s);
    }
}

template <int X, int NT, bool KC>
static void shapes()
{
    const int widths[] = {1, 2, 3, X / 2 - 1, X / 2, X - 1, X};
    for (int nx : widths) {
        for (int k_hi : {1, 2, 15, 16, 17, 33, 48, 63})  // no triangle, every k start
            for (int k_lo : {0, 1, 2, 16, 17})
                if (k_lo < k_hi)
                    for (int more : {0, 5}) operand<X, NT, KC, false>(0, nx, k_lo, k_hi, k_hi + more, false, false);
        for (int x0 : {0, X, 3, X + 7})  // bands start anywhere
            for (int unit = 0; unit < 2; ++unit) {
                const int n = x0 + nx;  // the last tile, and one with more rows after it
                for (int more : {0, 1, 40}) {
                    operand<X, NT, KC, false>(x0, nx, 0, n, n + more, true, unit);
                    operand<X, NT, KC, false>(x0, nx, x0, n, n + more, true, unit);      // a triangle by itself
                    operand<X, NT, KC, false>(x0, nx, x0 / 2, n, n + more, true, unit);  // a piece of a tile
                    operand<X, NT, KC, true>(x0, nx, x0, n + more, n + more, true, unit);
                }
            }
    }
}

int main()
{
    shapes<256, 1024, true>();
    shapes<128, 1024, false>();
    shapes<128, 512, true>();
    shapes<128, 512, false>();
    shapes<64, 256, true>();
    shapes<64, 256, false>();
    shapes<64, 512, true>();
    shapes<64, 512, false>();
    shapes<128, 256, true>();
    shapes<32, 256, false>();
    shapes<32, 512, false>();
    // full panels give way where a row is too long for 32-bit byte offsets
    CHECK((PanelIdx<256, 1024, true>::offsets_fit((1 << 21) - 2)), "256 rows");
    CHECK(!(PanelIdx<256, 1024, true>::offsets_fit((1 << 21) + 1)), "256 rows");
    if (fails) fprintf(stderr, "%d checks failed\n", fails);
    else printf("ok\n");
    return fails != 0;
}
