// Host-only check of the panels that a tile loads whole with 64-bit addresses
// (uvt_panel.hpp: whole() and clear(); built and run by
// tests/test_panel_wide_host.py, no GPU): for every operand shape of the kernels
// that do so, widths, k ranges and triangles, such a panel reads only elements
// of the matrix (at most one past a row's end, before the next row), inside [k_lo,
// k_hi), at their own place, and, of the triangle, none on or past the
// diagonal.  At long rows the places are those of 64-bit arithmetic.
#include <stdio.h>

#include <initializer_list>

#define __host__
#define __device__
#include "uvt_panel.hpp"

using namespace uvt;

static int fails = 0, wholes = 0;
#define CHECK(c, ...)                                          \
    do {                                                       \
        if (!(c) && ++fails <= 10) {                           \
            fprintf(stderr, "line %d: %s: ", __LINE__, #c);    \
            fprintf(stderr, __VA_ARGS__);                      \
            fprintf(stderr, "\n");                             \
        }                                                      \
    } while (0)

template <int X, int NT, bool KC, bool GE>
static void operand(int x0, int nx, int k_lo, int k_hi, int kmax, bool tri, int64_t ld)
{
    using I = PanelIdx<X, NT, KC>;
    for (int k0 = (k_lo & ~1); k0 < k_hi; k0 += kTileK) {
        if (!I::whole(k0, k_lo, k_hi, nx) || (tri && !I::template clear<GE>(k0, x0, nx))) continue;
        ++wholes;
        CHECK(I::inside(k0, k_lo, k_hi, nx, ld) == I::offsets_fit(ld), "k0 %d", k0);
        for (int t = 0; t < NT; ++t)
            for (int q = 0; q < I::VEC; ++q) {
                const int v = t + q * NT;
                if (I::PART && v >= I::PIECES) break;
                const int64_t x = I::full_x(v, nx), k = k0 + I::pk(v);
                for (int h = 0; h < 2; ++h) {
                    const int64_t xe = x + (KC ? 0 : h), ke = k + (KC ? h : 0);
                    CHECK(ke >= k_lo && ke < k_hi, "k %d", (int)ke);
                    const int64_t at = (KC ? x * ld + k : k * ld + x) + h;  // from element (x0, 0)
                    const int64_t end = KC ? (nx - 1) * ld + kmax - 1 : (kmax - 1) * ld + nx - 1;
                    CHECK(at >= 0 && at <= end, "x %d k %d at %lld", (int)xe, (int)ke, (long long)at);
                    CHECK(xe < nx ? at == (KC ? xe * ld + ke : ke * ld + xe) : !KC && xe == nx, "x %d", (int)xe);
                    if (tri && xe < nx) CHECK(GE ? ke > x0 + xe : ke < x0 + xe, "k %d x %d", (int)ke, (int)(x0 + xe));
                }
            }
    }
}

template <int X, int NT, bool KC>
static void shapes()
{
    const int widths[] = {1, 2, 3, X / 2 - 1, X / 2, X - 1, X};
    for (int nx : widths)
        for (int64_t more : {(int64_t)0, (int64_t)1, (int64_t)1 << 21, ((int64_t)1 << 25) + 1, (int64_t)1 << 30}) {
            for (int k_hi : {16, 17, 33, 48, 63})
                for (int k_lo : {0, 1, 16, 17})
                    if (k_lo < k_hi) operand<X, NT, KC, false>(0, nx, k_lo, k_hi, k_hi, false, (KC ? k_hi : nx) + more);
            for (int x0 : {0, X, 3 * X}) {
                const int n = x0 + nx;
                operand<X, NT, KC, false>(x0, nx, 0, n, n, true, n + more);
                operand<X, NT, KC, false>(x0, nx, x0 / 2, n, n, true, n + more);
                operand<X, NT, KC, true>(x0, nx, x0, n + 70, n + 70, true, n + 70 + more);
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
    if (wholes < 1000) ++fails;
    if (fails) fprintf(stderr, "%d checks failed\n", fails);
    else printf("ok\n");
    return fails != 0;
}
