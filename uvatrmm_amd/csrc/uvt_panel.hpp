// uvt_panel.hpp -- which elements of an operand an FP64 tile reads (host and
// device; the loads themselves are in uvt_f64_tile.hpp).
//
// A tile multiplies X rows of op(A) and X columns of op(B) over k in
// [k_lo, k_hi), kTileK deep panels from k_start = k_lo rounded down to even.
// An operand is k-contiguous in memory (KC: A, or B transposed; element
// (x, k) at x * ld + k) or x-contiguous (B, or A transposed; k * ld + x).
// Panels move as pairs along the contiguous direction.
//
//   full panels    pairs as they are, every row (column) past the tile's last
//                  one replaced by the last: no masks.  An odd last x of an
//                  x-contiguous operand reads its pair one element past the
//                  row's end, so such a panel never holds the matrix's last k
//                  row, and that element lies before the next row.
//   other panels   element by element, each at the nearest place inside the
//                  matrix, the k range and the triangle; what does not belong
//                  is zeroed on the way to LDS.
#pragma once

#include <stdint.h>

namespace uvt {

constexpr int kTileK = 16;  // k depth of one LDS panel (4 MFMA steps)

template <int X, int NT, bool KC>
struct PanelIdx {
    static constexpr int PIECES = X * kTileK / 2;         // pairs of a panel
    static constexpr int VEC = (PIECES + NT - 1) / NT;    // per thread
    static constexpr bool PART = PIECES < NT;             // the last threads hold none
    static_assert(PIECES % NT == 0 || PART, "uneven panel split");
    // Pieces of an x-contiguous panel that one thread holds sit KSTEP k rows
    // apart at the same x.
    static constexpr int KSTEP = KC ? 0 : NT / (X / 2);
    static_assert(KC || NT % (X / 2) == 0, "k rows per piece");

    // x and k of pair v (of its first element), relative to the panel.
    static __host__ __device__ int px(int v) { return KC ? v / (kTileK / 2) : (v % (X / 2)) * 2; }
    static __host__ __device__ int pk(int v) { return KC ? (v % (kTileK / 2)) * 2 : v / (X / 2); }
    // The x a full panel reads pair v at, with nx of the X inside the matrix.
    static __host__ __device__ int full_x(int v, int nx)
    {
        const int last = KC ? nx - 1 : (nx - 1) & ~1;
        return px(v) < last ? px(v) : last;
    }
    // Byte offsets of full panels fit 32 bits for every matrix but one whose
    // rows are 16 MB or longer; such a tile has no full panels.
    static __host__ __device__ bool offsets_fit(int64_t ld)
    {
        return ld <= (int64_t)(0xFFFFFFFFu / (8u * (KC ? X : kTileK))) - 1;
    }
    // Whether the panel at k0 lies wholly inside [k_lo, k_hi) and may be read
    // as a full one (whole: with 64-bit addresses).
    static __host__ __device__ bool whole(int k0, int k_lo, int k_hi, int nx)
    {
        return k0 >= k_lo && k0 + kTileK <= k_hi - (!KC && (nx & 1) ? 1 : 0);
    }
    static __host__ __device__ bool inside(int k0, int k_lo, int k_hi, int nx, int64_t ld)
    {
        return whole(k0, k_lo, k_hi, nx) && offsets_fit(ld);
    }
    // Whether it lies off the diagonal of the triangle (GE: k >= x, else k <=
    // x) whose x run from x0 on, nx of them.
    template <bool GE>
    static __host__ __device__ bool clear(int k0, int x0, int nx)
    {
        return GE ? k0 >= x0 + nx : k0 + kTileK <= x0;
    }
};

// The same for the tile of a single wave (uvt_f64_wave.hpp), whose operand is F
// blocks of 16 rows (columns).  A load of a full panel takes a pair along k (KC:
// 8 lanes on the 128 bytes of a row), a pair along x (PAIR: two blocks on
// alternate columns) or one element; the pairs along k are turned round through
// LDS rows of PITCH doubles.  Lane l's fragment of block f for MFMA step s is row
// row(f, l), k = 4 (l / 16) + s.
template <int F, bool KC>
struct WaveIdx {
    static constexpr bool PAIR = !KC && F == 2;
    static constexpr int LOADS = KC ? 2 * F : 4;
    static constexpr int PITCH = kTileK + 2;
    // x and k of load q (of its first element), with nx rows inside the matrix.
    static __host__ __device__ int load_x(int q, int lane, int nx)
    {
        const int x = KC ? 8 * q + (lane >> 3) : PAIR ? 2 * (lane & 15) : lane & 15;
        const int last = PAIR ? (nx - 1) & ~1 : nx - 1;
        return x < last ? x : last;
    }
    static __host__ __device__ int load_k(int q, int lane) { return KC ? 2 * (lane & 7) : 4 * (lane >> 4) + q; }
    static __host__ __device__ int row(int f, int lane) { return PAIR ? 2 * (lane & 15) + f : 16 * f + (lane & 15); }
    // Where in LDS load q's pair goes, and pair h of block f's fragment lies (KC).
    static __host__ __device__ int lds_write(int q, int lane) { return (8 * q + (lane >> 3)) * PITCH + 2 * (lane & 7); }
    static __host__ __device__ int lds_read(int f, int h, int lane)
    {
        return (16 * f + (lane & 15)) * PITCH + 4 * (lane >> 4) + 2 * h;
    }
    // Offsets of a full panel fit 32 bits for every matrix but one whose rows
    // are 256 MB (F = 2: 128 MB) or longer; such a tile has no full panels.
    static __host__ __device__ bool fits(int64_t ld) { return ld < (int64_t)(0xFFFFFFFFu / (8u * 16 * F)) - 16; }
};

// The k another panel reads element (x, k) at, x inside the matrix: the
// nearest below k_hi and, with tri, in the triangle (GE: k >= x, else k <= x).
template <bool GE>
__host__ __device__ inline int near_k(int k, int x, int k_hi, bool tri)
{
    k = k < k_hi ? k : k_hi - 1;
    if (tri) k = GE ? (k > x ? k : x) : (k < x ? k : x);
    return k;
}

// The tile's panels in the order it runs them, kt = 0 .. panels() - 1: up in k,
// or down (GE), so that the triangle's diagonal always comes last.
__host__ __device__ inline int panels(int k_lo, int k_hi)
{
    const int k_start = k_lo & ~1;
    return k_hi > k_start ? (k_hi - k_start + kTileK - 1) / kTileK : 0;
}
template <bool GE>
__host__ __device__ inline int panel_k0(int k_lo, int nk, int kt)
{
    return (k_lo & ~1) + (GE ? nk - 1 - kt : kt) * kTileK;
}

// Panels kt in [f0, f1) of that order need no masks: inside [k_lo, k_hi) (only
// the first can start below an odd k_lo, or pass k_hi on the way down), off
// the diagonal of the triangle whose x run from tx0 to tx1 (unit: the
// diagonal itself is replaced too), and away from the last k row where odd
// asks for it.  f0 is 0 or 1.  (GE: k_lo is even.)
struct FullPanels {
    int f0, f1;
};
template <bool GE>
__host__ __device__ inline FullPanels full_panels(int k_lo, int k_hi, bool tri, bool unit, int tx0, int tx1, bool odd)
{
    const int k_start = k_lo & ~1, nk = panels(k_lo, k_hi);
    int lim = k_hi, f0 = k_start < k_lo ? 1 : 0;
    if (tri && !GE) {
        const int d = tx0 + (unit ? 0 : 1);
        lim = lim < d ? lim : d;
    }
    if (tri && GE) {
        const int d = tx1 + (unit ? 1 : 0) - k_start;
        f0 = d > 0 ? (d + kTileK - 1) / kTileK : 0;
    }
    lim -= odd ? 1 : 0;
    const int f1 = lim > k_start ? (lim - k_start) / kTileK : 0;
    return GE ? FullPanels{nk - f1, nk - f0} : FullPanels{f0, f1};
}

}  // namespace uvt
