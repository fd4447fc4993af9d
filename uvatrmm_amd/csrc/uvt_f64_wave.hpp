// uvt_f64_wave.hpp -- FP64 products too small for workgroup tiles: one wave
// per (16 FM) x (16 FN) tile of C.
//
// A small product in 64x64 tiles leaves most of the chip idle (1000 x 777: 208
// workgroups on 256 compute units, one wave per SIMD) and pays a barrier and
// an LDS round trip per 16-deep panel of a long serial chain.  Here every
// wave works alone: it reads its operands from L1 and L2 (neighbouring waves
// share rows of A and columns of B) into registers, D panels ahead, and never
// waits for another wave.  The k order inside a panel, the panels' order and
// so every sum are those of f64_tile: same bits.
//
// What bounds it is how the loads split into cache lines.  A lane's fragment
// of an x-contiguous operand is one double of each of four k rows; two blocks
// take alternate columns, so that a lane loads them as one 16-byte pair and
// 16 lanes cover 256 contiguous bytes.  A fragment of a k-contiguous operand
// is four doubles of one row; loaded in that order every lane of a load
// touches another line (72 cycles per load measured, against 16), so a panel
// is loaded with 8 lanes on the 128 bytes of a row and turned round through
// a few KiB of LDS of the wave's own, which takes no barrier.
#pragma once

#include "uvt_f64_tile.hpp"

namespace uvt {

// F blocks of 16 rows of op(A) (columns of op(B)) as one wave's MFMA operand.
template <int F, bool KC, bool DOWN>
struct WaveOperand {
    using Idx = WaveIdx<F, KC>;
    static constexpr bool PAIR = Idx::PAIR;
    static constexpr int LOADS = Idx::LOADS;
    static constexpr int SLOT = 16 * F * Idx::PITCH;   // a panel in LDS
    static constexpr int LDS = KC ? 2 * SLOT : 0;      // doubles: two panels

    const UVT_GLOBAL double* p;  // element (x0, k = 0)
    int64_t ld;
    int nx, x0, lane;
    double* lds;
    const UVT_GLOBAL char* at;  // the full panel load() reads next
    uint32_t off[LOADS];        // byte offsets of this lane's loads in it

    __device__ __forceinline__ void init(const UVT_GLOBAL double* p_, int64_t ld_, int nx_, int x0_, double* lds_)
    {
        p = p_;
        ld = ld_;
        nx = nx_;
        x0 = x0_;
        lds = lds_;
        lane = threadIdx.x & 63;
#pragma unroll
        for (int q = 0; q < LOADS; ++q) {
            const uint32_t x = (uint32_t)Idx::load_x(q, lane, nx), k = (uint32_t)Idx::load_k(q, lane);
            off[q] = 8u * (KC ? x * (uint32_t)ld + k : k * (uint32_t)ld + x);
        }
    }
    // This lane's row (column) of block f.
    __device__ __forceinline__ int row(int f) const { return Idx::row(f, lane); }
    __device__ __forceinline__ void seek(int k0)
    {
        at = reinterpret_cast<const UVT_GLOBAL char*>(KC ? p + k0 : p + (int64_t)k0 * ld);
    }
    // The full panel at `at`, as it is loaded; then on to the next one (more)
    // or not.
    __device__ __forceinline__ void load(bool more, double (&r)[4 * F])
    {
#pragma unroll
        for (int q = 0; q < LOADS; ++q) {
            asm volatile("" : "+v"(off[q]));  // 32-bit offsets: see Panel::load
            if constexpr (KC || PAIR) {
                const dbl2 v = *reinterpret_cast<const UVT_GLOBAL dbl2u*>(at + off[q]);
                r[2 * q] = v.x;
                r[2 * q + 1] = v.y;
            } else {
                r[q] = *reinterpret_cast<const UVT_GLOBAL double*>(at + off[q]);
            }
        }
        const int64_t step = KC ? (int64_t)kTileK * 8 : ld * (kTileK * 8);
        if (more) at += DOWN ? -step : step;
    }
    // A loaded panel as fragments: v[f][s] for MFMA step s.  Through LDS for a
    // k-contiguous operand (slot 0 and 1 in turn): written and read by this
    // wave alone, whose LDS instructions run in order.
    __device__ __forceinline__ void fragments(const double (&r)[4 * F], int slot, double (&v)[F][4])
    {
        if constexpr (KC) {
            double* s = lds + slot * SLOT;
#pragma unroll
            for (int q = 0; q < LOADS; ++q)
                *reinterpret_cast<dbl2*>(&s[Idx::lds_write(q, lane)]) = dbl2{r[2 * q], r[2 * q + 1]};
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int f = 0; f < F; ++f)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const dbl2 w = *reinterpret_cast<const dbl2*>(&s[Idx::lds_read(f, h, lane)]);
                    v[f][2 * h] = w.x;
                    v[f][2 * h + 1] = w.y;
                }
        } else {
#pragma unroll
            for (int f = 0; f < F; ++f)
#pragma unroll
                for (int s = 0; s < 4; ++s) v[f][s] = r[PAIR ? 2 * s + f : s];
        }
    }
    // The fragments of any panel, read inside the matrix, below k_hi and inside
    // the triangle (near_k).
    template <bool GE>
    __device__ __forceinline__ void load_masked(int k0, int k_hi, bool tri, double (&v)[F][4]) const
    {
#pragma unroll
        for (int f = 0; f < F; ++f)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int xe = row(f), x = xe < nx ? xe : nx - 1;
                const int k = near_k<GE>(k0 + 4 * (lane >> 4) + s, x0 + x, k_hi, tri);
                v[f][s] = KC ? p[(int64_t)x * ld + k] : p[(int64_t)k * ld + x];
            }
    }
    // Zeros outside [k_lo, k_hi) and the triangle, and (unit) ones on its
    // diagonal.
    template <bool GE>
    __device__ __forceinline__ void mask(int k0, int k_lo, int k_hi, bool tri, bool unit, double (&v)[F][4]) const
    {
#pragma unroll
        for (int f = 0; f < F; ++f)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int x = x0 + row(f), k = k0 + 4 * (lane >> 4) + s;
                bool in = k >= k_lo && k < k_hi;
                if (tri) in = in && (GE ? k >= x : k <= x);
                v[f][s] = in ? v[f][s] : 0.0;
                if (unit && k == x) v[f][s] = 1.0;
            }
    }
};

// LDS of one wave's tile, in doubles.
template <int FM, int FN, class OPT>
constexpr int wave_lds()
{
    return WaveOperand<FM, OPT::A_KC, OPT::GE>::LDS + WaveOperand<FN, OPT::B_KC, OPT::GE>::LDS;
}

// One wave's tile (t.rows <= 16 FM rows from t.r0, columns from t.c0), by the
// 64 threads of the calling wave; lds: its own wave_lds() doubles, 16-byte
// aligned.  m: columns of C.
template <int FM, int FN, int D, class OPT = TileOpt<>>
__device__ __forceinline__ void f64_wave(const TileArgs& t, const UVT_GLOBAL double* __restrict__ A, int64_t lda,
                                         const UVT_GLOBAL double* __restrict__ B, int64_t ldb,
                                         UVT_GLOBAL double* __restrict__ C, int64_t ldc, int64_t m, double* lds,
                                         const TileEpi& epi = TileEpi())
{
    static_assert(D % 2 == 0, "the LDS slot of a panel is known at compile time");
    using OA = WaveOperand<FM, OPT::A_KC, OPT::GE>;
    using OB = WaveOperand<FN, OPT::B_KC, OPT::GE>;
    constexpr bool GE = OPT::GE, TRI_A = OPT::TRI_A;
    constexpr int TAIL = TRI_A ? FM : FN;  // panels on the diagonal (a partial last panel: one)
    const int lane = threadIdx.x & 63;
    const bool tri = OPT::TRI != kTriALe || (t.flags & kTileLower) != 0;
    const bool unit = OPT::UNIT && epi.unit;
    const int k_lo = t.k_lo, k_hi = t.k_hi;
    const int cols = (int64_t)t.c0 + 16 * FN <= m ? 16 * FN : (int)(m - t.c0);
    const int nk = panels(k_lo, k_hi);
    const int tx0 = TRI_A ? t.r0 : t.c0, tx1 = tx0 + (TRI_A ? t.rows : cols) - 1;
    const bool odd = (OA::PAIR && (t.rows & 1)) || (OB::PAIR && (cols & 1));
    const FullPanels fp = full_panels<GE>(k_lo, k_hi, tri, unit, tx0, tx1, odd);
    const int f0 = fp.f0, f1 = fp.f1 > f0 && OA::Idx::fits(lda) && OB::Idx::fits(ldb) ? fp.f1 : f0;

    OA pa;
    OB pb;
    pa.init(OPT::A_KC ? A + (int64_t)t.r0 * lda : A + t.r0, lda, t.rows, t.r0, lds);
    pb.init(OPT::B_KC ? B + (int64_t)t.c0 * ldb : B + t.c0, ldb, cols, t.c0, lds + OA::LDS);

    dbl4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
    auto multiply = [&](const double (&a)[FM][4], const double (&b)[FN][4]) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][s], b[j][s], acc[i][j], 0, 0, 0);
    };
    auto load_masked = [&](int kt, double (&a)[FM][4], double (&b)[FN][4]) {
        const int k0 = panel_k0<GE>(k_lo, nk, kt);
        pa.template load_masked<GE>(k0, k_hi, TRI_A && tri, a);
        pb.template load_masked<GE>(k0, k_hi, !TRI_A && tri, b);
    };
    auto multiply_masked = [&](int kt, double (&a)[FM][4], double (&b)[FN][4]) {
        const int k0 = panel_k0<GE>(k_lo, nk, kt);
        pa.template mask<GE>(k0, k_lo, k_hi, TRI_A && tri, TRI_A && unit, a);
        pb.template mask<GE>(k0, k_lo, k_hi, !TRI_A && tri, !TRI_A && unit, b);
        multiply(a, b);
    };

    // The first D full panels, then the diagonal's, are on their way before
    // the first product.
    double ra[D][4 * FM], rb[D][4 * FN];
    const int cnt = f1 - f0;
    pa.seek(panel_k0<GE>(k_lo, nk, f0));
    pb.seek(panel_k0<GE>(k_lo, nk, f0));
    // full panel i of cnt, or past the end the last one once more (unused)
    auto load = [&](int i, int d) {
        pa.load(i + 1 < cnt, ra[d]);
        pb.load(i + 1 < cnt, rb[d]);
    };
    if (cnt > 0) {
#pragma unroll
        for (int d = 0; d < D; ++d) load(d, d);
    }
    double ta[TAIL][FM][4], tb[TAIL][FN][4];
#pragma unroll
    for (int d = 0; d < TAIL; ++d)
        if (f1 + d < nk) load_masked(f1 + d, ta[d], tb[d]);
    if (f0 > 0 && nk > 0) {  // a partial first panel
        double ha[FM][4], hb[FN][4];
        load_masked(0, ha, hb);
        multiply_masked(0, ha, hb);
    }
    // fa, fb: the fragments of the panel to multiply next, taken from the
    // loaded panel during the products of the one before.
    double fa[FM][4], fb[FN][4];
    auto next = [&](int d) {
        pa.fragments(ra[d], d % 2, fa);
        pb.fragments(rb[d], d % 2, fb);
    };
    auto step = [&](int d) {  // multiplies panel i + d, turns panel i + d + 1 round
        double a[FM][4], b[FN][4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int i = 0; i < FM; ++i) a[i][s] = fa[i][s];
#pragma unroll
            for (int j = 0; j < FN; ++j) b[j][s] = fb[j][s];
        }
        next((d + 1) % D);
        multiply(a, b);
    };
    if (cnt > 0) next(0);
    int i = 0;
    for (; i + D <= cnt; i += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            step(d);
            load(i + D + d, d);
        }
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (i + d < cnt) step(d);
#pragma unroll
    for (int d = 0; d < TAIL; ++d)
        if (f1 + d < nk) multiply_masked(f1 + d, ta[d], tb[d]);
    for (int kt = f1 + TAIL; kt < nk; ++kt) {  // a last k row kept out of the full panels, or no full panels
        load_masked(kt, ta[0], tb[0]);
        multiply_masked(kt, ta[0], tb[0]);
    }

    // D layout: lane l, element v holds row l/16 + 4*v, column l%16 (see
    // f64_tile) of a block.
#pragma unroll
    for (int bi = 0; bi < FM; ++bi)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int in = (lane >> 4) + 4 * v, row = OA::PAIR ? 2 * in + bi : 16 * bi + in;
            if (row >= t.rows) continue;
#pragma unroll
            for (int bj = 0; bj < FN; ++bj) {
                const int col = OB::PAIR ? 2 * (lane & 15) + bj : 16 * bj + (lane & 15);
                if (col >= cols) continue;
                const double x = acc[bi][bj][v];
                UVT_GLOBAL double* p = C + (int64_t)(t.r0 + row) * ldc + (t.c0 + col);
                if constexpr (OPT::EPI) {
                    const double ax = epi.alpha * x;
                    *p = epi.beta == 0.0 ? ax : ax + epi.beta * *p;
                } else {
                    *p = x;
                }
            }
        }
}

}  // namespace uvt
