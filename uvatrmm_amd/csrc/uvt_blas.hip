// uvt_blas.hip -- device-resident BLAS forms of the two routines the
// reference calls per band (UVaTRMM/src/mm_triangular.c:347-360 cblas_dgemm,
// :374-387 cblas_dtrmm), row-major, every transpose / side / triangle / diagonal
// variant.  All of them run on the FP64 MFMA tile kernel of uvt_f64_tile.hpp:
//
//   dgemm  C = alpha op(A) op(B) + beta C
//          the rectangular tile walk; the tile reads either operand as it is
//          stored or transposed, and applies alpha and beta as it writes C
//          (C is not read when beta == 0).  No workspace, unless C shares
//          elements with A or B: then C is computed there and copied back.
//   dtrmm  B := alpha op(A) B  (left)  or  alpha B op(A)  (right), in place
//          B is copied to the workspace, then the tile walk multiplies the
//          copy into B (where A shares elements with B: B into the workspace,
//          which is then copied to B): the triangle masks either operand,
//          lower or upper, a transposed A is read as it is stored, and a unit
//          diagonal goes in on the way to LDS.
// (With op(A), op(B) and the triangle packed row-major and lower first, and
// the result unpacked afterwards, a dtrmm of a 2048 triangle on 3000 rows
// took 323 us, of which three packing passes were 57; now 241.  A 1500 x 2000
// x 3000 dgemm with A transposed and beta: 334 us, now 293.)
// Layout-only reductions (column-major input) are the caller's (the CBLAS
// shim): a column-major matrix is the transpose of a row-major one.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>

#include "uvt_f64_tile.hpp"
#include "uvt_f64_wave.hpp"
#include "uvt_internal.h"
#include "uvt_overlap.hpp"
#include "uvt_place.hpp"
#include "uvt_runtime.hpp"

using namespace uvt;

namespace {

// C = beta * C (beta == 0: zeros, C is not read).
__global__ __launch_bounds__(256) void k_scale(int64_t rows, int64_t cols, double beta, double* __restrict__ C,
                                               int64_t ldc)
{
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= cols) return;
    for (int64_t i = blockIdx.y; i < rows; i += gridDim.y) {
        double* c = C + i * ldc + j;
        *c = beta == 0.0 ? 0.0 : beta * *c;
    }
}

// dst[i][j] = src[i][j], rows x cols.  HBM-bound: 16 bytes per element moved.
__global__ __launch_bounds__(256) void k_copy(const double* __restrict__ src, int64_t lds, double* __restrict__ dst,
                                              int64_t ldd, int64_t rows, int64_t cols)
{
    const int64_t j = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);
    if (j >= cols) return;
    for (int64_t i0 = (int64_t)blockIdx.y * 16 + (threadIdx.x >> 6); i0 < rows; i0 += (int64_t)gridDim.y * 16) {
        double v[4];  // four rows in flight
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = i0 + 4 * q < rows ? src[(i0 + 4 * q) * lds + j] : 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (i0 + 4 * q < rows) dst[(i0 + 4 * q) * ldd + j] = v[q];
    }
}

// What a walk multiplies: C (M x N) from a reduction over K, and which
// operand is triangular (TriKind; kTriNone: neither); cus: the GPU's compute
// units.
struct Walk {
    int64_t M, N;
    int K, nrt, nct, cus;
};
constexpr int kTriNone = -1;

// One tile per workgroup, the deepest reductions first (left side: row tiles
// of the long end of the triangle; right side: column tiles), placed by
// walk_tile (uvt_place.hpp).
template <int TM, int TN, bool A_KC, bool B_KC, int TRI>
__global__ __launch_bounds__((64 * TileWaves<TM, TN>::M * TileWaves<TM, TN>::N), (TileWaves<TM, TN>::WAVES_PER_EU))
void k_blas_f64(Walk g, const double* __restrict__ A, int64_t lda, const double* __restrict__ B, int64_t ldb,
                double* __restrict__ C, int64_t ldc, TileEpi epi)
{
    using W = TileWaves<TM, TN>;
    constexpr bool kNone = TRI == kTriNone, kRight = TRI == kTriBLe || TRI == kTriBGe;
    using Opt = TileOpt<A_KC, B_KC, kNone ? kTriALe : (TriKind)TRI, !kNone, true, true, false>;
    __shared__ __attribute__((aligned(16))) double smem[F64Cfg<TM, TN, W::M, W::N, Opt>::SMEM_DOUBLES];
    const WalkTile wt = walk_tile((int)blockIdx.x, g.nrt * g.nct, kRight ? g.nrt : g.nct, g.cus, W::BLOCKS_PER_CU);
    int rt = kRight ? wt.inner : wt.outer, ct = kRight ? wt.outer : wt.inner;
    if (TRI == kTriALe) rt = g.nrt - 1 - rt;
    if (TRI == kTriBLe) ct = g.nct - 1 - ct;
    const int r0 = rt * TM, c0 = ct * TN;
    const int rows = (int)(g.M - r0 < TM ? g.M - r0 : TM), cols = (int)(g.N - c0 < TN ? g.N - c0 : TN);
    const int k_lo = TRI == kTriAGe ? r0 : TRI == kTriBGe ? c0 : 0;
    const int k_hi = TRI == kTriALe ? r0 + rows : TRI == kTriBLe ? c0 + cols : g.K;
    f64_tile<TM, TN, W::M, W::N, Opt>(TileArgs{r0, rows, c0, k_lo, k_hi, kNone ? 0 : kTileLower}, gbl(A), lda, gbl(B),
                                      ldb, gbl(C), ldc, g.N, smem, -1, nullptr, epi);
}

template <int TM, int TN, bool A_KC, bool B_KC, int TRI>
void launch_walk(Walk g, const double* A, int64_t lda, const double* B, int64_t ldb, double* C, int64_t ldc,
                 const TileEpi& epi, hipStream_t s)
{
    g.nrt = (int)((g.M + TM - 1) / TM);
    g.nct = (int)((g.N + TN - 1) / TN);
    const dim3 grid((unsigned)((int64_t)g.nrt * g.nct)), block(64 * TileWaves<TM, TN>::M * TileWaves<TM, TN>::N);
    hipLaunchKernelGGL((k_blas_f64<TM, TN, A_KC, B_KC, TRI>), grid, block, 0, s, g, A, lda, B, ldb, C, ldc, epi);
}

// The same walk in wave tiles, four to a workgroup, wn of them along the
// columns; every second run of `snake` workgroups is turned round, as the
// trapezoid walk's (uvt_api.hip).
template <int FM, int FN, int D, bool A_KC, bool B_KC, int TRI>
__global__ __launch_bounds__(256) void k_blas_waves_f64(Walk g, int wn, int snake, const double* __restrict__ A,
                                                        int64_t lda, const double* __restrict__ B, int64_t ldb,
                                                        double* __restrict__ C, int64_t ldc, TileEpi epi)
{
    constexpr bool kNone = TRI == kTriNone, kRight = TRI == kTriBLe || TRI == kTriBGe;
    using Opt = TileOpt<A_KC, B_KC, kNone ? kTriALe : (TriKind)TRI, !kNone, true>;
    __shared__ __attribute__((aligned(16))) double lds[4][wave_lds<FM, FN, Opt>() + 2];
    int b = (int)blockIdx.x;
    const int q = b / snake;
    if (q & 1) b = q * snake + min((q + 1) * snake, (int)gridDim.x) - 1 - b;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int rt = kRight ? b % g.nrt : b / g.nct, ct = kRight ? b / g.nrt : b % g.nct;
    if (TRI == kTriALe) rt = g.nrt - 1 - rt;
    if (TRI == kTriBLe) ct = g.nct - 1 - ct;
    const int64_t r0 = ((int64_t)rt * (4 / wn) + wave / wn) * (16 * FM), c0 = ((int64_t)ct * wn + wave % wn) * (16 * FN);
    if (r0 >= g.M || c0 >= g.N) return;
    const int rows = (int)(g.M - r0 < 16 * FM ? g.M - r0 : 16 * FM), cols = (int)(g.N - c0 < 16 * FN ? g.N - c0 : 16 * FN);
    const int k_lo = (int)(TRI == kTriAGe ? r0 : TRI == kTriBGe ? c0 : 0);
    const int k_hi = (int)(TRI == kTriALe ? r0 + rows : TRI == kTriBLe ? c0 + cols : g.K);
    f64_wave<FM, FN, D, Opt>(TileArgs{(int)r0, rows, (int)c0, k_lo, k_hi, kNone ? 0 : kTileLower}, gbl(A), lda, gbl(B),
                             ldb, gbl(C), ldc, g.N, lds[wave], epi);
}

template <int FM, int FN, int D, bool A_KC, bool B_KC, int TRI>
void launch_walk_waves(Walk g, const double* A, int64_t lda, const double* B, int64_t ldb, double* C, int64_t ldc,
                       const TileEpi& epi, int cus, hipStream_t s)
{
    const int64_t rt = (g.M + 16 * FM - 1) / (16 * FM), ct = (g.N + 16 * FN - 1) / (16 * FN);
    const int wn = ct > 1 ? (rt > 1 ? 2 : 4) : 1, wm = 4 / wn;
    g.nrt = (int)((rt + wm - 1) / wm);
    g.nct = (int)((ct + wn - 1) / wn);
    hipLaunchKernelGGL((k_blas_waves_f64<FM, FN, D, A_KC, B_KC, TRI>), dim3((unsigned)((int64_t)g.nrt * g.nct)),
                       dim3(256), 0, s, g, wn, cus, A, lda, B, ldb, C, ldc, epi);
}

// Which dgemm walks run in wave tiles, and in which (as uvt_wave_shape): all
// reductions are equally deep, so a second round of waves doubles the time,
// and each shape stops where the GPU holds no more of them (a wave per SIMD
// for 16x16 tiles, three for 16x32).  us, workgroup tiles / 16x16 / 16x32:
//     257 x 257 x 257      13.9 /  6.4 /  8.5   (289 tiles of 16x16)
//     512 x 512 x 512      22.9 /  9.5 / 12.2   (1024)
//     600 x 600 x 6000    233   / 164  / 107    (1444)
//    1024 x 1024 x 1024    43.6 / 50.6 / 39.1   (4096)
//    3000 x 500 x 800      57.1 / 62.7 / 48.4   (6016)
//    1300 x 1300 x 3000   205   / 345  / 289    (6724)
// Where C is only written, shallow products that fill the chip are bound by
// that, and go in workgroup tiles, which write whole lines:
//    1024 x 1024 x 16      4.9 /  6.5 /  5.5
//    1024 x 1024 x 64      6.7 /  9.0 /  7.0
//    3000 x 500 x 32       7.3 /  8.5 /  7.6
//    1001 x 1203 x 64      8.9 / 10.7 /  8.8
//    1001 x 1203 x 100    12.5 / 12.8 / 11.5
//    768 x 768 x 32        5.3 /  5.4 /  5.1    (2304)
//    1024 x 1024 x 64      8.2 /  9.6 /  8.0    (C read too)
int gemm_wave_shape(int64_t M, int64_t N, int64_t K, double beta)
{
    const int64_t tiles = ((M + 15) / 16) * ((N + 15) / 16);
    if (tiles > 2304 && K <= 64 && beta == 0.0) return 0;
    return tiles <= 1024 ? 11 : tiles <= 6144 ? 12 : 0;
}

// The tile shape for the walk: cfg as uvt_default_cfg / uvt_wide_tiles name
// it; on the right side 32 x 128 stands for 128 x 32 (B has few rows).
template <bool A_KC, bool B_KC, int TRI>
uvt_status launch_blas(int32_t cfg, const Walk& g, const double* A, int64_t lda, const double* B, int64_t ldb,
                       double* C, int64_t ldc, const TileEpi& epi, int cus, hipStream_t s)
{
    constexpr bool kRight = TRI == kTriBLe || TRI == kTriBGe;
    const int wave = TRI == kTriNone ? gemm_wave_shape(g.M, g.N, g.K, epi.beta)
                     : kRight        ? uvt_wave_shape(g.K, g.M, ldb, lda)
                                     : uvt_wave_shape(g.K, g.N, lda, ldb);
    if (wave) {
        if (wave == 11) launch_walk_waves<1, 1, 4, A_KC, B_KC, TRI>(g, A, lda, B, ldb, C, ldc, epi, cus, s);
        else if (wave == 12) launch_walk_waves<1, 2, 4, A_KC, B_KC, TRI>(g, A, lda, B, ldb, C, ldc, epi, cus, s);
        else launch_walk_waves<2, 2, 2, A_KC, B_KC, TRI>(g, A, lda, B, ldb, C, ldc, epi, cus, s);
        UVT_HIP(hipGetLastError());
        return UVT_OK;
    }
    const int64_t tm = kRight && cfg == UVT_CFG_128x32 ? 32 : uvt_cfg_tile_m(cfg);
    const int64_t tn = kRight && cfg == UVT_CFG_128x32 ? 128 : uvt_cfg_tile_n(cfg);
    if (((g.M + tm - 1) / tm) * ((g.N + tn - 1) / tn) > 0x7FFFFFFF) return UVT_ERR_SIZE;
    if (cfg == UVT_CFG_64x64) launch_walk<64, 64, A_KC, B_KC, TRI>(g, A, lda, B, ldb, C, ldc, epi, s);
    else if (cfg == UVT_CFG_128x32)
        launch_walk<kRight ? 32 : 128, kRight ? 128 : 32, A_KC, B_KC, TRI>(g, A, lda, B, ldb, C, ldc, epi, s);
    else if (cfg == UVT_CFG_128x128) launch_walk<128, 128, A_KC, B_KC, TRI>(g, A, lda, B, ldb, C, ldc, epi, s);
    else if constexpr (TRI != kTriNone)  // uvt_wide_tiles
        launch_walk<256, 128, A_KC, B_KC, TRI>(g, A, lda, B, ldb, C, ldc, epi, s);
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

void scale(int64_t rows, int64_t cols, double beta, double* C, int64_t ldc, hipStream_t s)
{
    const dim3 grid((unsigned)((cols + 255) / 256), (unsigned)std::min<int64_t>(rows, 32768));
    hipLaunchKernelGGL(k_scale, grid, dim3(256), 0, s, rows, cols, beta, C, ldc);
}

void copy(const double* src, int64_t lds, double* dst, int64_t ldd, int64_t rows, int64_t cols, hipStream_t s)
{
    const dim3 grid((unsigned)((cols + 63) / 64), (unsigned)std::min<int64_t>((rows + 15) / 16, 32768));
    hipLaunchKernelGGL(k_copy, grid, dim3(256), 0, s, src, lds, dst, ldd, rows, cols);
}

int64_t even(int64_t x) { return x + (x & 1); }
size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }

bool sizes_ok(int64_t a, int64_t b, int64_t c)
{
    const int64_t lim = 0x3FFFFFFF;
    return a <= lim && b <= lim && c <= lim;
}

}  // namespace

extern "C" uvt_status uvt_dgemm(uvt_handle h, uvt_trans ta, uvt_trans tb, int64_t m, int64_t n,
                                int64_t k, double alpha, const double* dA, int64_t lda,
                                const double* dB, int64_t ldb, double beta, double* dC,
                                int64_t ldc, void* stream)
{
    if (!h || m < 0 || n < 0 || k < 0) return UVT_ERR_ARG;
    if ((ta != UVT_NO_TRANS && ta != UVT_TRANS) || (tb != UVT_NO_TRANS && tb != UVT_TRANS))
        return UVT_ERR_ARG;
    const bool tA = ta == UVT_TRANS, tB = tb == UVT_TRANS;
    if (lda < std::max<int64_t>(1, tA ? m : k) || ldb < std::max<int64_t>(1, tB ? k : n) ||
        ldc < std::max<int64_t>(1, n))
        return UVT_ERR_ARG;
    if (m == 0 || n == 0) return UVT_OK;
    if (!dC || (k > 0 && alpha != 0.0 && (!dA || !dB))) return UVT_ERR_ARG;
    if (!sizes_ok(m, n, k)) return UVT_ERR_SIZE;
    UVT_HIP(hipSetDevice(h->device));
    hipStream_t s = (hipStream_t)stream;
    if (k == 0 || alpha == 0.0) {  // C = beta C, A and B not read
        scale(m, n, beta, dC, ldc, s);
        UVT_HIP(hipGetLastError());
        return UVT_OK;
    }
    const Walk g{m, n, (int)k, 0, 0, h->cus};
    TileEpi epi;
    epi.alpha = alpha;
    epi.beta = beta;
    const int32_t cfg = uvt_default_cfg(m, n);
    const auto walk = [&](double* R, int64_t ldr) {
        if (tA && tB) return launch_blas<false, true, kTriNone>(cfg, g, dA, lda, dB, ldb, R, ldr, epi, h->cus, s);
        if (tA) return launch_blas<false, false, kTriNone>(cfg, g, dA, lda, dB, ldb, R, ldr, epi, h->cus, s);
        if (tB) return launch_blas<true, true, kTriNone>(cfg, g, dA, lda, dB, ldb, R, ldr, epi, h->cus, s);
        return launch_blas<true, false, kTriNone>(cfg, g, dA, lda, dB, ldb, R, ldr, epi, h->cus, s);
    };
    if (!overlap(dC, m, n, ldc, dA, tA ? k : m, tA ? m : k, lda) &&
        !overlap(dC, m, n, ldc, dB, tB ? n : k, tB ? k : n, ldb))
        return walk(dC, ldc);
    // A tile would write C while others still read A or B there.
    const int64_t ldr = even(n);
    void* w = nullptr;
    uvt_status st = uvt_handle_workspace(h, (size_t)m * ldr * 8, &w);
    if (st != UVT_OK) return st;
    double* R = (double*)w;
    if (beta != 0.0) copy(dC, ldc, R, ldr, m, n, s);
    st = walk(R, ldr);
    if (st != UVT_OK) return st;
    copy(R, ldr, dC, ldc, m, n, s);
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

// ---- dtrmm ---------------------------------------------------------------------

// Scratch of uvt_dtrmm_noalloc: a fixed device array, one copy per device,
// held until the process ends.  Host code never passes `scratch` itself to a
// kernel (in host code it is only a stand-in for the device symbol); it uses
// the address hipGetSymbolAddress returned for the handle's device, which
// uvt_noalloc_setup stores in the handle.
constexpr size_t kNoAllocScratchBytes = (size_t)UVT_NOALLOC_SCRATCH_MB << 20;
static __device__ __align__(256) double scratch[kNoAllocScratchBytes / sizeof(double)];

namespace {

std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices];  // per device, set once

// One dtrmm call: the triangle's order nt on w columns (rows, right side) of
// B, and the workspace: B or the result with an even leading dimension.
struct DtrmmCall {
    bool right, tA, lower, unit;  // lower: op(A) is
    int64_t nt, w, ldw;
    size_t bytes;
    // What uvt_dtrmm_noalloc holds against its scratch: result, B where it is
    // transposed or reversed and the triangle where it is not plain lower,
    // each an array of its own.
    size_t declared;
};

// Validates the arguments and sizes the workspace.  UVT_OK with
// *nothing = true when B is empty (no work at all).
uvt_status dtrmm_prepare(uvt_handle h, uvt_side side, uvt_uplo uplo, uvt_trans ta, uvt_diag diag,
                         int64_t m, int64_t n, double alpha, const double* dA, int64_t lda,
                         double* dB, int64_t ldb, DtrmmCall* c, bool* nothing)
{
    *nothing = false;
    if (!h || m < 0 || n < 0) return UVT_ERR_ARG;
    if ((side != UVT_LEFT && side != UVT_RIGHT) || (uplo != UVT_LOWER && uplo != UVT_UPPER) ||
        (ta != UVT_NO_TRANS && ta != UVT_TRANS) || (diag != UVT_NON_UNIT && diag != UVT_UNIT))
        return UVT_ERR_ARG;
    c->right = side == UVT_RIGHT;
    c->nt = c->right ? n : m;  // order of the triangle
    c->w = c->right ? m : n;   // columns of X
    if (lda < std::max<int64_t>(1, c->nt) || ldb < std::max<int64_t>(1, n)) return UVT_ERR_ARG;
    if (m == 0 || n == 0) {
        *nothing = true;
        return UVT_OK;
    }
    if (!dB || (alpha != 0.0 && !dA)) return UVT_ERR_ARG;
    if (!sizes_ok(m, n, 1)) return UVT_ERR_SIZE;
    c->tA = ta == UVT_TRANS;
    c->lower = (uplo == UVT_LOWER) != c->tA;
    c->unit = diag == UVT_UNIT;
    c->ldw = even(n);
    c->bytes = up256((size_t)m * c->ldw * 8);
    const size_t rect = up256((size_t)c->nt * even(c->w) * 8), square = up256((size_t)c->nt * even(c->nt) * 8);
    const bool rev = c->lower == c->right;  // the triangle turned lower by reversal
    c->declared = rect + (c->right || rev ? rect : 0) + (c->tA != c->right || rev || c->unit ? square : 0);
    if (alpha == 0.0) c->bytes = c->declared = 0;  // no workspace: B = 0, A not read
    return UVT_OK;
}

// Enqueues the call on stream s with its workspace at wv.
uvt_status dtrmm_launch(const DtrmmCall& c, int64_t m, int64_t n, double alpha, const double* dA,
                        int64_t lda, double* dB, int64_t ldb, void* wv, int cus, hipStream_t s)
{
    if (alpha == 0.0) {  // B = 0, A not read
        scale(m, n, 0.0, dB, ldb, s);
        UVT_HIP(hipGetLastError());
        return UVT_OK;
    }
    // Where A shares elements with B, B is written only once A has been read.
    double* const W = (double*)wv;
    const bool late = overlap(dB, m, n, ldb, dA, c.nt, c.nt, lda);
    const double* X = late ? dB : W;
    double* R = late ? W : dB;
    const int64_t ldx = late ? ldb : c.ldw, ldr = late ? c.ldw : ldb;
    if (!late) copy(dB, ldb, W, c.ldw, m, n, s);
    const Walk g{m, n, (int)c.nt, 0, 0, cus};
    TileEpi epi;
    epi.alpha = alpha;
    epi.unit = c.unit;
    const auto walk = [&] {
        if (!c.right) {
            const int32_t cfg = uvt_wide_tiles(uvt_default_cfg(m, n), m, n);
            if (c.lower) {
                if (c.tA) return launch_blas<false, false, kTriALe>(cfg, g, dA, lda, X, ldx, R, ldr, epi, cus, s);
                return launch_blas<true, false, kTriALe>(cfg, g, dA, lda, X, ldx, R, ldr, epi, cus, s);
            }
            if (c.tA) return launch_blas<false, false, kTriAGe>(cfg, g, dA, lda, X, ldx, R, ldr, epi, cus, s);
            return launch_blas<true, false, kTriAGe>(cfg, g, dA, lda, X, ldx, R, ldr, epi, cus, s);
        }
        // B op(A): column j of the product needs k >= j where op(A) is lower
        const int32_t cfg = uvt_wide_tiles(uvt_default_cfg(n, m), m, n);
        if (c.lower) {
            if (c.tA) return launch_blas<true, true, kTriBGe>(cfg, g, X, ldx, dA, lda, R, ldr, epi, cus, s);
            return launch_blas<true, false, kTriBGe>(cfg, g, X, ldx, dA, lda, R, ldr, epi, cus, s);
        }
        if (c.tA) return launch_blas<true, true, kTriBLe>(cfg, g, X, ldx, dA, lda, R, ldr, epi, cus, s);
        return launch_blas<true, false, kTriBLe>(cfg, g, X, ldx, dA, lda, R, ldr, epi, cus, s);
    };
    const uvt_status st = walk();
    if (st != UVT_OK) return st;
    if (late) copy(W, c.ldw, dB, ldb, m, n, s);
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

}  // namespace

// Looks up this device's copy of `scratch` once per device (with the device
// current, as uvt_create leaves it) and stores its address in the handle.
uvt_status uvt_noalloc_setup(uvt_handle h)
{
    if (h->device < 0 || h->device >= kMaxDevices) return UVT_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[h->device]) {
        void* p = nullptr;
        UVT_HIP(hipSetDevice(h->device));
        UVT_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return UVT_ERR_HIP;
        g_scratch_ptr[h->device] = p;
    }
    h->scratch = g_scratch_ptr[h->device];
    return UVT_OK;
}

extern "C" uvt_status uvt_dtrmm(uvt_handle h, uvt_side side, uvt_uplo uplo, uvt_trans ta,
                                uvt_diag diag, int64_t m, int64_t n, double alpha,
                                const double* dA, int64_t lda, double* dB, int64_t ldb,
                                void* stream)
{
    DtrmmCall c;
    bool nothing = false;
    uvt_status st = dtrmm_prepare(h, side, uplo, ta, diag, m, n, alpha, dA, lda, dB, ldb, &c, &nothing);
    if (st != UVT_OK || nothing) return st;
    UVT_HIP(hipSetDevice(h->device));
    void* wv = nullptr;
    if (c.bytes) {
        st = uvt_handle_workspace(h, c.bytes, &wv);
        if (st != UVT_OK) return st;
    }
    return dtrmm_launch(c, m, n, alpha, dA, lda, dB, ldb, wv, h->cus, (hipStream_t)stream);
}

extern "C" uvt_status uvt_dtrmm_noalloc(uvt_handle h, uvt_side side, uvt_uplo uplo, uvt_trans ta,
                                        uvt_diag diag, int64_t m, int64_t n, double alpha,
                                        const double* dA, int64_t lda, double* dB, int64_t ldb,
                                        void* stream)
{
    DtrmmCall c;
    bool nothing = false;
    uvt_status st = dtrmm_prepare(h, side, uplo, ta, diag, m, n, alpha, dA, lda, dB, ldb, &c, &nothing);
    if (st != UVT_OK || nothing) return st;
    if (c.declared > kNoAllocScratchBytes) return UVT_ERR_SIZE;
    if (!h->scratch) return UVT_ERR_STATE;
    UVT_HIP(hipSetDevice(h->device));
    return dtrmm_launch(c, m, n, alpha, dA, lda, dB, ldb, h->scratch, h->cus, (hipStream_t)stream);
}
