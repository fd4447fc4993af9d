// uvt_api.hip -- C ABI of libuvt: device handle, FP64 TRMM launches, norm,
// input generators and small runtime helpers.  Declarations: include/uvt.h.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <new>
#include <vector>

#include "uvt_f64_tile.hpp"
#include "uvt_f64_wave.hpp"
#include "uvt_internal.h"
#include "uvt_place.hpp"
#include "uvt_runtime.hpp"
#include "uvt_sk.hpp"

using namespace uvt;

// ---------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------

namespace {  // kernels: internal to this file

// One workgroup of a plan launch: a plan tile (or a piece of its k range)
// and where its product goes: C (part < 0), or partial tile `part`, which a
// later k_add_parts launch adds to C.
struct LaunchTile {
    uvt_tile t;
    int32_t part;
};
// C[r0 + r][c0 + c] += partial tiles first, first + 1, ..., first + count - 1,
// in that order, for rows r < rows of a TM x TN tile.
struct PartSum {
    int32_t r0, rows, c0, first, count;
};

// PARTS: the records are LaunchTiles (some write partial tiles); else plain
// uvt_tiles, every one writing C.  WIDE: see TileOpt.
template <int TM, int TN, bool PARTS, bool WIDE>
__global__ __launch_bounds__((64 * TileWaves<TM, TN>::M * TileWaves<TM, TN>::N),
                             (TileWaves<TM, TN>::WAVES_PER_EU))
void k_trmm_tiles_f64(const void* __restrict__ tiles, const double* __restrict__ A, int64_t lda,
                      const double* __restrict__ B, int64_t ldb, double* __restrict__ C,
                      int64_t ldc, int64_t m, double* __restrict__ parts)
{
    using W = TileWaves<TM, TN>;
    using Opt = TileOpt<true, false, kTriALe, false, false, true, !PARTS, WIDE>;
    __shared__ __attribute__((aligned(16))) double smem[F64Cfg<TM, TN, W::M, W::N, Opt>::SMEM_DOUBLES];
    if constexpr (PARTS) {
        const LaunchTile lt = static_cast<const LaunchTile*>(tiles)[blockIdx.x];
        const uvt_tile& t = lt.t;
        UVT_GLOBAL double* part = lt.part >= 0 ? gbl(parts) + (int64_t)lt.part * (TM * TN) : nullptr;
        f64_tile<TM, TN, W::M, W::N, Opt>(TileArgs{t.r0, t.rows, t.c0, t.k_lo, t.k_hi, t.flags}, gbl(A), lda, gbl(B),
                                          ldb, gbl(C), ldc, m, smem, -1, part);
    } else {
        const uvt_tile t = static_cast<const uvt_tile*>(tiles)[blockIdx.x];
        f64_tile<TM, TN, W::M, W::N, Opt>(TileArgs{t.r0, t.rows, t.c0, t.k_lo, t.k_hi, t.flags}, gbl(A), lda, gbl(B),
                                          ldb, gbl(C), ldc, m, smem);
    }
}

// Adds the partial tiles of each record to C in the record's order (gridDim.y
// workgroups per record, each over its share of the rows; records cover
// disjoint parts of C), so the result does not depend on which workgroup
// finished first.  HBM-bound: 8 bytes per partial value, 16 per value of C
// (one workgroup per record: 35 us of the 383 of 9000 x 250).
__global__ __launch_bounds__(256) void k_add_parts(const PartSum* __restrict__ sums, int tn, int tile,
                                                   const double* __restrict__ parts, double* __restrict__ C,
                                                   int64_t ldc, int64_t m)
{
    const PartSum ps = sums[blockIdx.x];
    const UVT_GLOBAL double* P = gbl(parts) + (int64_t)ps.first * tile;
    const int per = (ps.rows + (int)gridDim.y - 1) / (int)gridDim.y;
    const int e_hi = min(ps.rows, ((int)blockIdx.y + 1) * per) * tn;
    for (int e = (int)blockIdx.y * per * tn + (int)threadIdx.x; e < e_hi; e += 256) {
        const int r = e / tn, c = e % tn;
        if ((int64_t)ps.c0 + c >= m) continue;
        UVT_GLOBAL double* p = gbl(C) + (int64_t)(ps.r0 + r) * ldc + (ps.c0 + c);
        double x = *p;
        int q = 0;
        for (; q + 4 <= ps.count; q += 4) {  // four loads in flight, added in order
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = P[(int64_t)(q + u) * tile + e];
#pragma unroll
            for (int u = 0; u < 4; ++u) x += v[u];
        }
        for (; q < ps.count; ++q) x += P[(int64_t)q * tile + e];
        *p = x;
    }
}

// The trapezoid walk without a tile list: longest reduction first, placed by
// walk_tile (uvt_place.hpp).
template <int TM, int TN>
__global__ __launch_bounds__((64 * TileWaves<TM, TN>::M * TileWaves<TM, TN>::N),
                             (TileWaves<TM, TN>::WAVES_PER_EU))
void k_trmm_trapezoid_f64(int64_t n, int64_t m, int nrt, int nct, int cus, const double* __restrict__ A,
                          int64_t lda, const double* __restrict__ B, int64_t ldb,
                          double* __restrict__ C, int64_t ldc)
{
    using W = TileWaves<TM, TN>;
    __shared__ __attribute__((aligned(16))) double smem[F64Cfg<TM, TN, W::M, W::N>::SMEM_DOUBLES];
    const WalkTile w = walk_tile((int)blockIdx.x, nrt * nct, nct, cus, W::BLOCKS_PER_CU);
    const int r0 = (nrt - 1 - w.outer) * TM;
    const int rows = (int)(n - r0 < TM ? n - r0 : TM);
    f64_tile<TM, TN, W::M, W::N>(TileArgs{r0, rows, w.inner * TN, 0, r0 + rows, kTileLower}, gbl(A), lda, gbl(B), ldb,
                                 gbl(C), ldc, m, smem);
}

// The trapezoid walk of a small product in wave tiles (uvt_f64_wave.hpp), four
// to a workgroup, wn of them along the columns: deepest first, every second
// run of `snake` workgroups turned round (as uvt_place.hpp's).
template <int FM, int FN, int D>
__global__ __launch_bounds__(256) void k_trmm_waves_f64(int64_t n, int64_t m, int nrt, int nct, int wn, int snake,
                                                        const double* __restrict__ A, int64_t lda,
                                                        const double* __restrict__ B, int64_t ldb,
                                                        double* __restrict__ C, int64_t ldc)
{
    int b = (int)blockIdx.x;
    const int g = b / snake;
    if (g & 1) b = g * snake + min((g + 1) * snake, (int)gridDim.x) - 1 - b;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rt = (nrt - 1 - b / nct) * (4 / wn) + wave / wn, ct = b % nct * wn + wave % wn;
    const int64_t r0 = (int64_t)rt * (16 * FM), c0 = (int64_t)ct * (16 * FN);
    __shared__ __attribute__((aligned(16))) double lds[4][wave_lds<FM, FN, TileOpt<>>()];
    if (r0 >= n || c0 >= m) return;
    const int rows = (int)(n - r0 < 16 * FM ? n - r0 : 16 * FM);
    f64_wave<FM, FN, D>(TileArgs{(int)r0, rows, (int)c0, 0, (int)r0 + rows, kTileLower}, gbl(A), lda, gbl(B), ldb,
                        gbl(C), ldc, m, lds[wave]);
}

// The trapezoid walk split stream-K (uvt_sk.hpp): workgroup w of group
// b = w / ncg runs the pieces of panels [b P / G, (b+1) P / G) one after
// another, in column tile w % ncg of each piece's row tile when the launch
// runs column groups; its first piece writes partial tile w if it starts
// inside its tile, every other piece starts at k = 0 and writes C.
template <int TM, int TN, bool WIDE>
__global__ __launch_bounds__((64 * TileWaves<TM, TN>::M * TileWaves<TM, TN>::N),
                             (TileWaves<TM, TN>::WAVES_PER_EU))
void k_trmm_sk_f64(SkGeo g, const double* __restrict__ A, int64_t lda, const double* __restrict__ B,
                   int64_t ldb, double* __restrict__ C, int64_t ldc, double* __restrict__ parts)
{
    using W = TileWaves<TM, TN>;
    using Opt = TileOpt<true, false, kTriALe, false, false, false, false, WIDE>;
    static_assert(kTileK == kSkPanel, "stream-K panels are the kernel's k panels");
    __shared__ __attribute__((aligned(16))) double smem[F64Cfg<TM, TN, W::M, W::N, Opt>::SMEM_DOUBLES];
    // The piece arithmetic (64-bit divisions) runs in vector registers; its
    // results are the same in every lane and go back to scalar registers, so
    // they do not take vector registers from the tile.
    auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    auto uni64 = [&](int64_t v) {
        return (int64_t)(((uint64_t)(uint32_t)uni((int)(v >> 32)) << 32) | (uint32_t)uni((int)v));
    };
    // The 8 XCDs take contiguous runs of the launch, so the workgroups that
    // share an XCD's L2 work on neighbouring tiles, or (column groups) on the
    // same rows of A at the same k.
    const int64_t w = sk_xcd_order(blockIdx.x, sk_launch(g));
    const int64_t b = w / g.ncg;
    const int cx = (int)(w % g.ncg) * TN;  // the member's column tile (0 without groups)
    int64_t x = uni64(sk_start(g, b));
    const int64_t xe = uni64(sk_start(g, b + 1));
    UVT_GLOBAL double* part = gbl(parts) + w * (TM * TN);
    bool first = true;
    while (x < xe) {
        const SkPiece s = sk_piece(g, x, xe);
        if (!first) __syncthreads();  // the LDS tile is reused by the next piece
        // the thread index, opaque per piece: the tile's per-thread offsets are
        // then computed inside each piece instead of held (and spilled) across
        // the piece loop
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        const TileArgs t{uni(s.r0), uni(s.rows), uni(s.c0 + cx), uni(s.k_lo), uni(s.k_hi), kTileLower};
        f64_tile<TM, TN, W::M, W::N, Opt>(t, gbl(A), lda, gbl(B), ldb, gbl(C), ldc, g.m, smem, tid,
                                          uni(s.p0 > 0) ? part : nullptr);
        first = false;
        x = uni64(s.next);
    }
}

// After k_trmm_sk_f64: for each tile split between workgroups, the
// workgroup b whose first piece is the tile's first partial tile adds
// partial tiles b, b+1, ... (k order) to C, which holds the k = 0 piece; with
// column groups, group b's member in each column tile does so in that column
// tile.  (gridDim.y workgroups per split tile, each over its share of the rows.)
template <int TM, int TN>
__global__ __launch_bounds__(256) void k_sk_fixup(SkGeo g, const double* __restrict__ parts,
                                                  double* __restrict__ C, int64_t ldc)
{
    const int64_t w = blockIdx.x;  // partial tile w: group b, column tile cx
    const int64_t b = w / g.ncg, cx = w % g.ncg;
    if (b == 0) return;
    const int64_t x = sk_start(g, b);
    const int j = sk_row(g, x);
    const int64_t d = sk_depth(g, j), off = x - sk_before(g, j), p0 = off % d;
    if (p0 == 0) return;                     // b starts its tile: it wrote C
    const int64_t tile0 = x - p0;
    if (sk_start(g, b - 1) > tile0) return;  // b - 1 holds this tile's first partial tile
    int64_t cnt = 1;
    while (b + cnt < g.G && sk_start(g, b + cnt) < tile0 + d) ++cnt;
    const int r0 = j * TM, rows = (int)(g.n - r0 < TM ? g.n - r0 : TM);
    const int64_t c0 = (off / d + cx) * TN;
    const UVT_GLOBAL double* P = gbl(parts) + w * (TM * TN);
    const int64_t step = g.ncg * (int64_t)(TM * TN);  // group b + q's partial tile in this column tile
    const int per = (rows + (int)gridDim.y - 1) / (int)gridDim.y;
    const int e_lo = (int)blockIdx.y * per * TN;
    const int e_hi = min(rows, ((int)blockIdx.y + 1) * per) * TN;
    for (int e = e_lo + (int)threadIdx.x; e < e_hi; e += 256) {
        const int r = e / TN, c = e % TN;
        if (c0 + c >= g.m) continue;
        UVT_GLOBAL double* p = gbl(C) + (int64_t)(r0 + r) * ldc + (c0 + c);
        double v = *p;
        for (int64_t q = 0; q < cnt; ++q) v += P[q * step + e];
        *p = v;
    }
}

// sum_j |c[j]| by one wave: lanes strided over columns, then a fixed
// butterfly, so the order (and the result) is the same on every run.
__device__ __forceinline__ double wave_abs_sum(const UVT_GLOBAL double* c, int64_t m, int lane)
{
    double s = 0.0;
    for (int64_t j = lane; j < m; j += 16 * 64) {  // sixteen loads in flight, added in order
        double v[16];
        if (j + 15 * 64 < m) {
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = c[j + 64 * u];
        } else {
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = j + 64 * u < m ? c[j + 64 * u] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) s += fabs(v[u]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    return s;
}

// One wave per row.
__global__ __launch_bounds__(256) void k_row_abs_sums(int64_t n, int64_t m,
                                                      const double* __restrict__ C, int64_t ldc,
                                                      double* __restrict__ out)
{
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= n) return;
    const double s = wave_abs_sum(gbl(C) + row * ldc, m, lane);
    if (lane == 0) out[row] = s;
}

// max_i sum_j |C[i][j]| in one launch, HBM-bound: every wave keeps the largest
// of its rows, every workgroup leaves one value in part, and the last one to
// finish (done, left at zero again) writes the largest to host memory.  (Row
// sums, a second launch for their maximum and a copy of 8 bytes took 21 us on
// the GPU at 2048 x 2048, and the host waited for each in turn.)
constexpr int kNormBlocks = 512, kNormWaves = 8;
__global__ __launch_bounds__(64 * kNormWaves) void k_inf_norm(int64_t n, int64_t m, const double* __restrict__ C, int64_t ldc,
                                                  double* __restrict__ part, unsigned* __restrict__ done,
                                                  double* __restrict__ out)
{
    __shared__ double best[kNormWaves];
    __shared__ bool last;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto block_max = [&](double v) {  // over the waves' values, in thread 0
        if (lane == 0) best[wave] = v;
        __syncthreads();
        for (int w = 1; w < kNormWaves; ++w) v = fmax(v, best[w]);
        return v;
    };
    double x = 0.0;
    for (int64_t row = (int64_t)blockIdx.x * kNormWaves + wave; row < n; row += (int64_t)gridDim.x * kNormWaves)
        x = fmax(x, wave_abs_sum(gbl(C) + row * ldc, m, lane));
    x = block_max(x);
    if (threadIdx.x == 0) {
        __hip_atomic_store(&part[blockIdx.x], x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1 == gridDim.x;
    }
    __syncthreads();
    if (!last) return;
    x = 0.0;
    for (int i = threadIdx.x; i < (int)gridDim.x; i += 64 * kNormWaves)
        x = fmax(x, __hip_atomic_load(&part[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x = fmax(x, __shfl_xor(x, off, 64));
    x = block_max(x);
    if (threadIdx.x == 0) {
        __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(out, x, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// mat_consecutive_values with MININUMS=1 (UVaTRMM/src/mm_triangular_common.c:1782-1805):
// value index row*n + column modulo VALUES_LIMIT=2341, plus one, reciprocal.
__global__ void k_fill_closed(int64_t n, int64_t rows, int64_t cols, int lower,
                              double* __restrict__ X, int64_t ldx)
{
    for (int64_t i = blockIdx.y; i < rows; i += gridDim.y)
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < cols;
         j += (int64_t)gridDim.x * blockDim.x) {
        double v;
        if (lower && j > i) {
            v = 0.0;
        } else {
            const int64_t idx = i * n + j;
            v = 1.0 / (double)(idx % 2341 + 1);
        }
        X[i * ldx + j] = v;
    }
}

__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

// Seeded generator, bit-identical to the host one: SplitMix64 (Steele, Lea,
// Flood 2014) applied to key + (idx+1)*gamma; 53 random bits -> U[-1,1);
// optional +2 on the diagonal; optional exact 2^e scaling, e in {-8..8}.
__global__ void k_fill_seeded(int64_t rows, int64_t cols, uint64_t key, int stream_is_a,
                              int spread, double* __restrict__ X, int64_t ldx)
{
    const uint64_t gamma = 0x9E3779B97F4A7C15ULL;
    for (int64_t i = blockIdx.y; i < rows; i += gridDim.y)
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < cols;
         j += (int64_t)gridDim.x * blockDim.x) {
        double v;
        if (stream_is_a && j > i) {
            v = 0.0;
        } else {
            const uint64_t idx = (uint64_t)(i * cols + j);
            const uint64_t z = mix64(key + (idx + 1) * gamma);
            const double u = (double)(z >> 11) * 0x1.0p-53;
            v = 2.0 * u - 1.0;
            if (stream_is_a && i == j) v = v + 2.0;
            if (spread) {
                const int e = (int)(mix64(z) % 17) - 8;
                v = v * __longlong_as_double((long long)((uint64_t)(1023 + e) << 52));
            }
        }
        X[i * ldx + j] = v;
    }
}

}  // namespace

// ---------------------------------------------------------------------
// Handle
// ---------------------------------------------------------------------

extern "C" uvt_status uvt_create(int device, uvt_handle* out)
{
    if (!out) return UVT_ERR_ARG;
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return UVT_ERR_UNSUPPORTED;
    if (device < 0 || device >= count) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(device));
    hipDeviceProp_t prop;
    UVT_HIP(hipGetDeviceProperties(&prop, device));
    uvt_handle h = new (std::nothrow) uvt_handle_s();  // zeros
    if (!h) return UVT_ERR_NOMEM;
    h->device = device;
    h->cus = prop.multiProcessorCount;
    h->vram = prop.totalGlobalMem;
    const uvt_status st = uvt_noalloc_setup(h);
    if (st != UVT_OK) {
        delete h;
        return st;
    }
    *out = h;
    return UVT_OK;
}

static void norm_free(uvt_handle h)
{
    if (h->norm_part) (void)hipFree(h->norm_part);
    if (h->norm_host) (void)hipHostFree(h->norm_host);
    h->norm_part = h->norm_host = nullptr;
}

extern "C" uvt_status uvt_destroy(uvt_handle h)
{
    if (!h) return UVT_ERR_ARG;
    (void)hipSetDevice(h->device);
    if (h->work) (void)hipFree(h->work);
    norm_free(h);
    for (int i = 0; i < 2; ++i) {
        if (h->pin_done[i]) (void)hipEventSynchronize(h->pin_done[i]);
        if (h->pin[i]) (void)hipHostFree(h->pin[i]);
        if (h->pin_done[i]) (void)hipEventDestroy(h->pin_done[i]);
    }
    delete h;
    return UVT_OK;
}

extern "C" int32_t uvt_device_cus(uvt_handle h) { return h ? h->cus : 0; }

uvt_status uvt_handle_workspace(uvt_handle h, size_t bytes, void** p)
{
    if (h->work_bytes < bytes) {
        if (h->work) {
            UVT_HIP(hipDeviceSynchronize());
            UVT_HIP(hipFree(h->work));
            h->work = nullptr;
            h->work_bytes = 0;
        }
        if (hipMalloc(&h->work, bytes) != hipSuccess) {
            (void)hipGetLastError();
            return UVT_ERR_NOMEM;
        }
        h->work_bytes = bytes;
    }
    *p = h->work;
    return UVT_OK;
}

// ---------------------------------------------------------------------
// Plans on the device
// ---------------------------------------------------------------------

extern "C" void uvt_plan_release_device(uvt_plan plan)
{
    if (!plan) return;
    void** bufs[3] = {&plan->dev_launch, &plan->dev_sums, &plan->dev_parts};
    for (void** b : bufs) {
        if (*b) {
            (void)hipSetDevice(plan->dev_id);
            (void)hipFree(*b);
            *b = nullptr;
        }
    }
    plan->nlaunch = plan->nsums = plan->nparts = plan->sk_grid = 0;
    plan->dev_id = -1;
}

namespace {

constexpr size_t kMaxPartBytes = (size_t)64 << 20;  // partial tiles of one plan
// Below this many flops a plan's launch time, not one tile's depth, bounds
// it, and the plan keeps whole tiles.
constexpr double kSplitMinFlops = 2e9;
// Stream-K walks run column groups (uvt_sk.hpp) where there are at least 8 of
// them.  Measured against one sequence over every tile (three alternating
// passes, one box): 8192 x 1024 1.20 -> 1.18 ms, 8165 x 939 1.30 -> 1.29 ms,
// 6772 x 1548 and 5000 x 2000 within 1 % either way.
constexpr bool kSkGroupCols = true;

int blocks_per_cu(int32_t cfg)
{
    if (cfg == UVT_CFG_256x128) return TileWaves<256, 128>::BLOCKS_PER_CU;
    if (cfg == UVT_CFG_64x64) return TileWaves<64, 64>::BLOCKS_PER_CU;
    if (cfg == UVT_CFG_128x32) return TileWaves<128, 32>::BLOCKS_PER_CU;
    return TileWaves<128, 128>::BLOCKS_PER_CU;
}

// The launch of a plan on a GPU of `cus` compute units: the whole tiles of the
// trapezoid walk, for either shape.  (A boxes plan's triangles were a second
// launch, which read and wrote C once more and waited for the first: N=2048,
// 4 bands, product and norm 193 us; now 170.)  Except for a plan whose longest
// reduction is much longer than an even share of the work would give a
// workgroup slot (narrow B, few tiles: the launch then lasts as long as its
// deepest tile).  Such a plan cuts every reduction longer than about half
// that share, kc, into pieces that run at once: the first piece writes C,
// the others write partial tiles, which k_add_parts adds to C afterwards in
// k order.  Measured at 9000 x 250 (the deepest tile 2.7x the share): 0.73
// -> 0.45 ms; at 4096 x 4096 (0.97x) cutting cost 7 %, between 0.9x and
// 1.6x it changed -1 to +7 %, so plans below 1.5x keep whole tiles (and the
// kernel without partial tiles); 64x64 tiles count three slots to a compute
// unit here, as those figures did, though four fit.  (A plan of 128x128 tiles
// whose whole tiles would not finish together runs stream-K instead, decided
// before this in plan_upload; so cuts serve the smaller tile shapes, where
// they were faster than stream-K.)
void build_launch(const uvt_plan_s& pl, int cus, std::vector<LaunchTile>& launch, std::vector<PartSum>& sums,
                  int64_t& nparts)
{
    launch.clear();
    sums.clear();
    nparts = 0;
    std::vector<uvt_tile> walk(uvt_plan_trapezoid_tiles(pl.n, pl.m, pl.cfg, nullptr));
    uvt_plan_trapezoid_tiles(pl.n, pl.m, pl.cfg, walk.data());  // deepest first
    const int64_t total = (int64_t)walk.size();
    const int nct = (int)((pl.m + uvt_cfg_tile_n(pl.cfg) - 1) / uvt_cfg_tile_n(pl.cfg));
    for (int64_t b = 0; b < total; ++b) {
        WalkTile w{(int)(b / nct), (int)(b % nct)};
        if (total <= 0x7FFFFFFF) w = walk_tile((int)b, (int)total, nct, cus, blocks_per_cu(pl.cfg));  // else not launched
        launch.push_back(LaunchTile{walk[(int64_t)w.outer * nct + w.inner], -1});
    }
    if (pl.flops < kSplitMinFlops || uvt_cfg_tile_n(pl.cfg) >= 128) return;
    int64_t work = 0, deepest = 0;  // k steps, summed over the tiles and the longest
    for (const uvt_tile& w : walk) {
        const int64_t len = (int64_t)w.k_hi - w.k_lo;
        work += len;
        deepest = len > deepest ? len : deepest;
    }
    const int64_t share = work / ((int64_t)cus * std::min(blocks_per_cu(pl.cfg), 3));
    if (2 * deepest < 3 * share) return;
    int64_t kc = (share / 2 + 127) / 128 * 128;
    kc = kc < 512 ? 512 : kc;
    std::vector<LaunchTile> cut;
    std::vector<PartSum> cut_sums;
    int64_t cut_parts = 0;
    for (const uvt_tile& t : walk) {
        const int64_t len = (int64_t)t.k_hi - t.k_lo;
        const int64_t np = len > kc ? (len + kc - 1) / kc : 1;
        if (np == 1) {
            cut.push_back(LaunchTile{t, -1});
            continue;
        }
        // piece boundaries on whole 16-deep panels, as even as that allows
        cut_sums.push_back(PartSum{t.r0, t.rows, t.c0, (int32_t)cut_parts, (int32_t)(np - 1)});
        for (int64_t q = 0; q < np; ++q) {
            uvt_tile piece = t;
            piece.k_lo = q == 0 ? t.k_lo : (int32_t)(t.k_lo + (len * q / np) / 16 * 16);
            piece.k_hi = q == np - 1 ? t.k_hi : (int32_t)(t.k_lo + (len * (q + 1) / np) / 16 * 16);
            cut.push_back(LaunchTile{piece, q == 0 ? -1 : (int32_t)cut_parts++});
        }
    }
    const size_t tile_bytes = (size_t)uvt_cfg_tile_m(pl.cfg) * uvt_cfg_tile_n(pl.cfg) * sizeof(double);
    if ((size_t)cut_parts * tile_bytes > kMaxPartBytes) return;
    // Deepest first, and of the pieces of one depth those that read the same
    // part of A (one for each column tile) one after another; then every 8 such
    // groups are dealt out to the XCDs, a group to each.  (A piece's column
    // neighbours on other XCDs each read A from memory: 9000 x 250 381 us, now
    // 367; 5000 x 300 158 and 151; 12000 x 128 350 and 342.)
    std::stable_sort(cut.begin(), cut.end(), [](const LaunchTile& a, const LaunchTile& b) {
        const int32_t la = a.t.k_hi - a.t.k_lo, lb = b.t.k_hi - b.t.k_lo;
        if (la != lb) return la > lb;
        return a.t.r0 != b.t.r0 ? a.t.r0 > b.t.r0 : a.t.k_lo < b.t.k_lo;
    });
    std::vector<LaunchTile> dealt;
    const int64_t run = (int64_t)kXcds * nct, full = (int64_t)cut.size() / run * run;
    for (int64_t i = 0; i < full; ++i) dealt.push_back(cut[i / run * run + i % kXcds * nct + i % run / kXcds]);
    cut.erase(cut.begin(), cut.begin() + full);
    dealt.insert(dealt.end(), cut.begin(), cut.end());
    cut.swap(dealt);
    launch.swap(cut);
    sums.swap(cut_sums);
    nparts = cut_parts;
}

}  // namespace

static uvt_status plan_upload(uvt_handle h, uvt_plan plan)
{
    if (plan->dev_id == h->device) return UVT_OK;
    uvt_plan_release_device(plan);
    // A plan whose whole tiles would not finish together runs stream-K:
    // nothing to upload but its partial tiles.
    const int64_t sk = uvt_sk_workgroups(plan->cfg, plan->n, plan->m, h->cus);
    if (sk > 0) {
        if (hipMalloc(&plan->dev_parts, uvt_sk_parts_bytes(plan->cfg, sk)) != hipSuccess) {
            (void)hipGetLastError();
            plan->dev_parts = nullptr;
            return UVT_ERR_NOMEM;
        }
        plan->dev_id = h->device;
        plan->sk_grid = sk;
        const SkGeo g =
            sk_geometry(plan->n, plan->m, uvt_cfg_tile_m(plan->cfg), uvt_cfg_tile_n(plan->cfg), sk, kSkGroupCols);
        for (int64_t b = 1; b < g.G; ++b)
            if (sk_piece(g, sk_start(g, b), sk_start(g, b + 1)).p0 > 0) plan->nparts += g.ncg;
        return UVT_OK;
    }
    std::vector<LaunchTile> launch;
    std::vector<PartSum> sums;
    int64_t nparts = 0;
    build_launch(*plan, h->cus, launch, sums, nparts);
    auto upload = [&](void** dst, const void* src, size_t bytes) -> uvt_status {
        if (!bytes) return UVT_OK;
        if (hipMalloc(dst, bytes) != hipSuccess) {
            (void)hipGetLastError();
            return UVT_ERR_NOMEM;
        }
        if (src && hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipGetLastError();
            return UVT_ERR_HIP;
        }
        return UVT_OK;
    };
    plan->dev_id = h->device;  // what is allocated below belongs to this device
    uvt_status st = UVT_OK;
    if (nparts > 0) {
        st = upload(&plan->dev_launch, launch.data(), launch.size() * sizeof(LaunchTile));
    } else {  // whole tiles: the plain records of the kernel without partial tiles
        std::vector<uvt_tile> plain;
        for (const LaunchTile& lt : launch) plain.push_back(lt.t);
        st = upload(&plan->dev_launch, plain.data(), plain.size() * sizeof(uvt_tile));
    }
    plan->nlaunch = (int64_t)launch.size();
    if (st == UVT_OK) st = upload(&plan->dev_sums, sums.data(), sums.size() * sizeof(PartSum));
    plan->nsums = (int64_t)sums.size();
    const int32_t tm = uvt_cfg_tile_m(plan->cfg), tn = uvt_cfg_tile_n(plan->cfg);
    if (st == UVT_OK) st = upload(&plan->dev_parts, nullptr, (size_t)nparts * tm * tn * sizeof(double));
    plan->nparts = nparts;
    if (st != UVT_OK) uvt_plan_release_device(plan);
    return st;
}

// ---------------------------------------------------------------------
// FP64 TRMM
// ---------------------------------------------------------------------

// Whether tiles of this shape have full panels with these leading dimensions
// (else: TileOpt::WIDE).
static bool full_panels_fit(int32_t cfg, int64_t lda, int64_t ldb)
{
    const int32_t rows = uvt_cfg_tile_m(cfg);
    return (rows == 256   ? PanelIdx<256, 64, true>::offsets_fit(lda)
            : rows == 128 ? PanelIdx<128, 64, true>::offsets_fit(lda)
                          : PanelIdx<64, 64, true>::offsets_fit(lda)) &&
           PanelIdx<128, 64, false>::offsets_fit(ldb);
}

// parts == nullptr: dtiles holds uvt_tiles; else LaunchTiles.
template <int TM, int TN, bool WIDE>
static void launch_tiles(const void* dtiles, int64_t ntiles, const double* A, int64_t lda, const double* B,
                         int64_t ldb, double* C, int64_t ldc, int64_t m, double* parts, hipStream_t s)
{
    const dim3 grid((unsigned)ntiles), block(64 * TileWaves<TM, TN>::M * TileWaves<TM, TN>::N);
    if constexpr (TN < 128) {  // only these are cut (build_launch)
        if (parts) {
            hipLaunchKernelGGL((k_trmm_tiles_f64<TM, TN, true, WIDE>), grid, block, 0, s, dtiles, A, lda, B, ldb, C,
                               ldc, m, parts);
            return;
        }
    }
    hipLaunchKernelGGL((k_trmm_tiles_f64<TM, TN, false, WIDE>), grid, block, 0, s, dtiles, A, lda, B, ldb, C, ldc, m,
                       parts);
}

static uvt_status launch_tiles_f64(int32_t cfg, const void* dtiles, int64_t ntiles,
                                   const double* A, int64_t lda, const double* B, int64_t ldb,
                                   double* C, int64_t ldc, int64_t m, double* parts, hipStream_t s)
{
    if (ntiles <= 0) return UVT_OK;
    if (ntiles > 0x7FFFFFFF) return UVT_ERR_SIZE;
    const auto launch = [&](auto wide) {
        constexpr bool W = decltype(wide)::value;
        if (cfg == UVT_CFG_256x128) launch_tiles<256, 128, W>(dtiles, ntiles, A, lda, B, ldb, C, ldc, m, parts, s);
        else if (cfg == UVT_CFG_64x64) launch_tiles<64, 64, W>(dtiles, ntiles, A, lda, B, ldb, C, ldc, m, parts, s);
        else if (cfg == UVT_CFG_128x32)  // WIDE: an A of 235 GB or more
            launch_tiles<128, 32, false>(dtiles, ntiles, A, lda, B, ldb, C, ldc, m, parts, s);
        else launch_tiles<128, 128, W>(dtiles, ntiles, A, lda, B, ldb, C, ldc, m, parts, s);
    };
    if (full_panels_fit(cfg, lda, ldb)) launch(std::false_type{});
    else launch(std::true_type{});
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

template <int TM, int TN>
static void launch_trapezoid(int64_t n, int64_t m, const double* A, int64_t lda, const double* B, int64_t ldb,
                             double* C, int64_t ldc, int cus, hipStream_t s)
{
    const int nrt = (int)((n + TM - 1) / TM), nct = (int)((m + TN - 1) / TN);
    const dim3 grid((unsigned)((int64_t)nrt * nct)), block(64 * TileWaves<TM, TN>::M * TileWaves<TM, TN>::N);
    hipLaunchKernelGGL((k_trmm_trapezoid_f64<TM, TN>), grid, block, 0, s, n, m, nrt, nct, cus, A, lda, B,
                       ldb, C, ldc);
}

// When a product runs in wave tiles, and in which (0: workgroup tiles): a rule
// on the 16x16 tiles of C and the flops.  Measured on MI355X, 68 shapes from
// 64 x 16 to 32000 x 32 (us; workgroup tiles / wave tiles of 16x16, 16x32,
// 32x32):
//     257 x 257      14.3 /   5.9    7.5   13.5     (289 tiles of 16x16)
//    1000 x 200      43.3 /  15.7   20.2   39.5     (819)
//     700 x 700      32.7 /  14.8   16.7   30.5     (1936)
//     400 x 1600     20.5 /  11.6   12.2   19.1     (2500)
//    1024 x 1024     44.9 /  28.7   22.9   42.0     (4096)
//    1200 x 1200     52.4 /  48.3   39.5   49.3     (5625)
//    1600 x 1600     98.4 / 108     91.7   80.0     (10000)
//    1800 x 1800    127   / 182    159    123       (12769)
//    2048 x 2048    136   / 202    154    155       (16384)
// and, deep and narrow, where a plan's workgroup tiles cut their reductions:
//    3000 x 300      67.1 /  89.3   65.2  116       (2.7e9 flops)
//    4000 x 250      88.9 / 114     80.2  152       (4.0e9)
//    5000 x 96       73.7 /  69.6   88.2  187       (2.4e9)
//    5000 x 160      93.6 / 117     91.2  188       (4.0e9)
//    5000 x 250     124   / 192    139    190       (6.2e9)
//    4000 x 400     136   / 183    143    154       (6.4e9)
// Small tiles share less per load, so each size's waves go from 16x16 to
// 16x32 to 32x32 as there are enough of them for every SIMD; 32x32 ones need
// reductions to spread (400 x 8192: 35.3 us in workgroup tiles, 34.4 in
// 16x32, 40.5 in 32x32).
int uvt_wave_shape(int64_t n, int64_t m, int64_t lda, int64_t ldb)
{
    const int64_t tiles = ((n + 15) / 16) * ((m + 15) / 16);
    const double flops = (double)m * (double)n * (double)n;
    if (n > 32768 || tiles > 13000 || flops >= (tiles > 7500 ? 8e9 : 6e9)) return 0;
    if (tiles <= 2500) return 11;
    if (tiles <= 7500 || n < 512) return 12;
    // Without full panels (rows of 128 MB or longer) 32x32 tiles lose: 1500 x
    // 1500 220 us, 136 in workgroup tiles; smaller tiles do not: 1024 x 400 40
    // and 82, 1200 x 1200 79 and 97.
    return WaveIdx<2, true>::fits(lda) && WaveIdx<2, false>::fits(ldb) ? 22 : 0;
}

namespace {

// Workgroups of four waves: wn of them along the columns, the rest along the
// rows.
struct WaveGrid {
    int nrt, nct, wn;
    int64_t launch() const { return (int64_t)nrt * nct; }
};
WaveGrid wave_grid(int shape, int64_t n, int64_t m)
{
    const int64_t tm = 16 * (shape / 10), tn = 16 * (shape % 10);
    const int64_t rt = (n + tm - 1) / tm, ct = (m + tn - 1) / tn;
    const int wn = ct > 1 ? 2 : 1, wm = 4 / wn;
    return WaveGrid{(int)((rt + wm - 1) / wm), (int)((ct + wn - 1) / wn), wn};
}

template <int FM, int FN, int D>
void launch_waves(int64_t n, int64_t m, const double* A, int64_t lda, const double* B, int64_t ldb, double* C,
                  int64_t ldc, int cus, hipStream_t s)
{
    const WaveGrid g = wave_grid(10 * FM + FN, n, m);
    hipLaunchKernelGGL((k_trmm_waves_f64<FM, FN, D>), dim3((unsigned)g.launch()), dim3(256), 0, s, n, m, g.nrt, g.nct,
                       g.wn, cus, A, lda, B, ldb, C, ldc);
}

}  // namespace

uvt_status uvt_launch_waves_f64(int shape, int64_t n, int64_t m, const double* A, int64_t lda, const double* B,
                                int64_t ldb, double* C, int64_t ldc, int cus, hipStream_t s)
{
    if (n <= 0 || m <= 0 || lda < n || ldb < m || ldc < m) return UVT_ERR_ARG;
    if (shape == 11) launch_waves<1, 1, 4>(n, m, A, lda, B, ldb, C, ldc, cus, s);
    else if (shape == 12) launch_waves<1, 2, 4>(n, m, A, lda, B, ldb, C, ldc, cus, s);
    else launch_waves<2, 2, 2>(n, m, A, lda, B, ldb, C, ldc, cus, s);
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

template <int TM, int TN, bool WIDE>
static void launch_trapezoid_sk(const SkGeo& g, const double* A, int64_t lda, const double* B, int64_t ldb,
                                double* C, int64_t ldc, double* parts, hipStream_t s)
{
    const dim3 grid((unsigned)sk_launch(g)), block(64 * TileWaves<TM, TN>::M * TileWaves<TM, TN>::N);
    hipLaunchKernelGGL((k_trmm_sk_f64<TM, TN, WIDE>), grid, block, 0, s, g, A, lda, B, ldb, C, ldc, parts);
    hipLaunchKernelGGL((k_sk_fixup<TM, TN>), dim3((unsigned)sk_launch(g), 4), dim3(256), 0, s, g, parts, C, ldc);
}

namespace {

// When the trapezoid walk runs stream-K (measured on MI355X, 26 shapes from
// 1500 x 1500 to 16384 x 4096 against whole tiles): with 128x128 tiles whose
// whole-tile span is 1.4-2.0x an even share (narrow B: 512-700 deep tiles on
// 512 slots), stream-K took 0.73-0.97x the time (3000 x 3500 at 1.42x: 1.0x);
// where whole tiles balance (span 1.0-1.1x) it took 1.05-1.23x, because its
// workgroups no longer go through k together and share less in L2; with 64x64
// tiles it took 1.02-1.25x at any span (there the partial-tile cut of the
// plan path is faster).  More workgroups than slots (2x, 4x) did not help.
constexpr double kSkMinFlops = 2e9;  // below: launch time, not balance, bounds a walk
constexpr double kSkGain = 1.3;      // whole-tile span over an even share that stream-K needs
                                     // (with column groups: 1-14 % slower up to 1.23, 2 % faster at 1.29)

// How long whole tiles take, in panels per workgroup slot: the launch hands
// tiles, deepest first, to the slot that frees first (list scheduling).
int64_t whole_tile_panels(const SkGeo& g, int64_t slots)
{
    std::vector<int64_t> heap(slots, 0);  // min-heap of the slots' finish times
    auto later = [](int64_t a, int64_t b) { return a > b; };
    int64_t span = 0;
    for (int j = g.nrt - 1; j >= 0; --j) {
        const int64_t d = sk_depth(g, j);
        for (int c = 0; c < g.nct; ++c) {
            std::pop_heap(heap.begin(), heap.end(), later);
            heap.back() += d;
            span = std::max(span, heap.back());
            std::push_heap(heap.begin(), heap.end(), later);
        }
    }
    return span;
}

}  // namespace

int64_t uvt_sk_workgroups(int32_t cfg, int64_t n, int64_t m, int cus)
{
    if (cfg != UVT_CFG_128x128 || (double)m * (double)n * (double)n < kSkMinFlops || n > 0x3FFFFFFF ||
        m > 0x3FFFFFFF)
        return 0;
    const int tm = uvt_cfg_tile_m(cfg), tn = uvt_cfg_tile_n(cfg);
    const int64_t slots = (int64_t)cus * blocks_per_cu(cfg);
    const SkGeo g = sk_geometry(n, m, tm, tn, slots);
    const int64_t tiles = (int64_t)g.nrt * g.nct;
    if (tiles > 16 * slots || g.G < slots) return 0;  // many tiles balance by themselves
    const int64_t even = (g.P + slots - 1) / slots;
    // List scheduling never takes longer than an even share plus the deepest
    // tile (Graham 1969), so with a deepest tile below (kSkGain - 1) x the
    // share the span cannot reach kSkGain x: no need to simulate it.
    if ((double)sk_depth(g, g.nrt - 1) < (kSkGain - 1.0) * (double)even) return 0;
    return (double)whole_tile_panels(g, slots) >= kSkGain * (double)even ? slots : 0;
}

size_t uvt_sk_parts_bytes(int32_t cfg, int64_t workgroups)
{
    return (size_t)workgroups * uvt_cfg_tile_m(cfg) * uvt_cfg_tile_n(cfg) * sizeof(double);
}

size_t uvt_sk_max_parts_bytes(int cus)
{
    return uvt_sk_parts_bytes(UVT_CFG_128x128, (int64_t)cus * blocks_per_cu(UVT_CFG_128x128));
}

uvt_status uvt_launch_trapezoid_sk_f64(int32_t cfg, int64_t n, int64_t m, const double* A, int64_t lda,
                                       const double* B, int64_t ldb, double* C, int64_t ldc,
                                       int64_t workgroups, double* parts, hipStream_t s)
{
    if (n <= 0 || m <= 0 || lda < n || ldb < m || ldc < m || workgroups <= 0 || !parts) return UVT_ERR_ARG;
    if (cfg != UVT_CFG_128x128) return UVT_ERR_ARG;  // stream-K runs 128x128 tiles (uvt_sk_workgroups)
    if (n > 0x3FFFFFFF || m > 0x3FFFFFFF || workgroups > 0x7FFFFFFF) return UVT_ERR_SIZE;
    const SkGeo g = sk_geometry(n, m, uvt_cfg_tile_m(cfg), uvt_cfg_tile_n(cfg), workgroups, kSkGroupCols);
    if (full_panels_fit(cfg, lda, ldb)) launch_trapezoid_sk<128, 128, false>(g, A, lda, B, ldb, C, ldc, parts, s);
    else launch_trapezoid_sk<128, 128, true>(g, A, lda, B, ldb, C, ldc, parts, s);
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

uvt_status uvt_launch_trapezoid_f64(int32_t cfg, int64_t n, int64_t m, const double* A, int64_t lda,
                                    const double* B, int64_t ldb, double* C, int64_t ldc, int cus,
                                    hipStream_t s)
{
    if (n <= 0 || m <= 0 || lda < n || ldb < m || ldc < m) return UVT_ERR_ARG;
    if (n > 0x3FFFFFFF || m > 0x3FFFFFFF) return UVT_ERR_SIZE;
    const int64_t tm = uvt_cfg_tile_m(cfg), tn = uvt_cfg_tile_n(cfg);
    if (((n + tm - 1) / tm) * ((m + tn - 1) / tn) > 0x7FFFFFFF) return UVT_ERR_SIZE;
    if (cfg == UVT_CFG_256x128) launch_trapezoid<256, 128>(n, m, A, lda, B, ldb, C, ldc, cus, s);
    else if (cfg == UVT_CFG_64x64) launch_trapezoid<64, 64>(n, m, A, lda, B, ldb, C, ldc, cus, s);
    else if (cfg == UVT_CFG_128x32) launch_trapezoid<128, 32>(n, m, A, lda, B, ldb, C, ldc, cus, s);
    else launch_trapezoid<128, 128>(n, m, A, lda, B, ldb, C, ldc, cus, s);
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

// Whether a plan that could run in wave tiles runs in workgroup tiles all the
// same: one whose reductions those cut (build_launch) and are so deep that a
// wave alone takes longer over its own.  us, cut workgroup tiles / wave tiles
// of 16x16 / 16x32:
//     6000 x 64       57.8 /  73.9 / 102      (2.3e9 flops)
//     6000 x 96       93.8 /  91.2 / 106      (3.5e9)
//     6000 x 160     127   / 158   / 122      (5.8e9)
//     7000 x 48       79.4 /  89.4 / 119      (2.4e9)
//     7000 x 96      118   / 132   / 123      (4.7e9)
//     9000 x 31       84.1 / 205   / 210      (2.5e9; uncut before: 153)
//    12500 x 33      227   / 435   / 321      (5.2e9)
//    16000 x 16      217   / 308   / 320      (4.1e9)
//    22000 x 9       413   / 450              (4.4e9)
//    26000 x 7       562   / 581              (4.7e9)
//    28000 x 7       653   / 640              (5.5e9; the reads of A bound both)
// and below 2e9 flops, where nothing is cut:
//     8000 x 31      406   / 133   / 158
//    10000 x 16      558   / 177   / 190
static bool deep_and_narrow(const uvt_plan_s& pl)
{
    return pl.n >= 7000 && pl.n < 27000 && pl.flops >= kSplitMinFlops;
}

extern "C" uvt_status uvt_trmm_f64(uvt_handle h, uvt_plan plan, const double* dA, int64_t lda,
                                   const double* dB, int64_t ldb, double* dC, int64_t ldc,
                                   void* stream)
{
    if (!h || !plan || !dA || !dB || !dC) return UVT_ERR_ARG;
    if (lda < plan->n || ldb < plan->m || ldc < plan->m) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    hipStream_t s = (hipStream_t)stream;
    // Wave tiles take no device memory: a deep plan without its records yet
    // runs in them too where memory cannot be had (none left, or a capture).
    const int shape = uvt_wave_shape(plan->n, plan->m, lda, ldb);
    const auto waves = [&] {
        return uvt_launch_waves_f64(shape, plan->n, plan->m, dA, lda, dB, ldb, dC, ldc, h->cus, s);
    };
    if (shape && !deep_and_narrow(*plan)) return waves();
    if (shape && plan->dev_id != h->device) {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        UVT_HIP(hipStreamIsCapturing(s, &capture));
        if (capture != hipStreamCaptureStatusNone) return waves();
    }
    uvt_status st = plan_upload(h, plan);
    if (shape && st == UVT_ERR_NOMEM) return waves();
    if (st != UVT_OK) return st;
    double* parts = (double*)plan->dev_parts;
    if (plan->sk_grid > 0)
        return uvt_launch_trapezoid_sk_f64(plan->cfg, plan->n, plan->m, dA, lda, dB, ldb, dC, ldc,
                                           plan->sk_grid, parts, s);
    if (plan->nsums > 0x7FFFFFFF) return UVT_ERR_SIZE;
    st = launch_tiles_f64(plan->cfg, plan->dev_launch, plan->nlaunch, dA, lda, dB, ldb, dC, ldc, plan->m,
                          plan->nparts > 0 ? parts : nullptr, s);
    if (st != UVT_OK) return st;
    if (plan->nsums > 0) {
        const int32_t tm = uvt_cfg_tile_m(plan->cfg), tn = uvt_cfg_tile_n(plan->cfg);
        hipLaunchKernelGGL(k_add_parts, dim3((unsigned)plan->nsums, 8), dim3(256), 0, s, (const PartSum*)plan->dev_sums,
                           (int)tn, (int)(tm * tn), (const double*)parts, dC, ldc, plan->m);
        UVT_HIP(hipGetLastError());
    }
    return UVT_OK;
}

// Of the tiles a launch runs (waves or the trapezoid walk; cut reductions are
// cut at whole panels), not of the plan's list.
extern "C" double uvt_plan_issued_flops(uvt_plan plan)
{
    if (!plan) return 0.0;
    const int shape = uvt_wave_shape(plan->n, plan->m, plan->n, plan->m);
    int64_t tm = uvt_cfg_tile_m(plan->cfg), tn = uvt_cfg_tile_n(plan->cfg);
    if (shape && !deep_and_narrow(*plan)) {
        tm = 16 * (shape / 10);
        tn = 16 * (shape % 10);
    }
    double s = 0.0;
    for (int64_t r0 = 0; r0 < plan->n; r0 += tm)
        s += (double)((std::min(r0 + tm, plan->n) + kTileK - 1) / kTileK * kTileK);
    return 2.0 * (double)tm * s * (double)((plan->m + tn - 1) / tn * tn);
}

extern "C" uvt_status uvt_plan_launch_info(uvt_handle h, uvt_plan plan, int64_t* workgroups,
                                           int64_t* partial_tiles)
{
    if (!h || !plan) return UVT_ERR_ARG;
    const int shape = uvt_wave_shape(plan->n, plan->m, plan->n, plan->m);
    if (shape && !deep_and_narrow(*plan)) {
        if (workgroups) *workgroups = wave_grid(shape, plan->n, plan->m).launch();
        if (partial_tiles) *partial_tiles = 0;
        return UVT_OK;
    }
    UVT_HIP(hipSetDevice(h->device));
    const uvt_status st = plan_upload(h, plan);
    if (st != UVT_OK) return st;
    if (workgroups)
        *workgroups = plan->sk_grid > 0 ? sk_launch(sk_geometry(plan->n, plan->m, uvt_cfg_tile_m(plan->cfg),
                                                                uvt_cfg_tile_n(plan->cfg), plan->sk_grid,
                                                                kSkGroupCols))
                                        : plan->nlaunch;
    if (partial_tiles) *partial_tiles = plan->nparts;
    return UVT_OK;
}

// ---------------------------------------------------------------------
// Norm
// ---------------------------------------------------------------------

extern "C" uvt_status uvt_row_abs_sums(uvt_handle h, int64_t n, int64_t m, const double* dC,
                                       int64_t ldc, double* d_rowsum, void* stream)
{
    if (!h || !dC || !d_rowsum || n <= 0 || m <= 0 || ldc < m) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    const int64_t blocks = (n + 3) / 4;
    if (blocks > 0x7FFFFFFF) return UVT_ERR_SIZE;
    hipLaunchKernelGGL(k_row_abs_sums, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       n, m, dC, ldc, d_rowsum);
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

extern "C" uvt_status uvt_inf_norm(uvt_handle h, int64_t n, int64_t m, const double* dC,
                                   int64_t ldc, double* norm, void* stream)
{
    if (!h || !dC || !norm || n <= 0 || m <= 0 || ldc < m) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    const int64_t want = (n + kNormWaves - 1) / kNormWaves;
    // Held until the result is read: the handle has one set of partial maxima
    // and one result, which the next call would write over.
    std::lock_guard<std::mutex> lk(h->norm_mu);
    if (!h->norm_part) {  // partial maxima and the counter, zeroed once
        void* d = nullptr;
        if (hipMalloc(&d, (kNormBlocks + 1) * sizeof(double)) != hipSuccess) {
            (void)hipGetLastError();
            return UVT_ERR_NOMEM;
        }
        if (hipMemsetAsync(d, 0, (kNormBlocks + 1) * sizeof(double), (hipStream_t)stream) != hipSuccess ||
            hipHostMalloc((void**)&h->norm_host, sizeof(double), hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipFree(d);
            h->norm_host = nullptr;
            return UVT_ERR_NOMEM;
        }
        h->norm_part = (double*)d;
    }
    hipLaunchKernelGGL(k_inf_norm, dim3((unsigned)std::min<int64_t>(want, kNormBlocks)), dim3(64 * kNormWaves), 0,
                       (hipStream_t)stream, n, m, dC, ldc, h->norm_part, (unsigned*)(h->norm_part + kNormBlocks),
                       h->norm_host);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize((hipStream_t)stream) != hipSuccess) {
        (void)hipGetLastError();
        norm_free(h);  // the counter may not be zero: the next call makes new ones
        return UVT_ERR_HIP;
    }
    *norm = *(volatile double*)h->norm_host;
    return UVT_OK;
}

// ---------------------------------------------------------------------
// Inputs
// ---------------------------------------------------------------------

static dim3 fill_grid(int64_t rows, int64_t cols)
{
    int64_t bx = (cols + 255) / 256;
    if (bx > 64) bx = 64;
    return dim3((unsigned)(bx < 1 ? 1 : bx), (unsigned)(rows < 32768 ? rows : 32768));
}

extern "C" uvt_status uvt_fill_closed_form(uvt_handle h, int64_t n, int64_t m, double* dA,
                                           int64_t lda, double* dB, int64_t ldb, void* stream)
{
    if (!h || n <= 0 || m <= 0) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    hipStream_t s = (hipStream_t)stream;
    if (dA) {
        if (lda < n) return UVT_ERR_ARG;
        hipLaunchKernelGGL(k_fill_closed, fill_grid(n, n), dim3(256), 0, s, n, n, n, 1, dA, lda);
    }
    if (dB) {
        if (ldb < m) return UVT_ERR_ARG;
        hipLaunchKernelGGL(k_fill_closed, fill_grid(n, m), dim3(256), 0, s, n, n, m, 0, dB, ldb);
    }
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

static uint64_t host_mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

extern "C" uvt_status uvt_fill_seeded(uvt_handle h, int64_t n, int64_t m, uint64_t seed,
                                      int32_t spread, double* dA, int64_t lda, double* dB,
                                      int64_t ldb, void* stream)
{
    if (!h || n <= 0 || m <= 0) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    hipStream_t s = (hipStream_t)stream;
    const uint64_t gamma = 0x9E3779B97F4A7C15ULL;
    if (dA) {
        if (lda < n) return UVT_ERR_ARG;
        hipLaunchKernelGGL(k_fill_seeded, fill_grid(n, n), dim3(256), 0, s, n, n,
                           host_mix64(seed ^ (1ULL * gamma)), 1, (int)spread, dA, lda);
    }
    if (dB) {
        if (ldb < m) return UVT_ERR_ARG;
        hipLaunchKernelGGL(k_fill_seeded, fill_grid(n, m), dim3(256), 0, s, n, m,
                           host_mix64(seed ^ (2ULL * gamma)), 0, (int)spread, dB, ldb);
    }
    UVT_HIP(hipGetLastError());
    return UVT_OK;
}

// ---------------------------------------------------------------------
// Runtime helpers
// ---------------------------------------------------------------------

extern "C" uvt_status uvt_malloc(uvt_handle h, size_t bytes, void** dptr)
{
    if (!h || !dptr) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    if (hipMalloc(dptr, bytes ? bytes : 1) != hipSuccess) {
        (void)hipGetLastError();
        *dptr = nullptr;
        return UVT_ERR_NOMEM;
    }
    return UVT_OK;
}

extern "C" uvt_status uvt_free(uvt_handle h, void* dptr)
{
    if (!h) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    if (dptr) UVT_HIP(hipFree(dptr));
    return UVT_OK;
}

// Bytes of each pinned bounce buffer of host copies (two per handle), and
// the size from which a contiguous host copy goes through them: staged
// through pinned memory a copy runs at about 37 GB/s on MI355X, a pageable
// one at about 27 GB/s.
constexpr size_t kPinBytes = (size_t)16 << 20;
constexpr size_t kPinMinBytes = (size_t)1 << 20;

static uvt_status pin_setup(uvt_handle h)
{
    if (h->pin[0]) return UVT_OK;
    for (int i = 0; i < 2; ++i) {
        if (hipHostMalloc(&h->pin[i], kPinBytes, hipHostMallocDefault) != hipSuccess ||
            hipEventCreateWithFlags(&h->pin_done[i], hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            for (int j = 0; j < 2; ++j) {
                if (h->pin[j]) (void)hipHostFree(h->pin[j]);
                if (h->pin_done[j]) (void)hipEventDestroy(h->pin_done[j]);
                h->pin[j] = nullptr;
                h->pin_done[j] = nullptr;
            }
            return UVT_ERR_NOMEM;
        }
        h->pin_used[i] = false;
    }
    return UVT_OK;
}

// Contiguous host <-> device copy through the handle's pinned buffers, a
// chunk in flight while the host fills (or drains) the other.
static uvt_status copy_pinned(uvt_handle h, char* dst, const char* src, size_t bytes, bool to_device)
{
    const size_t chunks = (bytes + kPinBytes - 1) / kPinBytes;
    auto len = [&](size_t c) { return std::min(kPinBytes, bytes - c * kPinBytes); };
    if (to_device) {
        for (size_t c = 0; c < chunks; ++c) {
            const int b = (int)(c & 1);
            if (h->pin_used[b]) UVT_HIP(hipEventSynchronize(h->pin_done[b]));
            memcpy(h->pin[b], src + c * kPinBytes, len(c));
            UVT_HIP(hipMemcpyAsync(dst + c * kPinBytes, h->pin[b], len(c), hipMemcpyHostToDevice, 0));
            UVT_HIP(hipEventRecord(h->pin_done[b], 0));
            h->pin_used[b] = true;
        }
        UVT_HIP(hipStreamSynchronize(0));
        return UVT_OK;
    }
    auto issue = [&](size_t c) -> hipError_t {
        const int b = (int)(c & 1);
        hipError_t e = hipMemcpyAsync(h->pin[b], src + c * kPinBytes, len(c), hipMemcpyDeviceToHost, 0);
        if (e == hipSuccess) e = hipEventRecord(h->pin_done[b], 0);
        h->pin_used[b] = true;
        return e;
    };
    UVT_HIP(issue(0));
    for (size_t c = 0; c < chunks; ++c) {
        if (c + 1 < chunks) UVT_HIP(issue(c + 1));
        const int b = (int)(c & 1);
        UVT_HIP(hipEventSynchronize(h->pin_done[b]));
        memcpy(dst + c * kPinBytes, h->pin[b], len(c));
    }
    return UVT_OK;
}

// Strided host <-> device copy through the handle's pinned buffers: rows are
// packed (or unpacked) on the host a chunk at a time, and each chunk moves as
// one rectangular copy on the null stream while the host packs the next.  A
// pageable strided copy instead pays a fixed cost per row (about 9 us on
// MI355X: 56 ms for the three 2048 x 2048 operand copies of one call).
static uvt_status copy_2d_pinned(uvt_handle h, char* dst, size_t dpitch, const char* src, size_t spitch,
                                 size_t width, size_t height, bool to_device)
{
    const size_t per = kPinBytes / width;
    if (to_device) {
        for (size_t r = 0, c = 0; r < height; r += per, ++c) {
            const size_t rows = std::min(per, height - r);
            const int b = (int)(c & 1);
            char* buf = (char*)h->pin[b];
            if (h->pin_used[b]) UVT_HIP(hipEventSynchronize(h->pin_done[b]));
            for (size_t i = 0; i < rows; ++i) memcpy(buf + i * width, src + (r + i) * spitch, width);
            if (dpitch == width)
                UVT_HIP(hipMemcpyAsync(dst + r * dpitch, buf, rows * width, hipMemcpyHostToDevice, 0));
            else
                UVT_HIP(hipMemcpy2DAsync(dst + r * dpitch, dpitch, buf, width, width, rows,
                                         hipMemcpyHostToDevice, 0));
            UVT_HIP(hipEventRecord(h->pin_done[b], 0));
            h->pin_used[b] = true;
        }
        UVT_HIP(hipStreamSynchronize(0));
        return UVT_OK;
    }
    // device -> host: chunk c + 1 is in flight while chunk c is unpacked
    auto issue = [&](size_t c) -> hipError_t {
        const size_t r = c * per, rows = std::min(per, height - r);
        const int b = (int)(c & 1);
        hipError_t e = spitch == width
                           ? hipMemcpyAsync(h->pin[b], src + r * spitch, rows * width, hipMemcpyDeviceToHost, 0)
                           : hipMemcpy2DAsync(h->pin[b], width, src + r * spitch, spitch, width, rows,
                                              hipMemcpyDeviceToHost, 0);
        if (e == hipSuccess) e = hipEventRecord(h->pin_done[b], 0);
        h->pin_used[b] = true;
        return e;
    };
    const size_t chunks = (height + per - 1) / per;
    UVT_HIP(issue(0));
    for (size_t c = 0; c < chunks; ++c) {
        if (c + 1 < chunks) UVT_HIP(issue(c + 1));
        const int b = (int)(c & 1);
        UVT_HIP(hipEventSynchronize(h->pin_done[b]));
        const size_t r = c * per, rows = std::min(per, height - r);
        const char* buf = (const char*)h->pin[b];
        for (size_t i = 0; i < rows; ++i) memcpy(dst + (r + i) * dpitch, buf + i * width, width);
    }
    return UVT_OK;
}

extern "C" uvt_status uvt_memcpy(uvt_handle h, void* dst, const void* src, size_t bytes,
                                 int32_t kind)
{
    if (!h || (!dst && bytes) || (!src && bytes)) return UVT_ERR_ARG;
    hipMemcpyKind k = kind == 0 ? hipMemcpyHostToDevice
                      : kind == 1 ? hipMemcpyDeviceToHost
                                  : hipMemcpyDeviceToDevice;
    if (kind < 0 || kind > 2) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    if (kind != 2 && bytes >= kPinMinBytes) {
        const uvt_status st = pin_setup(h);
        if (st != UVT_OK) return st;
        return copy_pinned(h, (char*)dst, (const char*)src, bytes, kind == 0);
    }
    if (bytes) UVT_HIP(hipMemcpy(dst, src, bytes, k));
    return UVT_OK;
}

extern "C" uvt_status uvt_memcpy_2d(uvt_handle h, void* dst, size_t dpitch, const void* src,
                                    size_t spitch, size_t width, size_t height, int32_t kind)
{
    if (!h || kind < 0 || kind > 2) return UVT_ERR_ARG;
    if (!width || !height) return UVT_OK;
    if (!dst || !src || dpitch < width || spitch < width) return UVT_ERR_ARG;
    const hipMemcpyKind k = kind == 0 ? hipMemcpyHostToDevice
                            : kind == 1 ? hipMemcpyDeviceToHost
                                        : hipMemcpyDeviceToDevice;
    UVT_HIP(hipSetDevice(h->device));
    if (dpitch == width && spitch == width)  // one contiguous block
        return uvt_memcpy(h, dst, src, width * height, kind);
    if (kind != 2 && width <= kPinBytes && height > 1) {
        const uvt_status st = pin_setup(h);
        if (st != UVT_OK) return st;
        return copy_2d_pinned(h, (char*)dst, dpitch, (const char*)src, spitch, width, height, kind == 0);
    }
    UVT_HIP(hipMemcpy2D(dst, dpitch, src, spitch, width, height, k));
    return UVT_OK;
}

extern "C" uvt_status uvt_memset(uvt_handle h, void* dptr, int32_t value, size_t bytes)
{
    if (!h || (!dptr && bytes)) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    if (bytes) UVT_HIP(hipMemset(dptr, value, bytes));
    return UVT_OK;
}

extern "C" uvt_status uvt_stream_create(uvt_handle h, void** stream)
{
    if (!h || !stream) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    hipStream_t s;
    UVT_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *stream = (void*)s;
    return UVT_OK;
}

extern "C" uvt_status uvt_stream_destroy(uvt_handle h, void* stream)
{
    if (!h) return UVT_ERR_ARG;
    if (stream) UVT_HIP(hipStreamDestroy((hipStream_t)stream));
    return UVT_OK;
}

extern "C" uvt_status uvt_stream_sync(uvt_handle h, void* stream)
{
    if (!h) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    UVT_HIP(hipStreamSynchronize((hipStream_t)stream));
    return UVT_OK;
}

extern "C" uvt_status uvt_event_create(uvt_handle h, void** event)
{
    if (!h || !event) return UVT_ERR_ARG;
    UVT_HIP(hipSetDevice(h->device));
    hipEvent_t e;
    UVT_HIP(hipEventCreate(&e));
    *event = (void*)e;
    return UVT_OK;
}

extern "C" uvt_status uvt_event_destroy(uvt_handle h, void* event)
{
    if (!h) return UVT_ERR_ARG;
    if (event) UVT_HIP(hipEventDestroy((hipEvent_t)event));
    return UVT_OK;
}

extern "C" uvt_status uvt_event_record(uvt_handle h, void* event, void* stream)
{
    if (!h || !event) return UVT_ERR_ARG;
    UVT_HIP(hipEventRecord((hipEvent_t)event, (hipStream_t)stream));
    return UVT_OK;
}

extern "C" uvt_status uvt_event_elapsed(uvt_handle h, void* start, void* end, float* ms)
{
    if (!h || !start || !end || !ms) return UVT_ERR_ARG;
    UVT_HIP(hipEventSynchronize((hipEvent_t)end));
    UVT_HIP(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)end));
    return UVT_OK;
}
