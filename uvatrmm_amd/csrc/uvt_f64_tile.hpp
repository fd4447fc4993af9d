// uvt_f64_tile.hpp -- FP64 MFMA tile of C = tril(A) * B for gfx950.
//
// One workgroup (WAVES_M x WAVES_N wave64 waves) computes a TM x TN tile of C over a k range
// [k_lo, k_hi), with A or B triangular or neither.  This one routine covers
// every product the reference issues per band
// (UVaTRMM/src/mm_triangular.c:347-393): its GEMM box and the triangle added to
// it are one masked tile, C[r0:r0+TM] = A[r0:, 0:r0+TM] * B with A[i][k] = 0
// for k > i.
//
// Data path: A and B k-panels (16 deep) stream from HBM with 16-byte loads
// into registers one panel ahead, are written to a
// double-buffered LDS tile, and each wave multiplies its (TM/WAVES_M) x
// (TN/WAVES_N) sub-tile with v_mfma_f64_16x16x4_f64 (one double of A and B
// per lane, four doubles of C per lane).  Each operand keeps its memory
// layout in LDS (struct Panel), so every LDS write is one 16-byte piece a
// thread loaded; the writes for the next panel are issued during the current
// panel's products (see compute()), and each lane reads its values of a
// k-contiguous operand as 16-byte pairs of one row.  (A transposed to k-major
// on the way in took four conflicting 8-byte writes per thread and cost about
// 10 % of the MFMA rate, measured register-only.)
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "uvt_panel.hpp"

namespace uvt {

typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef double dbl2 __attribute__((ext_vector_type(2)));

// Global-memory pointers.  A generic pointer (one read from a descriptor in
// memory, say) is accessed with flat instructions: 64-bit addresses, and
// their completion is counted together with LDS traffic, so a wait for an
// LDS read also waits for every load in flight.  Typed global, the same
// access compiles to a global load or store (scalar base + lane offset).
#define UVT_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ const UVT_GLOBAL T* gbl(const T* p)
{
    return (const UVT_GLOBAL T*)p;
}
template <typename T>
__device__ __forceinline__ UVT_GLOBAL T* gbl(T* p)
{
    return (UVT_GLOBAL T*)p;
}

constexpr int kTileLower = 1;  // UVT_TILE_LOWER

// Two doubles at an 8-byte aligned address: one 16-byte global load (global
// memory takes 16-byte accesses at any 4-byte alignment), so odd leading
// dimensions load like even ones.
typedef double dbl2u __attribute__((ext_vector_type(2), aligned(8)));

// One operand's panel of a tile on its way from memory to LDS (uvt_panel.hpp:
// which elements).  Its layout in LDS is the one it has in memory:
//   KC:  rows of kTileK + 2 doubles (144 B, 16-byte aligned; the 16 rows a
//        fragment read touches fall on distinct bank pairs);
//   !KC: k rows of X + 16 doubles; a fragment read touches four k rows
//        kTileK/4 apart (the k order of f64_tile), which share one half of
//        the 64 LDS banks (a pitch of X + 4, alternating halves, measured
//        the same).
// Edge tiles run the steady state like any other.  With every element of
// every panel of an edge tile checked instead, the edge tiles were the last
// to finish: 8165 x 939 took 1193 us instead of 1081, a 1500 x 2000 x 3000
// dgemm in 64x64 tiles 387 instead of 342 (same bits).
template <int X, int NT, bool KC, bool DOWN>
struct Panel {
    using Idx = PanelIdx<X, NT, KC>;
    static constexpr int LD = KC ? kTileK + 2 : X + 16;
    static constexpr int ELEMS = KC ? X * LD : kTileK * LD;
    static constexpr int PIECES = Idx::PIECES, VEC = Idx::VEC;
    static constexpr bool PART = Idx::PART;
    // Steady-state addresses: a wave-uniform base (scalar registers, moved from
    // panel to panel) plus a byte offset per thread that never changes; one
    // offset serves all of a thread's pieces of an x-contiguous panel.
    static constexpr int OFFS = KC ? VEC : 1;

    const UVT_GLOBAL double* p;  // element (x0, k = 0)
    int64_t ld;
    int nx;  // rows (columns) inside the matrix, 1 .. X
    int x0;  // the tile's first row (column): the triangle's coordinate
    const UVT_GLOBAL char* at;
    uint32_t off[OFFS];
    dbl2 r[VEC];

    __device__ __forceinline__ void init(int tid, const UVT_GLOBAL double* p_, int64_t ld_, int nx_, int x0_)
    {
        p = p_;
        ld = ld_;
        nx = nx_;
        x0 = x0_;
#pragma unroll
        for (int q = 0; q < OFFS; ++q) {
            const int v = tid + q * NT, x = Idx::full_x(v, nx), k = Idx::pk(v);
            off[q] = 8u * (KC ? (uint32_t)x * (uint32_t)ld + (uint32_t)k : (uint32_t)k * (uint32_t)ld + (uint32_t)x);
        }
    }

    static __device__ __forceinline__ int lds(int v)
    {
        return KC ? Idx::px(v) * LD + Idx::pk(v) : Idx::pk(v) * LD + Idx::px(v);
    }
    // load() reads the panel here next.
    __device__ __forceinline__ void seek(int k0)
    {
        at = reinterpret_cast<const UVT_GLOBAL char*>(KC ? p + k0 : p + (int64_t)k0 * ld);
    }
    // The next panel of the walk, a full one (DOWN: the walk goes down in k).
    __device__ __forceinline__ void load(int tid)
    {
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
            if (PART && tid + q * NT >= PIECES) break;
            // the 32-bit offset, opaque here: the access then takes it beside
            // the scalar base instead of a 64-bit sum in vector registers
            // (a copy of it in the 16-wave workgroups, whose loop the
            // compiler orders better so: 4096^2 992 us against 1007)
            if (NT == 1024) {
                uint32_t o = off[KC ? q : 0];
                asm volatile("" : "+v"(o));
                r[q] = *reinterpret_cast<const UVT_GLOBAL dbl2u*>(at + q * (Idx::KSTEP * 8) * ld + o);
                continue;
            }
            if (q < OFFS) asm volatile("" : "+v"(off[q]));
            r[q] = *reinterpret_cast<const UVT_GLOBAL dbl2u*>(at + q * (Idx::KSTEP * 8) * ld + off[KC ? q : 0]);
        }
        const int64_t step = KC ? (int64_t)kTileK * 8 : ld * (kTileK * 8);
        at += DOWN ? -step : step;
    }

    // Any panel: no load sits under a branch per element (such branches cost
    // a small product most of its time: 257 x 257 17.2 us, now 14.9).  An
    // operand without a triangle loads a panel inside the range as in the
    // steady state, so beside the diagonal only the triangle's own panels go
    // element by element.
    template <bool TRI, bool GE, bool WIDE>
    __device__ __forceinline__ void load_masked(int tid, int k0, int k_lo, int k_hi, bool tri)
    {
        if (!(TRI && tri) && Idx::inside(k0, k_lo, k_hi, nx, ld)) {
            seek(k0);
            load(tid);
            return;
        }
        if (WIDE && Idx::whole(k0, k_lo, k_hi, nx) && (!(TRI && tri) || Idx::template clear<GE>(k0, x0, nx))) {
#pragma unroll
            for (int q = 0; q < VEC; ++q) {
                const int v = tid + q * NT;
                if (PART && v >= PIECES) break;
                const int64_t x = Idx::full_x(v, nx), k = k0 + Idx::pk(v);
                r[q] = *reinterpret_cast<const UVT_GLOBAL dbl2u*>(p + (KC ? x * ld + k : k * ld + x));
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
            const int v = tid + q * NT;
            if (PART && v >= PIECES) break;
            double e[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int xe = KC ? Idx::px(v) : Idx::px(v) + h, ke = k0 + (KC ? Idx::pk(v) + h : Idx::pk(v));
                const int x = xe < nx ? xe : nx - 1, k = near_k<GE>(ke, x0 + x, k_hi, TRI && tri);
                e[h] = KC ? p[(int64_t)x * ld + k] : p[(int64_t)k * ld + x];
            }
            r[q] = dbl2{e[0], e[1]};
        }
    }

    __device__ __forceinline__ void store(int tid, double* s) const
    {
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
            const int v = tid + q * NT;
            if (PART && v >= PIECES) break;
            *reinterpret_cast<dbl2*>(&s[lds(v)]) = r[q];
        }
    }

    // The panel at k0 with zeros outside [k_lo, k_hi) and outside the
    // triangle, and (UNIT) ones on its diagonal.
    template <bool TRI, bool GE, bool UNIT, bool WIDE>
    __device__ __forceinline__ void store_masked(int tid, double* s, int k0, int k_lo, int k_hi, bool tri,
                                                 bool unit) const
    {
        if ((!(TRI && tri) || (WIDE && Idx::template clear<GE>(k0, x0, nx))) && k0 >= k_lo && k0 + kTileK <= k_hi) {
            store(tid, s);
            return;
        }
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
            const int v = tid + q * NT;
            if (PART && v >= PIECES) break;
            dbl2 w = r[q];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int x = x0 + (KC ? Idx::px(v) : Idx::px(v) + h), k = k0 + (KC ? Idx::pk(v) + h : Idx::pk(v));
                bool in = k >= k_lo && k < k_hi;
                if (TRI && tri) in = in && (GE ? k >= x : k <= x);
                w[h] = in ? w[h] : 0.0;
                if (UNIT && unit && k == x) w[h] = 1.0;
            }
            *reinterpret_cast<dbl2*>(&s[lds(v)]) = w;
        }
    }
};

// Which operand of a tile is triangular, and which part of it is kept.
enum TriKind {
    kTriALe,  // op(A)[i][k], k <= i (where the tile's flags hold kTileLower)
    kTriAGe,  // op(A)[i][k], k >= i
    kTriBLe,  // op(B)[k][j], k <= j
    kTriBGe   // op(B)[k][j], k >= j
};

// A_KC / B_KC: k contiguous in memory (A as it is; B transposed).
// UNIT_: the triangle's diagonal may be taken as ones (f64_tile's unit).
// EPI_: C = alpha * product + beta * C, else C = product.
// EDGE_IDLE: waves of an edge tile that hold no row or column of C run no
// products (off where a caller's own registers leave no room for the test:
// the stream-K kernel then spills inside its masked k loop).
// PIPE_MASKED: the masked panels run the software pipeline too.  Without it
// they leave 16 registers to their addresses and masks, which the kernels
// with more of their own need (8165 x 939 stream-K 1033 us with it, 1021
// without; 9000 x 250 in cut tiles 395 and 387; 512 problems in a batch, from
// one queue, 9.08 and 8.95 ms); the plain walks are faster with it (4096^2:
// 992 us, 1004 without).
// WIDE: an operand has rows too long for full panels (PanelIdx::offsets_fit);
// panels that no mask touches are then loaded with 64-bit addresses, not
// element by element.  A kernel of its own: in the others the extra branch
// costs registers (short batch tiles 4 % slower, dtrmm on the right 3-5 %).
template <bool A_KC_ = true, bool B_KC_ = false, TriKind TRI_ = kTriALe, bool UNIT_ = false, bool EPI_ = false,
          bool EDGE_IDLE_ = true, bool PIPE_MASKED_ = true, bool WIDE_ = false>
struct TileOpt {
    static constexpr bool A_KC = A_KC_, B_KC = B_KC_, UNIT = UNIT_, EPI = EPI_, EDGE_IDLE = EDGE_IDLE_,
                          PIPE_MASKED = PIPE_MASKED_, WIDE = WIDE_;
    static constexpr TriKind TRI = TRI_;
    static constexpr bool TRI_A = TRI == kTriALe || TRI == kTriAGe, GE = TRI == kTriAGe || TRI == kTriBGe;
};

template <int TM, int TN, int WAVES_M = 2, int WAVES_N = 2, class OPT = TileOpt<>>
struct F64Cfg {
    static constexpr int NT = 64 * WAVES_M * WAVES_N;
    static constexpr int WM = TM / WAVES_M, WN = TN / WAVES_N;
    static constexpr int FM = WM / 16, FN = WN / 16;
    using PA = Panel<TM, NT, OPT::A_KC, OPT::GE>;
    using PB = Panel<TN, NT, OPT::B_KC, OPT::GE>;
    static constexpr int SMEM_DOUBLES = 2 * (PA::ELEMS + PB::ELEMS);
    static_assert(FM >= 1 && FN >= 1, "wave tile below 16x16");
};

// The part of C a tile covers, its reduction range and what to do with it.
struct TileArgs {
    int r0, rows, c0, k_lo, k_hi, flags;
};
// C = alpha * product + beta * C (C not read when beta == 0); unit: ones on
// the triangle's diagonal.
struct TileEpi {
    double alpha = 1.0, beta = 0.0;
    bool unit = false;
};

// thread: the caller's thread index when it must stay opaque to the compiler
// (a persistent kernel running several tile shapes, whose per-thread offsets
// would otherwise be hoisted out of its tile loop for every shape at once
// and spilled); -1: threadIdx.x.
// part: if set, the tile's product goes there instead of to C, as a TM x TN
// row-major block (row r, column c of the tile at r * TN + c; only rows <
// rows and columns inside C are written), to be added to C later in a fixed
// order.
// m: columns of C (and of op(B)).
template <int TM, int TN, int WAVES_M, int WAVES_N, class OPT = TileOpt<>>
__device__ __forceinline__ void f64_tile(const TileArgs& t, const UVT_GLOBAL double* __restrict__ A, int64_t lda,
                                         const UVT_GLOBAL double* __restrict__ B, int64_t ldb,
                                         UVT_GLOBAL double* __restrict__ C, int64_t ldc, int64_t m, double* smem,
                                         int thread = -1, UVT_GLOBAL double* __restrict__ part = nullptr,
                                         const TileEpi& epi = TileEpi())
{
    using G = F64Cfg<TM, TN, WAVES_M, WAVES_N, OPT>;
    using PA = typename G::PA;
    using PB = typename G::PB;
    constexpr int BK = kTileK;
    constexpr bool GE = OPT::GE, TRI_A = OPT::TRI_A, UNIT = OPT::UNIT;
    const int tid = thread >= 0 ? thread : (int)threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: branches on it stay scalar
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    // kTriALe is the plans' kernel, whose boxes have no triangle; the other
    // kinds are launched for triangles only.
    const bool tri = OPT::TRI != kTriALe || (t.flags & kTileLower) != 0;
    const bool unit = UNIT && epi.unit;
    double* As = smem;                  // [2][PA::ELEMS]
    double* Bs = smem + 2 * PA::ELEMS;  // [2][PB::ELEMS]

    const int k_lo = t.k_lo, k_hi = t.k_hi;
    const int k_start = k_lo & ~1;
    const int nk = panels(k_lo, k_hi);
    auto k_at = [&](int kt) { return panel_k0<GE>(k_lo, nk, kt); };
    const int cols = (int64_t)t.c0 + TN <= m ? TN : (int)(m - t.c0);

    PA pa;
    PB pb;
    pa.init(tid, OPT::A_KC ? A + (int64_t)t.r0 * lda : A + t.r0, lda, t.rows, t.r0);
    pb.init(tid, OPT::B_KC ? B + (int64_t)t.c0 * ldb : B + t.c0, ldb, cols, t.c0);

    dbl4 acc[G::FM][G::FN];
#pragma unroll
    for (int i = 0; i < G::FM; ++i)
#pragma unroll
        for (int j = 0; j < G::FN; ++j) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};

    // full_tag: std::true_type for a panel that needs no masks at all (see
    // the panel ranges below); otherwise every element is checked.
    int mtid = tid;  // thread index of the masked panels
    auto load = [&](int k0, auto full_tag) {
        if constexpr (decltype(full_tag)::value) {
            pa.load(tid);  // panels of the steady state follow each other: see seek()
            pb.load(tid);
        } else {
            pa.template load_masked<TRI_A, GE, OPT::WIDE>(mtid, k0, k_lo, k_hi, tri);
            pb.template load_masked<!TRI_A, GE, OPT::WIDE>(mtid, k0, k_lo, k_hi, tri);
        }
    };
    auto store = [&](int buf, int k0, auto full_tag) {
        double* as = As + buf * PA::ELEMS;
        double* bs = Bs + buf * PB::ELEMS;
        if constexpr (decltype(full_tag)::value) {
            pa.store(tid, as);
            pb.store(tid, bs);
        } else {
            pa.template store_masked<TRI_A, GE, UNIT && TRI_A, OPT::WIDE>(mtid, as, k0, k_lo, k_hi, tri, unit);
            pb.template store_masked<!TRI_A, GE, UNIT && !TRI_A, OPT::WIDE>(mtid, bs, k0, k_lo, k_hi, tri, unit);
        }
    };

    // The products of the panel in LDS buffer buf; st() puts the registers
    // loaded for the next panel into buffer buf ^ 1.
    //
    // Software pipeline: the fragments of MFMA step s + 1 are read from LDS
    // during the products of step s, and those of the next panel's first step
    // during this panel's last one, behind the panel's one barrier.  (Read at
    // the head of their own step instead, they left the matrix units idle for
    // an LDS latency after each barrier, when every wave of a SIMD starts its
    // panel at once: 16384^2 took 61.7-62.5 ms against 60.4, 4096^2 1016-1027
    // us against 991, 2048^2 164 against 159, same bits.)  The source places the LDS
    // writes after the second of the four steps; after the first, the third,
    // or inside the second or third they measured 0-3 % slower (256x128
    // tiles).  The order inside a step is the compiler's: pinned with
    // __builtin_amdgcn_sched_barrier around each step's products, or with
    // s_setprio around them, the same loop was 4-5 % slower, and
    // sched_group_barrier (two products, one LDS read) changed nothing.
    //
    // k order inside a panel: at MFMA step s, lane group g = lane / 16 takes
    // k = g * BK/4 + s (A and B alike, so the four steps still cover the
    // panel's BK values of k once each).  A lane's values of a k-contiguous
    // operand for the whole panel are then BK/4 consecutive doubles of one
    // row, read as 16-byte pairs: half the LDS reads of one 8-byte read per
    // step (1.4 % on a register-only probe of this loop, 73.2 -> 74.3 TFLOP/s).
    // (Values of a k-contiguous operand come in pairs: steps s and s + 1 for
    // even s.)
    dbl2 a2[G::FM], b2[G::FN];
    double a1[G::FM], b1[G::FN];
    const int kg = (lane >> 4) * (BK / 4), xa = wm * G::WM + (lane & 15), xb = wn * G::WN + (lane & 15);
    const int ao = OPT::A_KC ? xa * PA::LD + kg : kg * PA::LD + xa;
    const int bo = OPT::B_KC ? xb * PB::LD + kg : kg * PB::LD + xb;
    auto read = [&](int buf, int s, auto& ra2, auto& rb2, auto& ra1, auto& rb1) {
        const double* as = As + buf * PA::ELEMS + ao;
        const double* bs = Bs + buf * PB::ELEMS + bo;
#pragma unroll
        for (int i = 0; i < G::FM; ++i) {
            if constexpr (OPT::A_KC) {
                if (s % 2 == 0) ra2[i] = *reinterpret_cast<const dbl2*>(&as[i * 16 * PA::LD + s]);
            } else {
                ra1[i] = as[s * PA::LD + i * 16];
            }
        }
#pragma unroll
        for (int j = 0; j < G::FN; ++j) {
            if constexpr (OPT::B_KC) {
                if (s % 2 == 0) rb2[j] = *reinterpret_cast<const dbl2*>(&bs[j * 16 * PB::LD + s]);
            } else {
                rb1[j] = bs[s * PB::LD + j * 16];
            }
        }
    };
    auto read0 = [&](int buf) { read(buf, 0, a2, b2, a1, b1); };
    auto multiply = [&](int s) {
#pragma unroll
        for (int i = 0; i < G::FM; ++i)
#pragma unroll
            for (int j = 0; j < G::FN; ++j) {
                const double a = OPT::A_KC ? a2[i][s % 2] : a1[i];
                const double b = OPT::B_KC ? b2[j][s % 2] : b1[j];
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[i][j], 0, 0, 0);
            }
    };
    auto compute = [&](int buf, auto&& st) {
#pragma unroll
        for (int s = 0; s < BK / 4; ++s) {
            dbl2 na2[G::FM], nb2[G::FN];
            double na1[G::FM], nb1[G::FN];
            if (s + 1 < BK / 4) {
                read(buf, s + 1, na2, nb2, na1, nb1);
            } else {
                __syncthreads();
                read(buf ^ 1, 0, na2, nb2, na1, nb1);
            }
            multiply(s);
            if (s == 1) st();
#pragma unroll
            for (int i = 0; i < G::FM; ++i) {
                if constexpr (OPT::A_KC) {
                    if (s % 2 == 1) a2[i] = na2[i];
                } else {
                    a1[i] = na1[i];
                }
            }
#pragma unroll
            for (int j = 0; j < G::FN; ++j) {
                if constexpr (OPT::B_KC) {
                    if (s % 2 == 1) b2[j] = nb2[j];
                } else {
                    b1[j] = nb1[j];
                }
            }
        }
    };
    // The masked panels (see PIPE_MASKED).
    auto compute_masked = [&](int buf, auto&& st) {
        if constexpr (OPT::PIPE_MASKED) {
            compute(buf, st);
            return;
        }
#pragma unroll
        for (int s = 0; s < BK / 4; ++s) {
            read(buf, s, a2, b2, a1, b1);
            multiply(s);
            if (s == 1) st();
        }
        __syncthreads();
    };

    // Panels [f0, f1) need no masks: the steady-state loop, free of per-panel
    // branches.  The rest (next to the diagonal, at the tile's k ends) run
    // masked.
    if (nk > 0) {
        const std::true_type full{};
        const std::false_type masked{};
        const bool odd = (!OPT::A_KC && (t.rows & 1)) || (!OPT::B_KC && (cols & 1));
        // first and last coordinate of the triangular operand
        const int tx0 = TRI_A ? t.r0 : t.c0, tx1 = tx0 + (TRI_A ? t.rows : cols) - 1;
        const FullPanels fp = full_panels<GE>(k_lo, k_hi, tri, unit, tx0, tx1, odd);
        const int f0 = fp.f0, f1 = PA::Idx::offsets_fit(lda) && PB::Idx::offsets_fit(ldb) ? fp.f1 : 0;
        pa.seek(k_at(f0));
        pb.seek(k_at(f0));

        const bool first_full = f0 == 0 && f1 > 0;
        if (first_full) {
            load(k_at(0), full);
            store(0, k_at(0), full);
        } else {
            load(k_at(0), masked);
            store(0, k_at(0), masked);
        }
        __syncthreads();
        // A panel whose k lies on the zero side of the triangle for all of a
        // wave's rows (columns) holds only zeros for it: the wave runs it
        // without products (it only stores the next panel), which leaves the
        // CU's matrix units to the other waves.  Panel counts are uniform over
        // the wave.  Skipping adds of exact zeros changes no result (the sign
        // of a zero aside).  Likewise a wave whose rows all lie past the
        // tile's last row, or whose columns all lie past C's last column,
        // writes nothing: outside the steady-state loop it runs no products.
        const bool idle = OPT::EDGE_IDLE && (wm * G::WM >= t.rows || wn * G::WN >= cols);
        int kt = 0;
        if (OPT::PIPE_MASKED || kt + 1 < f1) read0(kt & 1);
        if (idle) {  // this wave only feeds the others
            for (; kt + 1 < f1; ++kt) {
                load(k_at(kt + 1), full);
                store((kt & 1) ^ 1, 0, full);
                __syncthreads();
            }
        } else {
            for (; kt + 1 < f1; ++kt) {  // the next panel is full
                load(k_at(kt + 1), full);
                compute(kt & 1, [&] { store((kt & 1) ^ 1, 0, full); });
            }
        }
        // The masked panels' offsets are computed from here on, not held in
        // registers (or spilled) since the tile's first panel.
        asm volatile("" : "+v"(mtid));
        int nk_w = nk;
        if (idle) nk_w = kt;
        else if (tri && !GE) {
            // last row (column) of this wave
            const int last = tx0 + (TRI_A ? wm * G::WM + G::WM : wn * G::WN + G::WN) - 1;
            nk_w = last >= k_start ? (last - k_start) / BK + 1 : 0;
            nk_w = nk_w < kt ? kt : (nk_w > nk ? nk : nk_w);
        } else if (tri) {
            const int first = tx0 + (TRI_A ? wm * G::WM : wn * G::WN);  // first row (column) of this wave
            nk_w = nk - (first > k_start ? (first - k_start) / BK : 0);
            nk_w = nk_w < kt ? kt : nk_w;
        }
        for (; kt < nk_w; ++kt) {
            const bool more = kt + 1 < nk;
            if (more) load(k_at(kt + 1), masked);
            compute_masked(kt & 1, [&] {
                if (more) store((kt & 1) ^ 1, k_at(kt + 1), masked);
            });
        }
        for (; kt < nk; ++kt) {
            if (kt + 1 < nk) {
                load(k_at(kt + 1), masked);
                store((kt & 1) ^ 1, k_at(kt + 1), masked);
            }
            __syncthreads();
        }
    }

    // D layout of v_mfma_f64_16x16x4_f64 (measured on gfx950): lane l,
    // element v holds row l/16 + 4*v, column l%16 of the 16x16 block.
#pragma unroll
    for (int i = 0; i < G::FM; ++i) {
#pragma unroll
        for (int j = 0; j < G::FN; ++j) {
            const int col = wn * G::WN + j * 16 + (lane & 15);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = wm * G::WM + i * 16 + (lane >> 4) + 4 * v;
                if (col < cols && row < t.rows) {
                    const double x = acc[i][j][v];
                    if (part) {
                        part[row * TN + col] = x;
                    } else {
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
        }
    }
}

// Workgroup shapes of the FP64 tile kernels (waves along rows x columns and
// workgroups resident per CU).  A 128x128 tile runs as 8 waves of 32x64 (4
// waves per SIMD with two workgroups per CU, which hides global-load latency
// better than 4 waves of 64x64); 64x64 tiles (small problems) as 4 waves of
// 32x32; 128x32 tiles (narrow B) as 4 waves of 32x32 stacked along rows.
// WAVES_PER_EU (the second __launch_bounds__ argument on AMD) caps the
// registers per wave so that BLOCKS_PER_CU workgroups fit on one CU.
template <int TM, int TN> struct TileWaves;
template <> struct TileWaves<128, 128> {
    static constexpr int M = 4, N = 2, BLOCKS_PER_CU = 2, WAVES_PER_EU = 4;
};
// 256x128 tiles: 16 waves of 32x64; as 8 waves of 64x64 (a third fewer LDS
// reads, two waves per SIMD, 234 VGPRs) they measured 11-13 % slower.
template <> struct TileWaves<256, 128> {
    static constexpr int M = 8, N = 2, BLOCKS_PER_CU = 1, WAVES_PER_EU = 4;
};
template <> struct TileWaves<64, 64> {
    static constexpr int M = 2, N = 2, BLOCKS_PER_CU = 4, WAVES_PER_EU = 4;
};
template <> struct TileWaves<128, 32> {
    static constexpr int M = 4, N = 1, BLOCKS_PER_CU = 3, WAVES_PER_EU = 3;
};
template <> struct TileWaves<32, 128> {  // few rows: the right-side forms of the BLAS calls
    static constexpr int M = 1, N = 4, BLOCKS_PER_CU = 3, WAVES_PER_EU = 3;
};

}  // namespace uvt
