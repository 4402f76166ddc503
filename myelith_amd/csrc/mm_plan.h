// mm_plan.h -- launch planning of the byte-plane products (gemm_mfma2.h) and
// of the fragment-major products of decode batches (gemm_frag.h): block
// shapes, tile counts, the K split, grid and LDS sizes.  Plain C++
// with no HIP dependency: the launchers call these functions, and a host
// build of them runs under AddressSanitizer and UndefinedBehaviorSanitizer
// in the CPU tests (tests/test_launch_plan.py).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace myl {

// Block shape of an mm2 launch: MB x NB 32 x 32 accumulators per wave,
// WM_ x WN_ waves, STAGES LDS stages of KS bytes of K.
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS>
struct Mm2Dims {
    static_assert(KS == 64 || KS == 128, "stage width");
    static constexpr int kThreads = WM_ * WN_ * 64;
    static constexpr int BR = 32 * MB * WM_;   // A' rows per block (2 per token)
    static constexpr int BN = 32 * NB * WN_;   // weight rows per block
    static constexpr int kCpr = KS / 16;       // 16-byte chunks per stage row
    static constexpr int kRowsPerLoad = 64 / kCpr;
    static constexpr int kSwzRows = 256 / KS;  // rows sharing one swizzle slot
    static constexpr int kStageBytes = (BR + BN) * KS;
    static constexpr size_t kLds = (size_t)STAGES * kStageBytes;
    // 1 KiB wave loads per stage, dealt round-robin to the waves; every wave
    // issues kLoads (past the last group: that group again, the same bytes)
    static constexpr int kGroups = (BR + BN) / kRowsPerLoad;
    static constexpr int kLoads = (kGroups + kThreads / 64 - 1) / (kThreads / 64);
    static_assert((BR + BN) % kRowsPerLoad == 0, "whole 1 KiB loads");
    static_assert((STAGES - 1) * kLoads < 64, "a wait can count the loads in flight");
    // waves per SIMD the register budget must allow: two blocks per CU where
    // the stages leave room for them
    static constexpr int kMinWaves = std::max(1, (kLds <= 80 * 1024 ? 2 : 1) * (kThreads / 64) / 4);
};

// Grid of a launch over `items` work items: a multiple of 8 (the XCD count),
// so block b's XCD is b % 8 for every tile-order computation.
inline int mm2_grid_of(int items) { return 8 * ((items + 7) / 8); }

// The row tiles of a group of the grouped tile order (TileOrder): about `want`,
// so that no group is much smaller than the others.
inline int mm2_group_rows(int tiles_r, int want) {
    if (want < 1 || tiles_r <= want) return tiles_r;
    const int groups = (tiles_r + want - 1) / want;
    return (tiles_r + groups - 1) / groups;
}

// The K split of a product over M activation rows (A' = 2M plane rows), N
// weight rows and K (a multiple of KS): with fewer tiles than `fill` and
// room for the M x N i64 partial sums, K is cut into ns slices of kslice
// bytes (a multiple of KS, at least 512 bytes of K per slice, about two
// items per CU), else one slice covers K.
struct Mm2SplitPlan {
    int tiles_r = 0, ntiles = 0;  // row tiles, all output tiles
    int ks = 1;                   // requested split
    int kslice = 0, ns = 1;       // bytes of K per slice, slices
    int nitems = 0, grid = 0;     // work items (tiles x slices), blocks
    bool split = false;
};

template <int MB, int NB, int WM_, int WN_, int STAGES, int KS>
inline Mm2SplitPlan mm2_split_plan(int M, int N, int K, int cus, size_t acc_elems, int fill) {
    using S = Mm2Dims<MB, NB, WM_, WN_, STAGES, KS>;
    Mm2SplitPlan p;
    const int R2 = 2 * M;
    p.tiles_r = (R2 + S::BR - 1) / S::BR;
    p.ntiles = p.tiles_r * ((N + S::BN - 1) / S::BN);
    const int nkb = K / KS;
    if (p.ntiles < fill && (size_t)M * (size_t)N <= acc_elems)
        p.ks = std::max(1, std::min((2 * cus + p.ntiles - 1) / p.ntiles, nkb / (512 / KS)));
    p.split = p.ks > 1;
    p.kslice = p.split ? ((nkb + p.ks - 1) / p.ks) * KS : K;
    p.ns = p.split ? (K + p.kslice - 1) / p.kslice : 1;
    p.nitems = p.ntiles * p.ns;
    p.grid = mm2_grid_of(p.nitems);
    return p;
}

// Tiles of products of more than 32 rows with K % 128 == 0 (plane rows x weight
// rows, 128-byte K stages).  256 x 256 and 192 x 256 fill a CU's LDS with two
// stages and share their operands best; 128 x 128 and 64 x 128 with two stages
// run two and three blocks per CU; with three stages, 128 x 128 hides the
// memory latency of a lone block and 64 x 64 that of three small ones.
enum Mm2Tile { kMm2T256, kMm2T192, kMm2T128, kMm2T128s3, kMm2T64, kMm2T64s3 };

struct Mm2Pick {
    Mm2Tile tile = kMm2T256;
    bool split = false;  // K split of the 64 x 128 tiles through the accumulator
};

// The tile by the time of the busiest CU's queue of q tiles, measured on MI355X
// with weights from HBM, us at K = 3584: 256 x 256 53 q; 192 x 256 44.5 q;
// 128 x 128 22 alone (three stages; 28 with two), 17.6 q queued; 64 x 128 12 q
// queued; 64 x 64 14 alone, 19 for two, then 7 q + 6.  So the large tiles win
// where they fill whole rounds of the chip (down of the 7B layout over 1500 rows:
// 224 tiles of 192 x 256 258 us, 168 of 256 x 256 297, 672 of 128 x 128 261) and
// the small ones where few tiles would leave CUs idle (100 rows of o_proj: 224 of
// 64 x 64 13.9 us, 56 of 128 x 128 20.4, 14 of 256 x 256 49).  A K split adds
// about 5 us for the finish and its 64-bit atomics (about 180 a ns): 64 rows of
// the 7B down projection 35 us in 10 slices, 58 whole; 300 rows x 896 x 4864 20
// split, 17 whole.
inline Mm2Pick mm2_pick(int M, int N, int K, int cus, size_t acc_elems) {
    auto queue = [&](int br, int bn) {
        const int64_t t = (int64_t)((2 * (int64_t)M + br - 1) / br) * ((N + bn - 1) / bn);
        return (double)((t + cus - 1) / cus);
    };
    const double q2 = queue(128, 128), q4 = queue(64, 128), q5 = queue(64, 64);
    const double cost[6] = {53.0 * queue(256, 256),
                            44.5 * queue(192, 256),
                            q2 <= 1 ? 28.0 : 17.6 * q2,
                            q2 <= 1 ? 22.0 : 21.0 * q2,
                            q4 <= 1 ? 25.0 : q4 <= 2 ? 28.0 : 12.0 * q4,
                            q5 <= 1 ? 14.0 : q5 <= 2 ? 19.0 : 7.0 * q5 + 6.0};
    int best = 0;
    for (int i = 1; i < 6; ++i)
        if (cost[i] < cost[best]) best = i;
    Mm2Pick p;
    p.tile = (Mm2Tile)best;
    if (K >= 2048) {
        const Mm2SplitPlan sp = mm2_split_plan<1, 1, 2, 4, 2, 128>(M, N, K, cus, acc_elems, cus + 1);
        if (sp.split) {
            const double qs = (double)((sp.nitems + cus - 1) / cus);
            const double t = (double)sp.kslice / 3584.0 * (qs <= 1 ? 25.0 : qs <= 2 ? 28.0 : 12.0 * qs) + 5.0 +
                             (double)M * N * sp.ns / 180000.0;
            if (t < (double)K / 3584.0 * cost[best]) p.tile = kMm2T64, p.split = true;
        }
    }
    return p;
}

// ---- the fragment-major products of decode batches (gemm_frag.h) ----------

constexpr int kFragWaves = 8;
constexpr int kFragMaxRows = 32;  // token rows: 64 plane rows, RT = 4

// Plane-row tiles for R token rows (0: too many rows).
inline int frag_rt(int R) { return R <= 8 ? 1 : (R <= 16 ? 2 : (R <= kFragMaxRows ? 4 : 0)); }

// The LDS a launch needs: the reduction of ngb row groups and, for the
// staged epilogue, R x 16 ngb int16.  At least 81 KiB, so that one block
// runs per CU (the grid has one block per CU).
inline size_t frag_lds(int rt, int ngb, int R, bool staged) {
    const size_t red = (size_t)ngb * (rt * 256 + 16) * 4;
    const size_t stage = staged ? (size_t)R * 16 * ngb * 2 : 0;
    return std::max<size_t>(red + stage, 81 * 1024);
}
constexpr size_t kFragLdsMax = 160 * 1024;

// One K slice, the whole sum to the staged epilogue (gate/up with its SiLU):
// K <= 8 x 8 KiB (KT <= 64), N % 16 == 0.
inline bool frag_full_ok(int R, int K, int N, int cus) {
    if (frag_rt(R) == 0 || R < 1 || K <= 0 || K % 64 != 0 || K / 64 > kFragWaves * 8 || N <= 0 || N % 16 != 0) return false;
    const int NG = N / 16, ngb = (NG + cus - 1) / cus;
    return 16 * ngb <= kFragWaves * 64 && frag_lds(frag_rt(R), ngb, R, true) <= kFragLdsMax;
}

// Split-K plan: KPW K tiles per wave (8 or 5), S = ceil(KT / (8 KPW)) K
// slices of 8 KPW tiles, P = cus / S row parts; the plan whose busiest wave
// streams the fewest tiles (ceil(NG / P) row groups x KPW).  For the 7B down
// product (296 K tiles, 224 row groups): 5 x 8 slices, 7 row groups per block
// (the busiest wave 35 tiles; 8 tiles a wave in 5 slices: 40).
struct FragSplit {
    int kpw = 0, S = 0, P = 0, ngb = 0;
};
inline FragSplit frag_split_plan(int K, int N, int cus) {
    FragSplit best;
    const int KT = K / 64, NG = (N + 15) / 16;
    for (int kpw : {8, 5}) {
        const int S = (KT + kFragWaves * kpw - 1) / (kFragWaves * kpw);
        if (S > cus) continue;
        const int P = std::max(1, cus / S), ngb = (NG + P - 1) / P;
        if (best.kpw == 0 || ngb * kpw < best.ngb * best.kpw) best = FragSplit{kpw, S, P, ngb};
    }
    return best;
}

// The output policies map the block's 16 ngb columns onto its 512 threads
// (FragCols), so a plan needs 16 ngb <= 512.
inline bool frag_split_ok(int R, int K, int N, int cus, size_t acc_elems) {
    if (frag_rt(R) == 0 || R < 1 || K <= 0 || K % 64 != 0 || N <= 0 || (size_t)R * (size_t)N > acc_elems) return false;
    const FragSplit sp = frag_split_plan(K, N, cus);
    return sp.kpw != 0 && 16 * sp.ngb <= kFragWaves * 64 && frag_lds(frag_rt(R), sp.ngb, R, false) <= kFragLdsMax;
}

// ---- products of 2-32 rows on row-major weights (gemm_rows.h) ---------------

constexpr int kRowsWaves = 8;
constexpr int kRowsUnit = 2048;  // bytes of a unit: 16 weight rows x 128 bytes
constexpr int kRowsRing = 8;     // units a wave has in flight (a power of two)
constexpr int kRowsCpol = 2;     // the weights' cache policy: streaming
constexpr int kRowsOpsBytes = 8; // output operands of a column, kept in LDS
constexpr int kRowsMaxGroups = 80;  // row groups per block: their operands fit the LDS

// Row groups per epilogue window and the LDS of a launch: the waves' rings, two
// windows of plane sums (RT KiB a group), three of weight row sums, the
// activations' sums; a launch adds its columns' operands.
template <int RT>
struct RowsDims {
    static constexpr int G = RT <= 2 ? 4 : 2;
    static constexpr size_t kLds =
        (size_t)kRowsWaves * kRowsRing * kRowsUnit + (size_t)(2 * G * RT * 256 + 3 * G * 16 + RT * 16) * 4;
    static_assert(kLds + 16 * kRowsMaxGroups * kRowsOpsBytes <= 160 * 1024, "LDS of a CU");
};

// S K slices of csl columns (128 weight bytes) x P parts of the row groups, at
// most one block per CU; U columns per wave.  S == 0: not supported.
struct RowsPlan {
    int S = 0, P = 0, U = 0, C = 0, csl = 0, ngb = 0;
};

// Where lane l of load j (of two) of a unit fetches its 16 bytes: the byte offset
// within the block's rows (rowb bytes each) of row 16 g + 8 j + l / 8 and of the
// 16-byte chunk whose LDS slot is l % 8 (chunk c of row r sits at slot
// c ^ ((r / 2) % 8)) of column cb + u, as the lane's part and the unit's.  Their sum is
// the load's one offset, checked against the block's bytes: rows past N (the
// last group of N % 16 != 0) and the bytes past K of the last row's last
// column lie past them and read no memory.
constexpr uint32_t rows_lane_off(int j, int lane, uint32_t rowb, int cb) {
    const int row = 8 * j + (lane >> 3);
    return (uint32_t)row * rowb + (uint32_t)cb * 128u + (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) << 4);
}
constexpr uint32_t rows_unit_off(int g, int u, uint32_t rowb) { return (uint32_t)g * 16u * rowb + (uint32_t)u * 128u; }

// With one column per wave and four plane tiles, a unit's LDS adds (17 a wave)
// outlast its load; long row ranges then go to the plane tiles (151936 x 896 over
// 24 / 32 rows: 41.3 / 43.2 us here, 37.5 / 41.3 there; 32001 x 896: 15.0 / 15.4
// and 15.9 / 16.5).
inline bool rows_short_sums(int M, int U, int ngb, int wbytes) { return wbytes == 1 && M > 16 && U == 1 && ngb > 16; }

// The plan whose busiest block ends first.  A CU streams about 24 KB/us when all
// do (6.2 TB/s); a K split adds the finish launch (about 4 us) and its 64-bit
// atomics (about 90 a ns for the chip).  7B down: 8 slices x 32 parts of 7 row
// groups at 2-8 rows, 5 x 51 of 5 at 13-32; the 7B head (9504 groups) needs none.
// (8 slices at 13 rows measured 19.7 us against 20.7 with 5, in one run where
// the same plan differed by up to 2.5% between the sides: not taken.)
inline RowsPlan rows_plan(int M, int N, int K, int wbytes, int cus, size_t acc_elems) {
    RowsPlan best;
    if (M < 2 || M > kFragMaxRows || N < 1 || N >= (1 << 22) || K % 64 != 0 || K * wbytes < 128 || K >= 65536 || cus < 1 || cus > 1024)
        return best;
    const int C = (K * wbytes + 127) / 128, umax = wbytes == 1 ? 4 : 8, NG = (N + 15) / 16;
    double best_t = 0;
    for (int S = 1; S <= std::min(C, 16) && S <= cus; ++S) {
        if (S > 1 && (wbytes != 1 || (size_t)M * (size_t)N > acc_elems)) break;
        const int csl = (C + S - 1) / S, U = (csl + kRowsWaves - 1) / kRowsWaves;
        if (U > umax || (int64_t)(S - 1) * csl >= C) continue;
        const int P = std::min(cus / S, NG), ngb = (NG + P - 1) / P;
        if (rows_short_sums(M, U, ngb, wbytes)) continue;
        if (ngb > kRowsMaxGroups || (int64_t)ngb * 16 * K * wbytes >= (1ll << 31)) continue;
        const double t = (double)ngb * csl * kRowsUnit / 24200.0 + (S > 1 ? 4.0 + (double)M * N * S / 90000.0 : 0.0);
        if (best.S == 0 || t < best_t) best = RowsPlan{S, P, U, C, csl, ngb}, best_t = t;
    }
    return best;
}

// ---- the grouped expert products (moe.hip) ----------------------------------

// Byte-plane tiles (tokens x weight rows): 0: 128 x 256 (two 128-byte stages), 1:
// 128 x 128 (64-byte stages), 2: 64 x 128 (two 128-byte stages), 3: 32 x 64 (three).
constexpr int moe_tile_tokens(int tile) { return tile == 2 ? 64 : tile == 3 ? 32 : 128; }
constexpr int moe_tile_rows(int tile) { return tile == 0 ? 256 : tile == 3 ? 64 : 128; }

// Small tiles waste less on experts of few tokens and keep more blocks loading,
// large ones move fewer operand bytes; the whole 60-expert layer on MI355X, us:
//   tokens (rows per expert)   16 (1)  100 (7)  400 (27)  1000 (67)  2400 (160)  3001 (200)
//   tile 0                     157     261      316       426        664         795
//   tile 2                     125     210      265       379        647         807
//   tile 3                     114     202      283       444        878
// Tile 1 only where a K is not a multiple of 128 (k128 false).  R routed rows of E
// experts.
constexpr int kMoeRows2 = 14, kMoeRows0 = 180;  // rows per expert from which tiles 2 and 0 are taken
constexpr int moe_pick_tile(bool k128, int R, int E) {
    return !k128 ? 1 : R >= kMoeRows0 * E ? 0 : R >= kMoeRows2 * E ? 2 : 3;
}

// Work items of one grouped product over R routed rows of E experts, N weight
// rows: sum_e ceil(c_e / tokens) <= floor(R / tokens) + E token tiles.
constexpr int moe_max_items(int R, int E, int tile, int N) {
    return (R / moe_tile_tokens(tile) + E) * ((N + moe_tile_rows(tile) - 1) / moe_tile_rows(tile));
}
// Both products' (2 I and H weight rows).
constexpr int moe_work_items(int R, int E, int tile, int I, int H) {
    return moe_max_items(R, E, tile, 2 * I) + moe_max_items(R, E, tile, H);
}
// The most that a call over up to R rows needs: fewer rows take smaller tiles
// and can need more items, so a table sized for this is not grown again by a
// smaller call (growing frees and allocates, which a captured call must not).
inline int moe_work_cap(bool k128, int R, int E, int I, int H) {
    int most = moe_work_items(R, E, moe_pick_tile(k128, R, E), I, H);
    for (int b : {kMoeRows2 * E - 1, kMoeRows0 * E - 1})
        if (k128 && b < R) most = std::max(most, moe_work_items(b, E, moe_pick_tile(true, b, E), I, H));
    return most;
}

}  // namespace myl
