// gemm_mfma2.h -- the large-M W8A16 product on the int8 matrix cores.
//
// y[m][n] = epilogue(n, m, sum_k W[n][k] * x[m][k])  (exact i64 sums)
//
// The activations are split once, before the product, into byte planes laid
// out as interleaved rows of an int8 matrix A' [2M x K]: row 2m = hi(x_m) =
// x_m >> 8, row 2m + 1 = lo'(x_m) = (x_m & 255) - 128.  The product is then a
// plain int8 GEMM over 2M rows, C' = A' . W^T, and
//   sum_k w*x = 256 * C'[2m][n] + C'[2m+1][n] + 128 * sum_k W[n][k]
// with the row sums of W taken by v_dot4 on the B fragments.  In the 32x32
// accumulator layout rows 2m and 2m+1 land in registers r and r+1 of the same
// lane, so the combination needs no data movement.
//
// Tiling (gfx950, 160 KB LDS): a block of WM x WN waves owns BR = 32*MB*WM
// rows of A' and BN = 32*NB*WN weight rows; K advances KS = 64 or 128 bytes
// per stage through STAGES LDS buffers filled by direct global-to-LDS loads
// (global_load_lds_dwordx4: each wave instruction writes 1 KiB = 1024/KS rows
// x KS bytes): all STAGES buffers are filled before the loop, each is refilled
// as soon as the barrier that frees it is past, and a stage is awaited with an
// explicit vmcnt.  128-byte stages read whole cache lines of every row per load
// instruction and halve the barriers per K; 64-byte ones are kept for a K that
// is no multiple of 128.  The KS/16 chunks of LDS row r sit at slot
// chunk ^ ((r / (256/KS)) % (KS/16)), so the 16-byte fragment reads of 16
// consecutive rows cover all 64 banks once.  K must be a multiple of KS; rows
// past the matrix clamp to its last row (their outputs are discarded), so
// every load stays in bounds.
#pragma once

#include "gemm_mfma.h"
#include "internal.h"
#include "mm_plan.h"
#include "wave.h"

#include <algorithm>
#include <type_traits>

namespace myl {

typedef __attribute__((address_space(3))) void lds_void;

// x int16 [M x K] -> Ap int8 [2M x K]: row 2m = hi(x_m), row 2m+1 = lo'(x_m).
template <int = 0>
__global__ __launch_bounds__(256) void split_planes_kernel(const int16_t* __restrict__ x, int M, int ldx, int K, int8_t* __restrict__ Ap) {
    const int m = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;  // 8-element chunk
    if (m >= M || c * 8 >= K) return;
    const uint4 v = *reinterpret_cast<const uint4*>(x + (size_t)m * ldx + c * 8);
    uint2 h, l;
    split_planes8(v, h, l);
    *reinterpret_cast<uint2*>(Ap + (size_t)(2 * m) * K + c * 8) = h;
    *reinterpret_cast<uint2*>(Ap + (size_t)(2 * m + 1) * K + c * 8) = l;
}

// The wave's loads but the last N and its LDS reads done, then the block barrier.
template <int N>
__device__ inline void mm2_stage_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int MB, int NB, int WM_, int WN_, int STAGES, int KS = 64>
struct Mm2 : Mm2Dims<MB, NB, WM_, WN_, STAGES, KS> {
    using D = Mm2Dims<MB, NB, WM_, WN_, STAGES, KS>;
    __device__ static int slot(int row, int chunk) { return chunk ^ ((row / D::kSwzRows) & (D::kCpr - 1)); }
};

// Order of a product's output tiles over the grid.  mm_tile_index gives each
// XCD a contiguous range of tile numbers; here tile numbers run over groups
// of G row tiles (the last group may have fewer), the row tile fastest inside
// a group.  G = tiles_r is the plain order (all row tiles of one weight tile,
// then the next weight tile): the blocks an XCD runs at one time share one
// weight tile and read as many distinct A' tiles.  A small G makes them cover
// G row tiles x (blocks / G) weight tiles, so both operands are shared in the
// XCD's L2.
struct TileOrder {
    Divider span;        // G * tiles_n
    Divider g, g_last;   // row tiles of a group, of the last group
    uint32_t last;       // the last group
    static TileOrder of(int tiles_r, int tiles_n, int G) {
        G = mm2_group_rows(tiles_r, G);
        const int last = (tiles_r - 1) / G;
        return TileOrder{Divider::of((uint32_t)(G * tiles_n)), Divider::of((uint32_t)G),
                         Divider::of((uint32_t)(tiles_r - last * G)), (uint32_t)last};
    }
    __device__ inline void decode(uint32_t t, uint32_t& tn, uint32_t& tr) const {
        uint32_t grp, in, r;
        span.divmod(t, grp, in);
        if (grp < last) g.divmod(in, tn, r);
        else g_last.divmod(in, tn, r);
        tr = grp * g.d + r;
    }
};

// LDS layout of a stage: BR A' rows then BN weight rows, KS bytes each, the
// chunks of each row at Mm2::slot.
// The pipelined main loop: acc[i][j] = A' tile i x W tile j over K in
// [kb, ke) (multiples of KS); rs[j] = the lane's weight-row sum (summed over
// the lane pair l, l + 32 only after the loop).
// The fragments of the next 32 bytes of K are read from LDS while the current
// ones multiply (two register sets).  The switch to the next stage falls
// between the halves of a stage's last 32 bytes: by then the wave has read all
// of its current stage, so one barrier both publishes the next stage and
// frees the current buffer, and the second half of the multiplies covers the
// barrier and the first reads.
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS = 64>
__device__ inline void mm2_main(const int8_t* __restrict__ Ap, int R2, const int8_t* __restrict__ W, int N, int K,
                                int kb, int ke, int r0, int n0, int8_t* lds, v16i32_t (&acc)[MB][NB],
                                int32_t (&rs)[NB]) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    constexpr int SUB = KS / 32, L = S::kLoads;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM_, wn = wave / WM_;
    const int nk = (ke - kb) / KS;
    // Each wave-level load moves 1 KiB (64 lanes x 16 bytes) of 1024/KS rows:
    // lane l takes row l / (KS/16) of the group and the global chunk whose
    // swizzled slot is l % (KS/16) (the swizzle is its own inverse).
    auto group = [&](int i) { return min(wave + i * (S::kThreads / 64), S::kGroups - 1); };
    const int8_t* src[L];
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const int row = group(i) * S::kRowsPerLoad + lane / S::kCpr;  // A' rows first
        const int chunk = S::slot(row, lane & (S::kCpr - 1));
        const int8_t* p = row < S::BR ? Ap + (size_t)min(r0 + row, R2 - 1) * K : W + (size_t)min(n0 + row - S::BR, N - 1) * K;
        src[i] = p + kb + chunk * 16;
    }
    auto issue = [&](int kt) {
        int8_t* st = lds + (kt % STAGES) * S::kStageBytes;
#pragma unroll
        for (int i = 0; i < L; ++i)
            __builtin_amdgcn_global_load_lds((const void*)(src[i] + (size_t)kt * KS),
                                             (lds_void*)(st + group(i) * 1024), 16, 0, 0);
    };
    // A wave's fragments of 32 bytes of K: 16 bytes per lane, rows 32 apart
    // share a swizzle slot.
    int ao[SUB], bo[SUB];
#pragma unroll
    for (int s = 0; s < SUB; ++s) {
        const int chunk = 2 * s + (lane >> 5);
        const int ra = wm * MB * 32 + (lane & 31), rb = S::BR + wn * NB * 32 + (lane & 31);
        ao[s] = ra * KS + (S::slot(ra, chunk) << 4);
        bo[s] = rb * KS + (S::slot(rb, chunk) << 4);
    }
    v4i32_t a[2][MB], b[2][NB];
    auto read = [&](int kt, int s, v4i32_t (&fa)[MB], v4i32_t (&fb)[NB]) {
        const int8_t* st = lds + (kt % STAGES) * S::kStageBytes;
#pragma unroll
        for (int j = 0; j < NB; ++j) fb[j] = *reinterpret_cast<const v4i32_t*>(st + bo[s] + j * 32 * KS);
#pragma unroll
        for (int i = 0; i < MB; ++i) fa[i] = *reinterpret_cast<const v4i32_t*>(st + ao[s] + i * 32 * KS);
    };
    auto mul = [&](const v4i32_t (&fa)[MB], const v4i32_t (&fb)[NB], int j0, int j1) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (j < j0 || j >= j1) continue;
#pragma unroll
            for (int i = 0; i < MB; ++i) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) rs[j] = sdot4((uint32_t)fb[j][q], 0x01010101u, rs[j]);
        }
    };
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        rs[j] = 0;
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
    }
    // Loads retire in order, so with n later stages in flight a stage has
    // landed when at most n L loads of the wave are outstanding.  lgkmcnt(0):
    // the wave's reads of the buffer that the barrier frees are done.
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
        if (s < nk) issue(s);
    if (nk >= STAGES) mm2_stage_barrier<L*(STAGES - 1)>();
    else mm2_stage_barrier<0>();
    read(0, 0, a[0], b[0]);
    for (int kt = 0; kt < nk; ++kt) {
#pragma unroll
        for (int s = 0; s < SUB - 1; ++s) {
            read(kt, s + 1, a[(s + 1) & 1], b[(s + 1) & 1]);
            mul(a[s & 1], b[s & 1], 0, NB);
        }
        constexpr int cur = (SUB - 1) & 1, nxt = cur ^ 1;
        mul(a[cur], b[cur], 0, NB / 2);
        __builtin_amdgcn_sched_barrier(0);
        if (kt + 1 < nk) {
            if (kt + STAGES - 1 < nk) mm2_stage_barrier<L*(STAGES - 2)>();
            else mm2_stage_barrier<0>();
            if (kt + STAGES < nk) issue(kt + STAGES);
            read(kt + 1, 0, a[nxt], b[nxt]);
        }
        __builtin_amdgcn_sched_barrier(0);
        mul(a[cur], b[cur], NB / 2, NB);
    }
}

// Accumulator register r (even: the hi row of a token, r + 1 its lo' row) of a
// 32-row tile holds A' row mm2_row(r) + 4 (lane / 32) of the tile.
__device__ inline constexpr int mm2_row(int r) { return 8 * (r >> 2) + (r & 3); }

// 32-bit sums u * 256 + r need K < 2^16 (fixed.h, PlaneRescale).
constexpr int kPlaneSumK = 65536;

// One wave's part of a tile's epilogue.  Column operands are resolved once and
// an accumulator tile's element operands are all loaded before its first
// store: the stores may alias them, so loads left in the per-value code would
// wait out the memory latency once per value, and did: with 64-bit (multiplier:
// 128-bit) arithmetic under a branch per value the epilogue took 0.7 of the
// main loop's time (multiplier requant, 4001 x 18944 x 3584: 954 us of which
// 570 the loop).
template <int MB, int NB, bool FULL, class Sink>
__device__ inline void mm2_emit(const v16i32_t (&acc)[MB][NB], const int32_t (&rs)[NB], int R2, int N, int arow0,
                                int nw0, int lane, const Sink& sink) {
    // an element's place is a uniform offset plus the lane's own (32 bits)
    const int n_l = lane & 31, m_l = 2 * (lane >> 5), m0 = arow0 >> 1;
    uint32_t lo = (uint32_t)(sink.idx(n_l, m_l) - sink.idx(0, 0));
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int nj = nw0 + j * 32, n = nj + n_l;
        asm("" : "+v"(lo));  // no per-lane addresses kept from one j for the next: they cost two registers each
        const typename Sink::Col col = sink.col(FULL ? n : min(n, N - 1));
        const int32_t rs128 = (int32_t)((uint32_t)rs[j] << 7);
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const int mi = m0 + i * 16;
            typename Sink::Elt elt[8];
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const int d = mm2_row(r) >> 1;
                if (FULL || (2 * (mi + d + m_l) < R2 && n < N)) elt[r >> 1] = sink.elt(sink.idx(nj, mi + d), lo);
            }
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const int d = mm2_row(r) >> 1;
                if (!FULL && (2 * (mi + d + m_l) >= R2 || n >= N)) continue;
                const int32_t low = acc[i][j][r + 1] + rs128;
                sink.put(sink.idx(nj, mi + d), lo, acc[i][j][r] + (low >> 8), (uint32_t)low & 255u, col, elt[r >> 1]);
            }
        }
    }
}

// The same from 64-bit sums (a column's shift or K outside the 32-bit range),
// one register pair at a time.  The column's operands are loaded once: behind
// the stores, which may alias them, they cost a memory round trip per value.
template <int MB, int NB, class Sink>
__device__ inline void mm2_emit64(const v16i32_t (&acc)[MB][NB], const int32_t (&rs)[NB], int R2, int N, int arow0,
                                  int nw0, int lane, const Sink& sink) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int n = nw0 + j * 32 + (lane & 31);
        const auto ops = sink.ops(min(n, N - 1));
#pragma unroll
        for (int i = 0; i < MB; ++i) {
#pragma unroll 2
            for (int r = 0; r < 16; r += 2) {
                const int64_t v = (int64_t)acc[i][j][r] * 256 + (int64_t)acc[i][j][r + 1] + (int64_t)rs[j] * 128;
                const int m = ((arow0 + i * 32 + mm2_row(r)) >> 1) + 2 * (lane >> 5);
                if (2 * m < R2 && n < N) sink.put64(n, m, v, ops);
            }
        }
    }
}

// A multiplier sink whose columns' results fit 32 bits before their clamp: a wave
// of such columns skips the 64-bit clamp (4001 x 18944 x 3584, shifts 41-43: 586 us,
// 595 with it; in another run 576, and 583 with it in the ragged last tiles alone).
template <class Sink>
struct SinkNarrow {
    const Sink& s;
    using Col = PlaneMultNarrow;
    using Elt = typename Sink::Elt;
    __device__ inline Col col(int n) const { return Col{s.col(n)}; }
    __device__ inline Elt elt(size_t i, uint32_t lo) const { return s.elt(i, lo); }
    __device__ inline size_t idx(int n, int m) const { return s.idx(n, m); }
    __device__ inline void put(size_t i, uint32_t lo, int32_t u, uint32_t r, const Col& c, const Elt& x) const { s.put(i, lo, u, r, c, x); }
};

// K runs over [kb, ke) (multiples of KS).
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class Sink>
__device__ inline void mm2_tile(const int8_t* __restrict__ Ap, int R2, const int8_t* __restrict__ W, int N, int K,
                                int kb, int ke, int r0, int n0, int8_t* lds, const Sink& sink) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM_, wn = wave / WM_;
    v16i32_t acc[MB][NB];
    int32_t rs[NB];
    mm2_main<MB, NB, WM_, WN_, STAGES, KS>(Ap, R2, W, N, K, kb, ke, r0, n0, lds, acc, rs);
    const int arow0 = r0 + wm * MB * 32, nw0 = n0 + wn * NB * 32;
    if (arow0 >= R2 || nw0 >= N) return;
    bool fast = ke - kb < kPlaneSumK, narrow = true;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        rs[j] += __shfl_xor(rs[j], 32);
        const typename Sink::Col c = sink.col(min(nw0 + j * 32 + (lane & 31), N - 1));
        fast = fast && __all((int)c.fast);
        if constexpr (std::is_same_v<typename Sink::Col, PlaneMult>) narrow = narrow && __all(c.t + 8u >= kPlaneMultNarrow);
    }
    const bool whole = arow0 + MB * 32 <= R2 && nw0 + NB * 32 <= N;
    if constexpr (std::is_same_v<typename Sink::Col, PlaneMult>) {
        if (fast && narrow) {
            const SinkNarrow<Sink> sn{sink};
            if (whole) mm2_emit<MB, NB, true>(acc, rs, R2, N, arow0, nw0, lane, sn);
            else mm2_emit<MB, NB, false>(acc, rs, R2, N, arow0, nw0, lane, sn);
            return;
        }
    }
    if (!fast) mm2_emit64<MB, NB>(acc, rs, R2, N, arow0, nw0, lane, sink);
    else if (whole) mm2_emit<MB, NB, true>(acc, rs, R2, N, arow0, nw0, lane, sink);
    else mm2_emit<MB, NB, false>(acc, rs, R2, N, arow0, nw0, lane, sink);
}

template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class Epi>
__global__ __launch_bounds__(WM_ * WN_ * 64, (Mm2Dims<MB, NB, WM_, WN_, STAGES, KS>::kMinWaves)) void mm2_kernel(const int8_t* __restrict__ Ap, int R2, const int8_t* __restrict__ W,
                                                             int N, int K, TileOrder ord, int ntiles, Epi epi) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    extern __shared__ __align__(16) int8_t lds[];
    const int t = mm_tile_index(ntiles);
    if (t < 0) return;
    uint32_t tn, tr;
    ord.decode((uint32_t)t, tn, tr);
    mm2_tile<MB, NB, WM_, WN_, STAGES, KS>(Ap, R2, W, N, K, 0, K, (int)tr * S::BR, (int)tn * S::BN, lds, SinkEpi<Epi>{epi});
}

// A tile with a staged epilogue, for products whose output columns pair up
// (2i, 2i+1 -> element i of an output row): every sum is first reduced to an
// int16 by sink.stage and parked in LDS as a [BR/2 x BN] tile (the K
// stages are free by then); the block then hands sink.emit(m, i0, v) the 16
// staged values of columns 2 i0 .. 2 i0 + 15 of row m, for 8-column chunks of
// N / 2 (N % 16 == 0), so the outputs leave in whole 8-byte pieces.  The pairs
// are gate and up of the SiLU gate, whose table the sink names.
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class Sink>
__device__ inline void mm2_staged_tile(const int8_t* __restrict__ Ap, int R2, const int8_t* __restrict__ W, int N, int K,
                                       int r0, int n0, int8_t* lds, const Sink& sink) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    static_assert((size_t)(S::BR / 2) * S::BN * 2 <= S::kLds, "staged tile fits the stage buffers");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM_, wn = wave / WM_;
    v16i32_t acc[MB][NB];
    int32_t rs[NB];
    mm2_main<MB, NB, WM_, WN_, STAGES, KS>(Ap, R2, W, N, K, 0, K, r0, n0, lds, acc, rs);
    __syncthreads();  // every wave is past its last stage read
    int16_t* tile = reinterpret_cast<int16_t*>(lds);  // [BR / 2][BN]
    // The gate's table follows the tile in LDS when it fits in whole 1 KiB
    // loads, which run while the sums are staged: a wave's 64 lookups hit 64
    // lines, and a 32 KB table does not stay in the vector cache beside the
    // stores (1500 x 37888 x 3584: 458 us, 465 with lookups through it; the MoE
    // layer over 3001 tokens 702 and 720).
    constexpr uint32_t kTileBytes = (uint32_t)(S::BR / 2) * S::BN * 2;
    const uint32_t lut_bytes = sink.silu_table_len() * 2u;
    const bool lut_lds = lut_bytes % 1024 == 0 && kTileBytes + lut_bytes <= S::kLds && ((uintptr_t)sink.silu_table() & 15) == 0;
    int8_t* lut_l = lds + kTileBytes;
    if (lut_lds)
        for (uint32_t o = (uint32_t)wave * 1024u; o < lut_bytes; o += S::kThreads * 16u)
            __builtin_amdgcn_global_load_lds((const void*)(reinterpret_cast<const int8_t*>(sink.silu_table()) + o + lane * 16),
                                             (lds_void*)(lut_l + o), 16, 0, 0);
    // rows and columns past the matrix hold sums of clamped operands; in the
    // accumulator tiles that reach into it they are staged like the others and
    // never emitted.  Columns outside the 32-bit range (a hidden size of 448: shifts
    // of 8) take 64-bit sums; with their operand loaded again for each value and
    // every tile staged, one token of a 448-wide expert layer took 13.8 us here,
    // 9.4 before the 32-bit steps.
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        rs[j] += __shfl_xor(rs[j], 32);
        const int nl = (wn * NB + j) * 32 + (lane & 31), n = min(n0 + nl, N - 1);
        const typename Sink::Col col = sink.col(n);
        const bool fast = K < kPlaneSumK && __all((int)col.fast);
        const int32_t rs128 = (int32_t)((uint32_t)rs[j] << 7);
        int16_t* tj = tile + (wm * MB * 16 + 2 * (lane >> 5)) * S::BN + nl;
        if (fast) {
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                if (r0 + (wm * MB + i) * 32 >= R2) break;  // uniform
#pragma unroll
                for (int r = 0; r < 16; r += 2) {
                    const int32_t low = acc[i][j][r + 1] + rs128;
                    tj[((i * 32 + mm2_row(r)) >> 1) * S::BN] = sink.stage(col, acc[i][j][r] + (low >> 8), (uint32_t)low & 255u);
                }
            }
        } else {
            const auto op = sink.op(n);
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                if (r0 + (wm * MB + i) * 32 >= R2) break;
#pragma unroll 2
                for (int r = 0; r < 16; r += 2)
                    tj[((i * 32 + mm2_row(r)) >> 1) * S::BN] =
                        sink.stage64(op, n, (int64_t)acc[i][j][r] * 256 + (int64_t)acc[i][j][r + 1] + (int64_t)rs[j] * 128);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the wave's part of the table
    __syncthreads();
    constexpr int kChunks = S::BN / 16;  // 8-column output chunks per tile row
    const int m0 = r0 >> 1, i00 = n0 >> 1;
    auto emit_all = [&](const int16_t* lut) {
        for (int c = threadIdx.x; c < (S::BR / 2) * kChunks; c += S::kThreads) {
            const int ml = c / kChunks, ic = c % kChunks;  // powers of two
            const int m = m0 + ml, i0 = i00 + ic * 8;
            if (2 * m >= R2 || 2 * i0 >= N) continue;
            const uint4* src = reinterpret_cast<const uint4*>(tile + ml * S::BN + ic * 16);
            sink.emit(m, i0, src[0], src[1], lut);
        }
    };
    if (lut_lds) emit_all(reinterpret_cast<const int16_t*>(lut_l));
    else emit_all(sink.silu_table());
}

template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class Epi>
__global__ __launch_bounds__(WM_ * WN_ * 64, (Mm2Dims<MB, NB, WM_, WN_, STAGES, KS>::kMinWaves)) void mm2_staged_kernel(const int8_t* __restrict__ Ap, int R2,
                                                                    const int8_t* __restrict__ W, int N, int K,
                                                                    TileOrder ord, int ntiles, Epi epi) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    extern __shared__ __align__(16) int8_t lds[];
    const int t = mm_tile_index(ntiles);
    if (t < 0) return;
    uint32_t tn, tr;
    ord.decode((uint32_t)t, tn, tr);
    mm2_staged_tile<MB, NB, WM_, WN_, STAGES, KS>(Ap, R2, W, N, K, (int)tr * S::BR, (int)tn * S::BN, lds, epi);
}

// group: row tiles per group of the tile order (TileOrder; 0: the plain order).
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class Epi>
hipError_t mm2_staged_launch(const int8_t* Ap, int M, const int8_t* W, int N, int K, const Epi& epi, hipStream_t st,
                             int group = 0) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    const int R2 = 2 * M;
    const int tiles_r = (R2 + S::BR - 1) / S::BR, tiles_n = (N + S::BN - 1) / S::BN;
    const TileOrder ord = TileOrder::of(tiles_r, tiles_n, group);
    const int ntiles = tiles_r * tiles_n;
    auto kern = mm2_staged_kernel<MB, NB, WM_, WN_, STAGES, KS, Epi>;
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
    if (e != hipSuccess) return e;
    kern<<<8 * ((ntiles + 7) / 8), S::kThreads, S::kLds, st>>>(Ap, R2, W, N, K, ord, ntiles, epi);
    return hipGetLastError();
}

// int16 weights as byte planes: Wp [2N x K] with row 2n = hi(w_n), row
// 2n+1 = lo'(w_n), and wsum[n] = sum_k w_n[k]; likewise xsum[m] for the
// activations.  One int8 product over 2M x 2N plane rows yields the four
// plane products of each (m, n): in the 32x32 accumulator layout rows 2m and
// 2m+1 sit in registers r, r+1 of one lane and columns 2n, 2n+1 in lanes
// l, l^1, so a DPP swap of lane pairs assembles
//   x.w = 65536*hh + 256*(h lo' + lo' h) + lo' lo' + 128*(xsum + wsum) - 16384*K.
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class Epi>
__device__ inline void mm2w16_tile(const int8_t* __restrict__ Ap, int R2, const int8_t* __restrict__ Wp, int N2,
                                   int K, const int32_t* __restrict__ xsum, const int32_t* __restrict__ wsum, int r0,
                                   int n0, int8_t* lds, const Epi& epi) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM_, wn = wave / WM_;
    v16i32_t acc[MB][NB];
    int32_t rs[NB];
    mm2_main<MB, NB, WM_, WN_, STAGES, KS>(Ap, R2, Wp, N2, K, 0, K, r0, n0, lds, acc, rs);
    const bool even = (lane & 1) == 0;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int np = n0 + (wn * NB + j) * 32 + (lane & 31);
        const int n = np >> 1;
        const int nc = min(n, (N2 >> 1) - 1);
        const typename Epi::Ops o = epi.ops(nc);
        const int64_t nterm = 128 * (int64_t)wsum[nc] - 16384 * (int64_t)K;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const int arow0 = r0 + (wm * MB + i) * 32 + 4 * (lane >> 5);
            int32_t xs[8];  // ahead of the stores, as in mm2_emit
#pragma unroll
            for (int r = 0; r < 16; r += 2) xs[r >> 1] = xsum[min(arow0 + mm2_row(r), R2 - 2) >> 1];
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const int32_t a0 = acc[i][j][r], a1 = acc[i][j][r + 1];
                const int32_t b0 = dpp_mov<dpp::kXor1>(a0), b1 = dpp_mov<dpp::kXor1>(a1);
                const int arow = arow0 + mm2_row(r);
                if (even && arow < R2 && np < N2)
                    epi.one_ops(n, arow >> 1, 65536 * (int64_t)a0 + 256 * ((int64_t)a1 + (int64_t)b0) + (int64_t)b1 +
                                                  128 * (int64_t)xs[r >> 1] + nterm, o);
            }
        }
    }
}

template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class Epi>
__global__ __launch_bounds__(WM_ * WN_ * 64, (Mm2Dims<MB, NB, WM_, WN_, STAGES, KS>::kMinWaves)) void mm2w16_kernel(const int8_t* __restrict__ Ap, int R2,
                                                                const int8_t* __restrict__ Wp, int N2, int K,
                                                                const int32_t* __restrict__ xsum,
                                                                const int32_t* __restrict__ wsum, TileOrder ord,
                                                                int ntiles, Epi epi) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    extern __shared__ __align__(16) int8_t lds[];
    const int t = mm_tile_index(ntiles);
    if (t < 0) return;
    uint32_t tn, tr;
    ord.decode((uint32_t)t, tn, tr);
    mm2w16_tile<MB, NB, WM_, WN_, STAGES, KS>(Ap, R2, Wp, N2, K, xsum, wsum, (int)tr * S::BR, (int)tn * S::BN, lds,
                                          epi);
}

// x int16 [M x K] -> planes as split_planes_kernel, plus xsum[m] = sum_k x[m][k].
// One block per row.
template <int = 0>
__global__ __launch_bounds__(256) void split_planes_sum_kernel(const int16_t* __restrict__ x, int ldx, int K,
                                                               int8_t* __restrict__ Ap, int32_t* __restrict__ xsum) {
    __shared__ int32_t red[4];
    const int m = blockIdx.x;
    int32_t s = 0;
    for (int c = threadIdx.x; c * 8 < K; c += 256) {
        const uint4 v = *reinterpret_cast<const uint4*>(x + (size_t)m * ldx + c * 8);
        uint2 h, l;
        split_planes8(v, h, l);
        *reinterpret_cast<uint2*>(Ap + (size_t)(2 * m) * K + c * 8) = h;
        *reinterpret_cast<uint2*>(Ap + (size_t)(2 * m + 1) * K + c * 8) = l;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) s += (int32_t)(int16_t)(w[q] & 0xFFFFu) + (int32_t)(int16_t)(w[q] >> 16);
    }
    s = wave_sum_i32(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) xsum[m] = red[0] + red[1] + red[2] + red[3];
}

// Plane rows and sums of int16 rows (the weights of mm2w16, or activations).
inline hipError_t split_planes_sum(const int16_t* x, int M, int ldx, int K, int8_t* Ap, int32_t* xsum, hipStream_t st) {
    split_planes_sum_kernel<><<<M, 256, 0, st>>>(x, ldx, K, Ap, xsum);
    return hipGetLastError();
}

// The int16-weight product for two rows or more: A' and xsum from
// split_planes_sum, Wp and wsum prepared once the same way.  Up to 64 rows:
// 32- or 64-row plane tiles x 128 W' rows (the weight planes stream once);
// more: 256 A' rows x 256 W' rows with 128-byte stages when the grid holds
// at least four tiles per CU (and K % 128 == 0), else 256 x 128 tiles.
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class Epi>
hipError_t mm2w16_launch_cfg(const int8_t* Ap, const int32_t* xsum, int M, const int8_t* Wp, const int32_t* wsum,
                             int N, int K, const Epi& epi, hipStream_t st, int group = 0) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    const int R2 = 2 * M, N2 = 2 * N;
    const int tiles_r = (R2 + S::BR - 1) / S::BR, tiles_n = (N2 + S::BN - 1) / S::BN;
    const TileOrder ord = TileOrder::of(tiles_r, tiles_n, group);
    const int ntiles = tiles_r * tiles_n;
    auto kern = mm2w16_kernel<MB, NB, WM_, WN_, STAGES, KS, Epi>;
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
    if (e != hipSuccess) return e;
    kern<<<8 * ((ntiles + 7) / 8), S::kThreads, S::kLds, st>>>(Ap, R2, Wp, N2, K, xsum, wsum, ord, ntiles, epi);
    return hipGetLastError();
}

template <class Epi>
hipError_t mm2w16_launch(const int8_t* Ap, const int32_t* xsum, int M, const int8_t* Wp, const int32_t* wsum, int N,
                         int K, const Epi& epi, int cus, hipStream_t st) {
    // few rows: one plane-row tile streams the weight planes once
    if (M <= 16 && K % 128 == 0) return mm2w16_launch_cfg<1, 1, 1, 4, 3, 128>(Ap, xsum, M, Wp, wsum, N, K, epi, st);
    if (M <= 16) return mm2w16_launch_cfg<1, 1, 1, 4, 4, 64>(Ap, xsum, M, Wp, wsum, N, K, epi, st);
    if (M <= 32 && K % 128 == 0) return mm2w16_launch_cfg<2, 1, 1, 4, 2, 128>(Ap, xsum, M, Wp, wsum, N, K, epi, st);
    if (M <= 32) return mm2w16_launch_cfg<2, 1, 1, 4, 4, 64>(Ap, xsum, M, Wp, wsum, N, K, epi, st);
    if (M <= 64 && K % 128 == 0) return mm2w16_launch_cfg<2, 1, 2, 2, 3, 128>(Ap, xsum, M, Wp, wsum, N, K, epi, st);
    if (M <= 64) return mm2w16_launch_cfg<2, 1, 2, 4, 4, 64>(Ap, xsum, M, Wp, wsum, N, K, epi, st);
    using W = Mm2<4, 2, 2, 4, 2, 128>;
    const int wide_tiles = ((2 * M + W::BR - 1) / W::BR) * ((2 * N + W::BN - 1) / W::BN);
    if (K % 128 == 0 && wide_tiles >= 4 * cus)
        return mm2w16_launch_cfg<4, 2, 2, 4, 2, 128>(Ap, xsum, M, Wp, wsum, N, K, epi, st);
    return mm2w16_launch_cfg<2, 2, 4, 2, 3, 64>(Ap, xsum, M, Wp, wsum, N, K, epi, st);
}

// Split-K form: item t -> (slice t / ntiles, tile t % ntiles); the exact
// partial sums of each slice are added into acc [M x N] (i64, zero-kept; the
// finish kernel applies the epilogue and clears it).
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS = 64>
__global__ __launch_bounds__(WM_ * WN_ * 64, (Mm2Dims<MB, NB, WM_, WN_, STAGES, KS>::kMinWaves)) void mm2_splitk_kernel(const int8_t* __restrict__ Ap, int R2,
                                                                    const int8_t* __restrict__ W, int N, int K,
                                                                    Divider tiles_r, Divider ntiles, int nitems,
                                                                    int kslice, unsigned long long* __restrict__ acc) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    extern __shared__ __align__(16) int8_t lds[];
    const int t = mm_tile_index(nitems);
    if (t < 0) return;
    uint32_t ks, tile, tn, tr;
    ntiles.divmod((uint32_t)t, ks, tile);
    tiles_r.divmod(tile, tn, tr);
    const int kb = (int)ks * kslice, ke = min(K, kb + kslice);
    if (kb >= ke) return;
    mm2_tile<MB, NB, WM_, WN_, STAGES, KS>(Ap, R2, W, N, K, kb, ke, (int)tr * S::BR, (int)tn * S::BN, lds,
                                           SinkAtomic{acc, N});
}

// Work item of this block when the item count n is in device memory (written
// by an earlier kernel; grid = 8 ceil(max / 8) for an upper bound max): XCD x
// takes items [x per, (x + 1) per) with per = ceil(n / 8), as mm_tile_index
// does for a count known at launch; the other blocks get -1.
__device__ inline int mm_dyn_tile_index(const int* __restrict__ nwork) {
    const int n = __builtin_amdgcn_readfirstlane(*nwork);
    const int b = blockIdx.x, per = (n + 7) >> 3;
    const int t = (b & 7) * per + (b >> 3);
    return (b >> 3) < per && t < n ? t : -1;
}

// Grouped products (MoE experts): work item t = (expert e, token tile m0,
// weight tile n0) of the work table; expert e's rows are the byte-plane rows
// [2 offsets[e], 2 offsets[e+1]) of Ap and its weights W + e * w_stride
// [N x K].  The epilogue receives (e, n, row, sum) with row the activation
// row in Ap's token order (SinkGrouped).  The item count is read from
// *nwork on the device (the work table is built there); the grid covers
// maxwork items.  K % KS == 0.
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class EpiG>
__global__ __launch_bounds__(WM_ * WN_ * 64, (Mm2Dims<MB, NB, WM_, WN_, STAGES, KS>::kMinWaves)) void mm2_grouped_kernel(const int8_t* __restrict__ Ap,
                                                                     const int8_t* __restrict__ W, size_t w_stride,
                                                                     int N, int K, const int* __restrict__ offsets,
                                                                     const MmWork* __restrict__ work,
                                                                     const int* __restrict__ nwork, EpiG epi) {
    extern __shared__ __align__(16) int8_t lds[];
    const int t = mm_dyn_tile_index(nwork);
    if (t < 0) return;
    const MmWork wk = work[t];
    const int row0 = offsets[wk.e];
    const int Me = offsets[wk.e + 1] - row0;
    mm2_tile<MB, NB, WM_, WN_, STAGES, KS>(Ap + (size_t)2 * row0 * K, 2 * Me, W + (size_t)wk.e * w_stride, N, K, 0, K,
                                           2 * wk.m0, wk.n0, lds, SinkGrouped<EpiG>{epi, wk.e, row0});
}

// mm2_grouped_kernel with the staged epilogue (mm2_staged_tile): the sums of
// expert e reduce by EpiG::stage, and EpiG::emit takes the
// staged values with the activation row in Ap's token order.
template <class EpiG>
struct SinkGroupedStaged {
    const EpiG& epi;
    int e, row0;
    using Col = typename EpiG::Col;
    __device__ inline Col col(int n) const { return epi.col(e, n); }
    __device__ inline int16_t stage(const Col& c, int32_t u, uint32_t r) const { return epi.stage(c, u, r); }
    __device__ inline auto op(int n) const { return epi.op(e, n); }
    template <class Op>
    __device__ inline int16_t stage64(const Op& o, int n, int64_t v) const { return epi.stage64(o, n, v); }
    __device__ inline const int16_t* silu_table() const { return epi.silu; }
    __device__ inline uint32_t silu_table_len() const { return epi.silu_len; }
    __device__ inline void emit(int m, int i0, const uint4& a, const uint4& b, const int16_t* lut) const {
        epi.emit(e, row0 + m, i0, a, b, lut);
    }
};

template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class EpiG>
__global__ __launch_bounds__(WM_ * WN_ * 64, (Mm2Dims<MB, NB, WM_, WN_, STAGES, KS>::kMinWaves)) void mm2_grouped_staged_kernel(
    const int8_t* __restrict__ Ap, const int8_t* __restrict__ W, size_t w_stride, int N, int K,
    const int* __restrict__ offsets, const MmWork* __restrict__ work, const int* __restrict__ nwork, EpiG epi) {
    extern __shared__ __align__(16) int8_t lds[];
    const int t = mm_dyn_tile_index(nwork);
    if (t < 0) return;
    const MmWork wk = work[t];
    const int row0 = offsets[wk.e];
    mm2_staged_tile<MB, NB, WM_, WN_, STAGES, KS>(Ap + (size_t)row0 * 2 * K, 2 * (offsets[wk.e + 1] - row0),
                                                  W + (size_t)wk.e * w_stride, N, K, 2 * wk.m0, wk.n0, lds,
                                                  SinkGroupedStaged<EpiG>{epi, wk.e, row0});
}

template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class EpiG>
hipError_t mm2_grouped_staged_launch(const int8_t* Ap, const int8_t* W, size_t w_stride, int N, int K,
                                     const int* offsets, const MmWork* work, const int* nwork, int maxwork,
                                     const EpiG& epi, hipStream_t st) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    if (K % KS != 0 || N % 16 != 0) return hipErrorInvalidValue;
    if (maxwork <= 0) return hipSuccess;
    auto kern = mm2_grouped_staged_kernel<MB, NB, WM_, WN_, STAGES, KS, EpiG>;
    if (S::kLds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
        if (e != hipSuccess) return e;
    }
    kern<<<8 * ((maxwork + 7) / 8), S::kThreads, S::kLds, st>>>(Ap, W, w_stride, N, K, offsets, work, nwork, epi);
    return hipGetLastError();
}

// Token rows and weight rows of one grouped work item (for the work table).
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS>
struct Mm2GroupedShape {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    static constexpr int kTokens = S::BR / 2;
    static constexpr int kRows = S::BN;
};

template <int MB, int NB, int WM_, int WN_, int STAGES, int KS, class EpiG>
hipError_t mm2_grouped_launch(const int8_t* Ap, const int8_t* W, size_t w_stride, int N, int K, const int* offsets,
                              const MmWork* work, const int* nwork, int maxwork, const EpiG& epi, hipStream_t st) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    if (K % KS != 0) return hipErrorInvalidValue;
    if (maxwork <= 0) return hipSuccess;
    auto kern = mm2_grouped_kernel<MB, NB, WM_, WN_, STAGES, KS, EpiG>;
    if (S::kLds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
        if (e != hipSuccess) return e;
    }
    kern<<<8 * ((maxwork + 7) / 8), S::kThreads, S::kLds, st>>>(Ap, W, w_stride, N, K, offsets, work, nwork, epi);
    return hipGetLastError();
}

// K % KS == 0.
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS = 64, class Epi>
hipError_t mm2_launch(const int8_t* Ap, int M, const int8_t* W, int N, int K, const Epi& epi, hipStream_t st,
                      int group = 0) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    const int R2 = 2 * M;
    const int tiles_r = (R2 + S::BR - 1) / S::BR, tiles_n = (N + S::BN - 1) / S::BN;
    const TileOrder ord = TileOrder::of(tiles_r, tiles_n, group);
    const int ntiles = tiles_r * tiles_n;
    auto kern = mm2_kernel<MB, NB, WM_, WN_, STAGES, KS, Epi>;
    if (S::kLds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
        if (e != hipSuccess) return e;
    }
    kern<<<8 * ((ntiles + 7) / 8), S::kThreads, S::kLds, st>>>(Ap, R2, W, N, K, ord, ntiles, epi);
    return hipGetLastError();
}

// Weights stream once per row tile; K split across blocks when there are
// fewer tiles than `fill` (slices of at least 512 bytes), partial sums
// through the i64 accumulator.  A split product ends with fin(acc, st) (the
// finish kernel that applies the epilogue and clears acc) and sets *split;
// otherwise the tiles apply epi themselves.  K % KS == 0.
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS = 64, class Epi, class Fin>
hipError_t mm2_launch_splitk_fin(const int8_t* Ap, int M, const int8_t* W, int N, int K, const Epi& epi,
                                 const MmCtx* mm, int fill, hipStream_t st, const Fin& fin, bool* split) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    const Mm2SplitPlan p = mm2_split_plan<MB, NB, WM_, WN_, STAGES, KS>(M, N, K, mm->cus, mm->acc_elems, fill);
    *split = p.split;
    if (!p.split) return mm2_launch<MB, NB, WM_, WN_, STAGES, KS>(Ap, M, W, N, K, epi, st);
    auto kern = mm2_splitk_kernel<MB, NB, WM_, WN_, STAGES, KS>;
    if (S::kLds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
        if (e != hipSuccess) return e;
    }
    kern<<<p.grid, S::kThreads, S::kLds, st>>>(Ap, 2 * M, W, N, K, Divider::of((uint32_t)p.tiles_r),
                                               Divider::of((uint32_t)p.ntiles), p.nitems, p.kslice, mm->acc);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return fin(mm->acc, st);
}

template <int MB, int NB, int WM_, int WN_, int STAGES, int KS = 64, class Epi>
hipError_t mm2_launch_splitk(const int8_t* Ap, int M, const int8_t* W, int N, int K, const Epi& epi, const MmCtx* mm,
                             int fill, hipStream_t st) {
    bool split = false;
    auto fin = [&](unsigned long long* acc, hipStream_t s) {
        const int colb = (N + 255) / 256;
        const int rows = std::max(1, std::min(M, (mm->cus * 8 + colb - 1) / colb));
        mm_splitk_finish_kernel<Epi><<<dim3(colb, rows), 256, 0, s>>>(acc, M, N, epi);
        return hipGetLastError();
    };
    return mm2_launch_splitk_fin<MB, NB, WM_, WN_, STAGES, KS>(Ap, M, W, N, K, epi, mm, fill, st, fin, &split);
}

// Block tiles of a launch shape (for the dispatch's tile count).
template <int MB, int NB, int WM_, int WN_, int STAGES, int KS = 64>
inline int mm2_tiles(int M, int N) {
    using S = Mm2<MB, NB, WM_, WN_, STAGES, KS>;
    return ((2 * M + S::BR - 1) / S::BR) * ((N + S::BN - 1) / S::BN);
}


inline hipError_t split_planes(const int16_t* x, int M, int ldx, int K, int8_t* Ap, hipStream_t st) {
    split_planes_kernel<><<<dim3((K / 8 + 255) / 256, M), 256, 0, st>>>(x, M, ldx, K, Ap);
    return hipGetLastError();
}

}  // namespace myl
