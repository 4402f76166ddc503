// gemm_rows.h -- products of 2 to 32 activation rows with row-major weights:
// the weights stream once, at the rate of a plain read.
//
// y[m][n] = sum_k W[n][k] * x[m][k] exactly, int8 or int16 weights.  x is split
// into the byte planes of gemm_mfma2.h while it is loaded (plane row 2m =
// hi(x_m), 2m + 1 = lo'(x_m)), int16 weights into w = 256 wh + wl' + 128 while
// they leave LDS:
//   int8:   256 hi.w + lo'.w + 128 sum(w)
//   int16:  65536 hi.wh + 256 (hi.wl' + lo'.wh) + lo'.wl' + 128 (sum(x) + sum(w)) - 16384 K
// with the plane products on v_mfma_i32_16x16x64_i8 (plane sums of at most
// 2^16 K values: 32 bits) and the row sums from v_dot4 / v_dot2.
//
// What bounds it is the weight stream (N K bytes a weight byte), so the
// kernel is built around its loads.  One block of 8 waves per CU takes a K
// slice and a range of 16-row groups.  A wave owns U columns of 128 bytes of the
// slice, keeps their A' fragments in registers for the whole launch, and
// streams the units (row group, column): 16 rows x 128 bytes, two direct
// global-to-LDS loads of whole cache lines.  Each wave has its own ring of
// kRowsRing units in LDS, so no barrier orders the stream: 128 KiB per CU are in
// flight while the oldest unit multiplies.  Plane sums of the waves add up in
// LDS (exact in any order); every G row groups the block applies the output
// policy, two buffers alternating, so one barrier per G groups suffices and
// the stream's loads stay in flight across it.
#pragma once

#include "bufload.h"
#include "gemm_mfma.h"
#include "internal.h"
#include "mm_plan.h"
#include "wave.h"

namespace myl {

// LDS reads and writes done, then the block barrier (a fence would also wait
// for every load in flight).
__device__ inline void rows_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// LDS adds and writes beside loads to LDS in flight.  The compiler would put a
// wait for every such load before each of them (they might meet in LDS); here
// they never do: the loads fill the waves' rings only.  They return nothing,
// and rows_barrier waits for them.
__device__ inline uint32_t rows_lds_addr(const void* p) { return (uint32_t)(uintptr_t)(const buf_lds_void*)p; }
__device__ inline void rows_add32(uint32_t a, int32_t v) { asm volatile("ds_add_u32 %0, %1" ::"v"(a), "v"(v) : "memory"); }
__device__ inline void rows_add64(uint32_t a, int64_t v) { asm volatile("ds_add_u64 %0, %1" ::"v"(a), "v"(v) : "memory"); }
__device__ inline void rows_set32(uint32_t a, int32_t v) { asm volatile("ds_write_b32 %0, %1" ::"v"(a), "v"(v) : "memory"); }
__device__ inline void rows_set64(uint32_t a, uint64_t v) { asm volatile("ds_write_b64 %0, %1" ::"v"(a), "v"(v) : "memory"); }

// Activations: 16 values at k as raw int16, and as the bytes of a plane row.
struct RowsSrcX {
    const int16_t* x;  // [M x K], 16-byte aligned rows
    int ldx;
    struct Raw { uint4 a, b; };
    __device__ inline __amdgpu_buffer_rsrc_t rsrc(int M, int K) const {
        return weight_rsrc(x, ((uint32_t)(M - 1) * (uint32_t)ldx + (uint32_t)K) * 2u);
    }
    // zeros when !ok
    __device__ inline Raw load(const __amdgpu_buffer_rsrc_t& r, int m, int k, bool ok) const {
        const uint32_t o = ok ? ((uint32_t)m * (uint32_t)ldx + (uint32_t)k) * 2u : 0x7FFFFFC0u;
        return Raw{cload16(r, o), cload16(r, o + 16u)};
    }
    // the high bytes (lo false) or the low bytes - 128; zeros stay zeros when !ok
    __device__ inline static v4i32_t plane(const Raw& v, bool lo, bool ok) {
        const uint32_t sel = lo ? 0x06040200u : 0x07050301u, flip = lo && ok ? 0x80808080u : 0u;
        return v4i32_t{
            (int)(__builtin_amdgcn_perm(v.a.y, v.a.x, sel) ^ flip), (int)(__builtin_amdgcn_perm(v.a.w, v.a.z, sel) ^ flip),
            (int)(__builtin_amdgcn_perm(v.b.y, v.b.x, sel) ^ flip), (int)(__builtin_amdgcn_perm(v.b.w, v.b.z, sel) ^ flip)};
    }
};

// The same from byte planes [2M x K] (gemm_mfma2.h).
struct RowsSrcPlanes {
    const int8_t* Ap;
    int K;
    struct Raw { uint4 h, l; };
    __device__ inline __amdgpu_buffer_rsrc_t rsrc(int M, int) const { return weight_rsrc(Ap, 2u * (uint32_t)M * (uint32_t)K); }
    __device__ inline Raw load(const __amdgpu_buffer_rsrc_t& r, int m, int k, bool ok) const {
        const uint32_t o = 2u * (uint32_t)m * (uint32_t)K + (uint32_t)k;
        return Raw{cload16(r, ok ? o : 0x7FFFFFC0u), cload16(r, ok ? o + (uint32_t)K : 0x7FFFFFC0u)};
    }
    __device__ inline static v4i32_t plane(const Raw& v, bool lo, bool) {
        return lo ? v4i32_t{(int)v.l.x, (int)v.l.y, (int)v.l.z, (int)v.l.w} : v4i32_t{(int)v.h.x, (int)v.h.y, (int)v.h.z, (int)v.h.w};
    }
};

// Output policies.  ops(n), the operands of column n (at most 8 bytes), are
// fetched for all the block's columns before the stream and wait in LDS: loads
// retire in order, so one issued during the stream would wait for the whole
// ring.  put takes one exact sum.
template <class Epi>
struct RowsOutEpi {
    Epi e;
    using Ops = typename Epi::Ops;
    using Col = typename Epi::Col;
    __device__ inline Ops ops(int n) const { return e.ops(n); }
    __device__ inline Col col(const Ops& o) const { return e.col_of(o); }
    __device__ inline void put(const Col& c, const Ops& o, int n, int m, int32_t hi, int32_t low) const {
        if (c.fast) e.put(e.idx(n, m), 0, hi + (low >> 8), (uint32_t)low & 255u, c, e.elt(e.idx(n, m), 0));
        else e.one_ops(n, m, 256 * (int64_t)hi + (int64_t)low, o);
    }
};
// Products whose columns pair up (2i, 2i + 1 -> element i of an output row):
// each sum reduces to an int16, the odd column's goes to the even one's lane.
template <class Epi>
struct RowsOutPair {
    Epi e;
    struct Ops { typename Epi::Op o; };
    using Col = typename Epi::Col;
    __device__ inline Ops ops(int n) const { return Ops{e.op(n)}; }
    __device__ inline Col col(const Ops&) const { return Col{}; }
    __device__ inline void put(const Col&, const Ops& o, int n, int m, int32_t hi, int32_t low) const {
        const int32_t v = e.stage_with(o.o, n, 256 * (int64_t)hi + (int64_t)low);
        const int32_t up = dpp_mov<dpp::kXor1>(v);
        if ((n & 1) == 0) e.emit_one(m, n >> 1, (int16_t)v, (int16_t)up);
    }
};
struct RowsNoCol {};
// K slices: partial sums into acc [M x N] (zero-kept; the finish clears it).
struct RowsOutAcc {
    unsigned long long* acc;
    int ldn;
    using Ops = RowsNoCol;
    using Col = RowsNoCol;
    __device__ inline Ops ops(int) const { return Ops{}; }
    __device__ inline Col col(const Ops&) const { return Col{}; }
    __device__ inline void put(const Col&, const Ops&, int n, int m, int32_t hi, int32_t low) const {
        atomicAdd(acc + (size_t)m * ldn + n, (unsigned long long)(256 * (int64_t)hi + (int64_t)low));
    }
};
// int16 weights: the 64-bit sum.
template <class Epi>
struct RowsOutEpi64 {
    Epi e;
    using Ops = typename Epi::Ops;
    using Col = RowsNoCol;
    __device__ inline Ops ops(int n) const { return e.ops(n); }
    __device__ inline Col col(const Ops&) const { return Col{}; }
    __device__ inline void put64(const Ops& o, int n, int m, int64_t v) const { e.one_ops(n, m, v, o); }
};

// WB: bytes per weight; RT: tiles of 16 plane rows (8 token rows); U: columns
// of 128 weight bytes per wave; csl: columns per K slice; C: columns of a row.
template <int WB, int RT, int U, class Src, class Out>
__global__ __launch_bounds__(kRowsWaves * 64, 2) void rows_mm_kernel(Src src, int M, const void* __restrict__ W, int N, int K,
                                                                    int C, int csl, Divider P, Out out) {
    using D = RowsDims<RT>;
    constexpr int KT = 2 / WB;           // 64-K tiles per column
    constexpr int KC = 128 / WB;         // K per column
    constexpr int G = D::G;
    // Plane rows of a tile: with one tile, rows 2m, 2m + 1 are hi, lo' of token m
    // (8 tokens); with more, tile 2j holds hi and tile 2j + 1 lo' of tokens 16j ..
    // 16j + 15, so a lane's activations are loaded once for both.
    constexpr int RJ = (RT + 1) / 2;
    extern __shared__ __align__(16) int8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int8_t* ring = lds + wave * (kRowsRing * kRowsUnit);
    int32_t* red = reinterpret_cast<int32_t*>(lds + kRowsWaves * kRowsRing * kRowsUnit);  // [2][G][RT * 256]
    int32_t* rsl = red + 2 * G * RT * 256;                                                // [3][G * 16]
    int32_t* xsl = rsl + 3 * G * 16;                                                      // [RT * 16] (int16 weights)
    uint32_t s, p, g0u, g1u, rem;
    P.divmod(blockIdx.x, s, p);
    const uint32_t NG = (uint32_t)(N + 15) >> 4;
    P.divmod(p * NG, g0u, rem);  // p NG < 2^32: at most 2^10 parts, NG < 2^22
    P.divmod((p + 1) * NG, g1u, rem);
    const int g0 = (int)g0u, ngb = (int)(g1u - g0u);
    const int cb = (int)s * csl + wave * U;                                  // the wave's first column
    const int kn = max(0, min(U, min(C, ((int)s + 1) * csl) - cb));          // columns it owns
    const uint32_t rowb = (uint32_t)K * WB;
    // The columns' operands and the activations first: loads retire in order.
    uint64_t* ops_l = reinterpret_cast<uint64_t*>(xsl + RT * 16);  // [16 ngb]
    static_assert(sizeof(typename Out::Ops) <= kRowsOpsBytes && kRowsOpsBytes == 8, "operands of a column");
    auto ops_word = [&](int c) {
        const typename Out::Ops o = out.ops(min(16 * g0 + c, N - 1));
        uint64_t v = 0;
        __builtin_memcpy(&v, &o, sizeof(o));
        return v;
    };
    for (int i = threadIdx.x; i < 2 * G * RT * 256 + 3 * G * 16 + RT * 16; i += kRowsWaves * 64) red[i] = 0;
#pragma unroll 1
    for (int c = (int)threadIdx.x + kRowsWaves * 64; c < 16 * ngb; c += kRowsWaves * 64) ops_l[c] = ops_word(c);
    const uint64_t ops0 = ops_word((int)threadIdx.x);
    const __amdgpu_buffer_rsrc_t xr = src.rsrc(M, K);
    typename Src::Raw araw[U][KT][RJ];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int j = 0; j < RJ; ++j)
                araw[u][t][j] = src.load(xr, min(RT == 1 ? (lane & 15) >> 1 : 16 * j + (lane & 15), M - 1),
                                         (cb + u) * KC + 64 * t + 16 * (lane >> 4), u < kn && (cb + u) * KC + 64 * t < K);
    __builtin_amdgcn_sched_barrier(0);
    // The block's rows through a buffer descriptor, one offset per lane
    // (rows_lane_off, rows_unit_off): the fragment reads of 16 rows then cover all
    // 64 banks once.  Units past the block's rows or the wave's columns take an
    // offset past the descriptor, which reads no memory; rows past N and the
    // bytes past K of a row's last column meet discarded outputs and zero
    // fragments.
    const int rows_b = min(16 * ngb, N - 16 * g0);
    const __amdgpu_buffer_rsrc_t wr =
        weight_rsrc(reinterpret_cast<const int8_t*>(W) + (size_t)g0 * 16 * rowb, (uint32_t)max(rows_b, 0) * rowb);
    uint32_t voff[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) voff[j] = rows_lane_off(j, lane, rowb, cb);
    auto issue = [&](int g, int u, int slot) {
        const bool ok = g < ngb && u < kn;
        const uint32_t uo = rows_unit_off(g, u, rowb);
#pragma unroll
        for (int j = 0; j < 2; ++j)
            load_lds16<kRowsCpol>(wr, (buf_lds_void*)(ring + slot * kRowsUnit + j * 1024), ok ? voff[j] + uo : 0x7FFFFFF0u);
    };
#pragma unroll
    for (int d = 0; d < kRowsRing; ++d) issue(d / U, d % U, d);
    __builtin_amdgcn_sched_barrier(0);
    if ((int)threadIdx.x < 16 * ngb) rows_set64(rows_lds_addr(ops_l + threadIdx.x), ops0);
    // A' fragments (token rows past the matrix repeat its last row, their
    // outputs are discarded; tiles past K or past the wave's columns are zero)
    v4i32_t a[U][KT][RT];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int i = 0; i < RT; ++i)
                a[u][t][i] = Src::plane(araw[u][t][i >> 1], RT == 1 ? lane & 1 : i & 1, u < kn && (cb + u) * KC + 64 * t < K);
    rows_barrier();
    if (WB == 2 && kn > 0) {  // sum(x) by plane row: a product with ones, every column the same
        const v4i32_t ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            v4i32_t xs = {0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int t = 0; t < KT; ++t) xs = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u][t][i], ones, xs, 0, 0, 0);
            asm volatile("s_nop 15" : "+v"(xs));  // as below
            if ((lane & 15) == 0)
#pragma unroll
                for (int r = 0; r < 4; ++r) rows_add32(rows_lds_addr(xsl + 16 * i + 4 * (lane >> 4) + r), xs[r]);
        }
    }
    const int frow = lane & 15, fq = lane >> 4;
    int foff[2];  // the lane's two 16-byte reads of a unit
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int chunk = WB == 1 ? 4 * t + fq : 2 * fq + t;
        foff[t] = frow * 128 + ((chunk ^ ((frow >> 1) & 7)) << 4);
    }
    // the epilogue's fixed column of this thread
    const int ec = (int)threadIdx.x & (16 * G - 1), em0 = (int)threadIdx.x / (16 * G);
    constexpr int kEm = kRowsWaves * 64 / (16 * G);
    int slot = 0;
    for (int gw = 0; gw < ngb; gw += G) {
        const int win = gw / G;
        int32_t* rw = red + (win & 1) * (G * RT * 256);
        int32_t* rsw = rsl + (win % 3) * (G * 16);
        const int n = 16 * (g0 + gw) + ec;
        if (kn > 0) {
            for (int gg = 0; gg < G && gw + gg < ngb; ++gg) {
                const int g = gw + gg;
                v4i32_t acc[WB][RT];
#pragma unroll
                for (int b = 0; b < WB; ++b)
#pragma unroll
                    for (int i = 0; i < RT; ++i) acc[b][i] = v4i32_t{0, 0, 0, 0};
                int32_t rs = 0;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    // loads retire in order: the oldest unit has landed once
                    // only the younger ones' are outstanding; its bytes are in
                    // registers before the next unit may overwrite them
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (kRowsRing - 1)) : "memory");
                    const int8_t* up = ring + slot * kRowsUnit;
                    v4i32_t w0 = *reinterpret_cast<const v4i32_t*>(up + foff[0]);
                    v4i32_t w1 = *reinterpret_cast<const v4i32_t*>(up + foff[1]);
                    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w0), "+v"(w1)::"memory");
                    issue(g + (u + kRowsRing) / U, (u + kRowsRing) % U, slot);
                    slot = (slot + 1) & (kRowsRing - 1);
                    if (WB == 1) {
                        // whole tiles of K are valid or not
                        const uint32_t o0 = u < kn ? 0x01010101u : 0u;
                        const uint32_t o1 = u < kn && (cb + u) * KC + 64 < K ? 0x01010101u : 0u;
#pragma unroll
                        for (int i = 0; i < RT; ++i) {
                            acc[0][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u][0][i], w0, acc[0][i], 0, 0, 0);
                            acc[0][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u][KT - 1][i], w1, acc[0][i], 0, 0, 0);
                        }
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            rs = sdot4((uint32_t)w0[q], o0, rs);
                            rs = sdot4((uint32_t)w1[q], o1, rs);
                        }
                    } else {
                        v4i32_t wh, wl;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const uint32_t e0 = (uint32_t)(q < 2 ? w0 : w1)[2 * (q & 1)];
                            const uint32_t e1 = (uint32_t)(q < 2 ? w0 : w1)[2 * (q & 1) + 1];
                            wh[q] = (int)__builtin_amdgcn_perm(e1, e0, 0x07050301u);
                            wl[q] = (int)(__builtin_amdgcn_perm(e1, e0, 0x06040200u) ^ 0x80808080u);
                        }
#pragma unroll
                        for (int i = 0; i < RT; ++i) {
                            acc[0][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u][0][i], wh, acc[0][i], 0, 0, 0);
                            acc[WB - 1][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u][0][i], wl, acc[WB - 1][i], 0, 0, 0);
                        }
                        // sum(w) = 256 sum(wh) + sum(wl') + 128 K: the first two here
                        const uint32_t o = u < kn ? 0x01010101u : 0u;
                        int32_t sh = 0;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            sh = sdot4((uint32_t)wh[q], o, sh);
                            rs = sdot4((uint32_t)wl[q], o, rs);
                        }
                        rs += sh * 256;
                    }
                }
                // The compiler does not count the wait states between a matrix
                // (or dot) result and a use inside an asm block: 8-pass
                // products need 11 before LDS may read them.
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    if (WB == 1) asm volatile("s_nop 15" : "+v"(acc[0][i]));
                    else asm volatile("s_nop 15" : "+v"(acc[0][i]), "+v"(acc[WB - 1][i]));
                }
                asm volatile("s_nop 15" : "+v"(rs));
                // accumulator row 4 (lane / 16) + r of tile i, column lane % 16
                if (WB == 1) {
                    const uint32_t rg = rows_lds_addr(rw + gg * (RT * 256) + lane);
#pragma unroll
                    for (int i = 0; i < RT; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) rows_add32(rg + (i * 256 + r * 64) * 4, acc[0][i][r]);
                } else {
                    const uint32_t rg = rows_lds_addr(reinterpret_cast<int64_t*>(rw) + gg * (RT * 128) + lane);
                    auto whole = [](int32_t hh, int32_t lh, int32_t hl, int32_t ll) {
                        return 65536 * (int64_t)hh + 256 * ((int64_t)lh + (int64_t)hl) + (int64_t)ll;
                    };
                    if (RT == 1) {
#pragma unroll
                        for (int r = 0; r < 4; r += 2)
                            rows_add64(rg + r * 32 * 8, whole(acc[0][0][r], acc[0][0][r + 1], acc[WB - 1][0][r], acc[WB - 1][0][r + 1]));
                    } else {
#pragma unroll
                        for (int j = 0; j < RT / 2; ++j)
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                rows_add64(rg + (j * 256 + r * 64) * 8,
                                           whole(acc[0][2 * j][r], acc[0][(2 * j + 1) % RT][r], acc[WB - 1][2 * j][r],
                                                 acc[WB - 1][(2 * j + 1) % RT][r]));
                    }
                }
                rows_add32(rows_lds_addr(rsw + gg * 16 + frow), rs);
            }
        }
        rows_barrier();
        // the reader of a sum clears it for the window after the next
        if (n < N && gw + (ec >> 4) < ngb) {
            const int c = ec & 15;
            const int32_t rs = rsw[ec];
            typename Out::Ops ops;
            const uint64_t opw = ops_l[16 * gw + ec];
            __builtin_memcpy(&ops, &opw, sizeof(ops));
            const typename Out::Col col = out.col(ops);
#pragma unroll 1
            for (int m = em0; m < M; m += kEm) {
                // row r of a tile at (r % 4) 64 + (r / 4) 16
                const int t = m & 15;
                if constexpr (WB == 1) {
                    const int32_t* q0 = rw + (ec >> 4) * (RT * 256) + c +
                                        (RT == 1 ? (m & 1) * 128 + (m >> 1) * 16 : (m >> 4) * 512 + (t & 3) * 64 + (t >> 2) * 16);
                    constexpr int dlo = RT == 1 ? 64 : 256;
                    const int32_t hi = q0[0], lo = q0[dlo];
                    rows_set32(rows_lds_addr(q0), 0);
                    rows_set32(rows_lds_addr(q0 + dlo), 0);
                    out.put(col, ops, n, m, hi, lo + (int32_t)((uint32_t)rs << 7));
                } else {
                    const int64_t* q0 = reinterpret_cast<const int64_t*>(rw) + (ec >> 4) * (RT * 128) + c +
                                        (RT == 1 ? (m & 1) * 64 + (m >> 1) * 16 : (m >> 4) * 256 + (t & 3) * 64 + (t >> 2) * 16);
                    const int64_t v = *q0;
                    rows_set64(rows_lds_addr(q0), 0);
                    // the 128 K of sum(w) and of sum(x) and the -16384 K add up to 16384 K
                    const int32_t* xp = xsl + (RT == 1 ? 2 * m : (m >> 4) * 32 + t);
                    const int64_t xs = 256 * (int64_t)xp[0] + (int64_t)xp[RT == 1 ? 1 : 16];
                    out.put64(ops, n, m, v + 128 * (xs + (int64_t)rs) + 16384 * (int64_t)K);
                }
            }
        }
        // every reader of the previous window's row sums has passed this
        // window's barrier, and the next adds to them come after the next one
        if ((int)threadIdx.x < G * 16) rows_set32(rows_lds_addr(rsl + ((win + 2) % 3) * (G * 16) + threadIdx.x), 0);
    }
    // the ring's last loads (past the block's rows) have retired before its LDS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// ---- launches ---------------------------------------------------------------

// The activations' byte offsets fit the buffer descriptor.
inline bool rows_x_ok(int M, int ldx) { return (int64_t)M * ldx * 2 < 0x7FFFFF00ll; }

template <int WB, int RT, int U, class Src, class Out>
hipError_t rows_mm_launch(const RowsPlan& pl, const Src& src, int M, const void* W, int N, int K, const Out& out,
                          hipStream_t st) {
    const size_t lds = RowsDims<RT>::kLds + (size_t)16 * pl.ngb * kRowsOpsBytes;
    auto kern = rows_mm_kernel<WB, RT, U, Src, Out>;
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    kern<<<pl.S * pl.P, kRowsWaves * 64, lds, st>>>(src, M, W, N, K, pl.C, pl.csl, Divider::of((uint32_t)pl.P), out);
    return hipGetLastError();
}

template <int WB, class Src, class Out>
hipError_t rows_mm_run(const RowsPlan& pl, const Src& src, int M, const void* W, int N, int K, const Out& out,
                       hipStream_t st) {
    constexpr int U0 = WB == 1 ? 1 : 2, U1 = WB == 1 ? 2 : 4, U2 = WB == 1 ? 4 : 8;
#define MYL_ROWS_U(RTV)                                                                       \
    return pl.U <= U0   ? rows_mm_launch<WB, RTV, U0>(pl, src, M, W, N, K, out, st)           \
           : pl.U <= U1 ? rows_mm_launch<WB, RTV, U1>(pl, src, M, W, N, K, out, st)           \
                        : rows_mm_launch<WB, RTV, U2>(pl, src, M, W, N, K, out, st)
    switch (frag_rt(M)) {
    case 1: MYL_ROWS_U(1);
    case 2: MYL_ROWS_U(2);
    default: MYL_ROWS_U(4);
    }
#undef MYL_ROWS_U
}

// int8 weights: the whole sum per block, or K slices through mm's accumulator
// and the finish kernel.
template <class Src, class Epi>
hipError_t rows_mm_i8(const RowsPlan& pl, const Src& src, int M, const int8_t* W, int N, int K, const Epi& epi,
                      const MmCtx* mm, hipStream_t st) {
    if (pl.S == 1) return rows_mm_run<1>(pl, src, M, W, N, K, RowsOutEpi<Epi>{epi}, st);
    hipError_t e = rows_mm_run<1>(pl, src, M, W, N, K, RowsOutAcc{mm->acc, N}, st);
    if (e != hipSuccess) return e;
    const int colb = (N + 255) / 256;
    const int rows = std::max(1, std::min(M, (mm->cus * 8 + colb - 1) / colb));
    mm_splitk_finish_kernel<Epi><<<dim3(colb, rows), 256, 0, st>>>(mm->acc, M, N, epi);
    return hipGetLastError();
}

// int16 weights, whole sums only (pl.S == 1).
template <class Src, class Epi>
hipError_t rows_mm_i16(const RowsPlan& pl, const Src& src, int M, const int16_t* W, int N, int K, const Epi& epi,
                       hipStream_t st) {
    return rows_mm_run<2>(pl, src, M, W, N, K, RowsOutEpi64<Epi>{epi}, st);
}

}  // namespace myl
