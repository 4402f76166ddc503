// kernels.hip -- launchers for the GEMV and the op kernels of the integer
// forward path (gfx950).  Host-side shape checks live in abi.cpp; everything
// here assumes validated arguments.
#include "gemm_dispatch.h"
#include "../../include/myl_theta_v.h"
#include "ops.h"
#include "row_walk.h"
#include "wave.h"

namespace myl {

hipError_t linear_w8a16(const int16_t* x, int M, int ldx, const int8_t* W, int N, int K, const uint8_t* w_shifts,
                        uint8_t act_frac, uint8_t out_frac, const uint8_t* out_frac_pc, int16_t* out, int ldo,
                        hipStream_t st, const MmCtx* mm) {
    EpiShift e{w_shifts, out_frac_pc, act_frac, out_frac, out, ldo};
    return gemv_i8(x, M, ldx, W, N, K, e, st, mm);
}

hipError_t linear_w8a16_mult(const int16_t* x, int M, int ldx, const int8_t* W, int N, int K, const int32_t* mult,
                             const uint8_t* shift, int16_t* out, int ldo, hipStream_t st, const MmCtx* mm) {
    EpiMult e{mult, shift, out, ldo};
    return gemv_i8(x, M, ldx, W, N, K, e, st, mm);
}

hipError_t logits_w8(const int16_t* x, int M, int ldx, const int8_t* W, int N, int K, const uint8_t* row_shifts,
                     uint8_t norm_frac, uint8_t logit_frac, int32_t* out, int ldo, hipStream_t st, const MmCtx* mm) {
    EpiLogits e{row_shifts, norm_frac, logit_frac, out, ldo};
    return gemv_i8(x, M, ldx, W, N, K, e, st, mm);
}

hipError_t logits_w16(const int16_t* x, int M, int ldx, const int16_t* W, int N, int K, const uint8_t* row_shifts,
                      uint8_t norm_frac, uint8_t logit_frac, int32_t* out, int ldo, hipStream_t st, const MmCtx* mm) {
    EpiLogits e{row_shifts, norm_frac, logit_frac, out, ldo};
    return gemv_i16(x, M, ldx, W, N, K, e, st, mm);
}

hipError_t dot_raw_w8(const int16_t* x, int M, int ldx, const int8_t* W, int N, int K, int64_t* out, int ldo,
                      hipStream_t st, const MmCtx* mm) {
    EpiRaw e{out, ldo};
    return gemv_i8(x, M, ldx, W, N, K, e, st, mm);
}

// ---------------------------------------------------------------------------
// RMSNorm (rmsnorm.rs:61-161): one block per row.
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(kBlock) void rmsnorm_kernel(const int16_t* __restrict__ x, int ldx,
                                                        const uint8_t* __restrict__ xs, const int8_t* __restrict__ g,
                                                        const uint8_t* __restrict__ gs, int n, RmsParams p,
                                                        uint8_t out_frac, int16_t* __restrict__ out, int ldo) {
    __shared__ myl_i128 red128[kBlock];
    __shared__ int32_t red32[kBlock / 64];
    const int16_t* xr = x + (size_t)blockIdx.x * ldx;
    const RmsFactor f = rms_factor(xr, xs, n, p, red128, red32);
    int16_t* o = out + (size_t)blockIdx.x * ldo;
    for (int i = threadIdx.x; i < n; i += blockDim.x) o[i] = rms_out(xr[i], xs[i], g[i], gs[i], f, out_frac);
}

// Rows of up to kRmsThreads * kRmsPer elements: every element is loaded once,
// before the reductions, and stays in registers.
constexpr int kRmsThreads = 1024;
constexpr int kRmsPer = 4;
__global__ __launch_bounds__(kRmsThreads) void rmsnorm_fast_kernel(const int16_t* __restrict__ x, int ldx,
                                                                  const uint8_t* __restrict__ xs,
                                                                  const int8_t* __restrict__ g,
                                                                  const uint8_t* __restrict__ gs, int n, RmsParams p,
                                                                  uint8_t out_frac, int16_t* __restrict__ out, int ldo,
                                                                  int8_t* __restrict__ planes) {
    __shared__ myl_i128 red128[kRmsThreads / 64];
    __shared__ int32_t red32[kRmsThreads / 64];
    const int16_t* xr = x + (size_t)blockIdx.x * ldx;
    int16_t xv[kRmsPer];
    uint8_t sv[kRmsPer];
    int8_t gv[kRmsPer];
    uint8_t gsv[kRmsPer];
#pragma unroll
    for (int t = 0; t < kRmsPer; ++t) {
        const int i = threadIdx.x + t * kRmsThreads;
        const bool ok = i < n;
        xv[t] = ok ? xr[i] : (int16_t)0;
        sv[t] = ok ? xs[i] : (uint8_t)0;
        gv[t] = ok ? g[i] : (int8_t)0;
        gsv[t] = ok ? gs[i] : (uint8_t)0;
    }
    const RmsFactor f = rms_factor_regs<kRmsPer>(xv, sv, p, red128, red32);
    if (planes) {
        // byte planes of the output row: hi at row 2m, lo' at row 2m + 1
        int8_t* ph = planes + (size_t)(2 * blockIdx.x) * n;
#pragma unroll
        for (int t = 0; t < kRmsPer; ++t) {
            const int i = threadIdx.x + t * kRmsThreads;
            if (i < n) {
                const int32_t y = rms_out(xv[t], sv[t], gv[t], gsv[t], f, out_frac);
                ph[i] = (int8_t)(y >> 8);
                ph[n + i] = (int8_t)((y & 255) - 128);
            }
        }
        return;
    }
    int16_t* o = out + (size_t)blockIdx.x * ldo;
#pragma unroll
    for (int t = 0; t < kRmsPer; ++t) {
        const int i = threadIdx.x + t * kRmsThreads;
        if (i < n) o[i] = rms_out(xv[t], sv[t], gv[t], gsv[t], f, out_frac);
    }
}

// 256 threads per row, each thread owning PER chunks of 8
// consecutive elements loaded as one 16-byte (x) and 8-byte (shifts, gamma)
// vector each; rows of n % 8 == 0 elements, 16-byte aligned.  The sum of
// squares stays in 64 bits for elements at the largest shift (align 0) and
// takes the exact 128-bit path only for the others.
constexpr int kRowsThreads = 256;

__device__ inline uint8_t byte_of(const uint2& v, int q) {
    return (uint8_t)(((q < 4 ? v.x : v.y) >> (8 * (q & 3))) & 0xFFu);
}

template <int PER>
__global__ __launch_bounds__(kRowsThreads) void rmsnorm_rows_kernel(const int16_t* __restrict__ x, int ldx,
                                                                    const uint8_t* __restrict__ xs,
                                                                    const int8_t* __restrict__ g,
                                                                    const uint8_t* __restrict__ gs, int n,
                                                                    RmsParams p, uint8_t out_frac,
                                                                    int16_t* __restrict__ out, int ldo,
                                                                    int8_t* __restrict__ planes) {
    __shared__ myl_i128 red128[kRowsThreads / 64];
    __shared__ int32_t red32[kRowsThreads / 64];
    const int16_t* xr = x + (size_t)blockIdx.x * ldx;
    const int nc = n >> 3;
    uint4 xv[PER];
    uint2 sv[PER], gv[PER], gsv[PER];  // gamma and its shifts load with x
    int32_t mx = 0;
#pragma unroll
    for (int t = 0; t < PER; ++t) {
        const int c = threadIdx.x + t * kRowsThreads;
        xv[t] = make_uint4(0, 0, 0, 0);
        sv[t] = gv[t] = gsv[t] = make_uint2(0, 0);
        if (c < nc) {
            xv[t] = *reinterpret_cast<const uint4*>(xr + 8 * c);
            sv[t] = *reinterpret_cast<const uint2*>(xs + 8 * c);
            gv[t] = *reinterpret_cast<const uint2*>(g + 8 * c);
            gsv[t] = *reinterpret_cast<const uint2*>(gs + 8 * c);
        }
    }
#pragma unroll
    for (int t = 0; t < PER; ++t)
#pragma unroll
        for (int q = 0; q < 8; ++q) mx = max(mx, (int32_t)byte_of(sv[t], q));
    const uint8_t ref = (uint8_t)block_max_i32(mx, red32);
    uint64_t acc64 = 0;
    myl_i128 acc = 0;
#pragma unroll
    for (int t = 0; t < PER; ++t) {
        const uint32_t w[4] = {xv[t].x, xv[t].y, xv[t].z, xv[t].w};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int32_t xi = (int32_t)(int16_t)((w[q >> 1] >> (16 * (q & 1))) & 0xFFFFu);
            const uint32_t sq = (uint32_t)(xi * xi);   // <= 2^30
            const uint32_t align = 2u * (uint32_t)(uint8_t)(ref - byte_of(sv[t], q));
            if (align == 0) acc64 += sq;
            else acc = (myl_i128)((myl_u128)acc + (myl_u128)shl128((myl_i128)sq, align));
        }
    }
    // all lanes at the largest shift (the usual case): a 64-bit DPP sum
    // (each lane < 2^34, so the wave total < 2^40); else the 128-bit one
    if (__any(acc != 0)) acc = wave_sum_i128((myl_i128)((myl_u128)acc + (myl_u128)acc64));
    else acc = (myl_i128)wave_sum_u64(acc64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red128[threadIdx.x >> 6] = acc;
    __syncthreads();
    acc = 0;
#pragma unroll
    for (int i = 0; i < kRowsThreads / 64; ++i) acc = (myl_i128)((myl_u128)acc + (myl_u128)red128[i]);
    const RmsFactor f = rms_factor_of(acc, ref, p);
#pragma unroll
    for (int t = 0; t < PER; ++t) {
        const int c = threadIdx.x + t * kRowsThreads;
        if (c >= nc) continue;
        const uint32_t w[4] = {xv[t].x, xv[t].y, xv[t].z, xv[t].w};
        int32_t y[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            y[q] = rms_out((int16_t)((w[q >> 1] >> (16 * (q & 1))) & 0xFFFFu), byte_of(sv[t], q),
                           (int8_t)byte_of(gv[t], q), byte_of(gsv[t], q), f, out_frac);
        if (planes) {
            uint32_t h[2] = {0, 0}, l[2] = {0, 0};
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                h[q >> 2] |= ((uint32_t)(y[q] >> 8) & 0xFFu) << (8 * (q & 3));
                l[q >> 2] |= ((uint32_t)((y[q] & 255) - 128) & 0xFFu) << (8 * (q & 3));
            }
            int8_t* ph = planes + (size_t)(2 * blockIdx.x) * n + 8 * c;
            *reinterpret_cast<uint2*>(ph) = make_uint2(h[0], h[1]);
            *reinterpret_cast<uint2*>(ph + n) = make_uint2(l[0], l[1]);
        } else {
            uint32_t o[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                o[q] = ((uint32_t)y[2 * q] & 0xFFFFu) | ((uint32_t)y[2 * q + 1] << 16);
            *reinterpret_cast<uint4*>(out + (size_t)blockIdx.x * ldo + 8 * c) = make_uint4(o[0], o[1], o[2], o[3]);
        }
    }
}

// The row kernel's PER for n elements (0: not applicable).
inline int rms_rows_per(int n) {
    if (n % 8 != 0) return 0;
    const int nc = n / 8;
    return nc <= kRowsThreads ? 1 : nc <= 2 * kRowsThreads ? 2 : nc <= 4 * kRowsThreads ? 4 : 0;
}

// Row kernel launch when the layout allows it.
bool rmsnorm_rows(const int16_t* x, int M, int ldx, const uint8_t* xs, const int8_t* g, const uint8_t* gs, int n,
                  const RmsParams& p, uint8_t out_frac, int16_t* out, int ldo, int8_t* planes, hipStream_t st) {
    const int per = rms_rows_per(n);
    const bool aligned = ((uintptr_t)x % 16 == 0) && ldx % 8 == 0 && ((uintptr_t)xs % 8 == 0) &&
                         ((uintptr_t)g % 8 == 0) && ((uintptr_t)gs % 8 == 0) &&
                         (planes ? (uintptr_t)planes % 8 == 0 : ((uintptr_t)out % 16 == 0 && ldo % 8 == 0));
    if (M < 1 || per == 0 || !aligned) return false;
    if (per == 1)
        rmsnorm_rows_kernel<1><<<M, kRowsThreads, 0, st>>>(x, ldx, xs, g, gs, n, p, out_frac, out, ldo, planes);
    else if (per == 2)
        rmsnorm_rows_kernel<2><<<M, kRowsThreads, 0, st>>>(x, ldx, xs, g, gs, n, p, out_frac, out, ldo, planes);
    else
        rmsnorm_rows_kernel<4><<<M, kRowsThreads, 0, st>>>(x, ldx, xs, g, gs, n, p, out_frac, out, ldo, planes);
    return true;
}

hipError_t rmsnorm(const int16_t* x, int M, int ldx, const uint8_t* xs, const int8_t* g, const uint8_t* gs, int n,
                   const int16_t* lut, int lut_len, uint8_t lut_input_shift, uint8_t lut_output_frac,
                   int64_t inv_n_q20, uint8_t out_frac, int16_t* out, int ldo, hipStream_t st) {
    RmsParams p{lut, lut_len, lut_input_shift, lut_output_frac, inv_n_q20};
    if (rmsnorm_rows(x, M, ldx, xs, g, gs, n, p, out_frac, out, ldo, nullptr, st)) return hipGetLastError();
    if (n <= kRmsThreads * kRmsPer)
        rmsnorm_fast_kernel<<<M, kRmsThreads, 0, st>>>(x, ldx, xs, g, gs, n, p, out_frac, out, ldo, nullptr);
    else
        rmsnorm_kernel<<<M, kBlock, 0, st>>>(x, ldx, xs, g, gs, n, p, out_frac, out, ldo);
    return hipGetLastError();
}

bool rmsnorm_planes_ok(int n) { return n <= kRmsThreads * kRmsPer; }

hipError_t rmsnorm_planes(const int16_t* x, int M, int ldx, const uint8_t* xs, const int8_t* g, const uint8_t* gs,
                          int n, const int16_t* lut, int lut_len, uint8_t lut_input_shift, uint8_t lut_output_frac,
                          int64_t inv_n_q20, uint8_t out_frac, int8_t* planes, hipStream_t st) {
    if (!rmsnorm_planes_ok(n)) return hipErrorInvalidValue;
    RmsParams p{lut, lut_len, lut_input_shift, lut_output_frac, inv_n_q20};
    if (rmsnorm_rows(x, M, ldx, xs, g, gs, n, p, out_frac, nullptr, 0, planes, st)) return hipGetLastError();
    rmsnorm_fast_kernel<<<M, kRmsThreads, 0, st>>>(x, ldx, xs, g, gs, n, p, out_frac, nullptr, 0, planes);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Softmax (softmax.rs:24-64): one block per row.
// ---------------------------------------------------------------------------

__device__ inline void softmax_row(const int32_t* __restrict__ z, int n, const int16_t* __restrict__ lut,
                                   uint32_t lut_len, uint8_t lut_shift, uint8_t frac_bits, int32_t* __restrict__ out,
                                   int32_t* red32, uint32_t* redu) {
    const int32_t one = shl32(1, frac_bits);
    const int32_t lut_one = lut_len > 0 ? (int32_t)lut[0] : 1;
    int32_t mx = INT32_MIN;
    for (int i = threadIdx.x; i < n; i += blockDim.x) mx = max(mx, z[i]);
    const int32_t m = n > 0 ? block_max_i32(mx, red32) : 0;
    uint32_t s = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x)
        s += (uint32_t)exp_lookup(sat_sub32(m, z[i]), lut, lut_len, lut_shift, lut_one);
    const int32_t S = (int32_t)block_sum_u32(s, redu);
    if (S == 0) {
        // softmax.rs:42-48: uniform with the remainder on the lowest indices.
        // one / n without a divide: n * q <= one < n * (q + 1) by long division.
        uint32_t un = (uint32_t)n;
        uint32_t q = 0, r = 0;
        if (un) {
            uint64_t recip = recip32(un);
            uint32_t uone = one < 0 ? 0u - (uint32_t)one : (uint32_t)one;
            udivmod32(uone, un, recip, &q, &r);
        }
        int32_t base = one < 0 ? -(int32_t)q : (int32_t)q;
        int32_t rem = wsub32(one, wmul32(base, (int32_t)n));
        for (int i = threadIdx.x; i < n; i += blockDim.x)
            out[i] = base + (((uint64_t)i < (uint64_t)(int64_t)rem) ? 1 : 0);
        return;
    }
    const uint32_t us = S < 0 ? 0u - (uint32_t)S : (uint32_t)S;
    const uint64_t recip = recip32(us);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int32_t e = exp_lookup(sat_sub32(m, z[i]), lut, lut_len, lut_shift, lut_one);
        out[i] = softmax_div_round(wmul32(e, one), S, recip);
    }
}

__global__ __launch_bounds__(kBlock) void softmax_kernel(const int32_t* __restrict__ z, int n, int ldz,
                                                        const int16_t* __restrict__ lut, uint32_t lut_len,
                                                        uint8_t lut_shift, uint8_t frac_bits, int32_t* __restrict__ out,
                                                        int ldo) {
    __shared__ int32_t red32[kBlock / 64];
    __shared__ uint32_t redu[kBlock / 64];
    softmax_row(z + (size_t)blockIdx.x * ldz, n, lut, lut_len, lut_shift, frac_bits, out + (size_t)blockIdx.x * ldo,
                red32, redu);
}

hipError_t softmax(const int32_t* z, int M, int n, int ldz, const int16_t* lut, int lut_len, uint8_t lut_shift,
                   uint8_t frac_bits, int32_t* out, int ldo, hipStream_t st) {
    softmax_kernel<<<M, kBlock, 0, st>>>(z, n, ldz, lut, (uint32_t)lut_len, lut_shift, frac_bits, out, ldo);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Generic attention (attention.rs:42-90): one block per query row.
// scratch holds q_len x kv_len i32 scores followed by as many i32 probs.
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(kBlock) void attn_scores_kernel(const int16_t* __restrict__ q, const int16_t* __restrict__ k,
                                                            const uint8_t* __restrict__ mask, int kv_len, int hd,
                                                            int64_t score_mult, uint8_t score_shift,
                                                            int32_t* __restrict__ scores) {
    const int i = blockIdx.y;
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= kv_len) return;
    int32_t s;
    if (!mask || mask[(size_t)i * kv_len + j]) {
        const int16_t* qi = q + (size_t)i * hd;
        const int16_t* kj = k + (size_t)j * hd;
        uint64_t acc = 0;
        for (int d = 0; d < hd; ++d) acc += (uint64_t)((int64_t)qi[d] * (int64_t)kj[d]);
        s = (int32_t)rshift_round64(wmul64((int64_t)acc, score_mult), score_shift);
    } else {
        s = INT32_MIN;
    }
    scores[(size_t)i * kv_len + j] = s;
}

__global__ __launch_bounds__(kBlock) void attn_pv_kernel(const int32_t* __restrict__ probs, const int16_t* __restrict__ v,
                                                        int kv_len, int hd, uint8_t prob_frac,
                                                        int16_t* __restrict__ out) {
    const int i = blockIdx.y;
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= hd) return;
    const int32_t* p = probs + (size_t)i * kv_len;
    uint64_t acc = 0;
    for (int j = 0; j < kv_len; ++j) acc += (uint64_t)((int64_t)p[j] * (int64_t)v[(size_t)j * hd + d]);
    out[(size_t)i * hd + d] = clamp_i16_i64(rshift_round64((int64_t)acc, prob_frac));
}

hipError_t attention_generic(const int16_t* q, const int16_t* k, const int16_t* v, const uint8_t* mask, int q_len,
                             int kv_len, int hd, int64_t score_mult, uint8_t score_shift, const int16_t* lut,
                             int lut_len, uint8_t lut_shift, uint8_t prob_frac, int32_t* scratch, int16_t* out,
                             hipStream_t st) {
    int32_t* scores = scratch;
    int32_t* probs = scratch + (size_t)q_len * kv_len;
    attn_scores_kernel<<<dim3((kv_len + kBlock - 1) / kBlock, q_len), kBlock, 0, st>>>(q, k, mask, kv_len, hd,
                                                                                         score_mult, score_shift, scores);
    hipError_t rc = hipGetLastError();
    if (rc != hipSuccess) return rc;
    rc = softmax(scores, q_len, kv_len, kv_len, lut, lut_len, lut_shift, prob_frac, probs, kv_len, st);
    if (rc != hipSuccess) return rc;
    attn_pv_kernel<<<dim3((hd + kBlock - 1) / kBlock, q_len), kBlock, 0, st>>>(probs, v, kv_len, hd, prob_frac, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// RoPE (rope.rs:17-59): one thread per (row, pair); rows[] holds pos % n_pos.
// ---------------------------------------------------------------------------

__global__ void rope_kernel(int16_t* __restrict__ q, int16_t* __restrict__ k, int n, int hd,
                            const int16_t* __restrict__ cos_lut, const int16_t* __restrict__ sin_lut,
                            const int32_t* __restrict__ rows, uint8_t frac_bits) {
    const int half = hd >> 1;
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = blockIdx.y;
    if (j >= half || i >= n) return;
    const int32_t c = cos_lut[(size_t)rows[i] * half + j];
    const int32_t s = sin_lut[(size_t)rows[i] * half + j];
    for (int t = 0; t < 2; ++t) {
        int16_t* vec = (t == 0 ? q : k) + (size_t)i * hd;
        const int32_t x0 = vec[j], x1 = vec[j + half];
        vec[j] = clamp_i16(rshift_round32(wsub32(wmul32(x0, c), wmul32(x1, s)), frac_bits));
        vec[j + half] = clamp_i16(rshift_round32(wadd32(wmul32(x1, c), wmul32(x0, s)), frac_bits));
        if ((hd & 1) && j == 0) vec[hd - 1] = 0;
    }
}

hipError_t rope(int16_t* q, int16_t* k, int n, int hd, const int16_t* cos_lut, const int16_t* sin_lut,
                const int32_t* rows, uint8_t frac_bits, hipStream_t st) {
    const int half = hd >> 1;
    rope_kernel<<<dim3((half + 127) / 128, n), 128, 0, st>>>(q, k, n, hd, cos_lut, sin_lut, rows, frac_bits);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Bias (linear.rs:132-145), SiLU gating (mlp.rs:55-65), argmax (sampling.rs:8-18)
// ---------------------------------------------------------------------------

__global__ void bias_kernel(int16_t* __restrict__ out, const int16_t* __restrict__ b, const uint8_t* __restrict__ bs,
                            int n, uint8_t out_frac) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t br = rescale32((int32_t)b[i], bs[i], out_frac);
    out[i] = clamp_i16_i64((int64_t)out[i] + (int64_t)br);
}

hipError_t add_bias(int16_t* out, const int16_t* b, const uint8_t* bs, int n, uint8_t out_frac, hipStream_t st) {
    bias_kernel<<<(n + 255) / 256, 256, 0, st>>>(out, b, bs, n, out_frac);
    return hipGetLastError();
}

__device__ inline int16_t silu_gate(int16_t g, int16_t u, const int16_t* silu, uint32_t silu_len, uint8_t gate_frac,
                                    uint8_t up_frac, uint8_t down_in_frac, uint8_t silu_in_frac, int16_t silu_off,
                                    uint8_t silu_out_frac) {
    const int32_t g_dom = rescale32((int32_t)g, gate_frac, silu_in_frac);
    const int16_t act = lut_lookup_i16((int16_t)g_dom, silu, silu_len, silu_off);
    const int64_t prod = (int64_t)act * (int64_t)u;
    return clamp_i16_i64(rescale64(prod, (uint8_t)(silu_out_frac + up_frac), down_in_frac));
}

__global__ void silu_gate_kernel(const int16_t* __restrict__ gate, const int16_t* __restrict__ up, int n,
                                 const int16_t* __restrict__ silu, uint32_t silu_len, uint8_t gate_frac, uint8_t up_frac,
                                 uint8_t down_in_frac, uint8_t silu_in_frac, int16_t silu_off, uint8_t silu_out_frac,
                                 int16_t* __restrict__ h) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    h[i] = silu_gate(gate[i], up[i], silu, silu_len, gate_frac, up_frac, down_in_frac, silu_in_frac, silu_off,
                     silu_out_frac);
}

hipError_t silu_gate(const int16_t* gate, const int16_t* up, int n, const int16_t* silu, int silu_len,
                     uint8_t gate_frac, uint8_t up_frac, uint8_t down_in_frac, uint8_t silu_in_frac, int16_t silu_off,
                     uint8_t silu_out_frac, int16_t* h, hipStream_t st) {
    silu_gate_kernel<<<(n + 255) / 256, 256, 0, st>>>(gate, up, n, silu, (uint32_t)silu_len, gate_frac, up_frac,
                                                      down_in_frac, silu_in_frac, silu_off, silu_out_frac, h);
    return hipGetLastError();
}

// First maximum wins: the key orders by value, then by the smaller index.
__device__ inline uint64_t argmax_key(int32_t v, uint32_t idx) {
    return ((uint64_t)((uint32_t)v ^ 0x80000000u) << 32) | (uint64_t)(0xFFFFFFFFu - idx);
}

// Four consecutive values of a row: rows start at any 4-byte address (odd
// lengths and strides), which a 16-byte global load accepts.
typedef int32_t RowQuad __attribute__((ext_vector_type(4), aligned(4)));

// The passes over whole logit rows (row_walk.h) walk a row with the block's
// waves side by side: four 16-byte loads per lane and segment, two segments in
// flight, 128 KB per block, which is what one CU needs to draw its share of the
// memory rate with few rows in flight.

// Calls full(s, v) for each whole segment s of row[0, n) that falls to this
// wave, in ascending order (v[q][e] is value i = row_index(s, q, e), ascending
// in q and e), then tail(i0) on every wave for the partial last segment [i0, n),
// whose values the block's threads share (row_tail).
__device__ inline int row_index(int s, int q, int e) {
    return s * kRowSeg + q * 256 + (int)(threadIdx.x & 63) * 4 + e;
}
template <class Full, class Tail>
__device__ inline void row_segments(const int32_t* __restrict__ row, int n, const Full& full, const Tail& tail) {
    const int nfull = n / kRowSeg;
    auto load = [&](RowQuad (&v)[4], int s) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = *reinterpret_cast<const RowQuad*>(row + row_index(s, q, 0));
    };
    int s = threadIdx.x >> 6;
    for (; s + kRowWaves < nfull; s += 2 * kRowWaves) {
        RowQuad a[4], b[4];
        load(a, s);
        load(b, s + kRowWaves);
        full(s, a);
        full(s + kRowWaves, b);
    }
    if (s < nfull) {
        RowQuad a[4];
        load(a, s);
        full(s, a);
    }
    if (nfull * kRowSeg < n) tail(nfull * kRowSeg);
}

// The same with f(i, v) for every value and seg(s) after each segment (on each
// wave that had values of it).
template <class F, class Seg>
__device__ inline void row_values(const int32_t* __restrict__ row, int n, const F& f, const Seg& seg) {
    row_segments(
        row, n,
        [&](int s, const RowQuad (&v)[4]) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) f(row_index(s, q, e), v[q][e]);
            seg(s);
        },
        [&](int i0) {
            row_tail(i0, n, (int)threadIdx.x, kRowThreads, [&](int i) { f(i, row[i]); });
            if ((int)(threadIdx.x & ~63u) < n - i0) seg(i0 / kRowSeg);
        });
}

// f(i, v) for every value of a short row, ascending per thread.
template <class F>
__device__ inline void row_short(const int32_t* __restrict__ row, int n, const F& f) {
    row_quads(
        n, (int)threadIdx.x,
        [&](int i) {
            const RowQuad v = *reinterpret_cast<const RowQuad*>(row + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) f(i + e, v[e]);
        },
        [&](int i) { f(i, row[i]); });
}

// Bound by reading the row: 600 x 152064 values in 61 us (6.0 TB/s), 24 in 7.8
// us; 256 threads with one load in flight each and 64-bit keys throughout took
// 280 and 73 us.  A thread keeps its first maximum (ascending i, so strictly
// greater wins); keys order the threads'.
template <bool SHORT>
__global__ __launch_bounds__(SHORT ? kRowShortThreads : kRowThreads) void argmax_kernel(const int32_t* __restrict__ v, int n,
                                                                                       int ldv, int64_t* __restrict__ out) {
    constexpr int kWaves = (SHORT ? kRowShortThreads : kRowThreads) / 64;
    __shared__ uint64_t red[kWaves];
    const int32_t* row = v + (size_t)blockIdx.x * ldv;
    int32_t best = INT32_MIN;
    int at = -1;
    auto take = [&](int i, int32_t x) {
        const bool up = x > best || at < 0;
        best = up ? x : best;
        at = up ? i : at;
    };
    if constexpr (SHORT) row_short(row, n, take);
    else row_values(row, n, take, [](int) {});
    const uint64_t key = wave_max_u64(at < 0 ? 0 : argmax_key(best, (uint32_t)at));
    const int lane = threadIdx.x & 63;
    if (lane == 0) red[threadIdx.x >> 6] = key;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const uint64_t m = wave_max_u64(lane < kWaves ? red[lane] : 0);
    if (lane == 0) out[blockIdx.x] = (int64_t)(0xFFFFFFFFu - (uint32_t)(m & 0xFFFFFFFFu));
}

// Integer log-softmax of one row at its target (build-defined, see fixed.h):
//   m = max z;  S = sum_j lut[(m - z_j) << 2] (0 past the table; logits are
//   Q6 and the exp LUT's input is Q8);  lp = (z_target - m) * 2^10 - ln_q16(S)
// in Q16.  One block per row; targets < 0 give 0.
//
// Bound by reading the row, and S needs the maximum first, which read it
// twice.  The logits are whole numbers, so one pass counts them instead: a
// ring of kLogBins LDS counters indexed by z mod kLogBins (an LDS add where the
// second pass had an LDS table lookup), with the maximum and the least value
// counted.  Values kLogBins (128 logit units) or more below the largest of
// 1024 sampled ones are past the table whatever the maximum is and are not
// counted (masked tokens, say); a value that fills a segment, or half of it, is
// counted in registers.
// When the counted values lie less than kLogBins apart every counter stands
// for one value and S = sum over k of count[m - k] * lut[k << 2]; other rows,
// and tables longer than the ring, sum the table over a second pass.
// 600 x 152064 values in 80 us (4.6 TB/s); two passes of 256 threads took 385.
// Constant rows, rows wider than the ring, rows half masked with the least value
// and rows with all but 1% at one value in the ring take 78,
// 140, 83 and 92 us (189, 188, 346 and 193 with two passes; the last 402 with an add
// per value).
constexpr int kLogBins = 8192;
constexpr int kLogSame = 32;  // lanes of a wave with one value from which it is counted in registers

// One value's term of S, `below` under the maximum; the result from S.
__device__ inline int64_t logsoftmax_term(uint64_t below, const int16_t* lut, uint32_t lut_len) {
    const uint64_t d = below << (MYL_TV_EXP_INPUT_FRAC - MYL_TV_LOGIT_FRAC_BITS);
    return d < lut_len ? (int64_t)lut[d] : 0;
}
__device__ inline int64_t logsoftmax_at(const int32_t* row, int n, int64_t target, int32_t m, int64_t S) {
    if (target < 0 || target >= n) return 0;
    return ((int64_t)row[target] - (int64_t)m) * 1024 - ln_q16_of_sum(S < 1 ? 1u : (uint64_t)S);
}

__global__ __launch_bounds__(kRowThreads) void logsoftmax_kernel(const int32_t* __restrict__ z, int n, int ldz,
                                                                const int16_t* __restrict__ lut, uint32_t lut_len,
                                                                const int64_t* __restrict__ targets,
                                                                int64_t* __restrict__ out) {
    __shared__ int32_t reds[kRowWaves], redm[kRowWaves], redx[kRowWaves];
    __shared__ int64_t red64[kRowWaves];
    __shared__ uint32_t count[kLogBins];
    const int32_t* row = z + (size_t)blockIdx.x * ldz;
    const int tid = threadIdx.x;
    for (int i = tid; i < kLogBins; i += kRowThreads) count[i] = 0;
    static_assert(kRowThreads == 1024, "one sample per thread");
    const int32_t top = block_max_i32_dpp(row[((int64_t)tid * n) >> 10], reds);  // its barrier also clears the counts
    const int32_t least = (int32_t)max((int64_t)top - (kLogBins - 1), (int64_t)INT32_MIN);
    int32_t nm = INT32_MIN, mx = INT32_MIN;
    row_segments(
        row, n,
        [&](int, const RowQuad (&v)[4]) {
            int32_t smin = v[0][0], smax = v[0][0];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    smin = min(smin, v[q][e]);
                    smax = max(smax, v[q][e]);
                }
            mx = max(mx, smax);
            // A value that many lanes hold is counted in registers, and a second
            // one with it: the lanes' adds to one counter come one after another.
            const int32_t some = __builtin_amdgcn_readfirstlane(v[0][0]), low = __builtin_amdgcn_readfirstlane(smin),
                          high = __builtin_amdgcn_readfirstlane(smax);
            auto many = [&](int32_t x, int32_t y) {
                return (int)(y >= least) & (int)(__builtin_popcountll(__ballot(x == y)) >= kLogSame);
            };
            const int many_some = many(v[0][0], some), many_low = many(smin, low), many_high = many(smax, high);
            if (many_some | many_low | many_high) {  // uniform
                if (__all(smin == smax && smin == some)) {
                    nm = max(nm, ~some);
                    if ((tid & 63) == 0) atomicAdd(&count[(uint32_t)some % kLogBins], (uint32_t)kRowSeg);
                    return;
                }
                const int32_t a = many_some ? some : many_low ? low : high, b = high != a ? high : low;
                int32_t c = 0;  // of a | of b << 16
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int32_t x = v[q][e];
                        nm = x >= least ? max(nm, ~x) : nm;
                        c += x == a ? 1 : (x == b ? 0x10000 : 0);
                        if (x != a && x != b && x >= least) atomicAdd(&count[(uint32_t)x % kLogBins], 1u);
                    }
                c = wave_sum_i32(c);
                if ((tid & 63) == 0) {
                    atomicAdd(&count[(uint32_t)a % kLogBins], (uint32_t)c & 0xFFFFu);
                    if (b >= least) atomicAdd(&count[(uint32_t)b % kLogBins], (uint32_t)c >> 16);
                }
                return;
            }
            if (__all(smin >= least)) {
                nm = max(nm, ~smin);
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) atomicAdd(&count[(uint32_t)v[q][e] % kLogBins], 1u);
                return;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (v[q][e] >= least) {
                        nm = max(nm, ~v[q][e]);  // the minimum as ~max(~z)
                        atomicAdd(&count[(uint32_t)v[q][e] % kLogBins], 1u);
                    }
        },
        [&](int i0) {
            row_tail(i0, n, tid, kRowThreads, [&](int i) {
                const int32_t x = row[i];
                mx = max(mx, x);
                if (x < least) return;
                nm = max(nm, ~x);
                atomicAdd(&count[(uint32_t)x % kLogBins], 1u);
            });
        });
    const int32_t lo = ~block_max_i32_dpp(nm, redm);
    const int32_t m = block_max_i32_dpp(mx, redx);  // the barriers also publish the counts
    constexpr uint32_t sh = MYL_TV_EXP_INPUT_FRAC - MYL_TV_LOGIT_FRAC_BITS;
    auto term = [&](uint64_t below) { return logsoftmax_term(below, lut, lut_len); };
    int64_t s = 0;
    if ((int64_t)m - (int64_t)lo < kLogBins && lut_len <= ((uint32_t)kLogBins << sh)) {
        for (uint32_t k = tid; k < (uint32_t)kLogBins && ((uint64_t)k << sh) < lut_len; k += kRowThreads)
            s += (int64_t)count[((uint32_t)m - k) % kLogBins] * term(k);
    } else {
        // the table's every fourth entry in the counters' place
        int16_t* tab = reinterpret_cast<int16_t*>(count);
        for (uint32_t k = tid; k < (uint32_t)kLogBins; k += kRowThreads) tab[k] = (int16_t)term(k);
        __syncthreads();
        row_values(
            row, n,
            [&](int, int32_t x) {
                const uint64_t below = (uint64_t)((int64_t)m - (int64_t)x);
                s += below < (uint64_t)kLogBins ? (int64_t)tab[below] : term(below);
            },
            [](int) {});
    }
    s = wave_sum_i64(s);
    if ((tid & 63) == 0) red64[tid >> 6] = s;
    __syncthreads();
    if (tid >= 64) return;
    const int64_t S = wave_sum_i64(tid < kRowWaves ? red64[tid] : 0);
    if (tid == 0) out[blockIdx.x] = logsoftmax_at(row, n, targets[blockIdx.x], m, S);
}

// The same for short rows: the row is read twice, the second time from the
// cache, which costs less than clearing and summing the counters.  Past
// kLogTabRow values, the table's first entries (32 logit units) wait in LDS: 2000
// rows of 1000 / 8192 values 7.2 / 24.6 us (8.1 with the table for the first; 26.1
// for the second with the table copied before the row is read).
constexpr int kLogTab = 2048, kLogTabRow = 1024;
__global__ __launch_bounds__(kRowShortThreads) void logsoftmax_short_kernel(const int32_t* __restrict__ z, int n, int ldz,
                                                                           const int16_t* __restrict__ lut, uint32_t lut_len,
                                                                           const int64_t* __restrict__ targets,
                                                                           int64_t* __restrict__ out) {
    constexpr int kWaves = kRowShortThreads / 64;
    __shared__ int32_t redx[kWaves];
    __shared__ int64_t red64[kWaves];
    __shared__ int16_t tab[kLogTab];
    const int32_t* row = z + (size_t)blockIdx.x * ldz;
    const int tid = threadIdx.x;
    const uint64_t nt = n > kLogTabRow ? kLogTab : 0;
    constexpr int kTabEach = kLogTab / kRowShortThreads;
    int16_t own[kTabEach];  // the thread's entries, on their way while the row is read
    if (nt)
#pragma unroll
        for (int j = 0; j < kTabEach; ++j) own[j] = (int16_t)logsoftmax_term((uint64_t)(j * kRowShortThreads + tid), lut, lut_len);
    int32_t mx = INT32_MIN;
    row_short(row, n, [&](int, int32_t x) { mx = max(mx, x); });
    if (nt)
#pragma unroll
        for (int j = 0; j < kTabEach; ++j) tab[j * kRowShortThreads + tid] = own[j];
    const int32_t m = block_max_i32_dpp(mx, redx);  // its barrier also publishes the table
    int64_t s = 0;
    row_short(row, n, [&](int, int32_t x) {
        const uint64_t below = (uint64_t)((int64_t)m - (int64_t)x);
        s += below < nt ? (int64_t)tab[below] : logsoftmax_term(below, lut, lut_len);
    });
    s = wave_sum_i64(s);
    if ((tid & 63) == 0) red64[tid >> 6] = s;
    __syncthreads();
    if (tid >= 64) return;
    const int64_t S = wave_sum_i64(tid < kWaves ? red64[tid] : 0);
    if (tid == 0) out[blockIdx.x] = logsoftmax_at(row, n, targets[blockIdx.x], m, S);
}

hipError_t logsoftmax(const int32_t* z, int M, int n, int ldz, const int16_t* lut, int lut_len, const int64_t* targets,
                      int64_t* out, hipStream_t st) {
    if (row_short_logsoftmax(M, n)) logsoftmax_short_kernel<<<M, kRowShortThreads, 0, st>>>(z, n, ldz, lut, (uint32_t)lut_len, targets, out);
    else logsoftmax_kernel<<<M, kRowThreads, 0, st>>>(z, n, ldz, lut, (uint32_t)lut_len, targets, out);
    return hipGetLastError();
}

hipError_t argmax(const int32_t* v, int M, int n, int ldv, int64_t* out, hipStream_t st) {
    if (row_short_argmax(M, n)) argmax_kernel<true><<<M, kRowShortThreads, 0, st>>>(v, n, ldv, out);
    else argmax_kernel<false><<<M, kRowThreads, 0, st>>>(v, n, ldv, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Integer CDF sampling (sampling.rs:20-46): one block per row.
// ---------------------------------------------------------------------------

// SplitMix64 (prng.rs:7-14): advances the state, returns the output.
__device__ inline uint64_t splitmix64_next(uint64_t& state) {
    state += 0x9E3779B97F4A7C15ull;
    uint64_t z = state;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// n % d by binary long division (no hardware divide); 0 < d < 2^63.  The top
// bits of n that are together below d are the first remainder.
__device__ inline uint64_t umod64(uint64_t n, uint64_t d) {
    const int k = 64 - __builtin_clzll(d) - 1;  // 2^k <= d
    uint64_t r = k ? n >> (64 - k) : 0;
    for (int i = 63 - k; i >= 0; --i) {
        r = (r << 1) | ((n >> i) & 1u);
        if (r >= d) r -= d;
    }
    return r;
}

__device__ inline int64_t shfl_up_i64(int64_t v, int d) {
    const uint32_t lo = (uint32_t)__shfl_up((int)(uint32_t)v, d, 64);
    const uint32_t hi = (uint32_t)__shfl_up((int)(uint32_t)((uint64_t)v >> 32), d, 64);
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Exclusive prefix sum of one i64 per thread over the block (wrapping),
// and the block's total.  wt needs one slot per wave.
__device__ inline int64_t block_scan_i64(int64_t v, int64_t* wt, int64_t& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    int64_t inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t o = shfl_up_i64(inc, d);
        if (lane >= d) inc = (int64_t)((uint64_t)inc + (uint64_t)o);
    }
    if (lane == 63) wt[w] = inc;
    __syncthreads();
    int64_t before = 0, all = 0;
    for (int k = 0; k < nw; ++k) {
        const int64_t t = wt[k];
        if (k < w) before = (int64_t)((uint64_t)before + (uint64_t)t);
        all = (int64_t)((uint64_t)all + (uint64_t)t);
    }
    total = all;
    return (int64_t)((uint64_t)before + (uint64_t)inc - (uint64_t)v);
}

// Inclusive prefix sum of one i64 per lane over the wave (wrapping).
__device__ inline int64_t wave_scan_i64(int64_t v, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t o = shfl_up_i64(v, d);
        if (lane >= d) v = (int64_t)((uint64_t)v + (uint64_t)o);
    }
    return v;
}

// sample_integer_cdf (sampling.rs:27-46) of row blockIdx.x at state
// states[row]: weights w_i = z_i - min z + 1 (logits_to_weights,
// sampling.rs:20-24; i32 arithmetic, wrapping as the reference's release
// build does), total = sum w_i as i64; total <= 0 gives token 0 and the state
// unchanged; otherwise (state', r) = splitmix64(state), threshold = r % total
// and the token is the first i with threshold < w_0 + ... + w_i (the last
// index when there is none).
//
// Bound by reading the row, and with few rows by one block's loads in
// flight, so the row is read once: the pass keeps its minimum, its maximum
// and the sum of z of every group of 2^lg segments in LDS.  When no
// weight wraps (max - min + 1 < 2^31, as any logits of a model) the weights
// are positive, so the group's weight sums follow from those sums and the
// minimum, the running sum only rises, and the token lies in the first group
// whose running sum passes the threshold: only that group is read again, by
// one wave.  Rows with wrapped weights scan every value in order over tiles
// of 4 x kRowThreads positions, so the first such i is exact also when the
// running sums are not monotone.  24 x 152064: 17 us; three passes over the
// row with one load in flight per thread took 130 us.
constexpr int kSampleGroups = 1024;
__global__ __launch_bounds__(kRowThreads) void sample_cdf_kernel(const int32_t* __restrict__ z, int n, int ldz, int lg,
                                                                const uint64_t* __restrict__ states,
                                                                int64_t* __restrict__ tokens,
                                                                uint64_t* __restrict__ new_states) {
    __shared__ int32_t redm[kRowWaves], redx[kRowWaves];
    __shared__ int32_t redc[kRowWaves];
    __shared__ int64_t wt[kRowWaves];
    __shared__ int64_t s_thr;
    __shared__ unsigned long long gsum[kSampleGroups];
    const int32_t* row = z + (size_t)blockIdx.x * ldz;
    const int tid = threadIdx.x, lane = tid & 63;
    const int gvals = kRowSeg << lg;                                     // values per group
    const int ngroups = (int)(((int64_t)n + gvals - 1) / kRowSeg >> lg);  // <= kSampleGroups
    gsum[tid] = 0;
    __syncthreads();
    // the minimum as ~max(~z) (bitwise not reverses the signed order)
    int32_t nm = INT32_MIN, mx = INT32_MIN;
    int64_t part = 0;
    row_values(
        row, n,
        [&](int, int32_t x) {
            nm = max(nm, ~x);
            mx = max(mx, x);
            part += x;
        },
        [&](int s) {
            const int64_t t = wave_sum_i64(part);
            if (lane == 0) atomicAdd(&gsum[s >> lg], (unsigned long long)t);
            part = 0;
        });
    const int32_t m = ~block_max_i32_dpp(nm, redm);
    mx = block_max_i32_dpp(mx, redx);  // its barrier also publishes gsum
    uint64_t state = states[blockIdx.x];
    auto weight = [&](int32_t zi) -> int64_t { return (int64_t)(int32_t)((uint32_t)zi - (uint32_t)m + 1u); };
    if ((int64_t)mx - (int64_t)m + 1 <= (int64_t)INT32_MAX) {
        if (tid >= 64) return;
        // lane l: groups [16 l, 16 l + 16), their running weight sums
        constexpr int kPerLane = kSampleGroups / 64;
        const int64_t shift = (int64_t)m - 1;  // w = z - shift
        auto gw = [&](int g) -> int64_t {
            if (g >= ngroups) return 0;
            const int64_t len = min((int64_t)gvals, (int64_t)n - (int64_t)g * gvals);
            return (int64_t)gsum[g] - len * shift;
        };
        int64_t mine = 0;
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) mine += gw(lane * kPerLane + j);
        const int64_t inc = wave_scan_i64(mine, lane);
        const int64_t total = (int64_t)readlane_u64((uint64_t)inc, 63);  // >= n
        const uint64_t r = splitmix64_next(state);
        const int64_t thr = (int64_t)umod64(r, (uint64_t)total);  // total < 2^62: n < 2^31 weights below 2^31
        const uint64_t past = __ballot(thr < inc);                // the last lane's always is
        const int l0 = (int)__builtin_ctzll(past);
        int64_t base = (int64_t)readlane_u64((uint64_t)(inc - mine), l0);
        int g = l0 * kPerLane;
        for (int j = 0; j + 1 < kPerLane; ++j, ++g) {
            const int64_t wg = gw(g);
            if (thr < base + wg) break;
            base += wg;
        }
        int pick = n - 1;
        const int g0 = g * gvals, g1 = (int)min((int64_t)n, (int64_t)g0 + gvals);
        for (int k0 = 0; k0 < g1 - g0; k0 += 256) {
            int64_t w[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = row_group_index(g0, k0, lane) + e;
                w[e] = i < g1 ? (int64_t)row[i] - shift : 0;
            }
            const int64_t loc = w[0] + w[1] + w[2] + w[3];
            const int64_t sc = wave_scan_i64(loc, lane);
            const uint64_t hit = __ballot(thr < base + sc);
            if (hit) {  // uniform
                const int l = (int)__builtin_ctzll(hit);
                int64_t acc = base + sc - loc;
                int at = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc += w[e];
                    at += thr < acc ? 0 : 1;
                }
                pick = row_group_index(g0, k0, l) + readlane_i32(at, l);
                break;
            }
            base += (int64_t)readlane_u64((uint64_t)sc, 63);
        }
        if (lane == 0) {
            tokens[blockIdx.x] = pick;
            new_states[blockIdx.x] = state;
        }
        return;
    }
    part = 0;
    row_strided(n, tid, [&](int i) { part += weight(row[i]); });
    int64_t total = 0;
    (void)block_scan_i64(part, wt, total);
    if (total <= 0) {  // uniform: an empty or non-positive total keeps the state
        if (tid == 0) {
            tokens[blockIdx.x] = 0;
            new_states[blockIdx.x] = state;
        }
        return;
    }
    if (tid == 0) {
        const uint64_t r = splitmix64_next(state);
        s_thr = (int64_t)umod64(r, (uint64_t)total);  // total < 2^62: n < 2^31 weights below 2^31
        new_states[blockIdx.x] = state;
    }
    __syncthreads();
    const int64_t thr = s_thr;
    int64_t base = 0;
    int pick = n - 1;
    for (int64_t t0 = 0; t0 < n; t0 += 4 * kRowThreads) {
        const int64_t i0 = t0 + 4 * tid;
        int64_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = i0 + e < n ? weight(row[i0 + e]) : 0;
        const int64_t loc = w[0] + w[1] + w[2] + w[3];
        int64_t tile = 0;
        int64_t acc = base + block_scan_i64(loc, wt, tile);
        int cand = INT32_MAX;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc += w[e];
            if (i0 + e < n && thr < acc && cand == INT32_MAX) cand = (int)(i0 + e);
        }
        // the first candidate of the tile: a block minimum as ~max(~x)
        const int first = ~block_max_i32_dpp(~cand, redc);
        if (first != INT32_MAX) {  // uniform
            pick = first;
            break;
        }
        base += tile;
    }
    if (tid == 0) tokens[blockIdx.x] = pick;
}

// The same for rows of at most kRowShortThreads x EACH values, which stay in registers: one
// read, one scan over the block (wrapped weights included).  With the groups, a
// short row is mostly their two wave scans one after the other and the 16 waves'
// segment sums.  24 rows of 1000 / 4096 values: 5.0 / 6.8 us, 8.1 / 8.2 with the
// groups; 2000 rows of 1000: 11.6 and 20.6 (16 waves of four values a lane took
// 40 at 2000 x 2048: all of them work out the threshold's remainder).
template <int EACH>
__global__ __launch_bounds__(kRowShortThreads) void sample_short_kernel(const int32_t* __restrict__ z, int n, int ldz,
                                                                       const uint64_t* __restrict__ states,
                                                                       int64_t* __restrict__ tokens,
                                                                       uint64_t* __restrict__ new_states) {
    __shared__ int32_t redm[kRowShortThreads / 64], redc[kRowShortThreads / 64];
    __shared__ int64_t wt[kRowShortThreads / 64];
    const int32_t* row = z + (size_t)blockIdx.x * ldz;
    const int tid = threadIdx.x, i0 = EACH * tid;
    uint64_t state = states[blockIdx.x];
    int32_t v[EACH], nm = INT32_MIN;
#pragma unroll
    for (int e = 0; e < EACH; ++e) v[e] = row[min(i0 + e, n - 1)];  // past the row: the last value again
#pragma unroll
    for (int e = 0; e < EACH; ++e) nm = max(nm, ~v[e]);
    const int32_t m = ~block_max_i32_dpp(nm, redm);
    int64_t w[EACH], loc = 0;
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
        w[e] = i0 + e < n ? (int64_t)(int32_t)((uint32_t)v[e] - (uint32_t)m + 1u) : 0;
        loc += w[e];
    }
    int64_t total = 0;
    int64_t acc = block_scan_i64(loc, wt, total);
    if (total <= 0) {  // uniform: a non-positive total keeps the state
        if (tid == 0) {
            tokens[blockIdx.x] = 0;
            new_states[blockIdx.x] = state;
        }
        return;
    }
    const int64_t thr = (int64_t)umod64(splitmix64_next(state), (uint64_t)total);
    int cand = INT32_MAX;
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
        acc += w[e];
        if (i0 + e < n && thr < acc && cand == INT32_MAX) cand = i0 + e;
    }
    const int first = ~block_max_i32_dpp(~cand, redc);
    if (tid == 0) {
        tokens[blockIdx.x] = first == INT32_MAX ? n - 1 : first;
        new_states[blockIdx.x] = state;
    }
}

hipError_t sample_cdf(const int32_t* z, int M, int n, int ldz, const uint64_t* states, int64_t* tokens,
                      uint64_t* new_states, hipStream_t st) {
    if (n <= kRowShortThreads * 16) {
        if (n <= kRowShortThreads * 4) sample_short_kernel<4><<<M, kRowShortThreads, 0, st>>>(z, n, ldz, states, tokens, new_states);
        else sample_short_kernel<16><<<M, kRowShortThreads, 0, st>>>(z, n, ldz, states, tokens, new_states);
        return hipGetLastError();
    }
    // 2^lg segments per group, so that the row's groups fit the block's LDS sums
    int lg = 0;
    while (((int64_t)kSampleGroups * kRowSeg << lg) < n) ++lg;
    sample_cdf_kernel<<<M, kRowThreads, 0, st>>>(z, n, ldz, lg, states, tokens, new_states);
    return hipGetLastError();
}

// Best key of chunk blockIdx.x of row blockIdx.y.
__global__ __launch_bounds__(kBlock) void argmax_part_kernel(const int32_t* __restrict__ v, int n, int ldv,
                                                            uint64_t* __restrict__ part, int nch) {
    __shared__ uint64_t red[kBlock];
    const int32_t* row = v + (size_t)blockIdx.y * ldv;
    const int i0 = blockIdx.x * kArgChunk, i1 = min(n, i0 + kArgChunk);
    uint64_t best = 0;
    // 16-byte loads when the chunk starts aligned (kArgChunk is a multiple
    // of 4), the chunk's last partial quad and unaligned rows one by one
    const int q1 = ((uintptr_t)(row + i0) & 15) == 0 ? i0 + ((i1 - i0) & ~3) : i0;
#pragma unroll 4
    for (int i = i0 + 4 * (int)threadIdx.x; i < q1; i += 4 * kBlock) {
        const int4 q = *reinterpret_cast<const int4*>(row + i);
        const uint64_t k0 = argmax_key(q.x, (uint32_t)i), k1 = argmax_key(q.y, (uint32_t)i + 1);
        const uint64_t k2 = argmax_key(q.z, (uint32_t)i + 2), k3 = argmax_key(q.w, (uint32_t)i + 3);
        const uint64_t a = k0 > k1 ? k0 : k1, b = k2 > k3 ? k2 : k3, c = a > b ? a : b;
        best = c > best ? c : best;
    }
    for (int i = q1 + threadIdx.x; i < i1; i += kBlock) {
        const uint64_t key = argmax_key(row[i], (uint32_t)i);
        best = key > best ? key : best;
    }
    red[threadIdx.x] = best;
    __syncthreads();
    for (int s = blockDim.x >> 1; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] > red[threadIdx.x + s] ? red[threadIdx.x] : red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[(size_t)blockIdx.y * nch + blockIdx.x] = red[0];
}

__global__ __launch_bounds__(64) void argmax_final_kernel(const uint64_t* __restrict__ part, int nch,
                                                         int64_t* __restrict__ out) {
    uint64_t best = 0;
    for (int c = threadIdx.x; c < nch; c += 64) best = max(best, part[(size_t)blockIdx.x * nch + c]);
    best = wave_max_u64(best);
    if (threadIdx.x == 0) out[blockIdx.x] = (int64_t)(0xFFFFFFFFu - (uint32_t)(best & 0xFFFFFFFFu));
}

// One pass over `bytes` (a multiple of 16) of device memory: nontemporal
// 16-byte loads, four in flight per thread, grid-stride.  The thread's XOR of
// its words is stored only when it equals one arbitrary constant, so the
// loads cannot be dropped and at most a word is written.
__global__ __launch_bounds__(512) void read_probe_kernel(const uint4* __restrict__ p, size_t n16,
                                                         uint32_t* __restrict__ out) {
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    const size_t nthr = (size_t)gridDim.x * blockDim.x;
    uint32_t acc = 0;
    size_t i = tid;
    for (; i + 3 * nthr < n16; i += 4 * nthr) {
        v4u v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(p + i + u * nthr));
#pragma unroll
        for (int u = 0; u < 4; ++u) acc ^= v[u][0] ^ v[u][1] ^ v[u][2] ^ v[u][3];
    }
    for (; i < n16; i += nthr) {
        const uint4 v = p[i];
        acc ^= v.x ^ v.y ^ v.z ^ v.w;
    }
    if (acc == 0x9E3779B9u) out[0] = acc;
}

hipError_t read_probe(const void* p, size_t bytes, uint32_t* out, int cus, hipStream_t st) {
    read_probe_kernel<<<cus, 512, 0, st>>>(reinterpret_cast<const uint4*>(p), bytes / 16, out);
    return hipGetLastError();
}

hipError_t argmax_rows(const int32_t* v, int M, int n, int ldv, int64_t* out, uint64_t* part, hipStream_t st) {
    const int nch = (n + kArgChunk - 1) / kArgChunk;
    argmax_part_kernel<<<dim3(nch, M), kBlock, 0, st>>>(v, n, ldv, part, nch);
    argmax_final_kernel<<<M, 64, 0, st>>>(part, nch, out);
    return hipGetLastError();
}

}  // namespace myl
