// gemm_q8w.h -- weight-only int8 product with f32 activations,
//   C[m, n] = wscale[n] * sum_k A[m, k] * q[n, k],
// the device side of encoder.Q8Backend.MatmulBTQ8 (encoder/backend_use.go:59-83), whose CPU
// path widens the weight to f32 (f32(q) * wscale, linalg.DequantizeRowsInt8Into) and runs
// the f32 MatmulBT (encoder/linalg_q8.go:80-84). The activations are never quantized.
//
// Arithmetic. Each f32 activation is split exactly into three bf16 parts by truncation:
// b1 = the top 16 bits of a, b2 = the top 16 bits of a - b1, b3 = a - b1 - b2. a - b1 has at
// most 16 significant bits and a - b1 - b2 at most 8, so both subtractions are exact and b3
// is a bf16 value: a = b1 + b2 + b3 with no rounding, over f32's whole range (a part below
// 2^-126 may be flushed, an absolute error under 2^-126). A weight code q (any int8, -128
// included) is a bf16 value exactly. So every v_mfma_f32_32x32x16_bf16 product b_i q is exact
// and the sum over k (three MFMAs per 16-deep block) is accumulated in f32 in an order of its
// own; the channel scale multiplies the sum once at the end. The CPU rounds each widened weight and
// sums in f32 in its own order; the contract both meet is the reference's gate against a
// float64 dot product, worst |C - ref| <= 2e-4 max(|ref|, 1)
// (gpu/enccuda/backend_test.go:234-289). An infinite activation keeps b2 = b3 = 0, so its
// products are +-inf (or NaN against q = 0) as the reference's are; NaN stays NaN.
//
// Layout. The weight is the registered fragment-major int8 image (kernels.h frag_off:
// 1 KiB per 32 channels x 32 k, lane l holding channel l % 32, k 16 (l / 32) .. +15) and is
// read straight into registers, 16 bytes per lane per block. The MFMA's lane half h
// supplies depth 8h .. 8h + 7 of each 16-deep step, so step j of a 32-deep chunk takes
// bytes 8j .. 8j + 7 of the lane's 16, i.e. k = 16h + 8j + (0..7): the A operand is fed in
// the same k order, so the permutation cancels in the sum. A is row-major f32. Rows past M
// re-read row M - 1 and are not stored; k past K is zero in A (the weight image is zero there
// too); channels past N read the image's zero padding and are not stored.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "attention_f32.h"
#include "kernels.h"

#pragma clang fp contract(off)

namespace enchip {

// The exact split a = b1 + b2 + b3 of one f32 into the upper halves of t1, t2, t3 (the
// bf16 bit patterns are t >> 16).
__device__ __forceinline__ void q8w_split3(float a, uint32_t &t1, uint32_t &t2, uint32_t &t3) {
    const uint32_t u = __float_as_uint(a);
    t1 = u;
    float r1 = a - __uint_as_float(u & 0xFFFF0000u);
    r1 = __builtin_isinf(a) ? 0.0f : r1;  // inf - inf would be NaN
    t2 = __float_as_uint(r1);
    t3 = __float_as_uint(r1 - __uint_as_float(t2 & 0xFFFF0000u));
}

// bf16x2 word of the upper halves of lo (element 0) and hi (element 1).
__device__ __forceinline__ uint32_t q8w_pack(uint32_t lo, uint32_t hi) {
    return __builtin_amdgcn_perm(hi, lo, 0x07060302u);
}

// 4 int8 codes (bytes of w, element 0 lowest) -> 2 bf16x2 words, exactly.
__device__ __forceinline__ void q8w_widen4(uint32_t w, uint32_t &lo, uint32_t &hi) {
    const float f0 = (float)(int8_t)(w & 0xFFu), f1 = (float)(int8_t)((w >> 8) & 0xFFu);
    const float f2 = (float)(int8_t)((w >> 16) & 0xFFu), f3 = (float)(int8_t)(w >> 24);
    lo = q8w_pack(__float_as_uint(f0), __float_as_uint(f1));
    hi = q8w_pack(__float_as_uint(f2), __float_as_uint(f3));
}

// Grid: tilesM * tilesN workgroups (XCD-aware order). Block tile (32 TM WM) x (32 TN WN), WM x
// WN wavefronts of TM x TN 32 x 32 accumulators, K in chunks of KC: every thread loads 16-byte
// pieces of A's rows, splits them and stores the three parts as planes of [row][KC] bf16 (rows
// 16 bytes apart from a multiple of 128, so 32 rows' 16-byte operand reads fall in distinct
// banks), double-buffered. The 16-deep steps rotate over NACC sets of accumulators, added in
// order at the end: shorter sums, and MFMAs that do not wait for the one before.
// W: the fragment-major image of an Np x Kp weight (Kp a multiple of 64, Np of BN); ws[N].
// VEC: lda % 4 == 0, K % 4 == 0 and A 16-byte aligned (16-byte loads). Otherwise the chunks inside
// K load the same 16 bytes at 4-byte alignment, and the last one value by value (all of them did for
// a while: 8192 x 4096, K = 2047 417 us, 358 so; 4000 x 1000, K = 1001 53 and 38).
// What bounds it: with a block or two per CU the serial latency of a chunk, hence 32-row tiles
// and deep chunks; with many tiles the MFMA and the splitting's VALU work. Measured on MI355X
// against the form before (64 x 64 to 128 x 256 tiles, 32-deep chunks, branches around the
// next chunk's loads), us: 512 x 2304, K = 768 23.2 -> 14.6, 1024 x 768 21.1 -> 11.2, 2048 x
// 768, K = 3072 74.1 -> 44.3, all in 32 x 128 tiles; 32768 x 3072, K = 768 475 -> 440 (1.05
// PFLOP/s of bf16 products) and 32768 x 768, K = 3072 465 -> 404 in 128 x 256. Error against
// float64 at K = 768: 1.4e-7 with NACC = 4, 2.6e-7 with 1 (2.6e-7 before). 256 x 256 tiles
// with 8 or 16 wavefronts were no faster.
template <int TM, int TN, int WM, int WN, int KC, int NACC, bool VEC>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_q8w(
    const float *__restrict__ A, int64_t lda, const int8_t *__restrict__ W, const float *__restrict__ ws,
    float *__restrict__ C, int64_t ldc, int M, int N, int K, int Kp, int tilesN) {
    constexpr int NT = 64 * WM * WN, BM = 32 * TM * WM, BN = 32 * TN * WN, KB = KC / 32;
    constexpr int P = 2 * KC + 16, PL = BM * P, STAGE = 3 * PL;
    constexpr int LPR = KC / 4, AV = BM * LPR / NT;
    static_assert(AV >= 1 && BM * LPR % NT == 0, "tile");
    __shared__ __attribute__((aligned(16))) char lds[2 * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 31, hf = lane >> 5;
    const int logical = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int m0 = (logical / tilesN) * BM, n0 = (logical % tilesN) * BN;
    const int wm = wave / WN, wn = wave % WN;
    const int lk = 4 * (tid % LPR), lr = tid / LPR;
    const float *ga[AV];
#pragma unroll
    for (int i = 0; i < AV; ++i) ga[i] = A + (int64_t)min(m0 + lr + (NT / LPR) * i, M - 1) * lda;
    const int nk32 = Kp / 32;
    const int8_t *wb[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t) wb[t] = W + ((int64_t)((n0 >> 5) + TN * wn + t) * nk32) * 1024 + lane * 16;
    f32x4 ra[AV];
    u32x4 wr[KB][TN];
    auto load_a = [&](int c) {
        const int k = KC * c + lk;
        if (!VEC && KC * c + KC <= K) {  // uniform: all of the chunk, in unaligned 16-byte loads
#pragma unroll
            for (int i = 0; i < AV; ++i) ra[i] = f32x4{ga[i][k], ga[i][k + 1], ga[i][k + 2], ga[i][k + 3]};
            return;
        }
#pragma unroll
        for (int i = 0; i < AV; ++i) {
            if (VEC) ra[i] = *reinterpret_cast<const f32x4 *>(ga[i] + min(k, K - 4));
            else
                ra[i] = f32x4{ga[i][min(k, K - 1)], ga[i][min(k + 1, K - 1)], ga[i][min(k + 2, K - 1)],
                              ga[i][min(k + 3, K - 1)]};
        }
    };
    auto load_w = [&](int c) {
#pragma unroll
        for (int b = 0; b < KB; ++b)
#pragma unroll
            for (int t = 0; t < TN; ++t)
                wr[b][t] = *reinterpret_cast<const u32x4 *>(wb[t] + (int64_t)min(KB * c + b, nk32 - 1) * 1024);
    };
    auto store_a = [&](int c, char *st) {
        const int k = KC * c + lk;
#pragma unroll
        for (int i = 0; i < AV; ++i) {
            f32x4 v = ra[i];  // k past K counts as zero
            if (VEC) {
                if (k >= K) v = f32x4{0.f, 0.f, 0.f, 0.f};
            } else {
                v.x = k < K ? v.x : 0.f, v.y = k + 1 < K ? v.y : 0.f, v.z = k + 2 < K ? v.z : 0.f, v.w = k + 3 < K ? v.w : 0.f;
            }
            uint32_t a1[4], a2[4], a3[4];
            q8w_split3(v.x, a1[0], a2[0], a3[0]);
            q8w_split3(v.y, a1[1], a2[1], a3[1]);
            q8w_split3(v.z, a1[2], a2[2], a3[2]);
            q8w_split3(v.w, a1[3], a2[3], a3[3]);
            char *d = st + (lr + (NT / LPR) * i) * P + 2 * lk;
            *reinterpret_cast<uint2 *>(d) = make_uint2(q8w_pack(a1[0], a1[1]), q8w_pack(a1[2], a1[3]));
            *reinterpret_cast<uint2 *>(d + PL) = make_uint2(q8w_pack(a2[0], a2[1]), q8w_pack(a2[2], a2[3]));
            *reinterpret_cast<uint2 *>(d + 2 * PL) = make_uint2(q8w_pack(a3[0], a3[1]), q8w_pack(a3[2], a3[3]));
        }
    };
    f32x16 acc[NACC][TM][TN];
#pragma unroll
    for (int a = 0; a < NACC; ++a)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int t = 0; t < TN; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[a][i][t][e] = 0.0f;
    // Chunk c + 1 is split into the other stage while chunk c's MFMAs run, and its registers
    // take chunk c + 2. Past the last chunk the loads re-read it and the stage is not used: no
    // branch, so that all of an iteration is scheduled together.
    const int nc = (Kp + KC - 1) / KC, last = nc - 1;
    load_a(0);
    load_w(0);
    store_a(0, lds);
    load_a(min(1, last));
    lds_barrier();
    for (int c = 0; c < nc; ++c) {
        const char *cur = lds + (c & 1) * STAGE;
        char *nxt = lds + ((c & 1) ^ 1) * STAGE;
#pragma unroll
        for (int b = 0; b < KB; ++b) {
            bf16x8 wq[TN][2];
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                const uint32_t d[4] = {wr[b][t].x, wr[b][t].y, wr[b][t].z, wr[b][t].w};
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    uint32_t x[4];
                    q8w_widen4(d[2 * j], x[0], x[1]);
                    q8w_widen4(d[2 * j + 1], x[2], x[3]);
                    wq[t][j] = __builtin_bit_cast(bf16x8, (u32x4){x[0], x[1], x[2], x[3]});
                }
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                bf16x8 p[TM][3];
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        p[i][q] = *reinterpret_cast<const bf16x8 *>(cur + q * PL + (32 * (TM * wm + i) + r) * P + 64 * b +
                                                                    32 * hf + 16 * j);
#pragma unroll
                for (int q = 2; q >= 0; --q)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int t = 0; t < TN; ++t)
                            acc[(2 * b + j) % NACC][i][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                p[i][q], wq[t][j], acc[(2 * b + j) % NACC][i][t], 0, 0, 0);
            }
        }
        load_w(min(c + 1, last));
        store_a(c + 1, nxt);
        load_a(min(c + 2, last));
        lds_barrier();
    }
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        const int n = n0 + 32 * (TN * wn + t) + r;
        const float s = ws[min(n, N - 1)];
        if (n >= N) continue;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int mb = m0 + 32 * (TM * wm + i);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = mb + acc_row(e, lane);
                float v = acc[0][i][t][e];
#pragma unroll
                for (int a = 1; a < NACC; ++a) v += acc[a][i][t][e];
                if (m < M) C[(int64_t)m * ldc + n] = v * s;
            }
        }
    }
}

// Small form: one workgroup per 32-row x 32-channel tile, its 4 wavefronts
// splitting K (wavefront w takes the 32-deep chunks w, w + 4, w + 8, ...). Each lane loads
// its own MFMA operand values straight from HBM -- lane (row m, half h) the 16 activations
// a[m, 32 kc + 16 h ..], split in registers, and its 16 weight bytes -- so there is no LDS
// and no barrier in the main loop, and a ring of Q8W_RING chunks per wavefront keeps that
// many loads in flight. The four partial sums meet in LDS and are added in a fixed order
// (wavefront 0 + 1 + 2 + 3), so the result does not depend on timing. Same arithmetic,
// edges and preconditions as gemm_q8w.
constexpr int Q8W_RING = 4;

template <bool VEC>
__global__ __launch_bounds__(256) void gemm_q8w_small(const float *__restrict__ A, int64_t lda,
                                                      const int8_t *__restrict__ W, const float *__restrict__ ws,
                                                      float *__restrict__ C, int64_t ldc, int M, int N, int K, int Kp,
                                                      int tilesN) {
    __shared__ float red[4][16][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5;
    const int logical = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int m0 = (logical / tilesN) * 32, n0 = (logical % tilesN) * 32;
    const int nk = Kp / 32;
    const float *arow = A + (int64_t)min(m0 + (lane & 31), M - 1) * lda + 16 * h;
    const int8_t *wb = W + ((int64_t)(n0 >> 5) * nk) * 1024 + lane * 16;

    float av[Q8W_RING][16];
    u32x4 wr[Q8W_RING];
    // chunk kc into ring slot d (kc < nk, uniform per wavefront)
    auto load = [&](int d, int kc) {
        const int k0 = 32 * kc + 16 * h;
        if (32 * kc + 32 <= K) {
            if (VEC) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4 x = *reinterpret_cast<const f32x4 *>(arow + 32 * kc + 4 * i);
                    av[d][4 * i] = x.x;
                    av[d][4 * i + 1] = x.y;
                    av[d][4 * i + 2] = x.z;
                    av[d][4 * i + 3] = x.w;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) av[d][i] = arow[32 * kc + i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float x = arow[min(32 * kc + i, K - 1 - 16 * h)];
                av[d][i] = k0 + i < K ? x : 0.0f;
            }
        }
        wr[d] = *reinterpret_cast<const u32x4 *>(wb + (int64_t)kc * 1024);
    };

    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;

#pragma unroll
    for (int d = 0; d < Q8W_RING; ++d)
        if (wave + 4 * d < nk) load(d, wave + 4 * d);
    for (int kb = wave; kb < nk; kb += 4 * Q8W_RING) {
#pragma unroll
        for (int d = 0; d < Q8W_RING; ++d) {
            const int kc = kb + 4 * d;
            if (kc >= nk) break;  // uniform per wavefront
            // this chunk's operands out of the slot, then the slot's next chunk in flight
            bf16x8 ap[3][2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                uint32_t t1[8], t2[8], t3[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) q8w_split3(av[d][8 * j + e], t1[e], t2[e], t3[e]);
                ap[0][j] = __builtin_bit_cast(bf16x8, (u32x4){q8w_pack(t1[0], t1[1]), q8w_pack(t1[2], t1[3]),
                                                              q8w_pack(t1[4], t1[5]), q8w_pack(t1[6], t1[7])});
                ap[1][j] = __builtin_bit_cast(bf16x8, (u32x4){q8w_pack(t2[0], t2[1]), q8w_pack(t2[2], t2[3]),
                                                              q8w_pack(t2[4], t2[5]), q8w_pack(t2[6], t2[7])});
                ap[2][j] = __builtin_bit_cast(bf16x8, (u32x4){q8w_pack(t3[0], t3[1]), q8w_pack(t3[2], t3[3]),
                                                              q8w_pack(t3[4], t3[5]), q8w_pack(t3[6], t3[7])});
            }
            bf16x8 wq[2];
            const uint32_t dw[4] = {wr[d].x, wr[d].y, wr[d].z, wr[d].w};
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                uint32_t x[4];
                q8w_widen4(dw[2 * j], x[0], x[1]);
                q8w_widen4(dw[2 * j + 1], x[2], x[3]);
                wq[j] = __builtin_bit_cast(bf16x8, (u32x4){x[0], x[1], x[2], x[3]});
            }
            if (kc + 4 * Q8W_RING < nk) load(d, kc + 4 * Q8W_RING);
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 2; q >= 0; --q) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ap[q][j], wq[j], acc, 0, 0, 0);
        }
    }

    // ---- the four partial sums, added in wavefront order; wavefront w finishes the
    // accumulator registers 4w .. 4w + 3 (rows acc_row(r, lane))
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave][r][lane] = acc[r];
    __syncthreads();
    const int n = n0 + (lane & 31);
    const float s = ws[min(n, N - 1)];
    if (n >= N) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 4 * wave + i;
        const float v = ((red[0][r][lane] + red[1][r][lane]) + red[2][r][lane]) + red[3][r][lane];
        const int m = m0 + acc_row(r, lane);
        if (m < M) C[(int64_t)m * ldc + n] = v * s;
    }
}

}  // namespace enchip
