// gemm_f32.h -- f32 C = A . B^T on the gfx950 bf16 MFMA: the device side of
// encoder.Backend.MatmulBT (encoder/backend.go:19-28), used by attention for
// QK^T = qH . kH^T and scores . V = scores . (vHT)^T (encoder/attention.go:108,111).
//
// Batched and strided over two levels: problem (y, z) of a launch reads
// A + y*sa + z*sa2, B + y*sb + z*sb2 and writes C + y*sc + z*sc2, so one launch covers
// every (head, sequence) of a layer, each head read in place from the interleaved
// [L, D] activations (lda = D or 3D) with no extraction copy.
// B is [N, K] rows (MatmulBT's b, BKN = false) or [K, N] rows (BKN = true: V itself
// for scores . V, element (n, k) at B[k*ldb + n], so no transpose copy either).
//
// Arithmetic. Every operand value is split into three bf16 parts, x = h + m + l (h
// the bf16 nearest x, m the one nearest x - h, l the rest, which has at most 8 bits), and a
// product is six products of parts: h.h', h.m', m.h', m.m', h.l', l.h', each exact on
// v_mfma_f32_32x32x16_bf16 and summed in f32. The three left out, m.l', l.m' and l.l', come to at
// most 2^-24 |x y| (|m| <= 2^-8 |x|, |l| <= 2^-17 |x|; typically under 2^-26), what rounding the
// product once costs, and a 16-deep step rounds the sum 6 times where the f32 MFMA (32x32x2) rounds
// it 8 to 16 times.
// Measured against float64 (standard normal operands, relative 2-norm): K = 768 4.2e-7, or
// 2.1e-7 with K split over wavefronts, against the f32 MFMA's 5.0e-7; K = 3072 8.7e-7 /
// 4.3e-7 against 9.9e-7. The contract is the reference's gate against a float64 dot product
// (gpu/enccuda/backend_test.go:47-86).
// The split is exact for operands from 2^-110 up (bf16 subnormals are kept, in the conversions and
// in the MFMA). Outputs that can have lost by smaller ones are computed again on the f32 MFMA (see
// kBelow): with |a| near 2^-120 and |b| near 2^120 the worst relative error was 1.1e-5 without,
// 3.9e-7 with, as on the f32 MFMA throughout. The looking costs up to 3%: 4096 x 768, K = 768 40.0 ->
// 41.3 us, 512 x 3072 25.4 -> 26.0, 4096 x 3072, K = 3072 391 -> 395, K-split shapes none.
// An operand the split cannot hold (an infinity, or a value that rounds to one in bf16) or a
// sum that overflows leaves a non-finite output; those are computed again by f32_blocks on the f32
// MFMA, so infinities and overflow give what f32 arithmetic gives. The other outputs of the block
// keep their split sums.
//
// bf16 products run at 16 times the f32 MFMA's rate, so the six cost 0.38 of it; the f32
// kernel these replace reached 110-120 of its 154 TFLOP/s at 4096^2 and less than a third of
// that where its 128 x 128 tiles left CUs idle. Two forms, one result per shape:
//   gemm_f32_tile  block tiles with the parts staged in LDS;
//   gemm_f32_ksplit  K split over the wavefronts of small tiles, for shapes with so few
//                  tiles that the serial K loop is the time.
// The choice between them depends on M, N and K alone, and each gives the same bits for any
// tile size, batch, pitch, alignment and layout of the same operands.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"

#pragma clang fp contract(off)

namespace enchip {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Batch strides of one level (in floats).
struct F32Strides {
    int64_t a, b, c;
};

// A workgroup barrier that orders LDS accesses only: global loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The three bf16 parts of a (low half) and b (high half of each word); big: the largest magnitude
// so far.
__device__ __forceinline__ void split3_pair(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l, float &big) {
    big = fmaxf(fmaxf(fabsf(a), fabsf(b)), big);  // one v_max3
    h = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
    const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
    m = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{ra, rb}), bf16x2));
    const float sa = ra - __uint_as_float(m << 16), sb = rb - __uint_as_float(m & 0xffff0000u);
    l = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{sa, sb}), bf16x2));
}

// acc += the six products of one 16-deep step, smallest first; p[.][0..2] = h, m, l.
template <int TM, int TN>
__device__ __forceinline__ void mfma_parts(const bf16x8 (&pa)[TM][3], const bf16x8 (&pb)[TN][3], f32x16 (&acc)[TM][TN]) {
    constexpr int pi[6] = {2, 0, 1, 1, 0, 0}, qi[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int u = 0; u < 6; ++u)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int t = 0; t < TN; ++t)
                acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pa[i][pi[u]], pb[t][qi[u]], acc[i][t], 0, 0, 0);
}

// Where the parts are not the operand. bf16's last bit is 2^-133, so a nonzero operand under
// 2^-110 (kBelow, of the word below_split gives; zeros give the largest) may lose up to 2^-134. A
// sum of K products with every operand at most kBig then lost at most 2 K 2^-134 kBig = K 2^-109,
// under 2^-25 of any output from lost_below(K) up. So the main loop only looks for operands above
// kBig, and the end for outputs below that (zeros, as a rule): blocks with either have their
// operands searched for small ones, and f32_blocks computes the outputs that can have lost by it.
// (Looking for the small ones in the main loop cost up to 12%.)
constexpr uint32_t kBelow = ((127u - 110u) << 24) - 1u;
constexpr float kBig = 0x1p24f;
__device__ __forceinline__ uint32_t below_split(float x) { return (__float_as_uint(x) << 1) - 1u; }
__device__ __forceinline__ float lost_below(int K) { return (float)K * 0x1p-84f; }

// Whether any of the lane's outputs is infinite or NaN, and their smallest magnitude.
template <int TM, int TN>
__device__ __forceinline__ bool any_nonfinite(const f32x16 (&acc)[TM][TN], float &least) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                s = __builtin_fmaf(acc[i][t][e], 0.0f, s);
                least = fminf(fabsf(acc[i][t][e]), least);
            }
    return s != 0.0f;  // 0, or NaN
}

// For up to 32 rows of n values (row i at p + i * pitch, value k at k * step; those in mask), by one
// wavefront: which hold a nonzero value, one under 2^-110, one above kBig. Four rows at a time, for
// the loads in flight.
struct RowMarks {
    uint32_t live, small, big;
};
__device__ __forceinline__ RowMarks row_marks(const float *p, int64_t pitch, int64_t step, int n, uint32_t mask) {
    constexpr int R = 4, U = 4;
    const int lane = threadIdx.x & 63;
    RowMarks marks{0, 0, 0};
    while (mask != 0) {  // uniform
        int row[R];
        float most[R];
        uint32_t low[R];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            row[q] = __builtin_ctz(mask);
            if ((mask & (mask - 1)) != 0 || q == R - 1) mask &= mask - 1;  // else the last row again
            most[q] = 0.0f, low[q] = ~0u;
        }
        for (int k0 = 0; k0 < n; k0 += 64 * U) {
            float x[R][U];
#pragma unroll
            for (int q = 0; q < R; ++q)
#pragma unroll
                for (int u = 0; u < U; ++u) x[q][u] = p[row[q] * pitch + min(k0 + 64 * u + lane, n - 1) * step];
#pragma unroll
            for (int q = 0; q < R; ++q)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    most[q] = fmaxf(fabsf(x[q][u]), most[q]);
                    low[q] = min(below_split(x[q][u]), low[q]);
                }
        }
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const uint32_t bit = 1u << row[q];
            if (__builtin_amdgcn_ballot_w64(most[q] > 0.0f) != 0) marks.live |= bit;
            if (__builtin_amdgcn_ballot_w64(low[q] < kBelow) != 0) marks.small |= bit;
            if (__builtin_amdgcn_ballot_w64(most[q] > kBig) != 0) marks.big |= bit;
        }
    }
    return marks;
}

// Of the lane's 16 outputs of a 32 x 32 block, a bit each: those not finite, those under lost_below.
struct OutMarks {
    uint32_t bad, low;
};
__device__ __forceinline__ OutMarks out_marks(const f32x16 &v, int K) {
    OutMarks o{0, 0};
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        o.bad |= (uint32_t)!(fabsf(v[e]) < INFINITY) << e;
        o.low |= (uint32_t)(fabsf(v[e]) < lost_below(K)) << e;
    }
    return o;
}

// The TN 32 x 32 outputs at (m0, n0), (m0, n0 + 32), ..., stored from split sums, by one wavefront:
// those not finite, and those that can have lost by a small operand of their row or column, are
// computed again on the f32 MFMA with operands loaded value by value. Which ones depends on each
// output's own row, column and split sum, whatever the tile. any_big: the block has an operand above
// kBig. Rows of zeros, whose outputs are under lost_below, need no search of the columns.
template <int TN, bool BKN>
__device__ __forceinline__ void f32_blocks(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int64_t ldc,
                                        int M, int N, int K, int m0, int n0, bool any_big, const OutMarks (&marks)[TN]) {
    const int lane = threadIdx.x & 63, r = lane & 31, kh = 8 * (lane >> 5);
    if (m0 >= M) return;
    uint32_t in_rows = 0, doubt[TN], rows = 0;  // doubt: the lane's outputs that can have lost; rows: with any
#pragma unroll
    for (int e = 0; e < 16; ++e) in_rows |= (uint32_t)(m0 + acc_row(e, lane) < M) << e;
    uint32_t any = 0;
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        doubt[t] = n0 + 32 * t + r < N ? (any_big ? ~0u : marks[t].low) & in_rows : 0;
        any |= doubt[t];
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const uint64_t b = __builtin_amdgcn_ballot_w64((any >> e) & 1);
        rows |= (uint32_t)((uint32_t)b != 0) << acc_row(e, 0) | (uint32_t)((b >> 32) != 0) << acc_row(e, 32);
    }
    const RowMarks ra = row_marks(A + (int64_t)m0 * lda, lda, 1, K, rows);
#pragma unroll 1
    for (int t = 0; t < TN; ++t, n0 += 32) {
        uint32_t dt = doubt[0], low = marks[0].low, redo = marks[0].bad;
#pragma unroll
        for (int u = 1; u < TN; ++u)
            if (t == u) dt = doubt[u], low = marks[u].low, redo = marks[u].bad;
        redo &= n0 + r < N ? in_rows : 0;
        bool col = false;
#pragma unroll
        for (int e = 0; e < 16; ++e) col |= ((dt >> e) & (ra.live >> acc_row(e, lane)) & 1) != 0;
        if (__builtin_amdgcn_ballot_w64(col || redo != 0) == 0) continue;
        const uint64_t cb = __builtin_amdgcn_ballot_w64(col);
        const RowMarks rb = BKN ? row_marks(B + n0, 1, ldb, K, (uint32_t)cb | (uint32_t)(cb >> 32))
                                : row_marks(B + (int64_t)n0 * ldb, ldb, 1, K, (uint32_t)cb | (uint32_t)(cb >> 32));
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int at = acc_row(e, lane);
            const uint32_t small = ra.small >> at | rb.small >> r, big = ra.big >> at | rb.big >> r;
            redo |= (dt >> e & small & (low >> e | big) & 1) << e;
        }
        if (__builtin_amdgcn_ballot_w64(redo != 0) == 0) continue;
        const float *pa = A + (int64_t)min(m0 + r, M - 1) * lda;
        const int n = min(n0 + r, N - 1);
        f32x16 acc;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
        for (int k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int k = k0 + kh + s, kc = min(k, K - 1);
                const float a = pa[kc], b = BKN ? B[(int64_t)kc * ldb + n] : B[(int64_t)n * ldb + kc];
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(k < K ? a : 0.0f, k < K ? b : 0.0f, acc, 0, 0, 0);
            }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e)
            if ((redo >> e) & 1) C[(int64_t)(m0 + acc_row(e, lane)) * ldc + n0 + r] = acc[e];
    }
}

// Block tile (32 TM WM) x (32 TN WN), WM x WN wavefronts of TM x TN 32 x 32 accumulators, K in
// chunks of KC through two LDS stages. Every thread loads 16-byte pieces of the operands'
// rows, splits them into the three parts and stores those as planes of [row][KC] bf16; each
// operand value is split once per block and read back as 16-byte MFMA operands.
// What bounds it: at 4096 x 3072 x 3072 the MFMA, 400 us = 1.16 PFLOP/s of bf16 products (the
// f32 MFMA kernel took 637); with one block per CU the serial latency of a chunk (load, split,
// LDS round trip, MFMAs), which is why few tiles take deep chunks and 8 wavefronts: 512 x 3072,
// K = 768 in 64 x 128 tiles 22.9 us with 8 wavefronts and KC = 32, 25.8 with 4, 27.6 at KC =
// 16. Loads two or three chunks ahead and MFMAs interleaved with the split by hand gained
// nothing. Batched 512 x 64 x 512 over 384 heads: 168 -> 153 us, its f32 output's stores.
// VEC: K, pitches and strides multiples of 4, 16-byte aligned operands, and N % 4 == 0 for
// BKN; otherwise values are loaded one by one.
template <int TM, int TN, int WM, int WN, int KC, bool BKN, bool VEC>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_f32_tile(
    const float *__restrict__ A, int64_t lda, const float *__restrict__ B, int64_t ldb, float *__restrict__ C,
    int64_t ldc, F32Strides s1, F32Strides s2, int M, int N, int K, int tilesN) {
    constexpr int NT = 64 * WM * WN, BM = 32 * TM * WM, BN = 32 * TN * WN;
    constexpr int P = 2 * KC + 16;                // LDS bytes per row of a plane: 16-byte groups of 16 rows in distinct banks
    constexpr int PLA = BM * P, PLB = BN * P, STAGE = 3 * (PLA + PLB);
    constexpr int AV = BM * KC / 4 / NT;          // float4 per thread per chunk
    constexpr int KNI = (KC / 2) * (BN / 4);      // KN: (k pair, 4 columns) items of a chunk
    constexpr int BV = BKN ? 2 * ((KNI + NT - 1) / NT) : BN * KC / 4 / NT;
    static_assert(AV >= 1 && BV >= 1 && (KNI % NT == 0 || KNI < NT) && STAGE * 2 <= 128 * 1024, "tile");
    const bool kn_mine = KNI >= NT || (int)threadIdx.x < KNI;
    __shared__ __attribute__((aligned(16))) char lds[2 * STAGE];
    __shared__ int any_big;  // the block has an operand above kBig
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 31, hf = lane >> 5;
    if (tid == 0) any_big = 0;
    const int64_t y = blockIdx.y, z = blockIdx.z;
    A += y * s1.a + z * s2.a;
    B += y * s1.b + z * s2.b;
    C += y * s1.c + z * s2.c;
    const int logical = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int bm0 = (logical / tilesN) * BM, bn0 = (logical % tilesN) * BN;
    const int wm = wave / WN, wn = wave % WN;

    // Loader: KC / 4 consecutive threads per row, 16 bytes each, so rows are read in whole
    // KC * 4-byte runs. KN: thread items of two k rows x 4 columns, 4 items side by side.
    constexpr int LPR = KC / 4;
    const int lk = 4 * (tid % LPR), lr = tid / LPR;
    const float *ga[AV], *gb[BV];
#pragma unroll
    for (int i = 0; i < AV; ++i) ga[i] = A + (int64_t)min(bm0 + lr + (NT / LPR) * i, M - 1) * lda;
    // KN items: k pair pk, columns 4 pg ..
    constexpr int NPAIR = KC / 2;
    const int pk = (tid / 4) % NPAIR;
    auto pg = [&](int i) { return min(tid % 4 + 4 * ((tid / 4 + (NT / 4) * i) / NPAIR), BN / 4 - 1); };
#pragma unroll
    for (int i = 0; i < BV; ++i) {
        if (BKN) gb[i] = i < BV / 2 ? B + (VEC ? min(bn0 + 4 * pg(i), N - 4) : 0) : nullptr;
        else gb[i] = B + (int64_t)min(bn0 + lr + (NT / LPR) * i, N - 1) * ldb;
    }
    f32x4 ra[AV], rb[BV];
    float big = 0.0f;
    auto load_row = [&](const float *p, int k) -> f32x4 {
        if (VEC) return *reinterpret_cast<const f32x4 *>(p + min(k, K - 4));
        return f32x4{p[min(k, K - 1)], p[min(k + 1, K - 1)], p[min(k + 2, K - 1)], p[min(k + 3, K - 1)]};
    };
    auto load = [&](int c) {
        const int k = KC * c + lk;
#pragma unroll
        for (int i = 0; i < AV; ++i) ra[i] = load_row(ga[i], k);
        if (BKN) {
#pragma unroll
            for (int i = 0; i < BV / 2; ++i)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int64_t kr = (int64_t)min(KC * c + 2 * pk + u, K - 1) * ldb;
                    if (VEC) rb[2 * i + u] = *reinterpret_cast<const f32x4 *>(gb[i] + kr);
                    else {
                        const int n = bn0 + 4 * pg(i);
                        rb[2 * i + u] = f32x4{B[kr + min(n, N - 1)], B[kr + min(n + 1, N - 1)], B[kr + min(n + 2, N - 1)],
                                                    B[kr + min(n + 3, N - 1)]};
                    }
                }
        } else {
#pragma unroll
            for (int i = 0; i < BV; ++i) rb[i] = load_row(gb[i], k);
        }
    };
    auto put_row = [&](char *plane, int stride, int row, f32x4 v, int k) {
        // k >= K counts as zero
        if (VEC) {
            if (k >= K) v = f32x4{0.f, 0.f, 0.f, 0.f};
        } else {
            v.x = k < K ? v.x : 0.f, v.y = k + 1 < K ? v.y : 0.f, v.z = k + 2 < K ? v.z : 0.f, v.w = k + 3 < K ? v.w : 0.f;
        }
        uint32_t h0, m0, l0, h1, m1, l1;
        split3_pair(v.x, v.y, h0, m0, l0, big);
        split3_pair(v.z, v.w, h1, m1, l1, big);
        char *d = plane + row * P + 2 * lk;
        *reinterpret_cast<uint2 *>(d) = make_uint2(h0, h1);
        *reinterpret_cast<uint2 *>(d + stride) = make_uint2(m0, m1);
        *reinterpret_cast<uint2 *>(d + 2 * stride) = make_uint2(l0, l1);
    };
    auto store = [&](int c, char *st) {
#pragma unroll
        for (int i = 0; i < AV; ++i) put_row(st, PLA, lr + (NT / LPR) * i, ra[i], KC * c + lk);
        char *bp = st + 3 * PLA;
        if (BKN) {
#pragma unroll
            for (int i = 0; i < BV / 2; ++i) {
                if (!kn_mine) continue;
                f32x4 u = rb[2 * i], w = rb[2 * i + 1];
                const int k = KC * c + 2 * pk;
                if (k >= K) u = f32x4{0.f, 0.f, 0.f, 0.f};
                if (k + 1 >= K) w = f32x4{0.f, 0.f, 0.f, 0.f};
                const float uu[4] = {u.x, u.y, u.z, u.w}, ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t h, m, l;
                    split3_pair(uu[e], ww[e], h, m, l, big);
                    char *d = bp + (4 * pg(i) + e) * P + 4 * pk;
                    *reinterpret_cast<uint32_t *>(d) = h;
                    *reinterpret_cast<uint32_t *>(d + PLB) = m;
                    *reinterpret_cast<uint32_t *>(d + 2 * PLB) = l;
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < BV; ++i) put_row(bp, PLB, lr + (NT / LPR) * i, rb[i], KC * c + lk);
        }
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][t][e] = 0.0f;
    // Chunk c + 1 is split into the other stage while chunk c's MFMAs run, and its registers
    // take chunk c + 2. Past the last chunk the loads re-read it and the stage is not used: no
    // branch, so that all of an iteration is scheduled together.
    const int nc = (K + KC - 1) / KC, last = nc - 1;
    load(0);
    store(0, lds);
    load(min(1, last));
    lds_barrier();
    for (int c = 0; c < nc; ++c) {
        char *cur = lds + (c & 1) * STAGE, *nxt = lds + ((c & 1) ^ 1) * STAGE;
        bf16x8 pa[KC / 16][TM][3], pb[KC / 16][TN][3];
#pragma unroll
        for (int s = 0; s < KC / 16; ++s) {
            const char *ap = cur + (wm * 32 * TM + r) * P + 32 * s + 16 * hf;
            const char *bp = cur + 3 * PLA + (wn * 32 * TN + r) * P + 32 * s + 16 * hf;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
#pragma unroll
                for (int i = 0; i < TM; ++i) pa[s][i][q] = *reinterpret_cast<const bf16x8 *>(ap + q * PLA + 32 * i * P);
#pragma unroll
                for (int t = 0; t < TN; ++t) pb[s][t][q] = *reinterpret_cast<const bf16x8 *>(bp + q * PLB + 32 * t * P);
            }
        }
        store(c + 1, nxt);
        load(min(c + 2, last));
#pragma unroll
        for (int s = 0; s < KC / 16; ++s) mfma_parts<TM, TN>(pa[s], pb[s], acc);
        lds_barrier();
    }
    if (big > kBig) any_big = 1;
    lds_barrier();
    float least = INFINITY;
    const bool nonfinite = __builtin_amdgcn_ballot_w64(any_nonfinite<TM, TN>(acc, least)) != 0;
    const bool low = __builtin_amdgcn_ballot_w64(least < lost_below(K)) != 0;
    const int m0 = bm0 + 32 * TM * wm, n0 = bn0 + 32 * TN * wn;
    // The last loads, of a chunk already used, end here: left in flight, their registers' next use
    // waits in each store's branch, for the stores before it too (16 x 64 problems 3.6 -> 4.1 us).
#pragma unroll
    for (int i = 0; i < AV; ++i) asm volatile("" ::"v"(ra[i]));
#pragma unroll
    for (int i = 0; i < BV; ++i) asm volatile("" ::"v"(rb[i]));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            const int col = n0 + 32 * t + r;
            if (col >= N) continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + 32 * i + acc_row(e, lane);
                if (row < M) C[(int64_t)row * ldc + col] = acc[i][t][e];
            }
        }
    if (__builtin_expect(nonfinite || low || any_big != 0, 0)) {
        OutMarks marks[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int t = 0; t < TN; ++t) marks[i][t] = out_marks(acc[i][t], K);
#pragma unroll 1
        for (int i = 0; i < TM; ++i) {
            OutMarks mi[TN];
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                mi[t] = marks[0][t];
#pragma unroll
                for (int u = 1; u < TM; ++u)
                    if (i == u) mi[t] = marks[u][t];
            }
            f32_blocks<TN, BKN>(A, lda, B, ldb, C, ldc, M, N, K, m0 + 32 * i, n0, any_big != 0, mi);
        }
    }
}

// K split: 4 wavefronts per (32 TM) x (32 TN) tile, wavefront w taking the 32-deep chunks w, w +
// 4, ... Each lane loads its own MFMA operands (8 consecutive k of its row per step) and splits
// them in registers: no LDS and no barrier until the four partial sums are added in a fixed
// order. Bound by the row-per-lane loads (32 rows per instruction), so it only pays where the
// tiles are few and K is long: 128 x 768, K = 768 8.4 us against 17.8 in gemm_f32_tile's 64 x
// 64 tiles (61.5 on the f32 MFMA), 512 x 768 12.0 against 18.1, 512 x 768, K = 3072 36.8
// against 61.7; but 512 x 3072, K = 768 32.2 against 22.9. VEC as gemm_f32_tile's.
template <int TM, int TN, bool BKN, bool VEC>
__global__ __launch_bounds__(256, 2) void gemm_f32_ksplit(const float *__restrict__ A, int64_t lda,
                                                          const float *__restrict__ B, int64_t ldb, float *__restrict__ C,
                                                          int64_t ldc, F32Strides s1, F32Strides s2, int M, int N, int K,
                                                          int tilesN) {
    constexpr int WK = 4, NT = 256, BM = 32 * TM, BN = 32 * TN;
    constexpr int P = BN + 8;  // LDS row pitch: rows 4 apart start 32 banks apart
    __shared__ __attribute__((aligned(16))) float red[WK][BM * P];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t y = blockIdx.y, z = blockIdx.z;
    A += y * s1.a + z * s2.a;
    B += y * s1.b + z * s2.b;
    C += y * s1.c + z * s2.c;
    const int logical = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int m0 = (logical / tilesN) * BM, n0 = (logical % tilesN) * BN;
    const int r = lane & 31, hf = lane >> 5;

    const float *pa[TM], *pb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) pa[i] = A + (int64_t)min(m0 + 32 * i + r, M - 1) * lda;
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        const int n = min(n0 + 32 * t + r, N - 1);
        pb[t] = BKN ? B + n : B + (int64_t)n * ldb;
    }
    float ra[2][TM][8], rb[2][TN][8], big = 0.0f;
    auto load_row = [&](const float *p, int k, float (&v)[8]) {
        if (VEC) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f32x4 x = *reinterpret_cast<const f32x4 *>(p + min(k + 4 * q, K - 4));
                v[4 * q] = x.x, v[4 * q + 1] = x.y, v[4 * q + 2] = x.z, v[4 * q + 3] = x.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = p[min(k + e, K - 1)];
        }
    };
    auto load = [&](int j, int c) {  // step j of chunk c
        const int k = 32 * c + 16 * j + 8 * hf;
#pragma unroll
        for (int i = 0; i < TM; ++i) load_row(pa[i], k, ra[j][i]);
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            if (BKN) {
#pragma unroll
                for (int e = 0; e < 8; ++e) rb[j][t][e] = pb[t][(int64_t)min(k + e, K - 1) * ldb];
            } else {
                load_row(pb[t], k, rb[j][t]);
            }
        }
    };
    auto split8 = [&](const float (&x)[8], bf16x8 (&p)[3]) {
        uint32_t h[4], m[4], l[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) split3_pair(x[2 * i], x[2 * i + 1], h[i], m[i], l[i], big);
        p[0] = __builtin_bit_cast(bf16x8, (u32x4{h[0], h[1], h[2], h[3]}));
        p[1] = __builtin_bit_cast(bf16x8, (u32x4{m[0], m[1], m[2], m[3]}));
        p[2] = __builtin_bit_cast(bf16x8, (u32x4{l[0], l[1], l[2], l[3]}));
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][t][e] = 0.0f;
    const int nc = (K + 31) / 32;
    if (wave < nc) {  // uniform
        load(0, wave);
        load(1, wave);
        for (int c = wave; c < nc; c += WK) {
            const bool more = c + WK < nc;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (32 * c + 32 > K) {  // the last chunk: k past K counts as zero in both operands
                    const int k = 32 * c + 16 * j + 8 * hf;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
#pragma unroll
                        for (int i = 0; i < TM; ++i) ra[j][i][e] = k + e < K ? ra[j][i][e] : 0.0f;
#pragma unroll
                        for (int t = 0; t < TN; ++t) rb[j][t][e] = k + e < K ? rb[j][t][e] : 0.0f;
                    }
                }
                bf16x8 qa[TM][3], qb[TN][3];
#pragma unroll
                for (int i = 0; i < TM; ++i) split8(ra[j][i], qa[i]);
#pragma unroll
                for (int t = 0; t < TN; ++t) split8(rb[j][t], qb[t]);
                if (more) load(j, c + WK);
                mfma_parts<TM, TN>(qa, qb, acc);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) red[wave][(32 * i + acc_row(e, lane)) * P + 32 * t + r] = acc[i][t][e];
    __syncthreads();
    constexpr int RL = BN / 4, RP = NT / RL, NG = BM * RL / NT;  // 16-byte groups per row; rows per pass; passes
    static_assert(BM * RL % NT == 0 && WK == 4, "whole passes");
    const int c4 = 4 * (tid % RL), r0 = tid / RL, col = n0 + c4;
    const bool vst = ldc % 4 == 0 && N % 4 == 0 && ((uintptr_t)C & 15) == 0;
    float zeros = 0.0f, least = INFINITY;  // of the sums: NaN where one is not finite; the smallest
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int at = (r0 + RP * g) * P + c4, row = m0 + r0 + RP * g;
        f32x4 v = *reinterpret_cast<const f32x4 *>(&red[0][at]);
#pragma unroll
        for (int w = 1; w < WK; ++w) {
            const f32x4 o = *reinterpret_cast<const f32x4 *>(&red[w][at]);
            v.x += o.x, v.y += o.y, v.z += o.z, v.w += o.w;
        }
        const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            zeros += x[u] * 0.0f;
            least = fminf(fabsf(x[u]), least);
        }
        if (row >= M) continue;
        float *o = C + (int64_t)row * ldc + col;
        if (vst) {
            if (col < N) *reinterpret_cast<f32x4 *>(o) = v;
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (col + u < N) o[u] = x[u];
        }
    }
    if (__builtin_expect(__syncthreads_or(zeros != 0.0f || big > kBig || least < lost_below(K)), 0)) {
        const bool any_big = __syncthreads_or(big > kBig);
        for (int u = wave; u < TM * TN; u += WK) {
            const int mu = 32 * (u / TN), nu = 32 * (u % TN);
            f32x16 v;  // the sums again, each lane its f32 MFMA outputs
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int at = (mu + acc_row(e, lane)) * P + nu + r;
                v[e] = ((red[0][at] + red[1][at]) + red[2][at]) + red[3][at];
            }
            const OutMarks marks[1] = {out_marks(v, K)};
            f32_blocks<1, BKN>(A, lda, B, ldb, C, ldc, M, N, K, m0 + mu, n0 + nu, any_big, marks);
        }
    }
}

// C = 0 for a K = 0 product (the empty dot product), grid (ceil(M*N/256), inner, outer).
__global__ __launch_bounds__(256) void fill_zero_f32(float *__restrict__ C, int64_t ldc, int64_t sc1, int64_t sc2,
                                                     int M, int N) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)M * N) return;
    C[blockIdx.y * sc1 + blockIdx.z * sc2 + (i / N) * ldc + i % N] = 0.0f;
}

}  // namespace enchip
