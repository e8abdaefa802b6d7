// gemm_pieces.h -- the W8A8 GEMM for a few hundred to a few thousand rows: too many for the
// small-M kernels, too few for gemm_persistent.h's tiles to fill the chip.
//
// One workgroup per CM x CN piece of the output, its NW wavefronts splitting K: wavefront w
// takes the 64-deep stages w, w + NW, ..., for the whole piece. Both operands are fragment-
// major, so every load is 64 lanes x 16 contiguous bytes straight into MFMA registers: no
// LDS and no barrier in the main loop, each operand byte of a piece is loaded once, and a
// wavefront's ring of PW stages keeps its loads in flight. The exact int32 partial sums then
// meet in LDS, are added, and leave in row-major order as 16-byte stores, so the epilogue
// needs no other transpose.
//
// What bounds it: at these sizes a call is a few memory round trips long, whatever its
// arithmetic, so what counts is how many CUs take part and how few steps each wavefront
// runs one after the other. gemm_w8a8_pt's 64 x 256 tiles left most CUs idle there (96
// tiles for 512 x 3072 outputs). Measured on MI355X, per call in graph replay, outputs
// identical, pt -> pieces (us): bias only, K = 768: 64 x 768 6.4 -> 2.7, 512 x 768 6.5 ->
// 3.5, 512 x 3072 6.7 -> 5.7; K = 3072, 512 x 768 12.6 -> 4.9; K = 1536, 1024 x 384 8.5 ->
// 3.9; with the GELU, K = 768, 512 x 3072: 11.5 -> 7.0 at 7% erf tails and 21.2 -> 7.8 at
// 25%. (Rings of 3 stages, 8 wavefronts and 64 x 128 pieces were no faster.)
//
// Numerics are gemm_w8a8's (kernels.h): the int32 dot is exact in any order and the epilogue
// rounds in the reference's order, so the outputs are the same bits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_persistent.h"
#include "kernels.h"

#pragma clang fp contract(off)

namespace enchip {

constexpr int PC_BK = 64;  // K stage of one wavefront: two 32-deep MFMA steps

// GELUF32 of NG x 4 dequantized values per lane, in place in the wavefront's own LDS cells
// (cell4(i): the int4 cell of the lane's group i): the series branch for all, the values
// off it gathered into a wave-wide list (slot(e): list cell e, NG * 256 of them) and
// evaluated 64 at a time, two rounds interleaved. The same bits as gelu_f32 on each value.
template <int NG, typename Cell, typename Slot>
__device__ __forceinline__ void gelu_cells(int lane, const f32x4v (&y)[NG], int *base, Cell cell4, Slot slot, int4 (&v)[NG]) {
    static_assert(4 * NG <= 32, "one bit per value");
    uint32_t tail_mask = 0;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        uint32_t t4;
        const f32x4v gy = gelu_f32_series4(y[i], t4);
        v[i] = make_int4(__float_as_int(t4 & 1u ? y[i].x : gy.x), __float_as_int(t4 & 2u ? y[i].y : gy.y),
                         __float_as_int(t4 & 4u ? y[i].z : gy.z), __float_as_int(t4 & 8u ? y[i].w : gy.w));
        tail_mask |= t4 << (4 * i);
    }
    const int cnt = __builtin_popcount(tail_mask);  // up to 4 * NG: prefix sum bit by bit over ballots
    int excl = 0, total = 0;
#pragma unroll
    for (int b = 0; (1 << b) <= 4 * NG; ++b) {
        const uint64_t bm = __builtin_amdgcn_ballot_w64((cnt >> b) & 1);
        excl += (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u)) << b;
        total += __builtin_popcountll(bm) << b;
    }
    if (total == 0) return;  // uniform
#pragma unroll
    for (int i = 0; i < NG; ++i) *reinterpret_cast<int4 *>(base + cell4(i)) = v[i];
    int pos = excl;
    for (uint32_t m = tail_mask; m != 0u; m &= m - 1u, ++pos) {
        const int b = __builtin_ctz(m);
        *slot(pos) = (uint16_t)(cell4(b >> 2) + (b & 3));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int e = lane; e < total; e += 128) {
        const int i0 = *slot(e), i1 = *slot(min(e + 64, total - 1));
        const float g0 = gelu_f32_offseries(__int_as_float(base[i0]));
        const float g1 = gelu_f32_offseries(__int_as_float(base[i1]));
        base[i0] = __float_as_int(g0);
        if (e + 64 < total) base[i1] = __float_as_int(g1);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int i = 0; i < NG; ++i) v[i] = *reinterpret_cast<const int4 *>(base + cell4(i));
}

// The piece at rows m0.., columns n0... A is fragment-major at pitch Kp and read up to row
// m0 + CM - 1 (its buffer holds them: CM divides 128), the weights up to column n0 + CN - 1
// of their padded Np. VEC: N and ldo are multiples of 4 and out is 16-byte aligned.
template <int CM, int CN, int NW, int PW, int EPI, bool VEC>
__device__ __forceinline__ void w8a8_piece(const int8_t *__restrict__ A, const int8_t *__restrict__ Wf,
                                           const float *__restrict__ aS, const float *__restrict__ wS,
                                           const float *__restrict__ bias, void *__restrict__ out, int64_t ldo, int M,
                                           int N, int Kp, int m0, int n0) {
    constexpr int TM = CM / 32, TN = CN / 32, NT = 64 * NW;
    constexpr int P = CN + 8;             // LDS row pitch in ints: rows 4 apart start 32 banks apart
    constexpr int RL = CN / 4;            // 16-byte groups per row
    constexpr int ITEMS = CM * RL;        // 16-byte groups of the piece
    constexpr int NG = (ITEMS + NT - 1) / NT, RP = NT / RL;  // groups per thread; rows per pass
    static_assert(ITEMS % NT == 0 || ITEMS < NT, "whole passes, or one");
    static_assert((64 / RL) * P * 2 >= 256, "a pass's tail list fits the wavefront's rows of one partial sum");
    static_assert(NW >= 2, "the tail list lives in the second partial sum");
    __shared__ __attribute__((aligned(16))) int red[NW][CM * P];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nst = Kp / PC_BK, nk32 = Kp >> 5;
    const int8_t *ap[TM], *wp[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) ap[i] = A + (int64_t)(m0 / 32 + i) * nk32 * 1024 + lane * 16;
#pragma unroll
    for (int j = 0; j < TN; ++j) wp[j] = Wf + (int64_t)(n0 / 32 + j) * nk32 * 1024 + lane * 16;

    i32x4 a[PW][2][TM], w[PW][2][TN];
    auto load = [&](int slot, int s) {  // this wavefront's s-th stage
        const int64_t k32 = 2 * (int64_t)(wave + s * NW);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int i = 0; i < TM; ++i) a[slot][kb][i] = *reinterpret_cast<const i32x4 *>(ap[i] + (k32 + kb) * 1024);
#pragma unroll
            for (int j = 0; j < TN; ++j) w[slot][kb][j] = *reinterpret_cast<const i32x4 *>(wp[j] + (k32 + kb) * 1024);
        }
    };
    i32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
    auto mul = [&](int slot) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[slot][kb][i], w[slot][kb][j], acc[i][j], 0, 0, 0);
    };
    const int ns = nst > wave ? (nst - wave + NW - 1) / NW : 0;  // uniform
    if (ns > 0) {
        // the first PW stages (past the last one: the last again, not multiplied)
#pragma unroll
        for (int d = 0; d < PW; ++d) load(d, min(d, ns - 1));
        int s = 0;
        for (; s + 2 * PW <= ns; s += PW) {
#pragma unroll
            for (int d = 0; d < PW; ++d) {
                mul(d);
                load(d, s + PW + d);
            }
        }
#pragma unroll
        for (int d = 0; d < PW; ++d)
            if (s + d < ns) {
                mul(d);
                if (s + PW + d < ns) load(d, s + PW + d);
            }
#pragma unroll
        for (int d = 0; d < PW; ++d)
            if (s + PW + d < ns) mul(d);
    }

    // this thread's outputs: group tid % RL of rows tid / RL + RP * i; their constants are
    // loaded before the barrier
    const int c4 = 4 * (tid % RL), r0 = tid / RL, col = n0 + c4;
    const bool mine = ITEMS >= NT || tid < ITEMS;
    float as[NG], ws[4], bb[4];
#pragma unroll
    for (int i = 0; i < NG; ++i) as[i] = EPI == EPI_I32 ? 0.0f : aS[min(m0 + r0 + RP * i, M - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        ws[u] = EPI == EPI_I32 ? 0.0f : wS[min(col + u, N - 1)];
        bb[u] = EPI == EPI_I32 || bias == nullptr ? kNoBias : bias[min(col + u, N - 1)];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) red[wave][(32 * i + acc_row(r, lane)) * P + 32 * j + (lane & 31)] = acc[i][j][r];
    __syncthreads();
    if (!mine) return;  // whole wavefronts
    int4 v[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int at = (r0 + RP * i) * P + c4;
        int4 t = *reinterpret_cast<const int4 *>(&red[0][at]);
#pragma unroll
        for (int k = 1; k < NW; ++k) {
            const int4 o = *reinterpret_cast<const int4 *>(&red[k][at]);
            t.x += o.x, t.y += o.y, t.z += o.z, t.w += o.w;
        }
        v[i] = t;
    }
    if constexpr (EPI != EPI_I32) {
        f32x4v y[NG];
#pragma unroll
        for (int i = 0; i < NG; ++i)
            y[i] = f32x4v{dequant(v[i].x, as[i], ws[0], bb[0]), dequant(v[i].y, as[i], ws[1], bb[1]),
                          dequant(v[i].z, as[i], ws[2], bb[2]), dequant(v[i].w, as[i], ws[3], bb[3])};
        if constexpr (EPI == EPI_F32_GELU) {
            // rows RP * i + wave * 64 / RL .. of the partial sums were read by this wavefront alone
            const int wrow = wave * (64 / RL);
            gelu_cells<NG>(
                lane, y, red[0], [&](int i) { return (r0 + RP * i) * P + c4; },
                [&](int e) { return reinterpret_cast<uint16_t *>(&red[1][(wrow + RP * (e >> 8)) * P]) + (e & 255); }, v);
        } else {
#pragma unroll
            for (int i = 0; i < NG; ++i)
                v[i] = make_int4(__float_as_int(y[i].x), __float_as_int(y[i].y), __float_as_int(y[i].z), __float_as_int(y[i].w));
        }
    }
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int row = m0 + r0 + RP * i;
        if (row >= M) continue;
        int *o = reinterpret_cast<int *>(out) + (int64_t)row * ldo + col;
        if (VEC) {
            if (col < N) *reinterpret_cast<int4 *>(o) = v[i];
        } else {
            const int t[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (col + u < N) o[u] = t[u];
        }
    }
}

// The 64-row form of gemm_w8a8_pt with its BM x BN tiles cut into CM x CN pieces, one
// workgroup each (its preconditions: 16-byte row-major output stores, fragment-major A).
// Pieces of one 64-row band are consecutive, rows first, so a band's A and each group of
// weight columns are shared on one XCD.
template <int BM, int BN, int BK, int PW, int EPI, bool AF, int NW, int PRIO, int CM, int CN>
__global__ __launch_bounds__(64 * NW, 2) void gemm_w8a8_pt(const int8_t *__restrict__ A, const int8_t *__restrict__ Wf,
                                                           const float *__restrict__ aS, const float *__restrict__ wS,
                                                           const float *__restrict__ bias, void *__restrict__ out,
                                                           int64_t ldo, int M, int N, int Kp, int piecesN) {
    static_assert(AF && BK == PC_BK && BM % CM == 0 && BN % CN == 0 && PRIO == 0, "pieces of the fragment-major tile");
    const int l = xcd_logical_tile(blockIdx.x, gridDim.x), band = l / (piecesN * (BM / CM)), p = l % (piecesN * (BM / CM));
    const int m0 = band * BM + (p % (BM / CM)) * CM, n0 = (p / (BM / CM)) * CN;
    if (m0 >= M) return;
    w8a8_piece<CM, CN, NW, PW, EPI, true>(A, Wf, aS, wS, bias, out, ldo, M, N, Kp, m0, n0);
}

// The same pieces for outputs that gemm_w8a8_pt cannot store (N not a multiple of 4, an
// unaligned out) or whose K it cannot walk (an odd number of stages): any N and alignment.
template <int CM, int CN, int EPI, int NW, int PW>
__global__ __launch_bounds__(64 * NW, 2) void gemm_w8a8(const int8_t *__restrict__ A, const int8_t *__restrict__ Wf,
                                                        const float *__restrict__ aS, const float *__restrict__ wS,
                                                        const float *__restrict__ bias, void *__restrict__ out,
                                                        int64_t ldo, int M, int N, int Kp, int piecesN) {
    const int l = xcd_logical_tile(blockIdx.x, gridDim.x);
    w8a8_piece<CM, CN, NW, PW, EPI, false>(A, Wf, aS, wS, bias, out, ldo, M, N, Kp, (l / piecesN) * CM, (l % piecesN) * CN);
}

}  // namespace enchip
