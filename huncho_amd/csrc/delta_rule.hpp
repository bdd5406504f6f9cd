// delta_rule.hpp - the fp32 chunk computations that delta_rule.hip and delta_rule_split.hip share.
#pragma once
#include "common.hpp"
#include "kernel_args.hpp"

namespace hk {

constexpr int CH = 64;
constexpr int DK = 128;
constexpr int DV = 128;

// Inclusive prefix sum over the 64 lanes of a wave.
__device__ __forceinline__ float wave_incl_scan(float x, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        float y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    return x;
}

// 16x16 fp32 tiles on v_mfma_f32_16x16x4_f32: operand lane l holds row/column l % 16 and
// reduction index l / 16; accumulator lane l holds column l % 16, rows (l / 16) * 4 + j.
__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// D = X[16][K] . Y[K][16] from fp32 LDS tiles (K a multiple of 4).
__device__ __forceinline__ f32x4 tile16_mm(const float* X, int ldx, const float* Y, int ldy, int K, int lane) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    const int r = lane & 15, kq = lane >> 4;
    for (int k = 0; k < K; k += 4) acc = mfma16(X[r * ldx + k + kq], Y[(k + kq) * ldy + r], acc);
    return acc;
}

// D = -W[16][16] . Xacc where Xacc is a 16x16 accumulator tile: the reduction index of
// step j is paired with the accumulator row 4 * (l / 16) + j the lane already holds.
__device__ __forceinline__ f32x4 tile16_neg_mm_acc(const float* W, int ldw, f32x4 xacc, int lane) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    const int r = lane & 15, kq = lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = mfma16(-W[r * ldw + 4 * kq + j], xacc[j], acc);
    return acc;
}

__device__ __forceinline__ void tile16_store(float* D, int ldd, f32x4 acc, int lane) {
    const int c = lane & 15, r0 = (lane >> 4) * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) D[(r0 + j) * ldd + c] = acc[j];
}

// T = (I + A)^-1 for strictly lower A [64][lda] (fp32, LDS), all 4 waves, blocked:
//   1. wave w inverts the unit-lower diagonal block w (16x16) by forward substitution;
//   2. T[1][0] = -T11 A10 T00 and T[3][2] = -T33 A32 T22 (16 -> 32);
//   3. T[2:4][0:2] = -T[2:4][2:4] A[2:4][0:2] T[0:2][0:2] (32 -> 64), one 16x16 tile per wave.
// T is written to Tf [64][lda] with its upper triangle zeroed; Xs is a [32][ldx] scratch.
// Contains __syncthreads(): every thread of the workgroup must call it.
__device__ __forceinline__ void invert_unit_lower(const float* Am, float* Tf, int lda, float* Xs, int ldx, int wave, int lane) {
    {
        const int b = wave * 16;
        if (lane < 16) {
            float x[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float acc = (i == lane) ? 1.0f : 0.0f;
                const float* row = Am + (b + i) * lda + b;
#pragma unroll
                for (int k = 0; k < i; ++k) acc -= row[k] * x[k];
                x[i] = acc;
                Tf[(b + i) * lda + b + lane] = acc;
            }
        }
        // zero the blocks right of the diagonal in this block row
        for (int idx = lane; idx < 16 * (48 - b); idx += 64) {
            const int i = idx / (48 - b), j = idx % (48 - b);
            Tf[(b + i) * lda + b + 16 + j] = 0.0f;
        }
    }
    __syncthreads();
    if (wave < 2) {
        const int b = wave * 32;  // diagonal 32-block: [b, b+32)
        f32x4 x = tile16_mm(Am + (b + 16) * lda + b, lda, Tf + b * lda + b, lda, 16, lane);
        f32x4 t = tile16_neg_mm_acc(Tf + (b + 16) * lda + b + 16, lda, x, lane);
        tile16_store(Tf + (b + 16) * lda + b, lda, t, lane);
    }
    __syncthreads();
    {
        const int rt = wave >> 1, ct = wave & 1;
        f32x4 x = tile16_mm(Am + (32 + 16 * rt) * lda, lda, Tf + 16 * ct, lda, 32, lane);
        tile16_store(Xs + 16 * rt * ldx + 16 * ct, ldx, x, lane);
    }
    __syncthreads();
    {
        const int rt = wave >> 1, ct = wave & 1;
        f32x4 t = tile16_mm(Tf + (32 + 16 * rt) * lda + 32, lda, Xs + 16 * ct, ldx, 32, lane);
        t = -t;
        tile16_store(Tf + (32 + 16 * rt) * lda + 16 * ct, lda, t, lane);
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// fp32 variant
// ---------------------------------------------------------------------------
constexpr int F_KSTR = DK + 4;  // fp32 row stride of Kc/Qc
constexpr int F_ASTR = CH + 4;  // fp32 row stride of A/T and Aqk
constexpr int XSTR = 32 + 4;    // fp32 row stride of the inversion scratch
constexpr size_t GDN_F32_LDS = sizeof(float) * (2 * CH * F_KSTR + 3 * CH * F_ASTR + 32 * XSTR + 2 * CH);

// A and Aqk of a chunk [64][F_ASTR] from its q and k tiles
__device__ __forceinline__ void chunk_matrices_f32(const float* Qc, const float* Kc, const float* Gs, const float* Bs, float* Am,
                                                   float* Aq, int wave, int lane) {
    const int g = lane >> 5, col = lane & 31;
    // A (strictly lower, beta and decay folded in) and Aqk (lower incl. diagonal)
    if (wave < 3) {
        const int tb = wave == 0 ? 0 : 1, sb = wave == 2 ? 1 : 0;
        f32x16 kk = f32x16{}, qk = f32x16{};
        const float* ka = Kc + (tb * 32 + col) * F_KSTR + 2 * g;
        const float* qa = Qc + (tb * 32 + col) * F_KSTR + 2 * g;
        const float* kbp = Kc + (sb * 32 + col) * F_KSTR + 2 * g;
#pragma unroll 8
        for (int u = 0; u < 32; ++u) {
            f32x2 av = *(const f32x2*)(ka + 4 * u);
            f32x2 qv = *(const f32x2*)(qa + 4 * u);
            f32x2 bv = *(const f32x2*)(kbp + 4 * u);
            kk = mfma_f32(av[0], bv[0], kk);
            kk = mfma_f32(av[1], bv[1], kk);
            qk = mfma_f32(qv[0], bv[0], qk);
            qk = mfma_f32(qv[1], bv[1], qk);
        }
        const int s = sb * 32 + col;
        const float Gs_s = Gs[s];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int t = tb * 32 + acc_row(j, g);
            const float dec = s <= t ? __expf(Gs[t] - Gs_s) : 0.0f;
            Am[t * F_ASTR + s] = s < t ? Bs[t] * dec * kk[j] : 0.0f;
            Aq[t * F_ASTR + s] = s <= t ? dec * qk[j] : 0.0f;
        }
    } else {
        for (int idx = lane; idx < 32 * 32; idx += 64) {
            const int t = idx >> 5, s = 32 + (idx & 31);
            Am[t * F_ASTR + s] = 0.0f;
            Aq[t * F_ASTR + s] = 0.0f;
        }
    }
}

}  // namespace hk
