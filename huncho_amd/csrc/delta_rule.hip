// delta_rule.hip - chunked gated delta rule (Gated DeltaNet recurrence) for gfx950.
//
// Computes exactly the reference's per-token recurrence (crates/huncho-backend/src/
// delta_cpu.rs:95-131, == qwen3_5.rs:950-987): for each token t of a sequence and head,
//   S <- S * exp(g_t);  m = S^T k_t;  delta_t = (v_t - m) * beta_t;  S <- S + k_t delta_t^T;
//   o_t = S^T q_t
// with S [dk, dv] fp32, in the algebraically equal chunked form (chunk C = 64). With
// G_t = sum_{s<=t} g_s inside a chunk and S0 the state entering it:
//   A[t,s]   = beta_t exp(G_t - G_s) (k_t . k_s)        s < t   (strictly lower)
//   T        = (I + A)^-1                              (forward substitution, fp32)
//   delta    = T [ beta * (V - exp(G) * (K S0)) ]
//   O        = exp(G) * (Q S0) + Aqk delta,  Aqk[t,s] = exp(G_t - G_s) (q_t . k_s), s <= t
//   S_next   = exp(G_last) S0 + K^T [exp(G_last - G) * delta]
// Only decay ratios exp(G_t - G_s) with t >= s (each <= 1) are formed.
//
// One workgroup = one (sequence, head); 4 waves; wave w owns value columns 32w..32w+31 of
// the state, held as four 32x32 MFMA accumulators for the whole sequence, so the state
// never leaves registers between chunks and is read/written in HBM only at the start (an
// optional initial state) and the end (the optional final state). Every intermediate
// (K S, R, delta) stays in accumulator layout and feeds the next MFMA as its B operand:
// the reduction index of each product is permuted to match the accumulator's row order
// instead of transposing the data. Inputs stream from HBM once: q, k, v, g, beta in, o out.
//
// This file holds the fp32 variant (v_mfma_f32_32x32x2_f32, the fp32 model path); the 16-bit
// variants and the fused Gated DeltaNet layer kernel live in gdn16_kernel.hpp.
#include "delta_rule.hpp"

namespace hk {

__global__ __launch_bounds__(256, 1) void gdn_chunk_f32(GdnArgs a) {
    extern __shared__ __attribute__((aligned(16))) float smem_f[];
    float* Kc = smem_f;
    float* Qc = Kc + CH * F_KSTR;
    float* Am = Qc + CH * F_KSTR;
    float* Aq = Am + CH * F_ASTR;
    float* Tf = Aq + CH * F_ASTR;
    float* Xs = Tf + CH * F_ASTR;
    float* Gs = Xs + 32 * XSTR;
    float* Bs = Gs + CH;

    const int h = blockIdx.x, seq = blockIdx.y, H = a.H;
    const int t0 = a.cu_seqlens[seq];
    const int T = a.cu_seqlens[seq + 1] - t0;
    if (t0 < 0 || T < 0 || t0 + T > a.n_tokens) {
        if (threadIdx.x == 0) atomicOr(a.fault, 1);
        return;
    }
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 5, col = lane & 31;
    const int dvc = wave * 32 + col;  // this lane's value column
    const int kh = h / a.qk_rep;
    const float* qg = (const float*)a.q + (long)kh * DK;
    const float* kg = (const float*)a.k + (long)kh * DK;
    const float* vg = (const float*)a.v + (long)h * DV;
    float* og = (float*)a.o + (long)h * DV;
    // this sequence's state rows [H][dk][dv] (per-row pointer tables or contiguous arrays)
    const float* const s0 = a.init_rows ? a.init_rows[seq]
                                        : (a.initial_state ? a.initial_state + (long)seq * H * DK * DV : nullptr);
    float* const s1 = a.final_rows ? a.final_rows[seq]
                                   : (a.final_state ? a.final_state + (long)seq * H * DK * DV : nullptr);
    const long sbase = (long)h * DK * DV;

    f32x16 S[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int j = 0; j < 16; ++j)
            S[rb][j] = s0 ? s0[sbase + (long)(rb * 32 + acc_row(j, g)) * DV + dvc] : 0.0f;

    for (int c0 = 0; c0 < T; c0 += CH) {
        const int Lc = min(CH, T - c0);
        __syncthreads();
        {
            const int t = t0 + c0;
#include "delta_rule_load.inc"
        }
        __syncthreads();
        chunk_matrices_f32(Qc, Kc, Gs, Bs, Am, Aq, wave, lane);
        __syncthreads();
        invert_unit_lower(Am, Tf, F_ASTR, Xs, XSTR, wave, lane);
        // K S0 and Q S0 for this wave's value columns
        f32x16 ks[2], qs[2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            ks[tb] = f32x16{};
            qs[tb] = f32x16{};
            const float* kr = Kc + (tb * 32 + col) * F_KSTR + g * 4;
            const float* qr = Qc + (tb * 32 + col) * F_KSTR + g * 4;
#pragma unroll
            for (int rb = 0; rb < 4; ++rb)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    f32x4 kv = *(const f32x4*)(kr + rb * 32 + jj * 8);
                    f32x4 qv = *(const f32x4*)(qr + rb * 32 + jj * 8);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        ks[tb] = mfma_f32(kv[e], S[rb][jj * 4 + e], ks[tb]);
                        qs[tb] = mfma_f32(qv[e], S[rb][jj * 4 + e], qs[tb]);
                    }
                }
        }
        // R = beta * (V - exp(G) K S0); O starts as exp(G) Q S0
        f32x16 R[2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int t = tb * 32 + acc_row(j, g);
                const float eg = __expf(Gs[t]);
                const float vv = t < Lc ? vg[(long)(t0 + c0 + t) * a.v_tok + dvc] : 0.0f;
                R[tb][j] = Bs[t] * (vv - eg * ks[tb][j]);
                qs[tb][j] *= eg;
            }
        // delta = T R
        f32x16 dl[2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            dl[tb] = f32x16{};
            const float* tr = Tf + (tb * 32 + col) * F_ASTR + g * 4;
#pragma unroll
            for (int sb = 0; sb < 2; ++sb)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    f32x4 tv = *(const f32x4*)(tr + sb * 32 + jj * 8);
#pragma unroll
                    for (int e = 0; e < 4; ++e) dl[tb] = mfma_f32(tv[e], R[sb][jj * 4 + e], dl[tb]);
                }
        }
        // O = exp(G) Q S0 + Aqk delta -> HBM
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            const float* ar = Aq + (tb * 32 + col) * F_ASTR + g * 4;
#pragma unroll
            for (int sb = 0; sb < 2; ++sb)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    f32x4 av = *(const f32x4*)(ar + sb * 32 + jj * 8);
#pragma unroll
                    for (int e = 0; e < 4; ++e) qs[tb] = mfma_f32(av[e], dl[sb][jj * 4 + e], qs[tb]);
                }
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int t = tb * 32 + acc_row(j, g);
                if (t < Lc) og[(long)(t0 + c0 + t) * a.o_tok + dvc] = qs[tb][j];
            }
        }
        // S = exp(G_last) S + K^T (exp(G_last - G) delta)
        const float glast = Gs[CH - 1];
        const float eglast = __expf(glast);
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int j = 0; j < 16; ++j) dl[tb][j] *= __expf(glast - Gs[tb * 32 + acc_row(j, g)]);
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
#pragma unroll
            for (int j = 0; j < 16; ++j) S[rb][j] *= eglast;
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    S[rb] = mfma_f32(Kc[(tb * 32 + acc_row(j, g)) * F_KSTR + rb * 32 + col], dl[tb][j], S[rb]);
        }
    }
    if (s1) {
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int j = 0; j < 16; ++j) s1[sbase + (long)(rb * 32 + acc_row(j, g)) * DV + dvc] = S[rb][j];
    }
}

}  // namespace hk

extern "C" int hk_launch_gated_delta_chunked(int dtype, const hk::GdnArgs* args, int n_seqs, hipStream_t stream) {
    if (dtype != hk::DT_F32) return hk_launch_gdn16(dtype, 0, args, nullptr, n_seqs, stream);
    dim3 grid(args->H, n_seqs);
    // set once, under C++'s thread-safe static initialisation (replicas launch from several threads)
    static const bool configured = hipFuncSetAttribute((const void*)hk::gdn_chunk_f32,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)hk::GDN_F32_LDS) == hipSuccess;
    if (!configured) return HK_ERR_DEVICE;
    hipLaunchKernelGGL(hk::gdn_chunk_f32, grid, dim3(256), hk::GDN_F32_LDS, stream, *args);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}
