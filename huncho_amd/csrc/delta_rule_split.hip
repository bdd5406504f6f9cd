// delta_rule_split.hip - the fp32 chunked gated delta rule (delta_rule.hip) for few rows.
//
// gdn_chunk_f32 runs one workgroup per (sequence, head), whose four SIMDs take 33 us per 64-token chunk:
// 8.4 MFLOP of fp32 products at 256 FLOP per clock and CU are half of it. With one row that is 16
// workgroups on 256 CUs. Only K S0, T R and the state update depend on the chunk before, so, as for the
// 16-bit layer (gdn16_split.hip), three kernels share the work:
//   prep   (chunk, head), all at once: A, Aqk and T = (I + A)^-1 as gdn_chunk_f32 forms them
//   scan   (sequence, head, 16 value columns): the state through the chunks; four waves share the 16
//          columns, a quarter of each product's rows each, on 16x16x4 products whose operands pass
//          between the waves through LDS (S, R and delta, 16 columns of each)
//   out    (chunk, head, 64 value columns), all at once: O = e^G Q S0 + Aqk delta
// T, Aqk, delta and the state before each chunk pass between the kernels in the scratch, all fp32.
//
// Measured (16 heads, one row of 512 tokens with its final state): 268 -> 54 us, as far from the recurrence
// in 64 bits as before (9.6e-7). delta_split_takes (abi.cpp) has the rule and the times on both sides of it.
#include "chunk_slots.hpp"
#include "delta_rule.hpp"

namespace hk {
namespace delta_split {

// A slot of one (chunk, head), in floats
constexpr int SL_T = 0;                 // T [64][64]
constexpr int SL_Q = SL_T + CH * CH;    // Aqk [64][64]
constexpr int SL_G = SL_Q + CH * CH;    // e^G, beta, e^(G_last - G), e^G_last [4][64]
constexpr int SL_D = SL_G + 4 * CH;     // delta, transposed [value column 128][token 64]
constexpr int SL_S = SL_D + CH * DV;    // state before the chunk, transposed [value column 128][dk 128]
constexpr int SLOT = SL_S + DK * DV;
static_assert(SLOT * 4 == HK_DELTA_SPLIT_SLOT, "slot size in kernel_args.hpp");

constexpr int WC = 16;                  // value columns per scan workgroup
constexpr int SSTR = DK + 4, RSTR = CH + 4;

using chunk_slots::find_chunk;
using chunk_slots::first_chunk;
using chunk_slots::seq_rows;

__global__ __launch_bounds__(256, 1) void delta_split_prep(GdnArgs a, int n_seqs, float* scratch) {
    extern __shared__ __attribute__((aligned(16))) float smem_f[];
    float* Kc = smem_f;
    float* Qc = Kc + CH * F_KSTR;
    float* Am = Qc + CH * F_KSTR;
    float* Aq = Am + CH * F_ASTR;
    float* Tf = Aq + CH * F_ASTR;
    float* Xs = Tf + CH * F_ASTR;
    float* Gs = Xs + 32 * XSTR;
    float* Bs = Gs + CH;
    const int h = blockIdx.x, cid = blockIdx.y;
    int seq, c0, t0, Tn;
    if (!find_chunk(a, n_seqs, cid, seq, c0, t0, Tn)) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    {
        const int t = t0 + c0, Lc = min(CH, Tn - c0);
        const float* qg = (const float*)a.q + (long)(h / a.qk_rep) * DK;
        const float* kg = (const float*)a.k + (long)(h / a.qk_rep) * DK;
#include "delta_rule_load.inc"
    }
    __syncthreads();
    chunk_matrices_f32(Qc, Kc, Gs, Bs, Am, Aq, wave, lane);
    __syncthreads();
    invert_unit_lower(Am, Tf, F_ASTR, Xs, XSTR, wave, lane);
    float* const slot = scratch + ((long)cid * a.H + h) * SLOT;
    for (int i = tid; i < CH * CH / 4; i += 256) {
        const int r = i >> 4, c = (i & 15) * 4;
        *(f32x4*)(slot + SL_T + 4 * i) = *(const f32x4*)(Tf + r * F_ASTR + c);
        *(f32x4*)(slot + SL_Q + 4 * i) = *(const f32x4*)(Aq + r * F_ASTR + c);
    }
    const float glast = Gs[CH - 1];
    slot[SL_G + tid] = wave == 0 ? __expf(Gs[lane]) : wave == 1 ? Bs[lane] : wave == 2 ? __expf(glast - Gs[lane]) : __expf(glast);
}

// n_slots: chunks that the scratch holds; a row whose chunks lie past them (overlapping rows in a malformed
// cu_seqlens) is a fault.
__global__ __launch_bounds__(256, 1) void delta_split_scan(GdnArgs a, int n_slots, float* scratch) {
    __shared__ __attribute__((aligned(16))) float Ks[2][CH * F_KSTR];
    __shared__ __attribute__((aligned(16))) float Ts[2][CH * F_ASTR];
    __shared__ __attribute__((aligned(16))) float St[WC * SSTR];  // S, R and scaled delta, transposed:
    __shared__ __attribute__((aligned(16))) float Rt[WC * RSTR];  // [value column][dk or token]
    __shared__ __attribute__((aligned(16))) float Dt[WC * RSTR];
    __shared__ float Gx[2][4 * CH];
    const int h = blockIdx.x, cg = blockIdx.y, seq = blockIdx.z, H = a.H;
    int t0, Tn;
    const bool ok = seq_rows(a, seq, t0, Tn);
    const int first = first_chunk(a, seq), nc = ok ? (Tn + CH - 1) / CH : 0;
    if (!ok || first + nc > n_slots) {
        if (threadIdx.x == 0 && cg == 0) atomicOr(a.fault, FAULT_SEQLENS);
        return;
    }
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q4 = lane >> 4, j = lane & 15;
    const int col = WC * cg + j;
    const float* const kg = (const float*)a.k + (long)(h / a.qk_rep) * DK;
    const float* const vg = (const float*)a.v + (long)h * DV + col;
    const float* const s0 = a.init_rows ? a.init_rows[seq]
                                        : (a.initial_state ? a.initial_state + (long)seq * H * DK * DV : nullptr);
    float* const s1 = a.final_rows ? a.final_rows[seq]
                                   : (a.final_state ? a.final_state + (long)seq * H * DK * DV : nullptr);
    const long soff = (long)h * DK * DV + (long)(32 * wave + 4 * q4) * DV + col;
    float* const slots = scratch + ((long)first * H + h) * SLOT;
    const long step = (long)H * SLOT;

    // The next chunk's K, T, V and g rows, held in registers over a chunk. Rows past the sequence's end are
    // zero (beta is 0 there).
    f32x4 kr[8], tr[4];
    float vr[4], gr;
    auto fetch = [&](int c) {
        const int Lc = min(CH, Tn - c * CH);
        const float* const slot = slots + c * step;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int idx = tid + 256 * i, r = idx >> 5;
            kr[i] = r < Lc ? *(const f32x4*)(kg + (long)(t0 + c * CH + r) * a.k_tok + (idx & 31) * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) tr[i] = *(const f32x4*)(slot + SL_T + (tid + 256 * i) * 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = 16 * wave + 4 * q4 + r;
            vr[r] = t < Lc ? vg[(long)(t0 + c * CH + t) * a.v_tok] : 0.0f;
        }
        gr = slot[SL_G + tid];
    };
    auto stage = [&](int b) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int idx = tid + 256 * i;
            *(f32x4*)(Ks[b] + (idx >> 5) * F_KSTR + (idx & 31) * 4) = kr[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + 256 * i;
            *(f32x4*)(Ts[b] + (idx >> 4) * F_ASTR + (idx & 15) * 4) = tr[i];
        }
        Gx[b][tid] = gr;
    };

    f32x4 S[2];  // dk rows 32 wave + 16 i + 4 q4 + r of this lane's column
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] = s0 ? s0[soff + (16 * i + r) * DV] : 0.0f;
        *(f32x4*)(St + j * SSTR + 32 * wave + 16 * i + 4 * q4) = S[i];
    }
    if (nc > 0) {
        fetch(0);
        stage(0);
    }
    for (int c = 0; c < nc; ++c) {
        const int b = c & 1;
        float* const slot = slots + c * step;
        float vc[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) vc[r] = vr[r];
        if (c + 1 < nc) fetch(c + 1);
        __syncthreads();  // S, K, T and the g rows of chunk c are in LDS
        // the state before the chunk, for the out kernel: 16 columns of 128 floats
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int idx = tid + 256 * i, cc = idx >> 5, k = (idx & 31) * 4;
            *(f32x4*)(slot + SL_S + (WC * cg + cc) * DK + k) = *(const f32x4*)(St + cc * SSTR + k);
        }
        // (K S0) of tokens 16 wave ..; element e of lane group q4 of a 16-wide k-step is k = 16 kk + 4 q4 + e
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        {
            const float* const kp = Ks[b] + (16 * wave + j) * F_KSTR + 4 * q4;
            const float* const sp = St + j * SSTR + 4 * q4;
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
                const f32x4 kv = *(const f32x4*)(kp + 16 * kk), sv = *(const f32x4*)(sp + 16 * kk);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = mfma16(kv[e], sv[e], acc);
            }
        }
        const float* const G = Gx[b];
        {
            const f32x4 eg = *(const f32x4*)(G + 16 * wave + 4 * q4), bt = *(const f32x4*)(G + CH + 16 * wave + 4 * q4);
            f32x4 r4;
#pragma unroll
            for (int r = 0; r < 4; ++r) r4[r] = bt[r] * (vc[r] - eg[r] * acc[r]);
            *(f32x4*)(Rt + j * RSTR + 16 * wave + 4 * q4) = r4;
        }
        __syncthreads();
        // delta of tokens 16 wave ..: T is lower triangular, so k-steps 0 .. wave
        acc = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int kk = 0; kk <= wave; ++kk) {
            const f32x4 tv = *(const f32x4*)(Ts[b] + (16 * wave + j) * F_ASTR + 16 * kk + 4 * q4);
            const f32x4 rv = *(const f32x4*)(Rt + j * RSTR + 16 * kk + 4 * q4);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = mfma16(tv[e], rv[e], acc);
        }
        *(f32x4*)(slot + SL_D + col * CH + 16 * wave + 4 * q4) = acc;
        *(f32x4*)(Dt + j * RSTR + 16 * wave + 4 * q4) = acc * *(const f32x4*)(G + 2 * CH + 16 * wave + 4 * q4);
        __syncthreads();
        // S = e^G_last S + K^T (scaled delta) for dk rows 32 wave ..
        const float eglast = G[3 * CH];
#pragma unroll
        for (int i = 0; i < 2; ++i) S[i] *= eglast;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const f32x4 dv = *(const f32x4*)(Dt + j * RSTR + 16 * kk + 4 * q4);
            const float* const kp = Ks[b] + (16 * kk + 4 * q4) * F_KSTR + 32 * wave + j;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < 2; ++i) S[i] = mfma16(kp[e * F_KSTR + 16 * i], dv[e], S[i]);
        }
        // St was last read before the second barrier; K, T and the g rows of chunk c + 1 go to the buffer
        // last read in chunk c - 1
#pragma unroll
        for (int i = 0; i < 2; ++i) *(f32x4*)(St + j * SSTR + 32 * wave + 16 * i + 4 * q4) = S[i];
        if (c + 1 < nc) stage(b ^ 1);
    }
    if (s1) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) s1[soff + (16 * i + r) * DV] = S[i][r];
    }
}

__global__ __launch_bounds__(256, 2) void delta_split_out(GdnArgs a, int n_seqs, const float* scratch) {
    __shared__ __attribute__((aligned(16))) float Qs[CH * F_KSTR];
    __shared__ __attribute__((aligned(16))) float Aq[CH * F_ASTR];
    const int h = blockIdx.x, cid = blockIdx.y;
    int seq, c0, t0, Tn;
    if (!find_chunk(a, n_seqs, cid, seq, c0, t0, Tn)) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q4 = lane >> 4, j = lane & 15;
    const int Lc = min(CH, Tn - c0), col = 64 * blockIdx.z + 16 * wave + j;
    const float* const slot = scratch + ((long)cid * a.H + h) * SLOT;
    const float* const qg = (const float*)a.q + (long)(h / a.qk_rep) * DK;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int idx = tid + 256 * i, r = idx >> 5, k = (idx & 31) * 4;
        *(f32x4*)(Qs + r * F_KSTR + k) = r < Lc ? *(const f32x4*)(qg + (long)(t0 + c0 + r) * a.q_tok + k) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int idx = tid + 256 * i;
        *(f32x4*)(Aq + (idx >> 4) * F_ASTR + (idx & 15) * 4) = *(const f32x4*)(slot + SL_Q + 4 * idx);
    }
    f32x4 sv[8], dv[4], eg[4];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) sv[kk] = *(const f32x4*)(slot + SL_S + col * DK + 16 * kk + 4 * q4);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        dv[kk] = *(const f32x4*)(slot + SL_D + col * CH + 16 * kk + 4 * q4);
        eg[kk] = *(const f32x4*)(slot + SL_G + 16 * kk + 4 * q4);
    }
    __syncthreads();
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {  // tokens 16 tt + 4 q4 + r
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
            const f32x4 qv = *(const f32x4*)(Qs + (16 * tt + j) * F_KSTR + 16 * kk + 4 * q4);
#pragma unroll
            for (int e = 0; e < 4; ++e) o = mfma16(qv[e], sv[kk][e], o);
        }
        o *= eg[tt];
#pragma unroll
        for (int kk = 0; kk <= tt; ++kk) {
            const f32x4 av = *(const f32x4*)(Aq + (16 * tt + j) * F_ASTR + 16 * kk + 4 * q4);
#pragma unroll
            for (int e = 0; e < 4; ++e) o = mfma16(av[e], dv[kk][e], o);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = 16 * tt + 4 * q4 + r;
            if (t < Lc) ((float*)a.o + (long)h * DV)[(long)(t0 + c0 + t) * a.o_tok + col] = o[r];
        }
    }
}

}  // namespace delta_split
}  // namespace hk

// n_slots chunks of every head fit the scratch (n_slots * H * HK_DELTA_SPLIT_SLOT bytes); at least the
// batch's chunks: n_tokens / 64 + n_seqs.
extern "C" int hk_launch_delta_split(const hk::GdnArgs* a, int n_seqs, int n_slots, void* scratch, hipStream_t stream) {
    using namespace hk::delta_split;
    static const bool configured = hipFuncSetAttribute((const void*)delta_split_prep, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)hk::GDN_F32_LDS) == hipSuccess;
    if (!configured) return HK_ERR_DEVICE;
    hipLaunchKernelGGL(delta_split_prep, dim3(a->H, n_slots), dim3(256), hk::GDN_F32_LDS, stream, *a, n_seqs, (float*)scratch);
    hipLaunchKernelGGL(delta_split_scan, dim3(a->H, hk::DV / WC, n_seqs), dim3(256), 0, stream, *a, n_slots, (float*)scratch);
    hipLaunchKernelGGL(delta_split_out, dim3(a->H, n_slots, 2), dim3(256), 0, stream, *a, n_seqs, (const float*)scratch);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}
