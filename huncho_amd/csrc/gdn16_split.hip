// gdn16_split.hip - the fused Gated DeltaNet layer (gdn16_kernel.hpp) for few, long rows.
//
// gdn_chunk16 runs one workgroup per (sequence, head) through its chunks one after another. With one
// long row that is 16 workgroups on 256 CUs, each 12 us per 64-token chunk. Little of those 12 us
// depends on the chunk before: only delta = T [beta (V - e^G K S0)] and S1 = e^G_last S0 + K^T (..) do.
// So the layer runs as three kernels:
//   prep   (chunk, head), all chunks at once: conv, SiLU, l2norm, g scan, A, Aqk and the diagonal
//          blocks of T, left in a scratch slot in the layouts that the next two read
//   scan   (sequence, head, 32 value columns): the state through the chunks: K S0, R, delta and the
//          state update, nothing else; delta and the fp16 state before each chunk go to the slots
//   out    (chunk, head), all chunks at once: O = e^G Q S0 + Aqk delta, the gated RMSNorm, the store
// Every product keeps gdn_chunk16's operands, instruction and order, so the outputs, states and tails
// are the same bits as that kernel's.
//
// What bounds the whole is the scan's chain per chunk, about 1 us: 42 products, eight of them one after
// another, and the reads and conversions between them. A scan workgroup is two waves of 16 columns each (an S of 32 registers) and a third
// wave that only copies the next chunks' 42 KB from the slots into a ring of three LDS stages, so the
// computing waves issue no copies (at 13-17 clocks each they would add a third to a chunk's chain).
// Every operand sits in its slot in the order of the lanes, K in both orders it is used in: a read is
// one base register and an offset, 1 KB of consecutive LDS, without conflicts. (K as its LDS image,
// with the pair and transposing reads of gdn_chunk16, took 62-69 us for 43 chunks: their addresses
// spilled into accumulator registers.)
//
// Measured (bf16, 16 heads, one row of 2704 tokens with its state): prep 29, scan 44, out 15 us, the
// whole 521 -> 88 us. gdn_split_takes (abi.cpp) has the rule and the times on both sides of it.
#include "chunk_slots.hpp"
#include "gdn16_kernel.hpp"

namespace hk {
namespace gdn16 {

// A slot of one (chunk, head), byte offsets
constexpr int SL_Q = 0;                          // Q tile, the LDS image of gdn_chunk16
constexpr int SL_K = SL_Q + CH * RS * 2;         // K S0's K operand [k-step 4][token tile 4][lane] x 8
constexpr int SL_KT = SL_K + CH * DK * 2;        // the state update's K^T operand [k-step 2][row tile 8][lane] x 8
constexpr int SL_V = SL_KT + CH * DK * 2;        // V as R's accumulator layout [column tile 8][token tile 4][lane] x 4;
                                                 // the scan writes delta over it
constexpr int SL_A = SL_V + CH * DV * 2;         // -A_ij and T_ii operands [10 blocks][lane] x 4
constexpr int SL_G = SL_A + 10 * 64 * 8;         // fp32 [4][64]: e^G, beta, e^(G_last - G), e^G_last
constexpr int SL_AQ = SL_G + 1024;               // Aqk, the LDS image
constexpr int SL_S = SL_AQ + CH * TS * 2;        // state operand before the chunk [column tile 8][k-step 4][lane] x 8
constexpr int SLOT = SL_S + DK * DV * 2;
static_assert(SLOT % 1024 == 0 && SL_K % 1024 == 0 && SL_V % 1024 == 0 && SL_A % 1024 == 0, "1 KB copies");
static_assert(SLOT == HK_GDN_SPLIT_SLOT, "slot size in kernel_args.hpp");

constexpr int WCOLS = 32;                        // value columns per scan workgroup
constexpr int ST_KT = CH * DK * 2, ST_V = 2 * CH * DK * 2, ST_A = ST_V + 2 * 4 * 64 * 8, ST_G = ST_A + 10 * 64 * 8, STAGE = ST_G + 1024;
constexpr int N_STAGES = 3, COPIES = STAGE / 1024;
static_assert(STAGE % 1024 == 0 && COPIES <= 63, "vmcnt counts a stage of copies");

// The block (i, jj), jj <= i, of the lower triangle in the order the slots hold it
__device__ __forceinline__ int tri(int i, int jj) { return i * (i + 1) / 2 + jj; }

using chunk_slots::find_chunk;
using chunk_slots::first_chunk;
using chunk_slots::seq_rows;

// P0 of gdn_chunk16 as a function: here the compiler does better with it (row of 2704 tokens, bf16, 1 % of the layer)
template <typename T>
__device__ __forceinline__ void fused_rows(const GdnFusedArgs& fa, int t0, int Tn, int c0, int h, int kh, const T* hist,
                                           int wave, int q4, int j, f16* Qs, f16* Ks, f16* Vs) {
    typedef f16 CT;
    typedef typename M16<CT>::v8 v8;
    typedef typename M16<T>::v8 tv8;
    typedef typename M16<T>::v2 tv2;
#include "gdn16_rows.inc"
}

template <typename T>
__global__ __launch_bounds__(256, 2) void gdn_split_prep(GdnArgs a, GdnFusedArgs fa, int n_seqs, char* scratch) {
    typedef f16 CT;
    typedef typename M16<CT>::v8 v8;
    typedef typename M16<CT>::v4 v4;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    CT* Qs = (CT*)smem;
    CT* Ks = Qs + CH * RS;
    CT* Vs = Ks + CH * RS;
    float* Am = (float*)(Vs + CH * RS);
    CT* Aq = (CT*)(Am + CH * AS);
    float* Gs = (float*)(Aq + CH * TS);
    float* Bs = Gs + CH;
    const int h = blockIdx.x, cid = blockIdx.y;
    int seq, c0, t0, Tn;
    if (!find_chunk(a, n_seqs, cid, seq, c0, t0, Tn)) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q4 = lane >> 4, j = lane & 15;
    const int kh = h / a.qk_rep, Lc = min(CH, Tn - c0);
    const T* const hist = fa.hist_rows ? (const T*)fa.hist_rows[seq]
                                       : (fa.hist ? (const T*)fa.hist + (long)seq * fa.conv_dim * 3 : nullptr);
    fused_rows<T>(fa, t0, Tn, c0, h, kh, hist, wave, q4, j, Qs, Ks, Vs);
    if (wave == 3) {
        float gv = 0.0f, bv = 0.0f;
        if (lane < Lc) fused_g_beta<T>(fa, t0 + c0 + lane, h, gv, bv);
        Gs[lane] = wave_incl_scan(gv, lane);
        Bs[lane] = bv;
    }
    __syncthreads();
    chunk_tiles(Qs, Ks, Gs, Bs, Am, Aq, wave, q4, j);
    __syncthreads();
    // (inline: after a call, this compiler saved the thread index under a narrowed execution mask)
    solve_diagonal_blocks_inline(Am, wave, lane);
    __syncthreads();
    char* const slot = scratch + ((long)cid * a.H + h) * SLOT;
    // Q and Aqk as they lie in LDS
    for (int i = tid; i < SL_K / 16; i += 256) *(f32x4*)(slot + 16 * i) = *(const f32x4*)(smem + 16 * i);
    for (int i = tid; i < CH * TS * 2 / 16; i += 256)
        *(f32x4*)(slot + SL_AQ + 16 * i) = *(const f32x4*)((const char*)Aq + 16 * i);
    // K in the two operand orders: wave w takes k-step w of K S0 and row tiles 2 w, 2 w + 1 of K^T
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
        *(v8*)(slot + SL_K + ((wave * 4 + tt) * 64 + lane) * 16) = ld_pair<CT>(Ks, 16 * tt + j, 32 * wave + 4 * q4);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int kr = 32 * ks + 4 * q4 + (j >> 2), rb = 2 * wave + b;
            const i16x4 lo = lds_read_tr16(Ks + el(kr, 16 * rb + 4 * (j & 3)));
            const i16x4 hi = lds_read_tr16(Ks + el(kr + 16, 16 * rb + 4 * (j & 3)));
            *(i16x8*)(slot + SL_KT + ((ks * 8 + rb) * 64 + lane) * 16) = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    // V: rows 16 tt + 4 q4 + r of column 32 wave + 16 cw + j, by the transposing reads of gdn_chunk16
#pragma unroll
    for (int cw = 0; cw < 2; ++cw)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            const i16x4 v = lds_read_tr16(Vs + el(16 * tt + 4 * q4 + (j >> 2), 32 * wave + 16 * cw + 4 * (j & 3)));
            *(i16x4*)(slot + SL_V + (((2 * wave + cw) * 4 + tt) * 64 + lane) * 8) = v;
        }
    // -A_ij (j < i) and T_ii as fp16 operands
    for (int b = wave; b < 10; b += 4) {
        const int i = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, jj = b - tri(i, 0);
        const v4 x = jj < i ? ld_a4<CT, true>(Am, 16 * i + j, 16 * jj + 4 * q4)
                            : ld_a4<CT, false>(Am, 16 * i + j, 16 * i + 4 * q4);
        *(v4*)(slot + SL_A + (b * 64 + lane) * 8) = x;
    }
    const float glast = Gs[CH - 1];
    const float gx = wave == 0 ? __expf(Gs[lane]) : wave == 1 ? Bs[lane] : wave == 2 ? __expf(glast - Gs[lane]) : __expf(glast);
    *(float*)(slot + SL_G + tid * 4) = gx;
}

// n_slots: chunks that the scratch holds; a row whose chunks lie past them (overlapping rows in a
// malformed cu_seqlens) is a fault.
template <typename T>
__global__ __launch_bounds__(192, 2) void gdn_split_scan(GdnArgs a, GdnFusedArgs fa, int n_slots, char* scratch) {
    typedef f16 CT;
    typedef typename M16<CT>::v8 v8;
    typedef typename M16<CT>::v4 v4;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int H = a.H, h = blockIdx.x, cg = blockIdx.y, seq = blockIdx.z;
    int t0, Tn;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const bool ok = seq_rows(a, seq, t0, Tn);
    const int first = first_chunk(a, seq), nc = ok ? (Tn + CH - 1) / CH : 0;
    if (!ok || first + nc > n_slots) {
        if (threadIdx.x == 0 && cg == 0) atomicOr(a.fault, FAULT_SEQLENS);
        return;
    }
    char* const slots = scratch + ((long)first * H + h) * SLOT;
    const long step = (long)H * SLOT;

    if (wave == 2) {  // the copying wave
        const unsigned lds0 = lds_address(smem);
        auto copy_stage = [&](int c) {
            const char* s = slots + c * step + 16 * lane;
            const unsigned d = lds0 + (unsigned)(c % N_STAGES) * STAGE;
#pragma unroll
            for (int i = 0; i < ST_V / 1024; ++i) copy_x4(s + SL_K + 1024 * i, d + 1024 * i);  // K and K^T
#pragma unroll
            for (int i = 0; i < 4; ++i) copy_x4(s + SL_V + cg * 4096 + 1024 * i, d + ST_V + 1024 * i);
#pragma unroll
            for (int i = 0; i < 6; ++i) copy_x4(s + SL_A + 1024 * i, d + ST_A + 1024 * i);  // A, T and the g rows
        };
        for (int c = 0; c < min(N_STAGES - 1, nc); ++c) copy_stage(c);
        for (int c = 0; c < nc; ++c) {
            // stage c has landed once only the copies of the stages issued after it are in flight; the
            // barrier hands it over, and tells that chunk c - 1, whose stage is copied over next, is done
            const int later = min(N_STAGES - 2, nc - 1 - c);
            if (later == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COPIES) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            asm volatile("s_barrier" ::: "memory");
            if (c + N_STAGES - 1 < nc) copy_stage(c + N_STAGES - 1);
        }
        // the conv tail: 16 lanes x 8 channels for each of q, k and v
        T* const tail = fa.tail_rows ? (T*)fa.tail_rows[seq]
                                     : (fa.tail_out ? (T*)fa.tail_out + (long)seq * fa.conv_dim * 3 : nullptr);
        const int ts = lane >> 4, kh = h / a.qk_rep;
        if (tail && cg == 0 && ts < 3) {
            const T* const hist = fa.hist_rows ? (const T*)fa.hist_rows[seq]
                                               : (fa.hist ? (const T*)fa.hist + (long)seq * fa.conv_dim * 3 : nullptr);
            const long mc = ts < 2 ? ((long)ts * fa.Hk + kh) * 128 : (2L * fa.Hk + h) * 128;
            write_tail<T>(fa, t0, Tn, mc + 8 * (lane & 15), hist, tail);
        }
        return;
    }

    const int q4 = lane >> 4, j = lane & 15, ct = 2 * cg + wave;  // this wave's column tile
    const float* const s0 = a.init_rows ? a.init_rows[seq]
                                        : (a.initial_state ? a.initial_state + (long)seq * H * DK * DV : nullptr);
    float* const s1 = a.final_rows ? a.final_rows[seq]
                                   : (a.final_state ? a.final_state + (long)seq * H * DK * DV : nullptr);
    const long soff = (long)h * DK * DV + (long)(4 * q4) * DV + 16 * ct + j;
    f32x4 S[8];
#pragma unroll
    for (int rb = 0; rb < 8; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[rb][r] = s0 ? s0[soff + (16 * rb + r) * DV] : 0.0f;
    // The chunk's operands do not depend on the chain, so each group is read while the products before
    // its use run: K of chunk c + 1 under the state update of chunk c (barrier c + 1, which hands its
    // stage over, comes before that update: nothing of chunk c is read from LDS after it), everything
    // else under K S0.
    v8 Ko[4][4];
    auto read_k = [&](int c) {
        const char* const st = smem + (c % N_STAGES) * STAGE + lane * 16;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) Ko[s][tt] = *(const v8*)(st + (s * 4 + tt) * 1024);
    };
    if (nc > 0) {
        asm volatile("s_barrier" ::: "memory");
        read_k(0);
    }
    for (int c = 0; c < nc; ++c) {
        const char* const st = smem + (c % N_STAGES) * STAGE;
        char* const slot = slots + c * step;
        const float* G = (const float*)(st + ST_G);
        v8 Sb[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) Sb[s] = pack2<CT>(S[2 * s], S[2 * s + 1]);
        f32x4 ksa[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) ksa[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) ksa[tt] = M16<CT>::mma(Ko[s][tt], Sb[s], ksa[tt]);
        __builtin_amdgcn_sched_barrier(0);
        v4 At[10];
        f32x4 x[4];
        {
            v4 vv[4];
            f32x4 eg[4], bt[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                vv[i] = *(const v4*)(st + ST_V + ((wave * 4 + i) * 64 + lane) * 8);
                eg[i] = *(const f32x4*)(G + 16 * i + 4 * q4);
                bt[i] = *(const f32x4*)(G + 64 + 16 * i + 4 * q4);
            }
#pragma unroll
            for (int i = 0; i < 10; ++i) At[i] = *(const v4*)(st + ST_A + (i * 64 + lane) * 8);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) x[i][r] = rnd<CT>(bt[i][r] * (f(vv[i][r]) - eg[i][r] * ksa[i][r]));
        }
        __builtin_amdgcn_sched_barrier(0);
        v8 Kt[2][8];  // K^T operands of the state update
        f32x4 dc[4];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int rb = 0; rb < 8; ++rb) Kt[ks][rb] = *(const v8*)(st + ST_KT + (ks * 8 + rb) * 1024 + lane * 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) dc[i] = *(const f32x4*)(G + 128 + 16 * i + 4 * q4);
        const float eglast = G[3 * 64];
#pragma unroll
        for (int s = 0; s < 4; ++s) *(v8*)(slot + SL_S + ((ct * 4 + s) * 64 + lane) * 16) = Sb[s];
        f32x4 dl[4];
        v4 dbk[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            dl[i] = M16<CT>::mma16(At[tri(i, i)], pack1<CT>(x[i]), f32x4{0.f, 0.f, 0.f, 0.f});
            dbk[i] = pack1<CT>(dl[i]);
            *(v4*)(slot + SL_V + ((ct * 4 + i) * 64 + lane) * 8) = dbk[i];
            // column i of the substitution; the rows below meet their columns in the same order
#pragma unroll
            for (int k = i + 1; k < 4; ++k) x[k] = M16<CT>::mma16(At[tri(k, i)], dbk[i], x[k]);
        }
#pragma unroll
        for (int rb = 0; rb < 8; ++rb) S[rb] *= eglast;
        if (c + 1 < nc) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            read_k(c + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) dl[i] *= dc[i];
        const v8 Db[2] = {pack2<CT>(dl[0], dl[1]), pack2<CT>(dl[2], dl[3])};
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int rb = 0; rb < 8; ++rb) S[rb] = M16<CT>::mma(Kt[ks][rb], Db[ks], S[rb]);
    }
    if (s1) {
#pragma unroll
        for (int rb = 0; rb < 8; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) s1[soff + (16 * rb + r) * DV] = S[rb][r];
    }
}

constexpr int OUT_LDS = CH * RS * 2 + CH * TS * 2 + CH * RS * 2;

template <typename T>
__global__ __launch_bounds__(256, 2) void gdn_split_out(GdnArgs a, GdnFusedArgs fa, int n_seqs, const char* scratch) {
    typedef f16 CT;
    typedef typename M16<CT>::v8 v8;
    typedef typename M16<CT>::v4 v4;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    CT* Qs = (CT*)smem;
    CT* Aq = Qs + CH * RS;
    CT* Os = Aq + CH * TS;
    const int h = blockIdx.x, cid = blockIdx.y;
    int seq, c0, t0, Tn;
    if (!find_chunk(a, n_seqs, cid, seq, c0, t0, Tn)) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q4 = lane >> 4, j = lane & 15;
    const int Lc = min(CH, Tn - c0);
    const char* const slot = scratch + ((long)cid * a.H + h) * SLOT;
    // Q and Aqk into LDS: 17 and 9 copies of 1 KB over the four waves
    for (int i = wave; i < 26; i += 4)
        copy_x4(slot + (i < 17 ? SL_Q + 1024 * i : SL_AQ + 1024 * (i - 17)) + 16 * lane, lds_address(smem) + 1024 * i);
    v8 Sb[2][4];
    v4 dbk[2][4];
    float egj[4];
#pragma unroll
    for (int cw = 0; cw < 2; ++cw)
#pragma unroll
        for (int s = 0; s < 4; ++s) Sb[cw][s] = *(const v8*)(slot + SL_S + (((2 * wave + cw) * 4 + s) * 64 + lane) * 16);
#pragma unroll
    for (int cw = 0; cw < 2; ++cw)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) dbk[cw][tt] = *(const v4*)(slot + SL_V + (((2 * wave + cw) * 4 + tt) * 64 + lane) * 8);
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) egj[tt] = *(const float*)(slot + SL_G + (16 * tt + j) * 4);
    const int rsub = tid & 15, rrow = tid >> 4;
    float gz[4][8];
    gate_rows<T>(fa, t0, c0, Lc, h, rsub, rrow, gz);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
        f32x4 qsa[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const v8 qop = ld_pair<CT>(Qs, 16 * tt + j, 32 * s + 4 * q4);
#pragma unroll
            for (int cw = 0; cw < 2; ++cw) qsa[cw] = M16<CT>::mma(Sb[cw][s], qop, qsa[cw]);
        }
        f32x4 og[2];
#pragma unroll
        for (int cw = 0; cw < 2; ++cw)
#pragma unroll
            for (int r = 0; r < 4; ++r) og[cw][r] = egj[tt] * qsa[cw][r];
#pragma unroll
        for (int jj = 0; jj <= tt; ++jj) {
            const v4 aq = *(const v4*)(Aq + (16 * tt + j) * TS + 16 * jj + 4 * q4);
#pragma unroll
            for (int cw = 0; cw < 2; ++cw) og[cw] = M16<CT>::mma16(dbk[cw][jj], aq, og[cw]);
        }
#pragma unroll
        for (int cw = 0; cw < 2; ++cw) {
            const f16x2 lo = rnd_ct<T>(og[cw][0], og[cw][1]), hi = rnd_ct<T>(og[cw][2], og[cw][3]);
            *(v4*)(Os + el(16 * tt + j, 32 * wave + 16 * cw + 4 * q4)) = v4{lo[0], lo[1], hi[0], hi[1]};
        }
    }
    __syncthreads();
    char* const ob = (char*)a.o + ((long)t0 * a.o_tok + (long)h * DV) * (long)sizeof(T);
    bool range_bad = false;
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
        const int r = pass * 16 + rrow;
        const v8 ov = *(const v8*)(Os + el(r, 8 * rsub));
        if (store_gated<T>(fa, a.o_tok, ob, ov, gz[pass], c0 + r, r < Lc, rsub)) range_bad = true;
    }
    if (range_bad) atomicOr(a.fault, FAULT_RANGE);
}

template <typename T>
static int launch_split(const GdnArgs& a, const GdnFusedArgs& fa, int n_seqs, int n_slots, char* scratch, hipStream_t stream) {
    static const bool configured =
        hipFuncSetAttribute((const void*)gdn_split_prep<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES) ==
            hipSuccess &&
        hipFuncSetAttribute((const void*)gdn_split_scan<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            N_STAGES * STAGE) == hipSuccess &&
        hipFuncSetAttribute((const void*)gdn_split_out<T>, hipFuncAttributeMaxDynamicSharedMemorySize, OUT_LDS) == hipSuccess;
    if (!configured) return HK_ERR_DEVICE;
    hipLaunchKernelGGL(gdn_split_prep<T>, dim3(a.H, n_slots), dim3(256), LDS_BYTES, stream, a, fa, n_seqs, scratch);
    hipLaunchKernelGGL(gdn_split_scan<T>, dim3(a.H, DV / WCOLS, n_seqs), dim3(192), N_STAGES * STAGE, stream, a, fa, n_slots,
                       scratch);
    hipLaunchKernelGGL(gdn_split_out<T>, dim3(a.H, n_slots), dim3(256), OUT_LDS, stream, a, fa, n_seqs, (const char*)scratch);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}

}  // namespace gdn16
}  // namespace hk

// n_slots chunks of every head fit the scratch (n_slots * H * HK_GDN_SPLIT_SLOT bytes); at least the
// batch's chunks: n_tokens / 64 + n_seqs.
extern "C" int hk_launch_gdn16_split(int dtype16, const hk::GdnArgs* a, const hk::GdnFusedArgs* fa, int n_seqs, int n_slots,
                                     void* scratch, hipStream_t stream) {
    return dtype16 == 1 ? hk::gdn16::launch_split<hk::bf16>(*a, *fa, n_seqs, n_slots, (char*)scratch, stream)
                        : hk::gdn16::launch_split<hk::f16>(*a, *fa, n_seqs, n_slots, (char*)scratch, stream);
}
