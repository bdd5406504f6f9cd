// bert.hip - the ModernBERT encoder behind Huncho's Laya backend (candle ModernBERT,
// crates/huncho-backend/src/candle.rs:65-117, 319-416) on gfx950.
//
//   bidir_attn_16<T>   bidirectional softmax attention over an unpadded varlen batch, head dim
//                      64, optional window |i - j| <= w (local layers), q/k/v read straight
//                      from the fused Wqkv rows [tokens][3][heads][64]
//   bidir_attn_f32     the same in fp32 (the reference's execution precision)
//   layer_norm<T,VEC>  LayerNorm (ModernBERT's without bias; the Laya head's with), fp32 statistics
//   geglu<T,VEC>       gelu(x1) * x2 with the exact erf GELU
//   rope_qk<T,VEC>     NeoX rotate-half RoPE on the q and k parts of the Wqkv rows, in place
//   mean_pool_partial<T>, mean_pool_head<T>
//                      per-sequence mean of the final hidden rows (two deterministic passes),
//                      then a linear head (fp32)
//
// bidir_attn_16 design: one workgroup = one (sequence, head, 128 query positions); 4 waves x
// 32 queries; S^T = K Q^T on v_mfma_f32_32x32x16 (each lane owns a query column, K rows
// permuted so a lane's accumulator holds 16 consecutive keys that feed P.V directly); K and
// V tiles of 64 keys, copied straight from the q/k/v rows (global_load_lds_dwordx4, no staging
// registers), in double-buffered LDS with XOR chunk swizzles (K: (row >> 1) & 3 | bit 4 of row
// << 2; V: (row & 3) << 1 | (row >> 4) & 1, chosen so the permuted K reads, the transposing V
// reads (ds_read_b64_tr_b16) and the row writes all reach the LDS banks evenly); online softmax
// in base 2 with lazy rescaling; only tiles that intersect the block's key range are read.
#include "common.hpp"
#include "kernel_args.hpp"

namespace hk {
namespace bert {

constexpr int D = 64;                       // head dim
constexpr int BN = 64;                      // keys per tile
constexpr int TILE = BN * D;                // elements per K or V tile (8 KB in 16 bits)
constexpr size_t LDS16 = 4 * TILE * 2;      // K and V, double-buffered: 32 KB
constexpr float RESCALE_LOG2 = 8.0f;

__device__ __forceinline__ int perm_key(int m) { return ((m >> 2) & 1) * 16 + (m >> 3) * 4 + (m & 3); }
// LDS: 64 banks of 4 bytes, so a 128-byte row fills half a bank row. A 16-lane group of the
// S^T K reads (ds_read_b128) takes rows {0-7, 16-23} (or {8-15, 24-31}) at one logical chunk: the
// 8 even rows share one bank half and the 8 odd rows the other, and the swizzle gives each 8 a
// distinct chunk ((row >> 1) & 3 and row bit 4), so the 16 reads cover the 64 banks once (with
// row & 7, rows r and r + 16 met on the same chunk: a 2-way conflict on every K read). It does not
// change under the +32-row offset of the second key half.
__device__ __forceinline__ int kswz(int r) { return ((r >> 1) & 3) | (((r >> 4) & 1) << 2); }
__device__ __forceinline__ int vswz(int r) { return ((r & 3) << 1) | ((r >> 4) & 1); }
__device__ __forceinline__ int k_off(int r, int c) { return r * D + 8 * (c ^ kswz(r)); }
__device__ __forceinline__ int v_off(int r, int c) { return r * D + 8 * (c ^ vswz(r)); }

// NeoX rotate-half pair (x_i, x_{i+32}) at one position, in fp32, each result rounded to T; the
// same code in rope_qk and in the attention kernel's fused q rotation, so both round alike
template <typename T>
__device__ __forceinline__ void rope_pair(float a1, float a2, float c, float s, T& r1, T& r2) {
    r1 = from_f<T>(a1 * c - a2 * s);
    r2 = from_f<T>(a2 * c + a1 * s);
}

template <typename T>
__global__ __launch_bounds__(256, 2) void bidir_attn_16(BertAttnArgs a) {
    typedef typename Mma16<T>::v8 v8;
    typedef typename Mma16<T>::v4 v4;
    extern __shared__ __attribute__((aligned(16))) char bert_smem[];
    T* const lds = (T*)bert_smem;  // [buf][K | V][64][64]

    // XCD-aware order: workgroup i runs on XCD i % 8 as that XCD's (i / 8)-th. (sequence, head)
    // groups are striped over the XCDs (group x, x + 8, ... on XCD x) and all q-blocks of a
    // group run on its XCD back to back, sharing that XCD's L2 copy of the group's K/V rows
    const int slot = blockIdx.x >> 3;
    const int grp = (blockIdx.x & 7) + 8 * (slot / a.qblocks);
    if (grp >= a.heads * a.n_seqs) return;
    const int qb = slot % a.qblocks, h = grp % a.heads, seq = grp / a.heads;
    const int t0 = a.cu[seq];
    const int L = a.cu[seq + 1] - t0;
    if (t0 < 0 || L < 0 || t0 + L > a.n_tokens) {
        if (threadIdx.x == 0) atomicOr(a.fault, 1);
        return;
    }
    if (qb * 128 >= L) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 5, col = lane & 31;
    const int p = qb * 128 + wave * 32 + col;  // this lane's query position
    const bool q_valid = p < L;
    const int w = a.half_window;

    v8 qf[4];  // Q[p][16 ks + 8 g .. + 8]
    {
        const T* qp = (const T*)a.q + (long)(t0 + (q_valid ? p : 0)) * a.q_tok + (long)h * D;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) qf[ks] = q_valid ? *(const v8*)(qp + ks * 16 + g * 8) : v8{};
    }
    if (a.rope_cos) {
        // NeoX rotate-half RoPE of this lane's query row as it is loaded (the model's q RoPE;
        // rope_qk then rotates k only): dims 16 ks + 8 g + e, ks = 0, 1, pair with the dims 32
        // higher, which the same lane holds in qf[ks + 2]
        if (q_valid && p >= a.rope_max_pos) atomicOr(a.fault, 4);
        const int pr = min(q_valid ? p : 0, a.rope_max_pos - 1);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const float* cs = a.rope_cos + (long)pr * 32 + ks * 16 + g * 8;
            const float* sn = a.rope_sin + (long)pr * 32 + ks * 16 + g * 8;
            const f32x4 c0 = *(const f32x4*)cs, c1 = *(const f32x4*)(cs + 4);
            const f32x4 s0 = *(const f32x4*)sn, s1 = *(const f32x4*)(sn + 4);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                T r1, r2;
                rope_pair<T>((float)qf[ks][e], (float)qf[ks + 2][e], e < 4 ? c0[e] : c1[e - 4], e < 4 ? s0[e] : s1[e - 4],
                             r1, r2);
                qf[ks][e] = r1;
                qf[ks + 2][e] = r2;
            }
        }
    }
    // keys any query of the block may see
    const int blk_lo = qb * 128, blk_hi = min(L, qb * 128 + 128) - 1;
    const int k_lo = w < 0 ? 0 : max(0, blk_lo - w);
    const int k_hi = w < 0 ? L - 1 : min(L - 1, blk_hi + w);
    const int tile_lo = k_lo / BN, n_tiles = k_hi / BN - tile_lo + 1;

    int kro[4], vro[2];
    {
        const int r = perm_key(col);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) kro[ks] = k_off(r, 2 * ks + g);
        const int G = lane >> 4, j = lane & 15;
        const int vrow = (G >> 1) * 16 + (j >> 2);  // + 32 kb + 8 hh + 4 x, which leave vswz unchanged
        const int cl = 2 * (G & 1) + ((j & 3) >> 1);
#pragma unroll
        for (int db = 0; db < 2; ++db) vro[db] = vrow * D + 8 * ((4 * db + cl) ^ vswz(vrow)) + 4 * (j & 1);
    }

    // K / V tiles go straight from the q/k/v rows to LDS (global_load_lds_dwordx4): wave w
    // copies key rows 16 w .. 16 w + 15 of K and of V, 8 rows per copy; lane i of a copy writes
    // row r = base + i / 8 at physical chunk i % 8, so it reads logical chunk (i % 8) ^ swizzle(r).
    // Keys past the sequence end read its last row (finite; their scores are masked).
    const int crow = lane >> 3, cch = lane & 7;
    auto load_tile = [&](int tile, int buf) {
        const unsigned kb_ = lds_address(lds + buf * 2 * TILE), vb_ = kb_ + TILE * 2;
#pragma unroll
        for (int cp = 0; cp < 2; ++cp) {
            const int r0 = 16 * wave + 8 * cp, r = r0 + crow;
            const long key = t0 + min(tile * BN + r, L - 1);
            const unsigned dst = (unsigned)(r0 * D * 2);
            copy_x4((const T*)a.k + key * a.k_tok + (long)h * D + 8 * (cch ^ kswz(r)), kb_ + dst);
            copy_x4((const T*)a.v + key * a.v_tok + (long)h * D + 8 * (cch ^ vswz(r)), vb_ + dst);
        }
    };

    f32x16 acc_o[2];
    acc_o[0] = f32x16{};
    acc_o[1] = f32x16{};
    float m_use = -INFINITY, l_run = 0.0f;
    const float c = a.scale_log2;

    // Tile it of the block's key range. MASK: the tile reaches past the sequence end or outside
    // some query's window, so its scores take the compare. Masked and unmasked tiles run in loops
    // of their own (a runtime branch between the two forms made the compiler copy the 32 scores
    // at the merge, 32 extra VALU moves per tile).
    auto step = [&](int it, auto mask_c) {
        constexpr bool MASK = decltype(mask_c)::value;
        const int buf = it & 1, tile = tile_lo + it;
        if (it + 1 < n_tiles) load_tile(tile + 1, buf ^ 1);  // that buffer was last read in step it - 1
        const T* Kb = lds + buf * 2 * TILE;
        const T* Vb = Kb + TILE;
        // (the two accumulation chains alternate, so consecutive MFMAs are independent)
        f32x16 s[2] = {f32x16{}, f32x16{}};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                s[kb] = Mma16<T>::mma(*(const v8*)(Kb + kb * 32 * D + kro[ks]), qf[ks], s[kb]);
        // mask keys past the sequence end or outside this query's window; tiles that lie
        // inside every query's window skip the compare
        const int n0 = tile * BN;
        float mloc = -INFINITY;
        if (MASK) {
            // visible keys of this query: [lo, hi] (the window clipped to the sequence), as
            // offsets kb * 32 + jj from this lane's first key n0 + 16 g; one unsigned compare each
            const int lo = (w < 0 ? 0 : max(0, p - w)) - n0 - g * 16;
            const int hi = (w < 0 ? L - 1 : min(L - 1, p + w)) - n0 - g * 16;
            const unsigned span = (unsigned)(hi - lo);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int jj = 0; jj < 16; ++jj) {
                    if ((unsigned)(kb * 32 + jj - lo) > span) s[kb][jj] = -INFINITY;
                    mloc = fmaxf(mloc, s[kb][jj]);
                }
        } else {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int jj = 0; jj < 16; ++jj) mloc = fmaxf(mloc, s[kb][jj]);
        }
        const float m_tile = wave_max32(mloc);
        const bool grow = (m_tile - m_use) * c > RESCALE_LOG2;
        if (__any(grow)) {
            const float m_new = grow ? m_tile : m_use;
            // lanes that keep their max keep their sums (alpha 1; also avoids -inf - -inf)
            const float alpha = grow ? fast_exp2((m_use - m_new) * c) : 1.0f;
            m_use = m_new;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int jj = 0; jj < 16; ++jj) acc_o[db][jj] *= alpha;
        }
        // a query whose keys so far were all masked still has m_use = -inf: its scores are
        // all -inf and exp2 gives 0 with any finite offset
        const float mc = m_use == -INFINITY ? 0.0f : m_use * c;
        v8 pf[4];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                v8 t;
#pragma unroll
                for (int k = 0; k < 8; ++k) t[k] = (T)fast_exp2(fmaf(s[kb][hh * 8 + k], c, -mc));
                pf[kb * 2 + hh] = t;
            }
        // row sums of the rounded probabilities that P.V consumes (v_dot2 against ones)
        float lsum;
        {
            typedef typename Mma16<T>::v2 v2;
            const v2 one2 = {(T)1.0f, (T)1.0f};
            float l0 = 0.0f, l1 = 0.0f;
#pragma unroll
            for (int cc = 0; cc < 4; ++cc)
#pragma unroll
                for (int q = 0; q < 8; q += 4) {
                    l0 = dot2(v2{pf[cc][q], pf[cc][q + 1]}, one2, l0);
                    l1 = dot2(v2{pf[cc][q + 2], pf[cc][q + 3]}, one2, l1);
                }
            lsum = l0 + l1;
        }
        l_run += lsum;
        // (the two output blocks alternate, so consecutive MFMAs are independent)
#pragma unroll
        for (int cc = 0; cc < 4; ++cc)
#pragma unroll
            for (int db = 0; db < 2; ++db) {
                const T* vb = Vb + vro[db];
                const int kb = cc >> 1, hh = cc & 1;
                const i16x4 lo = lds_read_tr16(vb + (kb * 32 + hh * 8) * D);
                const i16x4 hi = lds_read_tr16(vb + (kb * 32 + hh * 8 + 4) * D);
                const v8 af = __builtin_bit_cast(v8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                acc_o[db] = Mma16<T>::mma(af, pf[cc], acc_o[db]);
            }
        // this wave's copies of the next tile; unconditional, so that no load is pending on the
        // loop's back edge
        __builtin_amdgcn_s_waitcnt(VMCNT0);
        __syncthreads();
    };
    // the tiles inside every query's window form one run [in_lo, in_hi) of the block's range
    auto inside = [&](int it) {
        const int n0 = (tile_lo + it) * BN;
        return n0 + BN - 1 < L && (w < 0 || (n0 >= blk_hi - w && n0 + BN - 1 <= blk_lo + w));
    };
    int in_lo = 0;
    while (in_lo < n_tiles && !inside(in_lo)) ++in_lo;
    int in_hi = in_lo;
    while (in_hi < n_tiles && inside(in_hi)) ++in_hi;
    std::integral_constant<bool, false> no_mask;
    std::integral_constant<bool, true> with_mask;

    load_tile(tile_lo, 0);
    __builtin_amdgcn_s_waitcnt(VMCNT0);  // Q and this wave's copies of the first tile
    __syncthreads();
    for (int it = 0; it < in_lo; ++it) step(it, with_mask);
    for (int it = in_lo; it < in_hi; ++it) step(it, no_mask);
    for (int it = in_hi; it < n_tiles; ++it) step(it, with_mask);
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    if (!q_valid) return;
    const float inv_l = 1.0f / l_tot;
    T* op = (T*)a.o + (long)(t0 + p) * a.o_tok + (long)h * D;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            v4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (T)(acc_o[db][jj * 4 + e] * inv_l);
            *(v4*)(op + db * 32 + jj * 8 + g * 4) = o;
        }
}

// fp32: one thread per query (q and the O accumulator in registers); 64 queries of one head
// share 32-key K and V tiles in LDS.
__global__ __launch_bounds__(64) void bidir_attn_f32(BertAttnArgs a) {
    __shared__ float Ks[32][D + 1];
    __shared__ float Vs[32][D + 1];
    const int qb = blockIdx.x, h = blockIdx.y, seq = blockIdx.z;
    const int t0 = a.cu[seq];
    const int L = a.cu[seq + 1] - t0;
    if (t0 < 0 || L < 0 || t0 + L > a.n_tokens) {
        if (threadIdx.x == 0) atomicOr(a.fault, 1);
        return;
    }
    if (qb * 64 >= L) return;
    const int tid = threadIdx.x;
    const int p = qb * 64 + tid;
    const bool q_valid = p < L;
    const int w = a.half_window;
    const float scale = a.scale_log2 * 0.69314718055994531f;  // natural-log scale
    float q[D], o[D];
    {
        const float* qp = (const float*)a.q + (long)(t0 + (q_valid ? p : 0)) * a.q_tok + (long)h * D;
#pragma unroll
        for (int e = 0; e < D; ++e) {
            q[e] = qp[e];
            o[e] = 0.0f;
        }
    }
    const int blk_lo = qb * 64, blk_hi = min(L, qb * 64 + 64) - 1;
    const int k_lo = w < 0 ? 0 : max(0, blk_lo - w);
    const int k_hi = w < 0 ? L - 1 : min(L - 1, blk_hi + w);
    float m = -INFINITY, l = 0.0f;
    for (int base = k_lo; base <= k_hi; base += 32) {
        __syncthreads();
        for (int idx = tid; idx < 32 * D; idx += 64) {
            const int r = idx / D, e = idx % D;
            const int key = min(base + r, L - 1);
            Ks[r][e] = ((const float*)a.k)[(long)(t0 + key) * a.k_tok + (long)h * D + e];
            Vs[r][e] = ((const float*)a.v)[(long)(t0 + key) * a.v_tok + (long)h * D + e];
        }
        __syncthreads();
        const int n = min(32, k_hi - base + 1);
        for (int r = 0; r < n; ++r) {
            const int key = base + r;
            const int dist = key > p ? key - p : p - key;
            if (w >= 0 && dist > w) continue;
            float sdot = 0.0f;
#pragma unroll
            for (int e = 0; e < D; ++e) sdot = fmaf(q[e], Ks[r][e], sdot);
            const float sv = sdot * scale;
            const float m_new = fmaxf(m, sv);
            const float alpha = __expf(m - m_new);
            const float pe = __expf(sv - m_new);
            l = l * alpha + pe;
#pragma unroll
            for (int e = 0; e < D; ++e) o[e] = fmaf(pe, Vs[r][e], o[e] * alpha);
            m = m_new;
        }
    }
    if (!q_valid) return;
    float* op = (float*)a.o + (long)(t0 + p) * a.o_tok + (long)h * D;
    const float inv = 1.0f / l;
#pragma unroll
    for (int e = 0; e < D; ++e) op[e] = o[e] * inv;
}

// 16-byte vector of T: 8 x 16-bit or 4 x fp32 elements.
template <typename T> struct Vec16 { typedef typename Mma16<T>::v8 type; static constexpr int N = 8; };
template <> struct Vec16<float> { typedef f32x4 type; static constexpr int N = 4; };

__device__ __forceinline__ float wave_sum(float s) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o);
    return s;
}

// LayerNorm (bias optional) over rows of `width` (<= 2048): one wave per row, two passes over
// registers (mean, then the centred sum of squares), statistics in fp32. VEC: 16-byte loads
// and stores (width a multiple of the vector, rows and weights 16-byte aligned).
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void layer_norm(LayerNormArgs a) {
    typedef typename Vec16<T>::type V;
    constexpr int N = VEC ? Vec16<T>::N : 1;
    constexpr int KM = 2048 / (64 * N);
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= a.rows) return;
    const T* x = (const T*)a.x + (long)row * a.x_tok;
    T* y = (T*)a.y + (long)row * a.y_tok;
    const int chunks = a.width / N;
    float v[KM][N];
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        const int c = lane + 64 * k;
        if constexpr (VEC) {
            V t = c < chunks ? *(const V*)(x + c * N) : V{};
#pragma unroll
            for (int e = 0; e < N; ++e) v[k][e] = (float)t[e];
        } else {
            v[k][0] = c < chunks ? to_f(x[c]) : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < N; ++e) s += v[k][e];
    }
    const float mean = wave_sum(s) / (float)a.width;
    float q = 0.0f;
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        const bool in = lane + 64 * k < chunks;
#pragma unroll
        for (int e = 0; e < N; ++e) {
            const float d = in ? v[k][e] - mean : 0.0f;
            q += d * d;
        }
    }
    const float inv = fast_rsqrt(wave_sum(q) / (float)a.width + a.eps);
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        const int c = lane + 64 * k;
        if (c >= chunks) continue;
        if constexpr (VEC) {
            V t;
#pragma unroll
            for (int h = 0; h < N; h += 4) {
                const f32x4 w = *(const f32x4*)(a.w + c * N + h);
                const f32x4 bb = a.b ? *(const f32x4*)(a.b + c * N + h) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; ++e) t[h + e] = from_f<T>(((v[k][h + e] - mean) * inv) * w[e] + bb[e]);
            }
            *(V*)(y + c * N) = t;
        } else {
            y[c] = from_f<T>(((v[k][0] - mean) * inv) * a.w[c] + (a.b ? a.b[c] : 0.0f));
        }
    }
}

// y[t][i] = gelu(x[t][i]) * x[t][I + i], fp32 arithmetic; VEC: N elements per thread with
// 16-byte accesses.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void geglu(GegluArgs a) {
    typedef typename Vec16<T>::type V;
    constexpr int N = VEC ? Vec16<T>::N : 1;
    const int wn = a.width / N;
    const long n = (long)a.rows * wn;
    for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < n; idx += (long)gridDim.x * blockDim.x) {
        const long t = idx / wn;
        const int i = (int)(idx % wn) * N;
        const T* row = (const T*)a.x + t * a.x_tok;
        T* out = (T*)a.y + t * a.y_tok + i;
        if constexpr (VEC) {
            const V g = *(const V*)(row + i), u = *(const V*)(row + a.width + i);
            V r;
#pragma unroll
            for (int e = 0; e < N; ++e) r[e] = from_f<T>(gelu_erf((float)g[e]) * (float)u[e]);
            *(V*)out = r;
        } else {
            *out = from_f<T>(gelu_erf(to_f(row[i])) * to_f(row[a.width + i]));
        }
    }
}

// RoPE on q (columns 0 .. heads*64) and k (heads*64 .. 2*heads*64) of each row, in place:
// x[i] = x[i] cos - x[i + 32] sin, x[i + 32] = x[i + 32] cos + x[i] sin (i < 32), at the
// token's position within its sequence. Grid (position blocks of 8, sequences); each work
// item rotates N consecutive pairs of one head (16-byte accesses when VEC).
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void rope_qk(RopeQkArgs a) {
    typedef typename Vec16<T>::type V;
    constexpr int N = VEC ? Vec16<T>::N : 1;
    constexpr int UPH = 32 / N;  // work items per head
    const int seq = blockIdx.y;
    const int t0 = a.cu[seq], L = a.cu[seq + 1] - t0;
    if (t0 < 0 || L < 0 || t0 + L > a.n_tokens) {
        if (threadIdx.x == 0 && blockIdx.x == 0) atomicOr(a.fault, 1);
        return;
    }
    const int p0 = blockIdx.x * 8, rows = min(L - p0, 8);
    if (rows <= 0) return;
    if (p0 + rows > a.max_pos) {
        if (threadIdx.x == 0) atomicOr(a.fault, 4);
        return;
    }
    const int per_tok = (a.k_only ? 1 : 2) * a.heads * UPH;
    for (int u = threadIdx.x; u < rows * per_tok; u += blockDim.x) {
        const int pp = p0 + u / per_tok, w = u % per_tok;
        const int hh = (a.k_only ? a.heads : 0) + w / UPH, i0 = (w % UPH) * N;
        T* xh = (T*)a.x + (long)(t0 + pp) * a.x_tok + hh * 64 + i0;
        const float* cs = a.cos + (long)pp * 32 + i0;
        const float* sn = a.sin + (long)pp * 32 + i0;
        if constexpr (VEC) {
            V x1 = *(const V*)xh, x2 = *(const V*)(xh + 32), r1, r2;
#pragma unroll
            for (int h = 0; h < N; h += 4) {
                const f32x4 c = *(const f32x4*)(cs + h), sv = *(const f32x4*)(sn + h);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    T t1, t2;
                    rope_pair<T>((float)x1[h + e], (float)x2[h + e], c[e], sv[e], t1, t2);
                    r1[h + e] = t1;
                    r2[h + e] = t2;
                }
            }
            *(V*)xh = r1;
            *(V*)(xh + 32) = r2;
        } else {
            const float c = cs[0], sv = sn[0];
            T t1, t2;
            rope_pair<T>(to_f(xh[0]), to_f(xh[32]), c, sv, t1, t2);
            xh[0] = t1;
            xh[32] = t2;
        }
    }
}

// Mean pooling in two deterministic passes. Pass 1, grid (sequences, POOL_PARTS): part j of a
// sequence of L rows sums rows [L j / P, L (j + 1) / P), P = min(POOL_PARTS, L), into the fp32
// slot row POOL_PARTS s + j of `pool` (every slot pass 2 reads is written first by pass 1, so
// the pool needs no clearing).

template <typename T>
__global__ __launch_bounds__(256) void mean_pool_partial(MeanPoolArgs a) {
    const int seq = blockIdx.x, j = blockIdx.y;
    const int t0 = a.cu[seq], L = a.cu[seq + 1] - t0;
    if (t0 < 0 || L <= 0 || t0 + L > a.n_tokens) {
        if (threadIdx.x == 0 && j == 0) atomicOr(a.fault, 1);
        return;
    }
    const int P = min(POOL_PARTS, L);
    if (j >= P) return;
    const long ta = t0 + (long)L * j / P, tb = t0 + (long)L * (j + 1) / P;
    const T* x = (const T*)a.x;
    float* const out = a.pool + ((long)seq * POOL_PARTS + j) * a.width;
    if (sizeof(T) == 2 && a.width % 8 == 0 && a.width <= 1024 && a.x_tok % 8 == 0 && ((uintptr_t)x & 15) == 0) {
        // 16-byte rows: thread c8 sums columns 8 c8 .. 8 c8 + 7 over the range's even rows and
        // thread c8 + 128 over its odd rows (eight independent sums each); the two halves are
        // added through LDS
        __shared__ float half1[1024];
        const int groups = a.width / 8, c8 = threadIdx.x & 127, parity = threadIdx.x >> 7;
        float acc[8] = {};
        if (c8 < groups && parity < 2) {
            for (long t = ta + parity; t < tb; t += 2) {
                const typename Vec16<T>::type v = *(const typename Vec16<T>::type*)(x + t * a.x_tok + 8 * c8);
#pragma unroll
                for (int e = 0; e < Vec16<T>::N; ++e) acc[e] += to_f(v[e]);
            }
            if (parity == 1)
#pragma unroll
                for (int e = 0; e < 8; ++e) half1[8 * c8 + e] = acc[e];
        }
        __syncthreads();
        if (c8 < groups && parity == 0)
#pragma unroll
            for (int e = 0; e < 8; ++e) out[8 * c8 + e] = acc[e] + half1[8 * c8 + e];
        return;
    }
    for (int i = threadIdx.x; i < a.width; i += blockDim.x) {
        float s0 = 0.0f, s1 = 0.0f;
        long t = ta;
        for (; t + 1 < tb; t += 2) {
            s0 += to_f(x[t * a.x_tok + i]);
            s1 += to_f(x[(t + 1) * a.x_tok + i]);
        }
        if (t < tb) s0 += to_f(x[t * a.x_tok + i]);
        out[i] = s0 + s1;
    }
}

// Pass 2, one workgroup per sequence: the parts summed in order, divided by L, then
// logits[s][o] = head_b[o] + sum_i head_w[o][i] * mean_i (fp32).
template <typename T>
__global__ __launch_bounds__(256) void mean_pool_head(MeanPoolArgs a) {
    extern __shared__ float pooled[];  // [width]
    const int seq = blockIdx.x;
    const int t0 = a.cu[seq], L = a.cu[seq + 1] - t0;
    if (t0 < 0 || L <= 0 || t0 + L > a.n_tokens) return;  // reported by pass 1
    const int P = min(POOL_PARTS, L);
    const float* const part = a.pool + (long)seq * POOL_PARTS * a.width;
    for (int i = threadIdx.x; i < a.width; i += blockDim.x) {
        // parts added in index order; eight loads are issued ahead of their adds
        float s = 0.0f;
        int j = 0;
        for (; j + 8 <= P; j += 8) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = part[(long)(j + k) * a.width + i];
#pragma unroll
            for (int k = 0; k < 8; ++k) s += v[k];
        }
        for (; j < P; ++j) s += part[(long)j * a.width + i];
        pooled[i] = s / (float)L;
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int o = wave; o < a.n_out; o += blockDim.x / 64) {
        float s = 0.0f;
        for (int i = lane; i < a.width; i += 64) s += to_f(((const T*)a.head_w)[(long)o * a.width + i]) * pooled[i];
        s = wave_sum(s);
        if (lane == 0) a.logits[(long)seq * a.n_out + o] = s + (a.head_b ? a.head_b[o] : 0.0f);
    }
}

}  // namespace bert
}  // namespace hk

#define HK_BERT_DISPATCH(dtype, KERNEL, grid, block, lds, stream, args)                                    \
    do {                                                                                                   \
        if ((dtype) == hk::DT_BF16)                                                                        \
            hipLaunchKernelGGL(hk::bert::KERNEL<hk::bf16>, grid, block, lds, stream, args);                \
        else if ((dtype) == hk::DT_F16)                                                                    \
            hipLaunchKernelGGL(hk::bert::KERNEL<hk::f16>, grid, block, lds, stream, args);                 \
        else                                                                                               \
            hipLaunchKernelGGL(hk::bert::KERNEL<float>, grid, block, lds, stream, args);                   \
    } while (0)

extern "C" int hk_launch_bidir_attention(int dtype, const hk::BertAttnArgs* a, int n_seqs, int max_len,
                                         hipStream_t stream) {
    if (dtype == hk::DT_F32) {
        hipLaunchKernelGGL(hk::bert::bidir_attn_f32, dim3((max_len + 63) / 64, a->heads, n_seqs), dim3(64), 0, stream,
                           *a);
        return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
    }
    // set once, under C++'s thread-safe static initialisation (replicas launch from several threads)
    static const bool configured =
        hipFuncSetAttribute((const void*)hk::bert::bidir_attn_16<hk::bf16>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)hk::bert::LDS16) == hipSuccess &&
        hipFuncSetAttribute((const void*)hk::bert::bidir_attn_16<hk::f16>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)hk::bert::LDS16) == hipSuccess;
    if (!configured) return HK_ERR_DEVICE;
    hk::BertAttnArgs b = *a;
    b.qblocks = (max_len + 127) / 128;
    const long groups = (long)b.heads * n_seqs;
    const long items = (groups + 7) / 8 * 8 * b.qblocks;  // 8 XCDs x ceil(groups / 8) x q-blocks
    if (items == 0) return HK_OK;
    if (items > (1L << 30)) return HK_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)items);
    if (dtype == hk::DT_BF16)
        hipLaunchKernelGGL(hk::bert::bidir_attn_16<hk::bf16>, grid, dim3(256), hk::bert::LDS16, stream, b);
    else
        hipLaunchKernelGGL(hk::bert::bidir_attn_16<hk::f16>, grid, dim3(256), hk::bert::LDS16, stream, b);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

#define HK_BERT_DISPATCH_VEC(dtype, vec, KERNEL, grid, block, lds, stream, args)                              \
    do {                                                                                                   \
        if ((dtype) == hk::DT_BF16) {                                                                      \
            if (vec) hipLaunchKernelGGL((hk::bert::KERNEL<hk::bf16, true>), grid, block, lds, stream, args); \
            else hipLaunchKernelGGL((hk::bert::KERNEL<hk::bf16, false>), grid, block, lds, stream, args);    \
        } else if ((dtype) == hk::DT_F16) {                                                                \
            if (vec) hipLaunchKernelGGL((hk::bert::KERNEL<hk::f16, true>), grid, block, lds, stream, args);  \
            else hipLaunchKernelGGL((hk::bert::KERNEL<hk::f16, false>), grid, block, lds, stream, args);     \
        } else {                                                                                           \
            if (vec) hipLaunchKernelGGL((hk::bert::KERNEL<float, true>), grid, block, lds, stream, args);    \
            else hipLaunchKernelGGL((hk::bert::KERNEL<float, false>), grid, block, lds, stream, args);       \
        }                                                                                                  \
    } while (0)

static int vec_elems(int dtype) { return dtype == hk::DT_F32 ? 4 : 8; }

extern "C" int hk_launch_layer_norm(int dtype, const hk::LayerNormArgs* a, hipStream_t stream) {
    if (a->rows == 0) return HK_OK;
    const int N = vec_elems(dtype);
    const bool vec = a->width % N == 0 && a->x_tok % N == 0 && a->y_tok % N == 0 && aligned16(a->x) &&
                     aligned16(a->y) && aligned16(a->w) && (!a->b || aligned16(a->b));
    HK_BERT_DISPATCH_VEC(dtype, vec, layer_norm, dim3((a->rows + 3) / 4), dim3(256), 0, stream, *a);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}

extern "C" int hk_launch_geglu(int dtype, const hk::GegluArgs* a, hipStream_t stream) {
    const int N = vec_elems(dtype);
    const bool vec = a->width % N == 0 && a->x_tok % N == 0 && a->y_tok % N == 0 && aligned16(a->x) && aligned16(a->y);
    const long n = (long)a->rows * (a->width / (vec ? N : 1));
    if (n == 0) return HK_OK;
    const int blocks = (int)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
    HK_BERT_DISPATCH_VEC(dtype, vec, geglu, dim3(blocks), dim3(256), 0, stream, *a);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}

extern "C" int hk_launch_rope_qk(int dtype, const hk::RopeQkArgs* a, int n_seqs, int max_len, hipStream_t stream) {
    if (max_len == 0) return HK_OK;
    const bool vec = a->x_tok % vec_elems(dtype) == 0 && aligned16(a->x) && aligned16(a->cos) && aligned16(a->sin);
    HK_BERT_DISPATCH_VEC(dtype, vec, rope_qk, dim3((max_len + 7) / 8, n_seqs), dim3(256), 0, stream, *a);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}

extern "C" int hk_launch_mean_pool_head(int dtype, const hk::MeanPoolArgs* a, int n_seqs, hipStream_t stream) {
    HK_BERT_DISPATCH(dtype, mean_pool_partial, dim3(n_seqs, hk::POOL_PARTS), dim3(256), 0, stream, *a);
    HK_BERT_DISPATCH(dtype, mean_pool_head, dim3(n_seqs), dim3(256), a->width * sizeof(float), stream, *a);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}

// ---------------------------------------------------------------------------------------------
// hk_mean_pool_head_noalloc: hk_mean_pool_head with its partial sums in a file-scope device
// array instead of a workspace, for callers that cannot allocate. The array holds 64 sequences
// x 32 partial sums x 2048 columns of fp32 (16 MiB per GPU, held until the process ends). Its
// device address comes from hipGetSymbolAddress, once per device with that device current
// (hk_noalloc_scratch_init, called by hk_ctx_create); host code uses only that address, never
// the array's name. The first context to call the entry point on a GPU owns that GPU's array
// until it is destroyed; calls from any other context on the same GPU are refused, so two
// contexts (replicas, each with its own stream) can never race on it. The owner's own calls are
// ordered on its stream; calls it makes from several streams overlap and race. Every slot the
// second pass reads is written by the first pass of the same call, so nothing needs clearing.
// ---------------------------------------------------------------------------------------------
#include <mutex>

#include "abi_internal.hpp"

namespace {
constexpr size_t kNoAllocFloats = (size_t)64 * hk::POOL_PARTS * 2048;
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
const hk_ctx* g_scratch_owner[kMaxDevices] = {};  // the context that uses each GPU's array
}  // namespace

// Gives up ctx's claim on its GPU's array (hk_ctx_destroy, after the stream has drained).
void hk_noalloc_scratch_release(const hk_ctx* ctx) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    for (auto& owner : g_scratch_owner)
        if (owner == ctx) owner = nullptr;
}

static __device__ __align__(256) float scratch[kNoAllocFloats];

// Resolves this device's scratch address (the caller has made `device` current). HK_OK once set.
int hk_noalloc_scratch_init(int device) {
    if (device < 0 || device >= kMaxDevices) return HK_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return HK_OK;
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return HK_ERR_DEVICE;
    g_scratch_ptr[device] = ptr;
    return HK_OK;
}

extern "C" int hk_mean_pool_head_noalloc(hk_ctx* ctx, int dtype, const void* x, long x_tok, const int32_t* cu,
                                         int n_seqs, int n_tokens, int width, const void* head_w, const float* head_b,
                                         int n_out, float* logits) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = hk_mean_pool_check(ctx, dtype, x, x_tok, cu, n_seqs, n_tokens, width, head_w, n_out, logits))
        return rc;
    if ((size_t)n_seqs * hk::POOL_PARTS * width > kNoAllocFloats)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED,
                       "mean pool without allocation: %d rows x %d columns exceed the fixed scratch of %zu partial "
                       "sums (64 rows x 32 parts x 2048 columns)",
                       n_seqs, width, kNoAllocFloats / hk::POOL_PARTS);
    if (hipSetDevice(ctx->device) != hipSuccess) return hk_fail(ctx, HK_ERR_DEVICE, "hipSetDevice failed");
    if (int rc = hk_noalloc_scratch_init(ctx->device))
        return hk_fail(ctx, rc, "hipGetSymbolAddress of the mean-pool scratch failed");
    void* ptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        const hk_ctx*& owner = g_scratch_owner[ctx->device];
        if (owner && owner != ctx)
            return hk_fail(ctx, HK_ERR_UNSUPPORTED,
                           "mean pool without allocation: GPU %d's scratch array belongs to another context until "
                           "that context is destroyed (use hk_mean_pool_head with a workspace here)",
                           ctx->device);
        owner = ctx;
        ptr = g_scratch_ptr[ctx->device];
    }
    hk::MeanPoolArgs pa{x, x_tok, cu, n_seqs, n_tokens, width, head_w, head_b, n_out, logits, ctx->fault_dev,
                        (float*)ptr};
    return hk_launch_mean_pool_head(dtype, &pa, n_seqs, ctx->stream) ? hk_fail(ctx, HK_ERR_DEVICE, "mean pool launch")
                                                                     : HK_OK;
}
