// attention.hip - paged GQA causal prefill attention for gfx950.
//
// Semantics follow the reference's dense path (crates/huncho-backend/src/qwen3_5.rs:669-703),
// its grouped/query-blocked variants (qwen3_5/attention.rs:6-111) and direct page attention
// (qwen3_5/kv_pages.rs:104-174): O = softmax(Q K^T * scale + causal mask) V, query head h
// reading KV head h / (Hq / Hkv), keys gathered through a block table (token j of a
// sequence lives in page block_tables[s][j / P], slot j % P; pool layout
// [page][kv_head][P][head_dim], the reference's Page tensor [1, Hkv, rows, d]).
//
// Design of the 16-bit kernel (one workgroup = one sequence x one KV head x a mirrored pair
// of 128-row query blocks):
//   * the 128 rows of a block are the GQA group's query heads x (128 / group) positions, so
//     every K/V tile gathered into LDS serves all query heads of its KV head;
//   * a workgroup runs q-blocks (n - 1 - z, z) of its sequence back to back on one tile
//     pipeline, so every workgroup of a sequence does the same n + 1 tiles;
//   * head widths 128 (NH = 1) and 256 (NH = 2): a 256-wide K or V tile is held as two
//     128-wide halves with the 128-wide layout, so the operand reads keep their bank pattern;
//     the 256-wide instance needs 128 KB of LDS and runs one workgroup per CU;
//   * 4 waves x 32 query rows; S^T = K Q^T on MFMA so that each lane owns one query
//     column and the softmax row statistics stay in-lane (one v_permlane32_swap per 32 keys);
//   * K rows are read into the MFMA A operand in a permuted order so that each lane's
//     accumulator holds 16 consecutive keys; P then feeds P.V directly as the B operand;
//   * K and V tiles sit row-major in double-buffered LDS with an XOR chunk swizzle; the V^T
//     operand of O^T = V^T P^T comes from transposing LDS reads (ds_read_b64_tr_b16);
//   * online softmax in base 2 with fp32 statistics and lazy rescaling; O^T accumulates in
//     fp32 registers; the output gate o *= sigmoid(gate) (qwen3_5.rs:706-714) is fused into
//     the epilogue.
// Grid = (kv_heads, q-block pairs, sequences): the pairs of one (sequence, KV head) are
// consecutive in dispatch order on one XCD and share its L2 copy of the K/V pages.
// The fp32 kernel keeps one workgroup per q-block, grid (kv_heads, sequences, q-blocks).
#include <type_traits>
#include "common.hpp"
#include "kernel_args.hpp"

namespace hk {

constexpr int D = 128;
constexpr int BN = 64;
constexpr int KS_STRIDE_F32 = D + 4;
constexpr int V_STRIDE_F32 = D + 4;

// Key row loaded by accumulator row m so that lane group g, element j sees key g*16 + j.
__device__ __forceinline__ int perm_key(int m) { return ((m >> 2) & 1) * 16 + (m >> 3) * 4 + (m & 3); }

// max of lane l and lane l ^ 32: v_permlane32_swap (gfx950) of a value with itself gives the low
// half's values in one result and the high half's in the other, in every lane
__device__ __forceinline__ float swap_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v),
                                                    false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}

__device__ __forceinline__ float sigmoidf_(float x) { return 1.0f / (1.0f + __expf(-x)); }


// Pool page of key `key` through the block table; -1 (and the fault flag) when the table
// entry lies past bt_stride or outside [0, num_pages).
__device__ __forceinline__ int page_of(const AttnArgs& a, const int* table, int key) {
    const int idx = key >> a.page_shift;
    const int page = idx < a.bt_stride ? table[idx] : -1;
    if ((unsigned)page >= (unsigned)a.num_pages) {
        atomicOr(a.fault, 2);
        return -1;
    }
    return page;
}

// ---------------------------------------------------------------------------
// 16-bit inputs (bf16 or fp16), fp32 accumulation
// ---------------------------------------------------------------------------
constexpr int KV_ROW = 128;                        // LDS row: one key's 128 dims (256 B, unpadded)
constexpr int TILE_ELEMS = BN * KV_ROW;            // one K or V tile: 16 KB
constexpr size_t ATTN16_LDS = 4 * TILE_ELEMS * 2;  // K and V, double-buffered: 65,536 B
constexpr float RESCALE_LOG2 = 8.0f;  // exponents may run up to 2^8 above the row max in use

// The 16-byte chunk c of key row r sits at chunk c ^ swz(r) in a V tile and c ^ swzk(r) in a
// K tile. The V swizzle depends only on row bits 0 and 1, so the transposing V reads of P.V can
// add key offsets of 4, 8 and 32 rows to one per-lane address; with XOR masks 0, 4, 8, 12 the 32
// lanes of each half of a ds_read_b64_tr_b16 (256 bytes) cover all 64 banks once (the earlier
// mask 2 (r & 3) + 8 bit4(r) left every half 2-way conflicted). The K swizzle serves the
// permuted-row reads of S^T = K Q^T: a 16-lane group reads rows {0-7, 16-23} (or {8-15, 24-31})
// at one logical chunk, and swzk maps those rows to 16 distinct chunks, one 16-byte slot each
// of the 256-byte bank row.
__device__ __forceinline__ int swz(int r) { return 4 * (r & 3); }
__device__ __forceinline__ int swzk(int r) { return (r & 7) | (((r >> 4) & 1) << 3); }
__device__ __forceinline__ int lds_off_k(int r, int c) { return r * KV_ROW + 8 * (c ^ swzk(r)); }

// Key-split launches: tiles per range of a q-block of nt tiles in a row of ctx keys, q_len of them new (nt: one
// range), and the first part of a q-block. A row is split by its own lengths, so that a row without cached
// tokens is finished in one range whatever batch or table it comes with.
__device__ __forceinline__ int split_range(const AttnArgs& a, int nt, int ctx, int q_len) {
    if (ctx <= (a.split_from - 1) * BN || (ctx >> 2) < q_len) return nt;
    return nt <= 4 * a.n_split ? min(nt, 4) : (nt + a.n_split - 1) / a.n_split;
}
__device__ __forceinline__ long part_index(const AttnArgs& a, int seq, int qb, int kvh) {
    return (((long)seq * a.n_qblocks + qb) * a.kv_heads + kvh) * a.n_split;
}

// Pipeline per 64-key tile (one barrier per tile): issue the direct-to-LDS copies of tile
// t+1 into buffer (t+1) % 2 (page read one tile earlier) and the block-table read of tile
// t+2; S^T = K Q^T, online softmax and O^T += V^T P^T on buffer t % 2; wait for this wave's
// copies; barrier.
// Softmax keeps the raw-score row max m and evaluates p = 2^(s c - m c) with one FMA
// (c = scale log2 e); the O / l rescale happens only when the max grew by more than 2^8
// (otherwise p <= 2^8 and the fp32 sums lose nothing), which is the same normalised result.
// The row sum l adds the probabilities as rounded for P.V (v_dot2 against ones), so the
// weights applied to V sum to one.
//
// SPLIT: a batch of few rows leaves most CUs idle (five 30-token questions over one 2,700-token state:
// 40 workgroups of 43 tiles, 54.9 us; split 17.4 and 4.7 for attn_combine). Then a workgroup takes one q-block and
// one range of its key tiles, and writes its unnormalised fp32 O rows with their max and sum; attn_combine adds the ranges of a
// row in their order. A q-block with a single range is finished here as in the unsplit kernel. A range
// may lie past a row's last visible key: its max stays -inf and its probabilities 0.
template <typename T, int NH, bool SPLIT>
__global__ __launch_bounds__(256, NH == 1 ? 2 : 1) void paged_prefill_attn_16(AttnArgs a) {
    typedef typename Mma16<T>::v8 v8;
    typedef typename Mma16<T>::v4 v4;
    typedef typename Mma16<T>::v2 v2;
    // NH 128-wide halves per head row (head_dim 128 NH): each K and V tile is held as NH
    // sub-tiles of 128 dims with the 128-wide layout and swizzles, so the operand reads and
    // their bank pattern are those of the 128-wide kernel
    constexpr int HD = 128 * NH;
    extern __shared__ __attribute__((aligned(16))) char attn_smem[];
    T* const lds = (T*)attn_smem;  // [buf][K half 0 .. NH - 1 | V half 0 .. NH - 1][64][128]

    // grid (kv_heads, q-block pairs, sequences): linear workgroup ids run KV head fastest,
    // and consecutive ids go round-robin to the 8 XCDs, so all q-block pairs of one
    // (sequence, KV head) run together on one XCD and share its L2 copy of the K/V pages
    // SPLIT: grid (kv_heads, sequences, n_split ranges of each q-block), range 0 of all sequences side by
    // side: where the contexts are short and have one range (a wide table), they spread over the chip as
    // in the unsplit launch (16 rows of 130 keys under 4,096: 12.3 us, 16.4 with the ranges side by side)
    const int kvh = blockIdx.x;
    const int z = SPLIT ? 0 : blockIdx.y;
    const int seq = SPLIT ? blockIdx.y : blockIdx.z;
    // SPLIT: the q-block, counted from the last, and its range
    const int zb = SPLIT && a.n_qblocks > 1 ? blockIdx.z / a.n_split : 0, zr = SPLIT ? blockIdx.z - zb * a.n_split : 0;
    const int q0 = a.cu_seqlens_q[seq];
    const int q_len = a.cu_seqlens_q[seq + 1] - q0;
    const int ctx = a.context_lens[seq];
    const int P = a.pos_per_block;  // 128 / group: a power of two
    const int p_shift = __builtin_ctz(P);
    if (q0 < 0 || q_len < 0 || q0 + q_len > a.n_tokens || q_len > ctx) {
        if (threadIdx.x == 0) atomicOr(a.fault, 1);
        return;
    }
    // this workgroup's q-blocks: the mirrored pair (nq - 1 - z, z), so every workgroup of a
    // sequence runs nq + 1 key tiles; the longer block goes first
    const int nq = SPLIT ? (q_len + P - 1) >> p_shift : (q_len + P - 1) / P;
    // (SPLIT: q-blocks past n_qblocks, rows longer than max_q_len, have no part)
    const int qb_a = SPLIT ? a.n_qblocks - 1 - zb : nq - 1 - z, qb_b = z;
    if (SPLIT ? qb_a >= nq : 2 * z >= nq) return;
    const int n_blocks = SPLIT || qb_a == qb_b ? 1 : 2;
    const int off = ctx - q_len;  // absolute position of the first new query
    const int* table = a.block_tables + (long)seq * a.bt_stride;
    const int pmask = (1 << a.page_shift) - 1;
    auto block_tiles = [&](int qb) { return (off + min(q_len, (qb + 1) * P) - 1) / BN + 1; };
    // SPLIT: tiles i0 .. nt_a - 1 of the block's
    const int nt_all = block_tiles(qb_a), range = SPLIT ? split_range(a, nt_all, ctx, q_len) : nt_all;
    const bool split = SPLIT && range < nt_all;
    const int i0 = zr * range;
    if (SPLIT && i0 >= nt_all) return;
    const int nt_a = SPLIT ? min(nt_all, i0 + range) : nt_all;
    const int n_sched = nt_a + (n_blocks == 2 ? block_tiles(qb_b) : 0);
    // schedule step i -> key tile: block a's tiles 0..nt_a-1, then block b's from 0
    auto sched_tile = [&](int i) { return i < nt_a ? i : i - nt_a; };

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63, g = lane >> 5, col = lane & 31;
    const int row = wave * 32 + col;  // this lane's query row: (head in group, position)
    const int hg = SPLIT ? row >> p_shift : row / P, p = SPLIT ? row & (P - 1) : row % P;
    const int head = kvh * a.group + hg;

    // per-lane LDS offsets (elements): K rows of S^T (row perm_key(col), chunk 2 ks + g) and
    // V^T transposing reads (16-lane group G: dims 32 db + 16 (G & 1) + 4 (j & 3), keys
    // 16 (G >> 1) + (j >> 2) + 4 r + 8 h + 32 kb; the key-independent part of the swizzle)
    int koff[8], vofs[4];
    {
        const int kr_ = perm_key(col);
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) koff[ks] = lds_off_k(kr_, 2 * ks + g);
        const int G = lane >> 4, j = lane & 15;
        const int vrow = (G >> 1) * 16 + (j >> 2);
        const int cl = 2 * (G & 1) + ((j & 3) >> 1);
#pragma unroll
        for (int db = 0; db < 4; ++db) vofs[db] = vrow * KV_ROW + 8 * ((4 * db + cl) ^ swz(vrow)) + 4 * (j & 1);
    }

    // K / V tiles go straight from the pool to LDS (global_load_lds_dwordx4): wave w copies
    // keys 16 w .. 16 w + 15 of a tile, which lie in one page (pages hold >= 16 keys), 4 rows
    // per copy; lane i of copy c writes row 16 w + 4 c + i / 16 at physical chunk i % 16, so it
    // reads logical chunk (i % 16) ^ swzk(row) of K and (i % 16) ^ swz(row) of V. Keys at or
    // past the context copy the context's last key: their scores are masked, so they add
    // 0 x a finite value. A page outside the table or the pool sets fault bit 2 and copies pool
    // row 0 instead.
    // The table entry of a tile is read one step before its copies and used only then: using
    // it in the step that reads it would wait for the copies issued just before (memory
    // loads complete in issue order), which would serialise every tile's copies with the
    // compute of the tile before.
    int pg = 0;      // this wave's page for the next tile to copy (wave-uniform)
    int e_next = 0;  // block-table entry of the tile after that (in flight)
    bool in_table = true;
    auto lookup = [&](int tile) {
        const int kc = min(tile * BN + 16 * wave, ctx - 1);
        const int idx = kc >> a.page_shift;
        in_table = idx < a.bt_stride;
        e_next = table[min(idx, a.bt_stride - 1)];
    };
    auto resolve = [&]() {
        int e = in_table ? e_next : -1;
        if ((unsigned)e >= (unsigned)a.num_pages) {
            if (lane == 0) atomicOr(a.fault, 2);
            e = 0;
        }
        pg = __builtin_amdgcn_readfirstlane(e);
    };
    const int crow = lane >> 4, cch = lane & 15;  // copy lane: row within a copy, physical chunk
    auto load_tile = [&](int tile, int buf) {
        const unsigned kb = lds_address(lds + buf * 2 * NH * TILE_ELEMS), vb = kb + NH * TILE_ELEMS * 2;
        const long page_row = ((long)pg * a.kv_heads + kvh) << a.page_shift;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int r = 16 * wave + 4 * c + crow;  // row of the tile = key offset
            const int key = min(tile * BN + r, ctx - 1);
            const long row_el = (page_row + (key & pmask)) * HD;
            const unsigned dst = (unsigned)((16 * wave + 4 * c) * KV_ROW * 2);
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                copy_x4((const T*)a.k_pool + row_el + 128 * h + 8 * (cch ^ swzk(r)), kb + h * TILE_ELEMS * 2 + dst);
                copy_x4((const T*)a.v_pool + row_el + 128 * h + 8 * (cch ^ swz(r)), vb + h * TILE_ELEMS * 2 + dst);
            }
        }
    };

    // per-block query state
    int qi = 0, qpos = 0, first_pos = 0;
    bool q_valid = false;
    v8 qf[8 * NH];  // Q[q][ks*16 + g*8 .. +8] for ks = 0 .. 8 NH - 1
    // Issued once the previous block's last S^T no longer needs qf. Rows past the sequence load
    // its last row (their columns of S^T, P and O^T are computed and never stored; each query
    // column is independent), so the loads need no select, which would make the compiler wait
    // for them on the spot.
    auto load_q = [&](int qb) {
        const int qi_ = min(qb * P + p, q_len - 1);
        const T* qp = (const T*)a.q + (long)(q0 + qi_) * a.q_tok + (long)head * a.q_head;
#pragma unroll
        for (int ks = 0; ks < 8 * NH; ++ks) qf[ks] = *(const v8*)(qp + ks * 16 + g * 8);
    };
    auto begin_block = [&](int qb) {
        qi = qb * P + p;  // index among the sequence's new queries
        q_valid = qi < q_len;
        qpos = off + (q_valid ? qi : q_len - 1);
        first_pos = off + qb * P;
    };

    // The epilogue's gate reads are unconditional (Q rows stand in when there is no gate), so
    // the compiler issues all of them before it waits for the first.
    const bool gated_out = a.gate != nullptr;
    const void* const tb = gated_out ? a.gate : a.q;
    const long tb_tok = gated_out ? a.g_tok : a.q_tok, tb_head = gated_out ? a.g_head : a.q_head;

    f32x16 acc_o[4 * NH];  // O^T dims 32 db .. + 31 (half db / 4)
#pragma unroll
    for (int db = 0; db < 4 * NH; ++db) acc_o[db] = f32x16{};
    float m_use = -INFINITY, l_run = 0.0f;
    const float c = a.scale_log2;
    // a range whose keys so far are all masked or -inf adds nothing; a whole row of them is NaN, as unsplit
    const float none = SPLIT && split ? 0.0f : -INFINITY;

    // Epilogue of block qb: o = O / l (both lane halves hold partial row sums), rounded to T,
    // then the output gate o = round(o) * round(sigmoid(gate)) as the reference rounds both.
    // O leaves its accumulator layout through LDS (the free K/V buffer `stg`, row-major with a
    // row XOR chunk swizzle), so the gate loads and output stores move whole 256-byte rows
    // (16 lanes x 16 bytes) instead of 32 rows x 16 bytes per instruction; the gate loads are
    // issued first and land while O is staged.
    auto finish_block = [&](int qb, int stg) {
        // [128 rows][HD] T in the free buffer (32 KB per half); half h of row R at R HD + 128 h
        T* const sb = lds + stg * 2 * NH * TILE_ELEMS;
        v8 gch[8 * NH];
        int orow[8 * NH];  // token index of each chunk's row (-1: past the sequence)
#pragma unroll
        for (int k = 0; k < 8 * NH; ++k) {
            const int id = tid + 256 * k, R = id / (16 * NH), ch = id % (16 * NH);
            const int qi_ = qb * P + (R & (P - 1));
            const int hd = kvh * a.group + (R >> p_shift);
            orow[k] = qi_ < q_len ? q0 + qi_ : -1;
            const T* gp = (const T*)tb + (long)(q0 + min(qi_, q_len - 1)) * tb_tok + (long)hd * tb_head + ch * 8;
            gch[k] = *(const v8*)gp;  // unconditional (a Q row when ungated): no select, no early wait
        }
        const float l_tot = l_run + __shfl_xor(l_run, 32);
        const float inv_l = 1.0f / l_tot;
#pragma unroll
        for (int db = 0; db < 4 * NH; ++db)
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                const int c16 = (db & 3) * 4 + jj;
                *(v4*)(sb + row * HD + 128 * (db >> 2) + 8 * (c16 ^ (row & 15)) + 4 * g) =
                    v4{(T)(acc_o[db][jj * 4] * inv_l), (T)(acc_o[db][jj * 4 + 1] * inv_l),
                       (T)(acc_o[db][jj * 4 + 2] * inv_l), (T)(acc_o[db][jj * 4 + 3] * inv_l)};
            }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 8 * NH; ++k) {
            const int id = tid + 256 * k, R = id / (16 * NH), ch = id % (16 * NH);
            v8 ov = *(const v8*)(sb + R * HD + 128 * (ch >> 4) + 8 * ((ch & 15) ^ (R & 15)));
            if (gated_out) {
#pragma unroll
                for (int e = 0; e < 8; ++e) ov[e] = (T)((float)ov[e] * (float)(T)fast_sigmoid((float)gch[k][e]));
            }
            if (orow[k] >= 0)
                *(v8*)((T*)a.o + (long)orow[k] * a.o_tok + (long)(kvh * a.group + (R >> p_shift)) * a.o_head + ch * 8) = ov;
        }
        __syncthreads();  // staging reads done before the buffer takes a K/V tile again
#pragma unroll
        for (int db = 0; db < 4 * NH; ++db) acc_o[db] = f32x16{};
        m_use = -INFINITY;
        l_run = 0.0f;
    };

    // Softmax pieces of one 32-key half (accumulator s, keys n0h ..): the causal mask (MASK:
    // only tiles that reach past the block's first query), the raw-score max of the half-wave
    // pair, and the lazy rescale when the max grew.
    auto half_max = [&](f32x16& sv, int n0h, auto mask_c) {
        constexpr bool MASK = decltype(mask_c)::value;
        float mloc = -INFINITY;
        if (MASK && n0h + 31 > first_pos) {
            const int lim = qpos - n0h - g * 16;  // key offset j is visible iff j <= lim
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                if (j > lim) sv[j] = -INFINITY;
                mloc = fmaxf(mloc, sv[j]);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) mloc = fmaxf(mloc, sv[j]);
        }
        return swap_max(mloc);
    };
    auto rescale = [&](float m_half) {
        const bool grow = (m_half - m_use) * c > RESCALE_LOG2;
        if (__any(grow)) {
            const float m_new = grow ? m_half : m_use;
            // lanes that keep their max keep their sums (alpha 1; also avoids -inf - -inf)
            const float alpha = grow ? fast_exp2((m_use - m_new) * c) : 1.0f;
            m_use = m_new;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < 4 * NH; ++db)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc_o[db][j] *= alpha;
        }
    };
    // probabilities of one half as the P.V operand (rounded to T), and their row sums
    auto half_p = [&](const f32x16& sv, v8* pf) {
        const float mc = SPLIT && m_use == -INFINITY ? none : m_use * c;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v8 t;
#pragma unroll
            for (int k = 0; k < 8; ++k) t[k] = (T)fast_exp2(fmaf(sv[h * 8 + k], c, -mc));
            pf[h] = t;
        }
        const v2 one2 = {(T)1.0f, (T)1.0f};
        float l0 = 0.0f, l1 = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 8; q += 4) {
                l0 = dot2(v2{pf[h][q], pf[h][q + 1]}, one2, l0);
                l1 = dot2(v2{pf[h][q + 2], pf[h][q + 3]}, one2, l1);
            }
        l_run += l0 + l1;
    };
    // O^T += V^T P^T for keys kb*32 + g*16 + h*8 + [0..7], dims db*32 + [0..31]
    auto pv = [&](const T* Vb, int kb, int h, const v8& p) {
#pragma unroll
        for (int db = 0; db < 4 * NH; ++db) {
            const T* vb = Vb + (db >> 2) * TILE_ELEMS + vofs[db & 3];
            const i16x4 lo = lds_read_tr16(vb + (kb * 32 + h * 8) * KV_ROW);
            const i16x4 hi = lds_read_tr16(vb + (kb * 32 + h * 8 + 4) * KV_ROW);
            const v8 af = __builtin_bit_cast(v8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            acc_o[db] = Mma16<T>::mma(af, p, acc_o[db]);
        }
    };

    // One 64-key tile of the schedule, ordered so that each wave has independent MFMA and
    // VALU work side by side: the copies of the next tile and the max of half 0 beside the
    // S^T MFMAs, the probabilities of half 0 beside the rest of half 1's S^T, the max of half 1
    // beside half 0's P.V, and the probabilities of half 1 beside its own P.V. The copies are
    // unconditional (the last step copies its own tile again into the free buffer) so that they
    // share the MFMAs' basic block; the table entry of a tile is read one step before its copies.
    auto step = [&](int i, auto mask_c) {
        const int buf = i & 1;
        const T* Kb = lds + buf * 2 * NH * TILE_ELEMS;  // K half h at Kb + h TILE_ELEMS
        const T* Vb = Kb + NH * TILE_ELEMS;
        // the first K fragments are read before the copies are issued (the copies' inline
        // assembly orders every LDS access around it), so their latency overlaps the copies
        v8 kf[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) kf[ks] = *(const v8*)(Kb + koff[ks]);
        resolve();
        load_tile(sched_tile(min(i + 1, n_sched - 1)), buf ^ 1);
        lookup(sched_tile(min(i + 2, n_sched - 1)));
        const int n0 = sched_tile(i) * BN;
        f32x16 s0 = f32x16{}, s1 = f32x16{};
        // k-step ks reads K half ks / 8 at its 128-wide offset koff[ks % 8]
        auto kfrag = [&](int ks, int row0) {
            return *(const v8*)(Kb + (ks >> 3) * TILE_ELEMS + row0 * KV_ROW + koff[ks & 7]);
        };
#pragma unroll
        for (int ks = 0; ks < 8 * NH; ++ks) {
            s0 = Mma16<T>::mma(ks < 4 ? kf[ks] : kfrag(ks, 0), qf[ks], s0);
            if (ks & 1) s1 = Mma16<T>::mma(kfrag(ks >> 1, 32), qf[ks >> 1], s1);
        }
        rescale(half_max(s0, n0, mask_c));
#pragma unroll
        for (int ks = 4 * NH; ks < 8 * NH; ++ks) s1 = Mma16<T>::mma(kfrag(ks, 32), qf[ks], s1);
        v8 p0[2], p1[2];
        half_p(s0, p0);
        pv(Vb, 0, 0, p0[0]);
        pv(Vb, 0, 1, p0[1]);
        rescale(half_max(s1, n0 + 32, mask_c));
        half_p(s1, p1);
        pv(Vb, 1, 0, p1[0]);
        pv(Vb, 1, 1, p1[1]);
        // this wave's copies of tile i + 1; unconditional, so that no load is pending on the
        // loop's back edge and the compiler adds no wait of its own inside the next step
        __builtin_amdgcn_s_waitcnt(VMCNT0);
        __syncthreads();
    };
    // tiles of a block before mask_from see only keys at or before the block's first query
    auto mask_from = [&](int qb) { return (off + qb * P + 1) / BN; };
    std::integral_constant<bool, false> no_mask;
    std::integral_constant<bool, true> with_mask;

    begin_block(qb_a);
    lookup(i0);  // issued before Q, so that resolving it waits for the table read alone
    load_q(qb_a);
    resolve();
    load_tile(i0, i0 & 1);
    lookup(sched_tile(min(i0 + 1, n_sched - 1)));
    __builtin_amdgcn_s_waitcnt(VMCNT0);  // Q and this wave's copies of tile 0
    __syncthreads();
    // The two blocks run as two loops whose bodies issue only the tile and table loads:
    // Q, gate and output traffic stays between them, so the compiler's wait counting never
    // holds a tile's S^T behind the next tile's prefetch.
    {
        const int mf = min(mask_from(qb_a), nt_a);
        for (int i = i0; i < mf; ++i) step(i, no_mask);
        for (int i = max(mf, i0); i < nt_a; ++i) step(i, with_mask);
    }
    if (SPLIT && split) {
        const float l_tot = l_run + __shfl_xor(l_run, 32);
        if (!q_valid) return;  // rows past the sequence have no part (short suffixes fill half a block)
        const long w = part_index(a, seq, qb_a, kvh) + zr;
        float* const op = a.part + (w * 128 + row) * HD + 4 * g;
#pragma unroll
        for (int db = 0; db < 4 * NH; ++db)
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
                *(f32x4*)(op + 32 * db + 8 * jj) = f32x4{acc_o[db][4 * jj], acc_o[db][4 * jj + 1], acc_o[db][4 * jj + 2],
                                                         acc_o[db][4 * jj + 3]};
        if (g == 0) *(f32x2*)(a.part_ml + (w * 128 + row) * 2) = f32x2{m_use, l_tot};
        return;
    }
    if (n_blocks == 2) load_q(qb_b);  // lands while block a's output is written
    finish_block(qb_a, (nt_a - 1) & 1);  // the buffer of block a's last tile is free
    if (n_blocks == 2) {
        begin_block(qb_b);
        __builtin_amdgcn_s_waitcnt(VMCNT0);  // Q of block b and block a's stores, once
        const int mf = nt_a + min(mask_from(qb_b), n_sched - nt_a);
        for (int i = nt_a; i < mf; ++i) step(i, no_mask);
        for (int i = mf; i < n_sched; ++i) step(i, with_mask);
        finish_block(qb_b, 0);
    }
}

// Adds the key ranges of RPP query rows of a q-block in their order and finishes them as the attention
// kernel does: o = sum_s 2^((m_s - m) c) O_s / l, rounded to T, times the gate. HD / 4 lanes per row.
template <typename T, int NH>
__global__ __launch_bounds__(256) void attn_combine(AttnArgs a) {
    typedef typename Mma16<T>::v4 v4;
    constexpr int HD = 128 * NH, LPR = HD / 4, RPP = 256 / LPR;  // lanes per row, rows per pass
    const int kvh = blockIdx.x, qb = blockIdx.y / (128 / RPP), seq = blockIdx.z;
    const int q0 = a.cu_seqlens_q[seq], q_len = a.cu_seqlens_q[seq + 1] - q0, ctx = a.context_lens[seq];
    const int P = a.pos_per_block;
    if (q0 < 0 || q_len < 0 || q0 + q_len > a.n_tokens || q_len > ctx || qb * P >= q_len) return;
    const int nt = (ctx - q_len + min(q_len, (qb + 1) * P) - 1) / BN + 1, range = split_range(a, nt, ctx, q_len);
    if (range >= nt) return;  // finished by the attention kernel
    const int ns = range == 4 ? (nt + 3) / 4 : (nt + range - 1) / range;
    const long w0 = part_index(a, seq, qb, kvh);
    const int row = RPP * (blockIdx.y % (128 / RPP)) + threadIdx.x / LPR, d = 4 * (threadIdx.x % LPR);
    const int qi = qb * P + (row & (P - 1)), head = kvh * a.group + (row >> __builtin_ctz(P));
    if (qi >= q_len) return;  // the same for a row's lanes
    // lane i of each 32 holds range i's max and sum: one load, then the weights by shuffle
    const int i = threadIdx.x & 31;
    const f32x2 v = *((const f32x2*)a.part_ml + (w0 + min(i, ns - 1)) * 128 + row);
    float m = i < ns ? v[0] : -INFINITY;
#pragma unroll
    for (int x = 1; x < 32; x <<= 1) m = fmaxf(m, __shfl_xor(m, x));
    // a range without a visible key adds nothing (also -inf - -inf); a NaN or +inf max stays one
    const float wgt = i >= ns || v[0] == -INFINITY ? 0.0f : fast_exp2((v[0] - m) * a.scale_log2);
    float l = i < ns ? wgt * v[1] : 0.0f;
#pragma unroll
    for (int x = 1; x < 32; x <<= 1) l += __shfl_xor(l, x);
    const float* const op = a.part + (w0 * 128 + row) * HD + d;
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < ns; s0 += 8) {  // 8 loads in flight
        f32x4 t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = *(const f32x4*)(op + (long)min(s0 + e, ns - 1) * 128 * HD);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float w = __shfl(wgt, s0 + e, 32);
            if (s0 + e < ns) o += w * t[e];
        }
    }
    const float inv = 1.0f / l;
    const long tok = q0 + qi;
    v4 r = v4{(T)(o[0] * inv), (T)(o[1] * inv), (T)(o[2] * inv), (T)(o[3] * inv)};
    if (a.gate) {
        const v4 gv = *(const v4*)((const T*)a.gate + tok * a.g_tok + (long)head * a.g_head + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = (T)((float)r[e] * (float)(T)fast_sigmoid((float)gv[e]));
    }
    *(v4*)((T*)a.o + tok * a.o_tok + (long)head * a.o_head + d) = r;
}

// ---------------------------------------------------------------------------
// fp32 inputs and accumulation (v_mfma_f32_32x32x2_f32)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256, 1) void paged_prefill_attn_f32(AttnArgs a) {
    __shared__ __attribute__((aligned(16))) float Ks[BN * KS_STRIDE_F32];
    __shared__ __attribute__((aligned(16))) float Vs[BN * V_STRIDE_F32];

    const int kvh = blockIdx.x;
    const int seq = blockIdx.y;
    const int qb = gridDim.z - 1 - blockIdx.z;
    const int q0 = a.cu_seqlens_q[seq];
    const int q_len = a.cu_seqlens_q[seq + 1] - q0;
    const int ctx = a.context_lens[seq];
    const int P = a.pos_per_block;
    if (q0 < 0 || q_len < 0 || q0 + q_len > a.n_tokens || q_len > ctx) {
        if (threadIdx.x == 0) atomicOr(a.fault, 1);
        return;
    }
    if (qb * P >= q_len) return;
    const int off = ctx - q_len;

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63, g = lane >> 5, col = lane & 31;
    const int row = wave * 32 + col;
    const int hg = row / P, p = row % P;
    const int qi = qb * P + p;
    const bool q_valid = qi < q_len;
    const int head = kvh * a.group + hg;
    const int qpos = off + (q_valid ? qi : q_len - 1);

    // Q fragment: Q[q][4u + 2g + e], u = 0..31, e = 0..1
    f32x2 qf[32];
    {
        const float* qp = (const float*)a.q + (long)(q0 + (q_valid ? qi : 0)) * a.q_tok + (long)head * a.q_head;
#pragma unroll
        for (int u = 0; u < 32; ++u) qf[u] = q_valid ? *(const f32x2*)(qp + 4 * u + 2 * g) : f32x2{0.f, 0.f};
    }

    const int last_pos = off + min(q_len, (qb + 1) * P) - 1;
    const int first_pos = off + qb * P;
    const int n_tiles = last_pos / BN + 1;
    const int* table = a.block_tables + (long)seq * a.bt_stride;
    const int pmask = (1 << a.page_shift) - 1;

    // tile = 64 rows x 128 floats = 2048 float4; thread t loads float4 chunk t + 256 i, i = 0..7
    float4 kr[8], vr[8];
    auto load_tile = [&](int tile) {
        const int n0 = tile * BN;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            int c = tid + 256 * i;
            int key = n0 + (c >> 5);
            int page = key < ctx ? page_of(a, table, key) : -1;
            if (page >= 0) {
                long base = ((((long)page * a.kv_heads + kvh) << a.page_shift) + (key & pmask)) * D + (c & 31) * 4;
                kr[i] = *(const float4*)((const float*)a.k_pool + base);
                vr[i] = *(const float4*)((const float*)a.v_pool + base);
            } else {
                kr[i] = float4{0.f, 0.f, 0.f, 0.f};
                vr[i] = float4{0.f, 0.f, 0.f, 0.f};
            }
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            int c = tid + 256 * i;
            *(float4*)(Ks + (c >> 5) * KS_STRIDE_F32 + (c & 31) * 4) = kr[i];
            *(float4*)(Vs + (c >> 5) * V_STRIDE_F32 + (c & 31) * 4) = vr[i];
        }
    };

    f32x16 acc_o[4];
#pragma unroll
    for (int db = 0; db < 4; ++db) acc_o[db] = f32x16{};
    float m_run = -INFINITY, l_run = 0.0f;

    load_tile(0);
    for (int tile = 0; tile < n_tiles; ++tile) {
        __syncthreads();
        store_tile();
        __syncthreads();
        if (tile + 1 < n_tiles) load_tile(tile + 1);

        f32x16 s[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            s[kb] = f32x16{};
            const float* krow = Ks + (kb * 32 + perm_key(col)) * KS_STRIDE_F32 + 2 * g;
#pragma unroll
            for (int u = 0; u < 32; ++u) {
                f32x2 kv = *(const f32x2*)(krow + 4 * u);
                s[kb] = mfma_f32(kv[0], qf[u][0], s[kb]);
                s[kb] = mfma_f32(kv[1], qf[u][1], s[kb]);
            }
        }
        const int n0 = tile * BN;
        const bool need_mask = n0 + BN - 1 > first_pos;
        float mloc = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                float v = s[kb][j] * a.scale_log2;
                if (need_mask && n0 + kb * 32 + g * 16 + j > qpos) v = -INFINITY;
                s[kb][j] = v;
                mloc = fmaxf(mloc, v);
            }
        const float m_new = fmaxf(m_run, wave_max32(mloc));
        const float alpha = exp2f(m_run - m_new);
        m_run = m_new;
        float lsum = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                float e = exp2f(s[kb][j] - m_new);
                s[kb][j] = e;
                lsum += e;
            }
        l_run = l_run * alpha + lsum;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc_o[db][j] *= alpha;
        // O^T[d][q] += V[key][d] P[q][key]; MFMA (kb, j) pairs k = g with key kb*32 + g*16 + j
#pragma unroll
        for (int db = 0; db < 4; ++db) {
            const float* vcol = Vs + g * 16 * V_STRIDE_F32 + db * 32 + col;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    acc_o[db] = mfma_f32(vcol[(kb * 32 + j) * V_STRIDE_F32], s[kb][j], acc_o[db]);
        }
    }

    const float l_tot = l_run + __shfl_xor(l_run, 32);
    const float inv_l = 1.0f / l_tot;
    if (!q_valid) return;
    float* op = (float*)a.o + (long)(q0 + qi) * a.o_tok + (long)head * a.o_head;
    const float* gp = a.gate ? (const float*)a.gate + (long)(q0 + qi) * a.g_tok + (long)head * a.g_head : nullptr;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const int d = db * 32 + jj * 8 + g * 4;
            f32x4 r;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = acc_o[db][jj * 4 + e] * inv_l;
                if (gp) v = v * sigmoidf_(gp[d + e]);
                r[e] = v;
            }
            *(f32x4*)(op + d) = r;
        }
}

}  // namespace hk

// ---------------------------------------------------------------------------
// launcher (called by the C ABI after validation)
// ---------------------------------------------------------------------------
extern "C" int hk_launch_paged_prefill_attention(int dtype, const hk::AttnArgs* args, int head_dim, int n_seqs,
                                                 int n_qblocks, hipStream_t stream) {
    using namespace hk;
    // set once, under C++'s thread-safe static initialisation (replicas launch from several threads);
    // head width 256 holds two 128-wide halves per K / V tile: 131,072 B, one workgroup per CU
    static const bool configured =
        hipFuncSetAttribute((const void*)paged_prefill_attn_16<bf16, 1, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)ATTN16_LDS) == hipSuccess &&
        hipFuncSetAttribute((const void*)paged_prefill_attn_16<f16, 1, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)ATTN16_LDS) == hipSuccess &&
        hipFuncSetAttribute((const void*)paged_prefill_attn_16<bf16, 2, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)(2 * ATTN16_LDS)) == hipSuccess &&
        hipFuncSetAttribute((const void*)paged_prefill_attn_16<f16, 2, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)(2 * ATTN16_LDS)) == hipSuccess;
    if (!configured) return HK_ERR_DEVICE;
    // 16-bit: one workgroup per mirrored pair of q-blocks (head width 128 or 256); fp32: one per
    // q-block (head width 128)
    if (dtype == DT_F32) {
        if (head_dim != 128) return HK_ERR_UNSUPPORTED;
        hipLaunchKernelGGL(paged_prefill_attn_f32, dim3(args->kv_heads, n_seqs, n_qblocks), dim3(256), 0, stream,
                           *args);
        return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
    }
    if (head_dim != 128 && head_dim != 256) return HK_ERR_UNSUPPORTED;
    const dim3 grid(args->kv_heads, (n_qblocks + 1) / 2, n_seqs);
    const bool bf = dtype == DT_BF16;
    if (head_dim == 128) {
        if (bf)
            hipLaunchKernelGGL((paged_prefill_attn_16<bf16, 1, false>), grid, dim3(256), ATTN16_LDS, stream, *args);
        else
            hipLaunchKernelGGL((paged_prefill_attn_16<f16, 1, false>), grid, dim3(256), ATTN16_LDS, stream, *args);
    } else {
        if (bf)
            hipLaunchKernelGGL((paged_prefill_attn_16<bf16, 2, false>), grid, dim3(256), 2 * ATTN16_LDS, stream, *args);
        else
            hipLaunchKernelGGL((paged_prefill_attn_16<f16, 2, false>), grid, dim3(256), 2 * ATTN16_LDS, stream, *args);
    }
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}

template <typename T, int NH>
static int launch_split(const hk::AttnArgs* a, int n_seqs, hipStream_t stream) {
    using namespace hk;
    auto kern = paged_prefill_attn_16<T, NH, true>;
    static const bool configured = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)(NH * ATTN16_LDS)) == hipSuccess;
    if (!configured) return HK_ERR_DEVICE;
    hipLaunchKernelGGL(kern, dim3(a->kv_heads, n_seqs, a->n_qblocks * a->n_split), dim3(256), NH * ATTN16_LDS, stream, *a);
    hipLaunchKernelGGL((attn_combine<T, NH>), dim3(a->kv_heads, a->n_qblocks * (128 / (NH == 1 ? 8 : 4)), n_seqs), dim3(256), 0,
                       stream, *a);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_DEVICE;
}

// 16-bit types, head_dim 128 or 256; the caller has sized part and part_ml
extern "C" int hk_launch_paged_prefill_attention_split(int dtype, const hk::AttnArgs* a, int head_dim, int n_seqs,
                                                       hipStream_t stream) {
    if (head_dim == 128)
        return dtype == hk::DT_BF16 ? launch_split<hk::bf16, 1>(a, n_seqs, stream) : launch_split<hk::f16, 1>(a, n_seqs, stream);
    if (head_dim == 256)
        return dtype == hk::DT_BF16 ? launch_split<hk::bf16, 2>(a, n_seqs, stream) : launch_split<hk::f16, 2>(a, n_seqs, stream);
    return HK_ERR_UNSUPPORTED;
}
