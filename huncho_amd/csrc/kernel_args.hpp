// kernel_args.hpp - argument blocks passed by value to the gfx950 kernels, and the
// launcher entry points the host side of the ABI calls after validation.
#pragma once

#include <hip/hip_runtime.h>

namespace hk {

struct AttnArgs {
    const void* q;
    long q_tok, q_head;
    const void* k_pool;
    const void* v_pool;
    int page_shift;  // log2(page_size)
    const int* block_tables;
    int bt_stride;
    const int* cu_seqlens_q;
    const int* context_lens;
    int q_heads, kv_heads, group, pos_per_block;
    float scale_log2;  // softmax scale * log2(e)
    const void* gate;
    long g_tok, g_head;
    void* o;
    long o_tok, o_head;
    int num_pages;
    int n_tokens;
    int* fault;
    // key-split kernel: the tiles of each q-block of a row of at least split_from tiles in at most n_split
    // ranges; part holds the ranges' unnormalised fp32 O rows, part_ml their (row max, row sum) pairs
    int n_split, split_from, n_qblocks;
    float* part;
    float* part_ml;
};

struct GdnArgs {
    const void* q;
    const void* k;
    const void* v;
    long q_tok, k_tok, v_tok;  // token strides (elements); head stride is dk (q,k) / dv (v)
    int qk_rep;                // value heads per key head
    const float* g;
    const float* beta;
    long gb_tok;
    const int* cu_seqlens;
    const float* initial_state;  // [n_seqs][H][dk][dv] or null
    float* final_state;          // [n_seqs][H][dk][dv] or null
    void* o;
    long o_tok;
    int H;
    int n_tokens;
    int* fault;
    // per-sequence state rows [H][dk][dv] (replace initial_state / final_state when set; a
    // null entry is a zero initial state / no final state)
    const float* const* init_rows;
    float* const* final_rows;
};

// Gated DeltaNet layer body read straight from the fused in_proj output (gdn16 FUSED mode).
struct GdnFusedArgs {
    const void* mixed;     // token rows [q(Hk*128) | k(Hk*128) | v(H*128) | ...]
    long mixed_tok;
    const float* conv_w;   // [conv_dim][4]
    int conv_dim;
    const void* hist;      // [n_seqs][conv_dim][3] cached conv tail or null
    void* tail_out;        // [n_seqs][conv_dim][3] new tail or null
    const void* ba;        // b at column b_col, a at column a_col of each token row
    long ba_tok;
    int b_col, a_col;
    const float* base_g;   // -exp(A_log) [H]
    const float* dt_bias;  // [H]
    float scale;           // q scale (128^-1/2)
    int Hk;
    const void* z;         // gate z at [t * z_tok + h * 128 + i]
    long z_tok;
    const float* norm_w;   // [128] gated-norm weight
    float eps;
    // per-sequence conv rows [conv_dim][3] (replace hist / tail_out when set; a null entry is
    // a zero history / no tail)
    const void* const* hist_rows;
    void* const* tail_rows;
};

// Scratch bytes of one (64-token chunk, head) of the fused layer for few, long rows (gdn16_split.hip)
constexpr int HK_GDN_SPLIT_SLOT = 114688;

// Scratch bytes of one (64-token chunk, head) of the fp32 delta rule for few rows (delta_rule_split.hip)
constexpr int HK_DELTA_SPLIT_SLOT = 4 * (2 * 64 * 64 + 4 * 64 + 64 * 128 + 128 * 128);

struct KvArgs {
    const void* q_in;
    long q_in_tok, q_in_head;
    const void* k_in;
    long k_in_tok;
    const void* v_in;
    long v_in_tok;
    const float* q_norm;  // (1 + w) or null
    const float* k_norm;
    float eps;
    const float* rope_cos;  // [max_pos][rd/2] or null
    const float* rope_sin;
    int rd, rope_max_pos;
    const int* cu_seqlens_q;
    const int* context_lens;
    int n_seqs, n_tokens;
    const int* block_tables;
    int bt_stride, num_pages, page_shift;
    int q_heads, kv_heads;
    void* q_out;
    long q_out_tok, q_out_head;
    void* k_pool;
    void* v_pool;
    int* fault;
    // [n_tokens] (sequence, absolute position) pairs, or null: then each token's pair is found
    // from cu_seqlens_q and context_lens
    const int* tok_sp;
};

struct PrepArgs {
    const void* mixed;
    long mixed_tok;
    const float* conv_w;  // [conv_dim][K]
    int K;
    const void* hist;  // [n_seqs][conv_dim][K-1] or null
    const void* ba;    // b at col b_col, a at col a_col of each token row
    long ba_tok;
    int b_col, a_col;
    const float* base_g;   // -exp(A_log) [Hv]
    const float* dt_bias;  // [Hv]
    const int* cu_seqlens;
    int n_seqs, n_tokens;
    int Hk, Hv;
    float scale;
    void* q_out;
    void* k_out;
    void* v_out;
    float* g_out;
    float* beta_out;
    int* fault;
    // per-sequence conv rows [conv_dim][K-1] (replace hist / the tail output when set; a null
    // entry is a zero history / no tail)
    const void* const* hist_rows;
    void* const* tail_rows;
    int dk, dv;  // head widths: q / k rows (Hk of dk) and v rows (Hv of dv), each at most 256
};

struct NormArgs {
    const void* x;
    long x_tok;
    const float* w;
    float eps;
    int rows, width;
    void* y;
    long y_tok;
    int x_f32;  // x is fp32 (a residual stream kept in fp32) instead of the dtype
};

struct GatedNormArgs {
    const void* x;  // [rows][width] contiguous (rows = tokens * heads)
    const void* z;  // token-strided: z[t * z_tok + h * width + i]
    long z_tok;
    int heads;
    const float* w;
    float eps;
    int rows, width;
    void* y;  // [rows][width]
};

struct SwigluArgs {
    const void* gu;  // gate at [t * gu_tok + i], up at [t * gu_tok + up_off + i]
    long gu_tok, up_off;
    int rows, width;
    void* y;
};

// ModernBERT encoder (bert.hip)
struct BertAttnArgs {
    const void* q;  // [tokens][heads][64] at token stride q_tok (elements)
    long q_tok;
    const void* k;
    long k_tok;
    const void* v;
    long v_tok;
    void* o;
    long o_tok;
    const int* cu;
    int n_seqs, n_tokens, heads;
    int half_window;   // keys with |i - j| <= half_window; < 0: the whole sequence
    float scale_log2;  // softmax scale * log2(e)
    int* fault;
    int qblocks;  // query blocks per (sequence, head) in the 16-bit grid (set by the launcher)
    // optional NeoX RoPE of q applied as the 16-bit kernel loads it ([max_pos][32] tables;
    // null: q is used as given)
    const float* rope_cos;
    const float* rope_sin;
    int rope_max_pos;
};

struct LayerNormArgs {
    const void* x;
    long x_tok;
    const float* w;
    float eps;
    int rows, width;
    void* y;
    long y_tok;
    const float* b;  // bias [width] or null (ModernBERT's LayerNorms have none)
};

// typed Laya head (laya_head.hip)
struct LayaTypeArgs {
    const void* x;  // [rows][width] at x_tok
    long x_tok;
    const float* type_emb;  // [n_types][width]
    const int* cu;          // [n_seqs + 1]
    int n_seqs;
    int qtype[64];          // per sequence
    int rows, width;
    void* y;
    long y_tok;
};
struct LayaBiasArgs {
    const void* x;
    long x_tok;
    const float* b;    // [width]
    const void* res;   // residual rows or null
    long res_tok;
    int rows, width;
    void* y;
    long y_tok;
};
struct LayaGatherArgs {
    const void* x;
    long x_tok;
    const int* cu;            // [n_seqs + 1] token rows
    const int* cu_positions;  // [n_seqs + 1] into positions
    const int* positions;     // relative to the sequence
    int n_seqs, n_positions, width;
    void* y;                  // [n_positions][width]
};
struct LayaScoreArgs {
    const void* y;  // [n_positions][width]
    const float* w;  // [width]
    float b;
    int n_positions, width;
    float* out;
};

struct GegluArgs {
    const void* x;  // x1 at [t * x_tok + i], x2 at [t * x_tok + width + i]
    long x_tok;
    int rows, width;
    void* y;
    long y_tok;
};

struct RopeQkArgs {
    void* x;  // rows [q (heads x 64) | k (heads x 64) | ...] at token stride x_tok
    long x_tok;
    const float* cos;  // [max_pos][32]
    const float* sin;
    int max_pos, heads;
    const int* cu;
    int n_seqs, n_tokens;
    int* fault;
    int k_only;  // rotate only the k part (q is rotated by the attention kernel as it loads it)
};

// Mean-pool partial sums per sequence (slot rows of MeanPoolArgs::pool).
constexpr int POOL_PARTS = 32;

struct MeanPoolArgs {
    const void* x;
    long x_tok;
    const int* cu;
    int n_seqs, n_tokens, width;
    const void* head_w;  // [n_out][width], model dtype
    const float* head_b;  // [n_out] or null
    int n_out;
    float* logits;  // [n_seqs][n_out]
    int* fault;
    float* pool;  // [n_seqs][32][width] fp32 partial sums (sequence s: slot rows 32 s .. 32 s + min(32, L) - 1)
};

// Readout at request positions (Qwen3_5Backend::readout, qwen3_5.rs:3196-3255): the
// final-normed hidden row at each position and, with a pointer head, its fp32 score.
struct ReadoutArgs {
    const void* x;              // residual stream before the final norm [tokens][width]
    long x_tok;
    const int* cu;              // token cu_seqlens [n_seqs + 1]
    const int* cu_pos;          // [n_seqs + 1] offsets into positions
    const int* positions;       // [n_positions], relative to each row's tokens
    int n_seqs, n_positions, width;
    const float* w_eff;         // final norm (1 + w) [width]
    float eps;
    void* hidden_out;           // [n_positions][width] model dtype, or null
    const float *q_w, *q_b, *k_w, *k_b;  // pointer head [head_dim][width] / [head_dim], fp32
    int head_dim;
    float scale;                // 1 / sqrt(head_dim)
    float* scores;              // [n_positions] fp32, or null
    int* fault;
    int x_f32;                  // x is fp32 (a residual stream kept in fp32) instead of the dtype
};

// Dense projection Y = X W^T with a fused epilogue (gemm.hip; gemm_few_rows.hip for few rows, which
// also has EPI_RESIDUAL_F32: fp32 rows of c and y, the fp32 residual stream; and EPI_GEGLU: y =
// T(gelu(T(g)) * T(u)) of w's first and second N / 2 rows).
enum { EPI_STORE = 0, EPI_RESIDUAL = 1, EPI_SWIGLU = 2, EPI_RESIDUAL_F32 = 3, EPI_GEGLU = 4 };
struct GemmArgs {
    const void* x;  // [M][K], row stride ldx
    const void* w;  // [N][K], row stride ldw
    const void* c;  // EPI_RESIDUAL: [M][N], row stride ldc (may alias y)
    void* y;        // [M][N] (EPI_SWIGLU: [M][N / 2])
    long ldx, ldw, ldc, ldy;
    int M, N, K;
    // gemm_few_rows.hip, EPI_STORE: a second projection of the same x rows, Y2 = X W2^T (row stride of
    // w2 = ldw); N2 = 0: none
    const void* w2;
    void* y2;
    long ldy2;
    int N2;
};

}  // namespace hk

extern "C" {
int hk_launch_paged_prefill_attention(int dtype, const hk::AttnArgs* args, int head_dim, int n_seqs, int n_qblocks,
                                      hipStream_t stream);
int hk_launch_paged_prefill_attention_split(int dtype, const hk::AttnArgs* args, int head_dim, int n_seqs,
                                            hipStream_t stream);
int hk_launch_gated_delta_chunked(int dtype, const hk::GdnArgs* args, int n_seqs, hipStream_t stream);
int hk_launch_gdn16(int dtype16, int fused, const hk::GdnArgs* a, const hk::GdnFusedArgs* fa, int n_seqs,
                    hipStream_t stream);
int hk_launch_qk_norm_rope_kv_write(int dtype, const hk::KvArgs* args, int head_dim, hipStream_t stream);
int hk_launch_gdn_prep(int dtype, const hk::PrepArgs* a, void* tail_out, hipStream_t st);
int hk_launch_rms_norm(int dtype, const hk::NormArgs* a, hipStream_t st);
int hk_launch_gated_rms_norm(int dtype, const hk::GatedNormArgs* a, hipStream_t st);
int hk_launch_swiglu(int dtype, const hk::SwigluArgs* a, hipStream_t st);
int hk_launch_embed(int dtype, int x_f32, const int* ids, int n, const void* table, int vocab, int width, void* out,
                    int* fault, hipStream_t st);
int hk_launch_final_norm_head(int dtype, int x_f32, const void* x, long x_tok, const int* cu, int n_seqs,
                              const float* w_eff, float eps, int width, const void* head_w, const float* head_b,
                              int n_out, float* logits, void* h_out, hipStream_t st);
int hk_launch_seq_lens(const int* cu, int n, int* out, hipStream_t st);
// out[t] = (sequence of token t, its absolute position ctxl[s] - q_len + (t - q0)) as int pairs;
// a sequence whose range lies outside [0, n_tokens) sets fault bit 1 and writes nothing
int hk_launch_token_seq_pos(const int* cu, const int* ctxl, int n_seqs, int n_tokens, int* out, int* fault,
                            hipStream_t st);
int hk_launch_readout(int dtype, const hk::ReadoutArgs* a, hipStream_t st);
int hk_launch_delta_split(const hk::GdnArgs* a, int n_seqs, int n_slots, void* scratch, hipStream_t stream);
int hk_launch_gdn16_split(int dtype16, const hk::GdnArgs* a, const hk::GdnFusedArgs* fa, int n_seqs, int n_slots,
                          void* scratch, hipStream_t stream);
int hk_launch_gemm(int dtype16, int epi, const hk::GemmArgs* a, hipStream_t stream);
float hk_gemm_few_rows_cost(int epi, const hk::GemmArgs* a);
int hk_launch_gemm_few_rows(int dtype16, int epi, const hk::GemmArgs* a, hipStream_t stream);
int hk_launch_gemm_few_rows_tile(int dtype16, int epi, const hk::GemmArgs* a, int i, int deep, hipStream_t stream);
int hk_launch_lora_merge(int dtype, void* w, long rows, int cols, const float* a, const float* b, int rank, float scale,
                         hipStream_t st);
int hk_launch_bidir_attention(int dtype, const hk::BertAttnArgs* a, int n_seqs, int max_len, hipStream_t stream);
int hk_launch_layer_norm(int dtype, const hk::LayerNormArgs* a, hipStream_t stream);
int hk_launch_laya_type_add(int dtype, const hk::LayaTypeArgs* a, hipStream_t stream);
int hk_launch_laya_bias_act(int dtype, int act, const hk::LayaBiasArgs* a, hipStream_t stream);
int hk_launch_laya_gather(int dtype, const hk::LayaGatherArgs* a, hipStream_t stream);
int hk_launch_laya_score(int dtype, const hk::LayaScoreArgs* a, hipStream_t stream);
int hk_launch_geglu(int dtype, const hk::GegluArgs* a, hipStream_t stream);
int hk_launch_rope_qk(int dtype, const hk::RopeQkArgs* a, int n_seqs, int max_len, hipStream_t stream);
int hk_launch_mean_pool_head(int dtype, const hk::MeanPoolArgs* a, int n_seqs, hipStream_t stream);
// general.hip: head widths other than 128 (each at most 256)
int hk_launch_kv_write_gen(int dtype, const hk::KvArgs* a, int hd, hipStream_t st);
int hk_launch_attention_gen(int dtype, const hk::AttnArgs* a, int hd, int n_seqs, hipStream_t st);
int hk_launch_delta_gen(int dtype, const hk::GdnArgs* a, int dk, int dv, int n_seqs, hipStream_t st);
size_t hk_delta_gen_lds(int dk, int dv);
int hk_launch_rope_qk_gen(int dtype, const hk::RopeQkArgs* a, int hd, int n_seqs, int max_len, hipStream_t st);
int hk_launch_bidir_gen(int dtype, const hk::BertAttnArgs* a, int hd, hipStream_t st);
}
