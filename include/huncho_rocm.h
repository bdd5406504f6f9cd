/*
 * huncho_rocm.h - C ABI of libhuncho_rocm, the MI355X (gfx950) implementation of Huncho's
 * Kev/Qwen3.5 scoring-forward (prefill) path.
 *
 * The reference boundary is the Rust `huncho_core::backend::Backend` trait
 * (crates/huncho-core/src/backend.rs:213-438) implemented for Kev by `Qwen3_5Backend`
 * (crates/huncho-backend/src/qwen3_5.rs:2514-2935). A thin Rust FFI crate binds this header
 * and keeps that trait's contract (see INTEGRATION.md in the repository). Each entry point
 * below names the reference function whose numerics it replaces.
 *
 * Conventions
 *   - Every pointer argument named *_dev is device memory owned by the caller; nothing is
 *     retained after the call returns. Host pointers are named *_host.
 *   - All work is stream-ordered on the context's stream (hk_ctx_set_stream), so calls
 *     return before the GPU finishes; hk_ctx_synchronize waits.
 *   - Returns HK_OK (0) or an error code; hk_ctx_last_error() gives the message. Shapes,
 *     strides and dtypes are validated before any launch. Data-dependent faults found on
 *     the device (block-table entry or token id out of range, malformed cu_seqlens) skip
 *     the offending writes and set the context's fault flag, read and cleared by
 *     hk_ctx_take_faults (no partial cache commit: the caller commits only after a clean
 *     forward, as qwen3_5.rs:2747-2751 does).
 *   - Activations are token-major: [tokens][heads][head_dim]; varlen batches are
 *     delimited by cu_seqlens (int32, n_seqs + 1 entries, cu[0] = 0).
 *   - Paged KV pools are [num_pages][kv_heads][page_size][head_dim]: one pool page holds
 *     what one reference Page holds ([1, Hkv, rows, d], qwen3_5/kv_pages.rs:18-22). Token j
 *     of sequence s lives in page block_tables[s * bt_stride + j / page_size], slot
 *     j % page_size. page_size is a power of two in 16..256 (qwen3_5.rs parsers,
 *     huncho-cli/src/load.rs:679-747).
 *   - A context is used by one thread at a time (the engine serialises calls per model,
 *     crates/huncho-core/src/engine.rs:175-178); distinct contexts are independent.
 */
#ifndef HUNCHO_ROCM_H
#define HUNCHO_ROCM_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define HK_OK 0
#define HK_ERR_INVALID 1     /* bad argument, shape or stride  -> Error::Backend / Request */
#define HK_ERR_UNSUPPORTED 2 /* shape or dtype this build does not implement -> Error::Unsupported */
#define HK_ERR_DEVICE 3      /* HIP runtime / launch failure -> Error::Backend */
#define HK_ERR_NOMEM 4       /* allocation failed (context, model creation, hk_buffer_alloc) */

#define HK_F32 0
#define HK_BF16 1
#define HK_F16 2

/* Device fault bits reported by hk_ctx_take_faults. */
#define HK_FAULT_SEQLENS 1   /* cu_seqlens / context_lens inconsistent for a token */
#define HK_FAULT_PAGE 2      /* block-table entry outside [0, num_pages) or past bt_stride */
#define HK_FAULT_ROPE 4      /* position beyond the RoPE table */
#define HK_FAULT_TOKEN 8     /* token id outside the vocabulary */
#define HK_FAULT_RANGE 16    /* a non-finite Gated DeltaNet output row: an fp16 MFMA operand of the
                                16-bit recurrence (|x| > 65504) overflowed */

typedef struct hk_ctx hk_ctx;

typedef struct {
    char name[64];          /* gcnArchName, e.g. "gfx950:sramecc+:xnack-" */
    int compute_units;
    int clock_khz;
    int mem_clock_khz;
    int mem_bus_width;
    size_t total_mem;
    size_t lds_per_block;
    int l2_bytes;
} hk_device_info_t;

/* ---- context (replaces device selection, crates/huncho-backend/src/device.rs:12-72) ---- */
/* Fails with HK_ERR_UNSUPPORTED when no GPU is visible (hipGetDeviceCount == 0).
 * The context holds 512 MiB of device scratch for batches of few, long rows (hk_gdn_fused,
 * hk_gated_delta_chunked in fp32, hk_paged_prefill_attention on suffixes, and the models' layers), from
 * here to hk_ctx_destroy (another 512 MiB once it has used it on two streams). Which kernel a call takes follows from its sizes,
 * and whether its stream is being captured: a captured call runs without the scratch, as does a context
 * that could not have it. For the fp32 delta rule and the suffix attention the two differ by the
 * rounding of their sums. */
int hk_ctx_create(int device_ordinal, hk_ctx** out);
int hk_ctx_destroy(hk_ctx* ctx);
/* Work is ordered on this hipStream_t from now on (NULL: HIP's null stream). A new
 * context uses its own default-priority stream, returned by hk_ctx_own_stream. */
int hk_ctx_set_stream(hk_ctx* ctx, void* hip_stream);
void* hk_ctx_stream(hk_ctx* ctx);
void* hk_ctx_own_stream(hk_ctx* ctx);
int hk_ctx_synchronize(hk_ctx* ctx);
const char* hk_ctx_last_error(hk_ctx* ctx);
int hk_ctx_device_info(hk_ctx* ctx, hk_device_info_t* out);
/* Synchronises, returns the OR of HK_FAULT_* bits raised since the last call, clears them. */
int hk_ctx_take_faults(hk_ctx* ctx, int* faults_out);
int hk_device_count(int* out);
const char* hk_version(void);

/* ---- dense projections ------------------------------------------------------------
 * The context's GEMM algorithm per shape is a deterministic function of the shape by default:
 * the library's own few-row kernel where a 16-bit product has few rows, else a solution pinned for
 * the shape at build time, else hipBLASLt's heuristic first choice. The GEMM handle and workspace are created with the first model on the context, so a forward
 * never allocates, times or synchronises. hk_ctx_set_gemm_autotune(ctx, 1) makes shapes first
 * seen afterwards time every supported hipBLASLt solution instead (allocates scratch and synchronises
 * on that first use; the choice then follows the device's timing). No reference counterpart:
 * candle's Linear (qwen3_5.rs:306-515) calls its BLAS with the library's own choice.
 * hk_ctx_gemm_plans writes one line per cached plan ("dtype= out= n= in= ... index= source")
 * into buf (NUL-terminated, truncated to len) and the full length + 1 into *needed. */
int hk_ctx_set_gemm_autotune(hk_ctx* ctx, int enable);
int hk_ctx_gemm_plans(hk_ctx* ctx, char* buf, size_t len, size_t* needed);

/* Dense projection on the library's own MFMA kernel (candle Linear, qwen3_5.rs:306-515), 16-bit
 * dtypes: y [rows][.] = epilogue(x [rows][in] . w [out][in]^T), fp32 accumulation, with
 *   epilogue 0: y = acc                      (y [rows][out])
 *   epilogue 1: y = acc + c                  (the residual add of DecoderLayer::forward,
 *                                             1083-1104; c [rows][out] may alias y)
 *   epilogue 2: y = silu(g) * u              (Mlp::forward 1020-1031 and gate_cpu::silu_mul 8-47,
 *                                             g and u rounded to the dtype first as the reference
 *                                             stores them; w holds blocks of 32 rows [16 gate rows |
 *                                             the 16 matching up rows], y [rows][out / 2], output
 *                                             column 16 b + i from w rows 32 b + i and 32 b + 16 + i)
 * out must be a multiple of 256 and in of 64; rows and pointers 16-byte aligned. */
int hk_linear(hk_ctx* ctx, int dtype, int epilogue, const void* x_dev, long ldx, const void* w_dev, long ldw,
              int rows, int out, int in, const void* c_dev, long ldc, void* y_dev, long ldy);

/* ---- device memory for callers without a HIP binding (the Rust FFI crate): plain
 * hipMalloc / hipFree on the context's device, stream-ordered copies on the context's
 * stream. hk_memcpy_d2h returns after the copy has completed. -------------------------- */
int hk_buffer_alloc(hk_ctx* ctx, size_t bytes, void** dev_out);
int hk_buffer_free(hk_ctx* ctx, void* dev);
int hk_memcpy_h2d(hk_ctx* ctx, void* dev_dst, const void* host_src, size_t bytes);
int hk_memcpy_d2h(hk_ctx* ctx, void* host_dst, const void* dev_src, size_t bytes);

/* ---- RoPE tables (qwen3_5.rs:220-247: inv_freq = theta^(-2i/rd) in f32, cos/sin of
 * pos * inv_freq in f32, cast to the model dtype) -----------------------------------------------
 * Host-side helper: fills cos_host/sin_host [max_pos][rd/2] for upload; round_dtype HK_BF16 /
 * HK_F16 rounds the values to that type (HK_F32: no rounding). */
int hk_rope_fill_table(int rotary_dim, double theta, int max_pos, int round_dtype, float* cos_host,
                       float* sin_host);

/* ---- fused q/k norm + partial RoPE + paged KV append -------------------------------------
 * Replaces qwen3_5.rs:596-624 (q/gate split, q_norm/k_norm, apply_partial_rotary, page
 * append) and kv_pages.rs:307-341. New token i of sequence s has absolute position
 * context_lens[s] - q_len(s) + i. q_norm_eff/k_norm_eff are (1 + w) in fp32, or NULL to
 * skip the norm; rope_cos/rope_sin NULL skips RoPE. head_dim 1..256 (128 and 256 on the
 * vectorised kernel for HK_BF16 / HK_F16 with 16-byte aligned rows and tables, other widths
 * and cases on a general one). q_out may alias q_in (the q half of the fused projection is
 * rotated in place). */
int hk_qk_norm_rope_kv_write(hk_ctx* ctx, int dtype, const void* q_in_dev, long q_in_tok, long q_in_head,
                             const void* k_in_dev, long k_in_tok, const void* v_in_dev, long v_in_tok,
                             const float* q_norm_eff_dev, const float* k_norm_eff_dev, float eps,
                             const float* rope_cos_dev, const float* rope_sin_dev, int rotary_dim,
                             int rope_max_pos, const int32_t* cu_seqlens_q_dev, const int32_t* context_lens_dev,
                             int n_seqs, int n_tokens, const int32_t* block_tables_dev, int bt_stride,
                             int num_pages, int page_size, int q_heads, int kv_heads, int head_dim,
                             void* q_out_dev, long q_out_tok, long q_out_head, void* k_pool_dev,
                             void* v_pool_dev);

/* ---- paged KV append only (kv_pages.rs:307-341): k/v [n_tokens][kv_heads][head_dim] ---- */
int hk_paged_kv_write(hk_ctx* ctx, int dtype, const void* k_dev, const void* v_dev,
                      const int32_t* cu_seqlens_q_dev, const int32_t* context_lens_dev, int n_seqs,
                      int n_tokens, const int32_t* block_tables_dev, int bt_stride, int num_pages,
                      int page_size, int kv_heads, int head_dim, void* k_pool_dev, void* v_pool_dev);

/* ---- paged GQA causal prefill attention ----------------------------------------------------
 * Replaces the attention core of Attention::forward (qwen3_5.rs:626-703), grouped GQA and
 * query blocks (qwen3_5/attention.rs:6-111) and direct page attention
 * (qwen3_5/kv_pages.rs:104-174): O = softmax(Q K^T * scale + causal) V with query head h
 * reading KV head h / (q_heads / kv_heads). Sequence s has q_len(s) new queries at
 * positions context_lens[s] - q_len(s) .. context_lens[s] - 1 and keys 0..pos through its
 * block table. max_q_len bounds q_len over the batch. gate_dev (optional) applies
 * o *= sigmoid(gate) (qwen3_5.rs:706-714). head_dim 1..256 and any q_heads / kv_heads group:
 * head_dim 128 (any dtype) or 256 (HK_BF16 / HK_F16) with a group of 1, 2, 4 or 8 runs on the
 * MFMA kernels (16-byte aligned rows required), every other shape on a general kernel (one wave
 * per query row, keys in order).
 * dtype HK_F32: fp32 everywhere; HK_BF16 / HK_F16: 16-bit in/out, fp32 accumulation and softmax. */
int hk_paged_prefill_attention(hk_ctx* ctx, int dtype, const void* q_dev, long q_tok, long q_head,
                               const void* k_pool_dev, const void* v_pool_dev, int num_pages, int page_size,
                               const int32_t* block_tables_dev, int bt_stride, const int32_t* cu_seqlens_q_dev,
                               const int32_t* context_lens_dev, int n_seqs, int n_tokens, int max_q_len,
                               int q_heads, int kv_heads, int head_dim, float scale, const void* gate_dev,
                               long gate_tok, long gate_head, void* o_dev, long o_tok, long o_head);

/* ---- chunked gated delta rule ------------------------------------------------------------------
 * Replaces recurrent_gated_delta (qwen3_5.rs:950-987) / delta_cpu::recurrent
 * (delta_cpu.rs:29-138). q,k [tokens][k_heads][dk] (token strides q_tok/k_tok),
 * v [tokens][heads][dv], g/beta fp32 [tokens][heads], value head h reads key head
 * h / (heads / k_heads). initial_state (optional, fp32 [n_seqs][heads][dk][dv], the carried
 * cache state) and final_state (optional, same shape) may alias. o [tokens][heads][dv] with
 * token stride o_tok. dk = dv = 128 runs an equal chunked (C = 64) MFMA algorithm (16-bit rows
 * 16-byte aligned); other widths (each 1..256, dk * dv <= 32768) run the per-token recurrence
 * itself on a general kernel. */
int hk_gated_delta_chunked(hk_ctx* ctx, int dtype, const void* q_dev, long q_tok, const void* k_dev, long k_tok,
                           const void* v_dev, long v_tok, const float* g_dev, const float* beta_dev,
                           const int32_t* cu_seqlens_dev, int n_seqs, int n_tokens, int heads, int k_heads,
                           int dk, int dv, const float* initial_state_dev, float* final_state_dev, void* o_dev,
                           long o_tok);

/* ---- GDN input prep -----------------------------------------------------------------------------
 * Replaces LinearAttn::forward up to the recurrence (qwen3_5.rs:846-925): causal depthwise
 * conv (conv_w [conv_dim][K] fp32, ascending taps, conv_cpu.rs:34-48) + SiLU over the
 * q|k|v channels of `mixed` (token stride mixed_tok), with the cached conv tail
 * (conv_hist, [n_seqs][conv_dim][K-1], optional) prepended; l2norm of q and k per head,
 * q * dk^-1/2; beta = sigmoid(b); g = base_g * softplus(a + dt_bias) with
 * base_g = -exp(A_log). b and a are read at columns b_col/a_col of `ba` rows. Outputs
 * q,k [tokens][k_heads][128], v [tokens][heads][128], g/beta fp32 [tokens][heads], and the
 * new conv tail (optional). conv_dim = (2 * k_heads + heads) * 128. */
int hk_gdn_prep(hk_ctx* ctx, int dtype, const void* mixed_dev, long mixed_tok, const float* conv_w_dev, int conv_k,
                const void* conv_hist_dev, const void* ba_dev, long ba_tok, int b_col, int a_col,
                const float* base_g_dev, const float* dt_bias_dev, const int32_t* cu_seqlens_dev, int n_seqs,
                int n_tokens, int heads, int k_heads, void* q_out_dev, void* k_out_dev, void* v_out_dev,
                float* g_out_dev, float* beta_out_dev, void* conv_tail_out_dev);

/* ---- fused Gated DeltaNet layer body (16-bit dtypes) ------------------------------------------
 * Replaces LinearAttn::forward between in_proj and out_proj (qwen3_5.rs:846-940) in one
 * kernel: causal depthwise conv (conv_w [conv_dim][4] fp32, cached tail conv_hist
 * [n_seqs][conv_dim][3] optional) + SiLU over the q|k|v channels at the start of each
 * `mixed` row, l2norm of q and k, q * 128^-1/2, beta = sigmoid(b), g = base_g *
 * softplus(a + dt_bias), the chunked gated delta rule (states as in
 * hk_gated_delta_chunked), and the gated RMSNorm rms(o) * norm_w * silu(z) (193-201).
 * out [tokens][heads][128] (token stride out_tok) is the out_proj input. Rows of mixed / z /
 * out must be 16-byte aligned with strides that are multiples of 8 elements. */
int hk_gdn_fused(hk_ctx* ctx, int dtype, const void* mixed_dev, long mixed_tok, const float* conv_w_dev, int conv_k,
                 const void* conv_hist_dev, void* conv_tail_out_dev, const void* ba_dev, long ba_tok, int b_col,
                 int a_col, const float* base_g_dev, const float* dt_bias_dev, const void* z_dev, long z_tok,
                 const float* norm_w_dev, float eps, const int32_t* cu_seqlens_dev, int n_seqs, int n_tokens,
                 int heads, int k_heads, const float* initial_state_dev, float* final_state_dev, void* out_dev,
                 long out_tok);

/* ---- norms and gates (qwen3_5.rs:184-201, 1020-1031) -------------------------------------------- */
int hk_rms_norm(hk_ctx* ctx, int dtype, const void* x_dev, long x_tok, const float* w_eff_dev, float eps, int rows,
                int width, void* y_dev, long y_tok);
int hk_gated_rms_norm(hk_ctx* ctx, int dtype, const void* x_dev, const void* z_dev, long z_tok, int heads,
                      const float* w_dev, float eps, int rows, int width, void* y_dev);
int hk_swiglu(hk_ctx* ctx, int dtype, const void* gu_dev, long gu_tok, long up_off, int rows, int width, void* y_dev);

/* ---- Kev-shaped hybrid model (qwen3_5.rs:1283-1553 forward; Backend::forward_batch,
 * qwen3_5.rs:3138-3194) -------------------------------------------------------------------------------*/
typedef struct {
    int hidden, n_layers, n_heads, n_kv_heads, head_dim, intermediate, vocab;
    float eps;
    double rope_theta;
    int rotary_dim;
    int conv_k, lin_key_dim, lin_n_k_heads, lin_n_v_heads, lin_v_dim;
    int page_size;          /* KV pool page (power of two 16..256) */
    int max_context;        /* longest sequence the model accepts (RoPE table size) */
    int n_out;              /* decision-head outputs (0 = no head) */
    const int32_t* layer_types_host; /* per layer: 0 = Gated DeltaNet, 1 = full attention */
    /* 16-bit models only: 0 keeps the residual stream in the model dtype, rounded after every
     * residual add as the reference stores it (DecoderLayer::forward, qwen3_5.rs:1083-1104);
     * 1 keeps it in fp32: the embedding rows are widened, the output projections (o_proj,
     * out_proj, down_proj) add their fp32 products to it unrounded, and the norms read it in
     * fp32. Mixer and MLP internals keep the model dtype's storage points either way. */
    int residual_fp32;
} hk_kev_config;

/* Per-layer weights, device memory in the model dtype unless noted, PyTorch [out][in]
 * layout. Norm weights are the raw checkpoint values (the model bakes 1 + w itself). */
typedef struct {
    const void *input_norm, *post_norm;                 /* [hidden] */
    const void *gate_proj, *up_proj, *down_proj;
    const void *in_qkv, *in_z, *in_b, *in_a, *out_proj; /* linear attention */
    const void *conv_w;                                 /* [conv_dim][1][K] */
    const void *norm_w, *a_log, *dt_bias;
    const void *q_proj, *k_proj, *v_proj, *o_proj;      /* full attention */
    const void *q_norm, *k_norm;
} hk_kev_layer_weights;

/* LoRA merge at load time (merge_lora_into_map, qwen3_5.rs:1597-1640): in place,
 * w = dtype(w + scale * (b . a)) with the delta formed and added in fp32. w [rows][cols] in dtype
 * (the base weight, PyTorch [out][in]); a = lora_A [rank][cols] and b = lora_B [rows][rank] as
 * fp32; scale = lora_alpha / r. Run on the staged checkpoint tensors before hk_kev_model_create,
 * as the reference merges before building its model. */
int hk_lora_merge(hk_ctx* ctx, int dtype, void* w_dev, int rows, int cols, const float* a_dev, const float* b_dev,
                  int rank, float scale);

typedef struct hk_kev_model hk_kev_model;

/* Loads (copies and fuses) the weights; the caller's buffers may be freed afterwards. Waits for
 * the work queued on the context's stream first (staged tensors may come from it) and returns
 * once the copies are complete (load time only: model and head creation block the host).
 * head_w [n_out][hidden] (model dtype), head_b [n_out] fp32 or NULL. Head widths: head_dim,
 * lin_key_dim and lin_v_dim each 1..256 with lin_key_dim * lin_v_dim <= 32768; 128-wide heads
 * run on the MFMA kernels (16-bit models: the fused Gated DeltaNet layer), other widths on the
 * general kernels. hidden and intermediate are multiples of 8, hidden at most 16380. */
int hk_kev_model_create(hk_ctx* ctx, int dtype, const hk_kev_config* cfg, const hk_kev_layer_weights* layers_host,
                        const void* embed_dev, const void* final_norm_dev, const void* head_w_dev,
                        const float* head_b_dev, hk_kev_model** out);
int hk_kev_model_destroy(hk_kev_model* m);
/* Workspace bytes for a forward over n_tokens tokens in n_seqs sequences. */
int hk_kev_workspace_size(hk_kev_model* m, int n_tokens, int n_seqs, size_t* bytes_out);
/* Full scoring forward of a fresh (uncached) varlen batch: ids [n_tokens], cu_seqlens
 * [n_seqs + 1] on device and on host (the host copy sizes the launch grids). Writes the
 * decision logits [n_seqs][n_out] fp32 and, if hidden_last_dev != NULL, the final-normed
 * last-token hidden rows [n_seqs][hidden]. Page assignment: sequence s uses pool pages
 * block_tables_dev[s * bt_stride ...]; the pools live in the workspace, which must be 16-byte
 * aligned (HK_ERR_INVALID otherwise; device allocations are). */
int hk_kev_forward(hk_kev_model* m, const int32_t* ids_dev, const int32_t* cu_seqlens_dev,
                   const int32_t* cu_seqlens_host, int n_seqs, const int32_t* block_tables_dev, int bt_stride,
                   int num_pages, void* workspace_dev, size_t workspace_bytes, float* logits_dev,
                   void* hidden_last_dev);

/* Execution identity (the keys Capabilities.extra carries, qwen3_5.rs:2540-2653, which the
 * engine matches against the calibration key, engine.rs:218-226): sorted "key=value" lines such as
 * device, native_execution, device_path, attention_execution, delta_rule_execution and
 * activation_dtype, written to buf (NUL-terminated, truncated to len); *needed = full length + 1. */
int hk_kev_model_identity(hk_kev_model* m, char* buf, size_t len, size_t* needed);

/* ---- readout at the request's positions (Qwen3_5Backend::readout, qwen3_5.rs:3196-3255;
 * ForwardInput.positions, crates/huncho-core/src/backend.rs:52-58) -----------------------------
 * Row s reads positions[cu_positions[s] .. cu_positions[s + 1]), each relative to that row's new
 * tokens (the reference's `position < input.tokens.len()` check, qwen3_5.rs:2688-2696; rows may
 * read no position). hidden_dev receives the final-normed hidden row at each position in the
 * model dtype (the reference's `selected`); pointer_scores_dev the Kev PointerHead score
 * (W_k h_pos + b_k) . (W_q h_last + b_q) / sqrt(head_dim) in fp32, h_last the row's final-normed
 * last token (kev.rs:161-165; the model needs hk_kev_model_set_pointer_head). Either output may
 * be NULL. Host and device copies of both index arrays are required; the host copies are
 * validated before any work. */
typedef struct {
    const int32_t* cu_positions_host;  /* [n_seqs + 1], cu_positions_host[0] = 0, non-decreasing */
    const int32_t* positions_host;     /* [n_positions] */
    const int32_t* cu_positions_dev;   /* the same arrays on the device */
    const int32_t* positions_dev;
    void* hidden_dev;                  /* [n_positions][hidden] or NULL */
    float* pointer_scores_dev;         /* [n_positions] or NULL */
} hk_kev_readout;

/* Copies a Kev PointerHead (kev.rs:112-165): q and k projections [head_dim][hidden] with biases
 * [head_dim], fp32 device buffers (head_dim <= 1024; the caller's buffers may be freed after).
 * Replaces a previously set head. */
int hk_kev_model_set_pointer_head(hk_kev_model* m, int head_dim, const float* q_w_dev, const float* q_b_dev,
                                  const float* k_w_dev, const float* k_b_dev);
/* hk_kev_forward with the readout at positions; logits_dev (the decision head of the last token
 * per row) may be NULL. */
int hk_kev_forward_readout(hk_kev_model* m, const int32_t* ids_dev, const int32_t* cu_seqlens_dev,
                           const int32_t* cu_seqlens_host, int n_seqs, const int32_t* block_tables_dev, int bt_stride,
                           int num_pages, void* workspace_dev, size_t workspace_bytes, const hk_kev_readout* readout,
                           float* logits_dev);

/* ---- prefix cache: cached sequences that continue, fork and are released (the Backend trait's
 * cache surface, crates/huncho-core/src/backend.rs:333-437: prefill / fork / release_cache;
 * crates/huncho-backend/src/qwen3_5.rs:2655-2757 forward with fork_from, 2818-2847; pages and
 * copy-on-write tails as qwen3_5/kv_pages.rs:18-98, 307-341). A handle holds its tokens' K/V in
 * pages of a pool shared by all handles (reference counted), plus the recurrent state and conv
 * tail of every Gated DeltaNet layer. Handles are process-unique, never reused (lib.rs:64-76).
 * Models of every activation dtype with conv kernel 4. Calls on one cache are not thread-safe
 * (the engine serialises them). --- */
typedef struct hk_kev_cache hk_kev_cache;
/* Pools of max_pages pages (page_size tokens of every KV head of every attention layer) and at
 * most max_handles live handles (the reference: 64). All device storage is allocated here: the
 * pools and max_handles + 17 state slots (two fp32 recurrent states and two conv tails each,
 * 39.5 MB per slot at the Kev shape), for the live handles and the retained snapshots. Open, fork
 * and release then allocate, free and synchronise nothing; released pages and slots are reused
 * in stream order on the context's stream. */
int hk_kev_cache_create(hk_kev_model* m, int max_pages, int max_handles, hk_kev_cache** out);
int hk_kev_cache_destroy(hk_kev_cache* c);
/* A new empty handle (zero tokens, zero state). */
int hk_kev_cache_open(hk_kev_cache* c, uint64_t* handle_out);
/* A private branch of `parent`: shares its pages, copies its recurrent state and conv tails.
 * Later continuations of either never change the other (a shared partial page is copied
 * before it is appended to). */
int hk_kev_cache_fork(hk_kev_cache* c, uint64_t parent, uint64_t* child_out);
/* Frees the handle's state; its pages return to the pool when no other handle holds them. */
int hk_kev_cache_release(hk_kev_cache* c, uint64_t handle);
int hk_kev_cache_tokens(hk_kev_cache* c, uint64_t handle, int* tokens_out);
int hk_kev_cache_stats(hk_kev_cache* c, int* live_handles, int* free_pages);
int hk_kev_cache_workspace_size(hk_kev_cache* c, int n_tokens, int n_seqs, size_t* bytes_out);
/* Continues up to 64 distinct handles with their new tokens (row s: ids[cu[s] .. cu[s+1]),
 * nonempty, appended after the handle's cached tokens) and writes each row's decision logits
 * (and, if hidden_last_dev != NULL, final-normed last-token hidden rows) as hk_kev_forward does.
 * Synchronises the context's stream: the handles' tokens, pages and state change only when the
 * call returns HK_OK (device faults included: nothing is committed). HK_ERR_NOMEM when the pool
 * has too few free pages. */
int hk_kev_forward_cached(hk_kev_cache* c, const uint64_t* handles_host, int n_seqs, const int32_t* ids_dev,
                          const int32_t* cu_seqlens_dev, const int32_t* cu_seqlens_host, void* workspace_dev,
                          size_t workspace_bytes, float* logits_dev, void* hidden_last_dev);

/* hk_kev_forward_cached with the readout at positions (relative to each row's new tokens, as
 * ForwardInput.positions are for a fork_from continuation, backend.rs:66-69). */
int hk_kev_forward_cached_readout(hk_kev_cache* c, const uint64_t* handles_host, int n_seqs, const int32_t* ids_dev,
                                  const int32_t* cu_seqlens_dev, const int32_t* cu_seqlens_host, void* workspace_dev,
                                  size_t workspace_bytes, const hk_kev_readout* readout, float* logits_dev);

/* Work counters of the prefill calls (PrefillWork, crates/huncho-core/src/backend.rs:85-89):
 * native forward calls (failed attempts included), tokens processed, and prefills that took a
 * second chunk. */
typedef struct hk_prefill_work {
    uint64_t forward_calls;
    uint64_t processed_tokens;
    uint64_t chunked_prefills;
} hk_prefill_work;

/* Backend::prefill_cached / prefill_cached_with_work (backend.rs:371-395; qwen3_5.rs:2850-2865,
 * 2937-3041): a new handle holding a prefix, given on the host (ids_host: the key and the checks)
 * and on the device (ids_dev: the same ids). With max_bytes > 0 an identical retained prefix is
 * cloned (hit = 1, no model work). Otherwise the prefix is computed in chunks of chunk_tokens (0:
 * one forward) and, if its charged bytes (8 per token + 512, and per layer 512 plus its pages,
 * recurrent state and conv tail: ModelCache::retention_bytes, qwen3_5.rs:1161-1185) fit
 * max_bytes, kept as an immutable snapshot; older snapshots are evicted first in, first out to
 * make room, and at most 16 are kept (qwen3_5.rs:1215-1234). Snapshots hold pool pages (shared
 * with the handles cloned from them) until evicted or cleared. workspace: at least
 * hk_kev_cache_workspace_size(c, largest chunk, 1) bytes. Synchronises the stream. work may be
 * NULL. */
int hk_kev_cache_prefill_cached(hk_kev_cache* c, const int32_t* ids_host, const int32_t* ids_dev, int n_tokens,
                                size_t max_bytes, int chunk_tokens, void* workspace_dev, size_t workspace_bytes,
                                uint64_t* handle_out, int* hit_out, hk_prefill_work* work);
/* Backend::begin_resumable_prefill (backend.rs:399-414; qwen3_5.rs:2873-2897): validates the
 * prefix and returns either a clone of an identical retained prefix (hit = 1, complete) or an
 * empty pending handle (hit = 0; no model work). A pending handle cannot be forked or continued
 * until it is complete; releasing it cancels the prefill. */
int hk_kev_cache_begin_resumable(hk_kev_cache* c, const int32_t* ids_host, int n_tokens, size_t max_bytes,
                                 uint64_t* handle_out, int* hit_out);
/* Backend::advance_resumable_prefill (backend.rs:416-425; qwen3_5.rs:2899-2934): appends the next
 * chunk (at most chunk_tokens > 0) of a pending prefix (ids_dev: the whole prefix on the device).
 * complete = 1 once the prefix is whole; it is then retained as by prefill_cached and the handle
 * is an ordinary one. A failed chunk commits nothing and still counts as work. */
int hk_kev_cache_advance_resumable(hk_kev_cache* c, uint64_t handle, const int32_t* ids_dev, int chunk_tokens,
                                   void* workspace_dev, size_t workspace_bytes, hk_prefill_work* work,
                                   int* complete_out);
/* Backend::clear_prefix_cache (backend.rs:427-430): drops every retained snapshot; handles
 * cloned from them keep their own state and page references. */
int hk_kev_cache_clear_prefixes(hk_kev_cache* c);
/* The number of retained snapshots and their charged bytes. */
int hk_kev_cache_prefix_stats(hk_kev_cache* c, int* count_out, size_t* bytes_out);

/* ---- ModernBERT encoder (the Laya backend: candle ModernBert, crates/huncho-backend/src/
 * candle.rs:65-117 load, 319-416 forward; config normalisation 157-203) ----------------------
 * LayerNorm without bias: y = (x - mean) / sqrt(var + eps) * w, w fp32 [width], width <= 2048. */
int hk_layer_norm(hk_ctx* ctx, int dtype, const void* x_dev, long x_tok, const float* w_dev, float eps, int rows,
                  int width, void* y_dev, long y_tok);
/* Bidirectional softmax attention inside each sequence of an unpadded varlen batch, the
 * sequence-local part of ModernBERT's attention: q, k, v [tokens][heads][head_dim] at their
 * token strides, key j visible to query i iff half_window < 0 or |i - j| <= half_window (local
 * layers: local_attention / 2). o [tokens][heads][head_dim]. max_len >= the longest sequence.
 * head_dim 64 runs on the tile kernels (16-bit: q/k/v rows 16-byte and o rows 8-byte aligned),
 * other widths 1..256 on a general kernel. */
int hk_bidir_attention(hk_ctx* ctx, int dtype, const void* q_dev, long q_tok, const void* k_dev, long k_tok,
                       const void* v_dev, long v_tok, const int32_t* cu_seqlens_dev, int n_seqs, int n_tokens,
                       int max_len, int heads, int head_dim, int half_window, float scale, void* o_dev, long o_tok);

typedef struct {
    int hidden, n_layers, n_heads, intermediate, vocab;  /* head dim = hidden / n_heads: even, <= 256 */
    float eps;             /* layer_norm_eps (1e-5) */
    int global_every;      /* layer i is global iff i % global_every == 0 */
    int local_window;      /* local_attention: local layers see |i - j| <= local_window / 2 */
    double global_theta, local_theta;
    int max_context;       /* longest sequence (RoPE table size) */
    int n_out;             /* mean-pooled linear head outputs (0 = none) */
} hk_bert_config;

/* Per-layer weights in the model dtype, [out][in] (checkpoint names model.layers.{i}.*). */
typedef struct {
    const void* attn_norm;         /* attn_norm.weight [H], or NULL for an identity */
    const void *wqkv, *wo;         /* attn.Wqkv.weight [3H][H], attn.Wo.weight [H][H] */
    const void* mlp_norm;          /* mlp_norm.weight [H] */
    const void *wi, *wo2;          /* mlp.Wi.weight [2I][H], mlp.Wo.weight [H][I] */
} hk_bert_layer_weights;

typedef struct hk_bert_model hk_bert_model;

/* Copies the weights (the caller's buffers may be freed afterwards). head_w [n_out][H] in the
 * model dtype, head_b [n_out] fp32 device or NULL. 64-wide heads run on the tile kernels (the
 * 16-bit attention rotates q as it loads it), other even widths up to 256 on the general
 * kernels; the RoPE tables are [max_context][head_dim / 2]. */
int hk_bert_model_create(hk_ctx* ctx, int dtype, const hk_bert_config* cfg, const hk_bert_layer_weights* layers_host,
                         const void* embed_dev, const void* emb_norm_dev, const void* final_norm_dev,
                         const void* head_w_dev, const float* head_b_dev, hk_bert_model** out);
int hk_bert_model_destroy(hk_bert_model* m);
int hk_bert_workspace_size(hk_bert_model* m, int n_tokens, size_t* bytes_out);
/* Execution identity of the encoder (as hk_kev_model_identity; candle.rs:272-302 capabilities). */
int hk_bert_model_identity(hk_bert_model* m, char* buf, size_t len, size_t* needed);
/* Encoder forward of an unpadded varlen batch: ids [n_tokens], cu_seqlens on device and
 * host. Writes the mean-pooled head's logits [n_seqs][n_out] (fp32) and, if hidden_out_dev
 * != NULL, the final-normed hidden states [n_tokens][hidden] in the model dtype. The workspace
 * must be 16-byte aligned. */
int hk_bert_forward(hk_bert_model* m, const int32_t* ids_dev, const int32_t* cu_seqlens_dev,
                    const int32_t* cu_seqlens_host, int n_seqs, void* workspace_dev, size_t workspace_bytes,
                    float* logits_dev, void* hidden_out_dev);

/* ---- the typed Laya decision head (LayaHead, candle.rs:500-694; built from the checkpoint's
 * `type_emb.weight`, `head.layers.{i}.*` and `scorer.*` tensors, candle.rs:596-649) -------------
 * z = hidden + type_emb[qtype]; each head layer is a pre-norm nn.TransformerEncoderLayer
 * (LayerNorm eps 1e-5 with bias; in_proj q|k|v with bias; max(d / 64, 1) heads of d / heads over
 * the whole sequence, candle.rs:606-609; out_proj with bias; residual; LayerNorm; linear1 + ReLU;
 * linear2; residual;
 * LayaLayer::forward 520-585); the rows at the readout positions then go through the scorer
 * LayerNorm -> Linear(d -> a) -> GELU (erf) -> Linear(a -> 1) (660-694). */
typedef struct hk_laya_head_config {
    int d;              /* encoder width: a multiple of 8 up to 2048 that max(d / 64, 1) heads divide */
    int n_layers;       /* head layers (the reference fixture: 2) */
    int ffn;            /* linear1 rows */
    int scorer_hidden;  /* scorer.1 rows */
    int n_types;        /* type_emb rows */
} hk_laya_head_config;
/* Device pointers in the model dtype; weights row-major [out][in], as in the checkpoint. */
typedef struct hk_laya_head_layer_weights {
    const void *in_proj_w, *in_proj_b, *out_proj_w, *out_proj_b;
    const void *norm1_w, *norm1_b, *norm2_w, *norm2_b;
    const void *linear1_w, *linear1_b, *linear2_w, *linear2_b;
} hk_laya_head_layer_weights;
typedef struct hk_laya_head hk_laya_head;
/* Copies the head (the caller's buffers may be freed after). */
int hk_laya_head_create(hk_ctx* ctx, int dtype, const hk_laya_head_config* cfg, const void* type_emb_dev,
                        const hk_laya_head_layer_weights* layers_host, const void* scorer_ln_w_dev,
                        const void* scorer_ln_b_dev, const void* scorer_w1_dev, const void* scorer_b1_dev,
                        const void* scorer_w2_dev, const void* scorer_b2_dev, hk_laya_head** out);
int hk_laya_head_destroy(hk_laya_head* h);
int hk_laya_head_workspace_size(hk_laya_head* h, int n_tokens, int n_positions, size_t* bytes_out);
/* LayaHead::forward for each sequence of an unpadded varlen batch (1..64 sequences): hidden
 * [n_tokens][d] (the encoder's final-normed rows, model dtype), qtype per sequence,
 * positions[cu_positions[s] .. cu_positions[s + 1]) relative to sequence s (host and device
 * copies). Writes one fp32 score per position (the reference's [n, 1] output). hidden and the
 * workspace (hk_laya_head_workspace_size bytes) are 16-byte aligned; an unknown qtype, an empty
 * sequence or a position outside its sequence is HK_ERR_INVALID before any work. */
int hk_laya_head_forward(hk_laya_head* h, const void* hidden_dev, const int32_t* cu_seqlens_dev,
                         const int32_t* cu_seqlens_host, int n_seqs, const int32_t* qtype_host,
                         const int32_t* cu_positions_dev, const int32_t* cu_positions_host,
                         const int32_t* positions_dev, const int32_t* positions_host, void* workspace_dev,
                         size_t workspace_bytes, float* scores_dev);

/* Mean-pooled linear head of the encoder workload over un-padded hidden rows (candle.rs:399-414
 * hands each row's own tokens to the readout; this head pools them): logits[s][o] = head_b[o] +
 * head_w[o] . mean of rows cu[s] .. cu[s + 1] - 1 of x, in fp32, each row's sum taken as up to
 * 32 partial sums added in a fixed order (deterministic). x [n_tokens][width] at token stride
 * x_tok and head_w [n_out][width] in dtype, head_b [n_out] fp32 or NULL, width <= 2048. The
 * partial sums go to workspace_dev (hk_mean_pool_workspace_size bytes). */
int hk_mean_pool_workspace_size(int n_seqs, int width, size_t* bytes_out);
int hk_mean_pool_head(hk_ctx* ctx, int dtype, const void* x_dev, long x_tok, const int32_t* cu_seqlens_dev, int n_seqs,
                      int n_tokens, int width, const void* head_w_dev, const float* head_b_dev, int n_out,
                      float* logits_dev, void* workspace_dev, size_t workspace_bytes);

/* hk_mean_pool_head without a workspace: no counterpart in the reference. It is for callers that
 * cannot allocate (code under HIP graph capture, tight serving loops). The partial sums live in a
 * fixed device array of the library (64 rows x 32 parts x 2048 columns fp32, 16 MiB per GPU, held
 * until the process ends), so it allocates nothing and calls nothing that does; n_seqs * width
 * beyond 64 * 2048 returns HK_ERR_UNSUPPORTED before any launch. The first context to call it on
 * a GPU owns that GPU's array until hk_ctx_destroy; other contexts on that GPU get
 * HK_ERR_UNSUPPORTED. The owner's calls on its stream are ordered; its calls from several
 * streams at once race on the array. Results equal hk_mean_pool_head's bit for bit. */
int hk_mean_pool_head_noalloc(hk_ctx* ctx, int dtype, const void* x_dev, long x_tok, const int32_t* cu_seqlens_dev,
                              int n_seqs, int n_tokens, int width, const void* head_w_dev, const float* head_b_dev,
                              int n_out, float* logits_dev);

/* ---- calibration (crates/huncho-core/src/calibration.rs:42-60, 170-173) --------------------------
 * Host-side: fp32 exp((x - max) / T), fp64 ordered sum and divide, fp32 result. Returns
 * HK_ERR_INVALID for a non-finite logit or a non-positive / non-finite temperature. */
int hk_calibrate(const float* logits_host, int n, float temperature, float* probs_host);

/* ---- synthetic inputs (seeded, host-side; identical streams to the test oracle) -------------
 * splitmix64 -> two 24-bit uniforms per draw -> Box-Muller in double precision. */
int hk_synth_normal(uint64_t seed, uint64_t stream, float* out_host, size_t n, float mean, float std);
int hk_synth_normal_bf16(uint64_t seed, uint64_t stream, uint16_t* out_host, size_t n, float mean, float std);
int hk_synth_uniform_int(uint64_t seed, uint64_t stream, int32_t* out_host, size_t n, int32_t lo, int32_t hi);
int hk_synth_permutation(uint64_t seed, uint64_t stream, int32_t* out_host, int32_t n);

#ifdef __cplusplus
}
#endif
#endif
