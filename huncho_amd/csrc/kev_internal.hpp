// kev_internal.hpp - the Kev model object and the forward entry shared by kev_model.cpp
// (fresh batches) and kev_cache.cpp (cached continuation, forks).
#pragma once

#include <vector>

#include "abi_internal.hpp"

namespace hk_kev {

struct Layer {
    int type = 0;
    float *in_norm = nullptr, *post_norm = nullptr;
    void *w_gu = nullptr, *w_down = nullptr;
    void *w_in = nullptr, *w_ba = nullptr, *w_out = nullptr;
    float *conv_w = nullptr, *norm_w = nullptr, *base_g = nullptr, *dt_bias = nullptr;
    void *w_qkv = nullptr, *w_o = nullptr;
    float *q_norm = nullptr, *k_norm = nullptr;
};

}  // namespace hk_kev

struct hk_kev_model {
    hk_ctx* ctx = nullptr;
    int dtype = HK_BF16;
    size_t esz = 2;
    bool x_f32 = false;  // residual stream in fp32 (16-bit models with cfg.residual_fp32)
    hk_kev_config cfg{};
    std::vector<int> layer_types;
    std::vector<hk_kev::Layer> layers;
    std::vector<void*> owned;
    void* embed = nullptr;
    float* final_norm = nullptr;
    void* head_w = nullptr;
    float* head_b = nullptr;
    float *rope_cos = nullptr, *rope_sin = nullptr;
    // Kev PointerHead (kev.rs:112-165), fp32: q/k weights [ptr_hd][hidden], biases [ptr_hd]
    float *ptr_qw = nullptr, *ptr_qb = nullptr, *ptr_kw = nullptr, *ptr_kb = nullptr;
    int ptr_hd = 0;
    // derived sizes
    int key_dim = 0, value_dim = 0, conv_dim = 0, gdn_rows = 0, ba_rows = 0, attn_rows = 0;
    // MLP gate|up on the library's own GEMM with the SwiGLU epilogue (16-bit models whose
    // intermediate size is a multiple of 128): w_gu then holds 32-row blocks [16 gate | 16 up]
    bool mlp_fused = false;
};

// Per-call view of cached state for a continuation forward (all pointers owned by the cache).
struct KevCacheView {
    const int32_t* ctx_lens_dev;         // [n_seqs] cached + new tokens per sequence
    int max_ctx = 0;                     // the longest of them
    std::vector<void*> k_pools, v_pools;  // one pool per attention layer, in layer order
    // one device array of n_seqs pointers per Gated DeltaNet layer, in layer order
    std::vector<const float* const*> init_rows;
    std::vector<float* const*> final_rows;
    std::vector<const void* const*> hist_rows;
    std::vector<void* const*> tail_rows;
};

// The scoring forward (fresh batch when view == nullptr). Returns an HK_* status.
// readout (optional): rows and pointer scores at request positions, validated before any work.
int kev_forward_impl(hk_kev_model* m, const int32_t* ids, const int32_t* cu_dev, const int32_t* cu_host, int n_seqs,
                     const int32_t* bt, int bt_stride, int num_pages, void* workspace, size_t workspace_bytes,
                     float* logits, void* hidden_last, const KevCacheView* view, const hk_kev_readout* readout);
// Host-side validation of a readout against the rows' new-token counts (HK_OK or an error set on
// the context).
int kev_validate_readout(hk_kev_model* m, const int32_t* cu_host, int n_seqs, const hk_kev_readout* r);
// Workspace bytes of a forward over n tokens in n_seqs sequences with num_pages workspace pages
// (0 when the pools belong to a cache).
size_t kev_workspace_bytes(const hk_kev_model* m, int n, int n_seqs, int num_pages);

// The fused Gated DeltaNet layer with optional per-sequence row tables (abi.cpp).
int hk_gated_delta_chunked_rows(hk_ctx* ctx, int dtype, const void* q, long q_tok, const void* k, long k_tok,
                                const void* v, long v_tok, const float* g, const float* beta, const int32_t* cu,
                                int n_seqs, int n_tokens, int heads, int k_heads, int dk, int dv,
                                const float* initial_state, float* final_state, void* o, long o_tok,
                                const float* const* init_rows, float* const* final_rows);
int hk_gdn_prep_rows(hk_ctx* ctx, int dtype, const void* mixed, long mixed_tok, const float* conv_w, int conv_k,
                     const void* conv_hist, const void* ba, long ba_tok, int b_col, int a_col, const float* base_g,
                     const float* dt_bias, const int32_t* cu, int n_seqs, int n_tokens, int heads, int k_heads,
                     int dk, int dv, void* q_out, void* k_out, void* v_out, float* g_out, float* beta_out,
                     void* conv_tail_out, const void* const* hist_rows, void* const* tail_rows);
int hk_gdn_fused_rows(hk_ctx* ctx, int dtype, const void* mixed, long mixed_tok, const float* conv_w, int conv_k,
                      const void* conv_hist, void* conv_tail_out, const void* ba, long ba_tok, int b_col, int a_col,
                      const float* base_g, const float* dt_bias, const void* z, long z_tok, const float* norm_w,
                      float eps, const int32_t* cu, int n_seqs, int n_tokens, int heads, int k_heads,
                      const float* initial_state, float* final_state, void* out, long out_tok,
                      const float* const* init_rows, float* const* final_rows, const void* const* hist_rows,
                      void* const* tail_rows);
