// abi_internal.hpp - context object and helpers shared by the host-side ABI files.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <utility>
#include <vector>

#include "../../include/huncho_rocm.h"
#include "kernel_args.hpp"

struct hk_blas;  // GEMM state (hipBLASLt), created lazily per context

struct hk_ctx {
    int device = 0;
    hipDeviceProp_t prop{};
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    int* fault_dev = nullptr;
    std::string last_error;
    hk_blas* blas = nullptr;
    // Scratch of the kernels that split few, long rows over the chip (gdn16_split.hip, delta_rule_split.hip, the
    // key-split attention): kSplitScratch bytes from hk_ctx_create on (null if they could not be had), so that
    // which kernel a call takes follows from its sizes. Work on it is ordered by the stream (split_stream: of
    // the last use). split_done, from the context's first use on a second stream on: the end of the last use;
    // split_first: the block of the uses before that.
    void* split_scratch = nullptr;
    void* split_first = nullptr;
    hipStream_t split_stream = nullptr;
    hipEvent_t split_done = nullptr;
    bool split_used = false;
};
constexpr int kAttnParts = 512;  // most parts of a key-split attention launch, of at most half as many q-blocks
constexpr size_t kSplitScratch = 512u << 20;
// Bytes for the chunks of n_tokens tokens in n_seqs rows.
size_t hk_gdn_split_bytes(int n_tokens, int n_seqs, int heads);
size_t hk_delta_split_bytes(int n_tokens, int n_seqs, int heads);

int hk_fail(hk_ctx* ctx, int code, const char* fmt, ...);
int hk_check_hip(hk_ctx* ctx, hipError_t e, const char* what);
void hk_blas_release(hk_ctx* ctx);
// Creates the context's hipBLASLt handle and GEMM workspace (once; called at model creation so
// that no forward allocates).
int hk_blas_prepare(hk_ctx* ctx);
float hk_host_f16_to_f32(uint16_t b);
uint16_t hk_host_f32_to_f16(float x);

// Row-major Y[n][out] = alpha * X[n][in] . W[out][in]^T + beta * C (C may alias Y or be null).
// dtype HK_BF16: bf16 in/out, fp32 accumulation; HK_F32: fp32.
int hk_gemm_xwt(hk_ctx* ctx, int dtype, int n, int out, int in, const void* x, long ldx, const void* w, long ldw,
                void* y, long ldy, const void* c, long ldc, float alpha, float beta);
// The same with C and Y of dtype cd_dtype (HK_F32 with 16-bit operands: a residual stream kept
// in fp32 takes the product unrounded).
int hk_gemm_xwt_cd(hk_ctx* ctx, int dtype, int cd_dtype, int n, int out, int in, const void* x, long ldx,
                   const void* w, long ldw, void* y, long ldy, const void* c, long ldc, float alpha, float beta);

// hk_paged_prefill_attention with a bound on the batch's context lengths (0: what the block tables can hold).
int hk_paged_prefill_attention_impl(hk_ctx* ctx, int dtype, const void* q, long q_tok, long q_head, const void* k_pool,
                                    const void* v_pool, int num_pages, int page_size, const int32_t* bt, int bt_stride,
                                    const int32_t* cu, const int32_t* ctxl, int n_seqs, int n_tokens, int max_q_len,
                                    int q_heads, int kv_heads, int head_dim, float scale, const void* gate,
                                    long gate_tok, long gate_head, void* o, long o_tok, long o_head, int max_ctx);

// Two projections of the same x rows, Y = X W^T and Y2 = X W2^T (contiguous weights and outputs).
int hk_gemm_xwt_pair(hk_ctx* ctx, int dtype, int n, int in, const void* x, long ldx, int out, const void* w, void* y,
                     int out2, const void* w2, void* y2);

// y [n][inter] = gelu(x Wg^T) * (x Wu^T) of the stacked weight [Wg | Wu] [2 inter][in], each product rounded to
// the dtype first, in one launch for few rows; false (nothing launched) where the projection and the
// GeGLU pass on their own are the way.
bool hk_gemm_geglu_few_rows(hk_ctx* ctx, int dtype, int n, int inter, int in, const void* x, const void* w, void* y, int* rc);

// hk_qk_norm_rope_kv_write with an optional per-token (sequence, position) table (int pairs,
// hk_launch_token_seq_pos), which replaces the kernel's search of cu_seqlens
int hk_qk_norm_rope_kv_write_impl(hk_ctx* ctx, int dtype, const void* q_in, long q_in_tok, long q_in_head,
                                  const void* k_in, long k_in_tok, const void* v_in, long v_in_tok, const float* q_norm,
                                  const float* k_norm, float eps, const float* rope_cos, const float* rope_sin, int rd,
                                  int rope_max_pos, const int32_t* cu, const int32_t* ctxl, int n_seqs, int n_tokens,
                                  const int32_t* bt, int bt_stride, int num_pages, int page_size, int q_heads,
                                  int kv_heads, int head_dim, void* q_out, long q_out_tok, long q_out_head,
                                  void* k_pool, void* v_pool, const int32_t* tok_sp);
// Argument checks shared by hk_mean_pool_head and its variants (HK_OK or an error set on ctx).
int hk_mean_pool_check(hk_ctx* ctx, int dtype, const void* x, long x_tok, const int32_t* cu, int n_seqs, int n_tokens,
                       int width, const void* head_w, int n_out, const float* logits);
// Resolves the no-allocation scratch array's address on `device` (current); bert.hip.
int hk_noalloc_scratch_init(int device);
// Gives up ctx's claim on its GPU's no-allocation scratch array (hk_ctx_destroy).
void hk_noalloc_scratch_release(const hk_ctx* ctx);
// Writes sorted "key=value" lines (NUL-terminated, truncated to len) and the full length + 1.
int hk_write_identity(std::vector<std::pair<std::string, std::string>> kv, char* buf, size_t len, size_t* needed);
// The library's MFMA GEMM with a fused epilogue (hk::EPI_*); HK_ERR_UNSUPPORTED, with no error
// message set, for shapes or dtypes it does not cover.
int hk_gemm_native(hk_ctx* ctx, int dtype, int epi, int n, int out, int in, const void* x, long ldx, const void* w,
                   long ldw, void* y, long ldy, const void* c, long ldc);
