// kev_model.cpp - the Kev/Qwen3.5 hybrid scoring forward on one MI355X.
//
// Mirrors Model::forward_inner / DecoderLayer::forward (crates/huncho-backend/src/
// qwen3_5.rs:1083-1104, 1533-1553) for a fresh varlen batch (the native batch path,
// forward_independent_batch 3138-3194, without right padding):
//   x = embed(ids)
//   per layer: h = rms(x) ; x += mixer(h) ; h = rms(x) ; x += down(silu(gate(h)) * up(h))
//   mixer = Gated DeltaNet (LinearAttn::forward 846-946) or gated full attention
//           (Attention::forward 586-726)
//   final: rms of each sequence's last token, then the decision head (fp32).
// Load-time layout work (done once, qwen3_5.rs:2185-2348 is the reference loader):
//   * projections that read the same input are fused into one GEMM weight:
//     GDN in_proj_qkv | in_proj_z (and in_proj_b | in_proj_a as a second, narrow GEMM, so
//     the wide one keeps a multiple of 256 columns), attention q_proj | k_proj | v_proj,
//     MLP gate_proj | up_proj;
//   * zero-centred norm weights become (1 + w) in fp32 (effective_norm_weight, 180-182),
//     conv weights, the gated-norm weight and dt_bias become fp32, A_log becomes
//     base_g = -exp(A_log) in fp32 (788-790);
//   * a RoPE cos/sin table in the model dtype covers positions 0..max_context-1.
// Residual adds are folded into the GEMM epilogue (beta = 1 onto the residual stream). With
// cfg.residual_fp32 a 16-bit model keeps that stream in fp32: the GEMM's C and D operands are
// fp32, so each output projection's fp32 accumulator is added without rounding, and the norms
// read fp32 rows.
#include <math.h>
#include <string.h>

#include <cmath>
#include <cstdio>
#include <string>

#include <vector>

#include "kev_internal.hpp"

namespace {

using hk_kev::Layer;

inline float bf16_to_f32(uint16_t b) {
    uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

}  // namespace

static int dev_alloc(hk_kev_model* m, size_t bytes, void** out) {
    if (hipMalloc(out, bytes) != hipSuccess) return hk_fail(m->ctx, HK_ERR_NOMEM, "model allocation of %zu bytes failed", bytes);
    m->owned.push_back(*out);
    return HK_OK;
}

// Reads `count` elements of the model dtype at src (device) into fp32 on the host.
static int read_as_f32(hk_kev_model* m, const void* src, size_t count, std::vector<float>& out) {
    out.resize(count);
    if (m->dtype == HK_F32)
        return hk_check_hip(m->ctx, hipMemcpy(out.data(), src, count * 4, hipMemcpyDeviceToHost), "weight read");
    std::vector<uint16_t> tmp(count);
    if (int rc = hk_check_hip(m->ctx, hipMemcpy(tmp.data(), src, count * 2, hipMemcpyDeviceToHost), "weight read"))
        return rc;
    for (size_t i = 0; i < count; ++i) out[i] = m->dtype == HK_F16 ? hk_host_f16_to_f32(tmp[i]) : bf16_to_f32(tmp[i]);
    return HK_OK;
}

static int upload_f32(hk_kev_model* m, const std::vector<float>& v, float** out) {
    if (int rc = dev_alloc(m, v.size() * 4, (void**)out)) return rc;
    return hk_check_hip(m->ctx, hipMemcpy(*out, v.data(), v.size() * 4, hipMemcpyHostToDevice), "weight upload");
}

// fp32 copy of a small weight, optionally transformed.
template <typename F>
static int small_f32(hk_kev_model* m, const void* src, size_t count, float** out, F&& f) {
    if (!src) return hk_fail(m->ctx, HK_ERR_INVALID, "missing small weight");
    std::vector<float> v;
    if (int rc = read_as_f32(m, src, count, v)) return rc;
    for (auto& x : v) x = f(x);
    return upload_f32(m, v, out);
}

// Stacks row-major [rows_i][in] weights into one [sum rows][in] buffer, followed by zero rows
// up to pad_rows rows when pad_rows is larger.
static int fuse_rows(hk_kev_model* m, std::initializer_list<std::pair<const void*, int>> parts, int in, void** out,
                     size_t pad_rows = 0) {
    size_t rows = 0;
    for (auto& p : parts) {
        if (!p.first) return hk_fail(m->ctx, HK_ERR_INVALID, "missing projection weight");
        rows += p.second;
    }
    const size_t total = pad_rows > rows ? pad_rows : rows;
    if (int rc = dev_alloc(m, total * in * m->esz, out)) return rc;
    if (total > rows &&
        hipMemset((char*)*out + rows * in * m->esz, 0, (total - rows) * in * m->esz) != hipSuccess)
        return hk_fail(m->ctx, HK_ERR_DEVICE, "weight padding failed");
    size_t off = 0;
    for (auto& p : parts) {
        size_t bytes = (size_t)p.second * in * m->esz;
        if (int rc = hk_check_hip(m->ctx, hipMemcpy((char*)*out + off, p.first, bytes, hipMemcpyDeviceToDevice),
                                  "weight fuse"))
            return rc;
        off += bytes;
    }
    return HK_OK;
}

// gate_proj and up_proj [I][in] as the fused SwiGLU GEMM's weight (gemm.hip): 32-row blocks
// [gate rows 16 b .. 16 b + 15 | up rows 16 b .. 16 b + 15], I a multiple of 16
static int fuse_swiglu_rows(hk_kev_model* m, const void* gate, const void* up, int I, int in, void** out) {
    if (!gate || !up) return hk_fail(m->ctx, HK_ERR_INVALID, "missing projection weight");
    if (int rc = dev_alloc(m, (size_t)2 * I * in * m->esz, out)) return rc;
    const size_t blk = (size_t)16 * in * m->esz;
    if (int rc = hk_check_hip(m->ctx, hipMemcpy2D(*out, 2 * blk, gate, blk, blk, I / 16, hipMemcpyDeviceToDevice),
                              "gate weight blocks"))
        return rc;
    return hk_check_hip(m->ctx, hipMemcpy2D((char*)*out + blk, 2 * blk, up, blk, blk, I / 16, hipMemcpyDeviceToDevice),
                        "up weight blocks");
}

extern "C" int hk_kev_model_destroy(hk_kev_model* m) {
    if (!m) return HK_ERR_INVALID;
    hipSetDevice(m->ctx->device);
    hipStreamSynchronize(m->ctx->stream);
    for (void* p : m->owned) hipFree(p);
    for (float* p : {m->ptr_qw, m->ptr_qb, m->ptr_kw, m->ptr_kb})
        if (p) hipFree(p);
    delete m;
    return HK_OK;
}

extern "C" int hk_kev_model_create(hk_ctx* ctx, int dtype, const hk_kev_config* cfg, const hk_kev_layer_weights* lw,
                                   const void* embed, const void* final_norm, const void* head_w, const float* head_b,
                                   hk_kev_model** out) {
    if (!ctx || !cfg || !lw || !embed || !final_norm || !out) return HK_ERR_INVALID;
    *out = nullptr;
    if (dtype != HK_BF16 && dtype != HK_F16 && dtype != HK_F32) return hk_fail(ctx, HK_ERR_UNSUPPORTED, "dtype %d", dtype);
    const hk_kev_config& c = *cfg;
    // 128-wide heads run on the MFMA kernels; other widths up to 256 on the general kernels
    if (c.head_dim < 1 || c.head_dim > 256 || c.lin_key_dim < 1 || c.lin_key_dim > 256 || c.lin_v_dim < 1 ||
        c.lin_v_dim > 256 || c.lin_key_dim * c.lin_v_dim > 32768)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED,
                       "head dims %d/%d/%d: each in 1..256 with linear key x value dims <= 32768 are implemented",
                       c.head_dim, c.lin_key_dim, c.lin_v_dim);
    if (c.hidden <= 0 || c.hidden % 8 || c.intermediate <= 0 || c.intermediate % 8 || c.n_layers <= 0 || c.vocab <= 0 ||
        c.n_heads <= 0 || c.n_kv_heads <= 0 || c.n_heads % c.n_kv_heads || c.lin_n_k_heads <= 0 ||
        c.lin_n_v_heads % c.lin_n_k_heads || c.conv_k < 1 || c.max_context <= 0 || c.n_out < 0 ||
        !c.layer_types_host || c.rotary_dim < 2 || c.rotary_dim > c.head_dim || c.rotary_dim % 2)
        return hk_fail(ctx, HK_ERR_INVALID, "invalid model configuration");
    if (c.n_out > 0 && !head_w) return hk_fail(ctx, HK_ERR_INVALID, "missing decision head");
    // the final norm + head kernel stages one fp32 hidden row and four partial sums in 64 KiB of LDS
    if (c.hidden > 16380)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "hidden size %d: at most 16380 is supported", c.hidden);
    hipSetDevice(ctx->device);
    hipStreamSynchronize(ctx->stream);  // staged tensors written by queued work are complete
    if (int rc = hk_blas_prepare(ctx)) return rc;  // GEMM handle + workspace, before any forward
    hk_kev_model* m = new hk_kev_model();
    m->ctx = ctx;
    m->dtype = dtype;
    m->esz = dtype == HK_F32 ? 4 : 2;
    m->x_f32 = dtype != HK_F32 && c.residual_fp32 != 0;
    m->mlp_fused = dtype != HK_F32 && c.intermediate % 128 == 0 && c.hidden % 64 == 0;
    m->cfg = c;
    m->layer_types.assign(c.layer_types_host, c.layer_types_host + c.n_layers);
    m->cfg.layer_types_host = m->layer_types.data();
    m->key_dim = c.lin_n_k_heads * c.lin_key_dim;
    m->value_dim = c.lin_n_v_heads * c.lin_v_dim;
    m->conv_dim = 2 * m->key_dim + m->value_dim;
    // GDN in_proj as two GEMMs: [qkv | z] (a multiple of the GEMM's 256-column tiles at the
    // Kev shape, 8192) and [b | a] (2 Hv columns); both padded to a multiple of 8 rows
    // (16-byte aligned rows for the fused layer)
    m->gdn_rows = (m->conv_dim + m->value_dim + 7) / 8 * 8;
    m->ba_rows = (2 * c.lin_n_v_heads + 7) / 8 * 8;
    m->attn_rows = 2 * c.n_heads * c.head_dim + 2 * c.n_kv_heads * c.head_dim;
    const int H = c.hidden, I = c.intermediate;
    int rc = HK_OK;
    auto fail = [&](int code) {
        hk_kev_model_destroy(m);
        return code;
    };
    auto eff = [](float w) { return 1.0f + w; };
    auto same = [](float w) { return w; };
    auto negexp = [](float w) { return -expf(w); };
    for (int l = 0; l < c.n_layers; ++l) {
        const hk_kev_layer_weights& w = lw[l];
        Layer L;
        L.type = m->layer_types[l];
        if ((rc = small_f32(m, w.input_norm, H, &L.in_norm, eff))) return fail(rc);
        if ((rc = small_f32(m, w.post_norm, H, &L.post_norm, eff))) return fail(rc);
        if (m->mlp_fused) {
            if ((rc = fuse_swiglu_rows(m, w.gate_proj, w.up_proj, I, H, &L.w_gu))) return fail(rc);
        } else if ((rc = fuse_rows(m, {{w.gate_proj, I}, {w.up_proj, I}}, H, &L.w_gu))) {
            return fail(rc);
        }
        if ((rc = fuse_rows(m, {{w.down_proj, H}}, I, &L.w_down))) return fail(rc);
        if (L.type == 0) {
            const int Hv = c.lin_n_v_heads;
            if ((rc = fuse_rows(m, {{w.in_qkv, m->conv_dim}, {w.in_z, m->value_dim}}, H, &L.w_in, m->gdn_rows)))
                return fail(rc);
            if ((rc = fuse_rows(m, {{w.in_b, Hv}, {w.in_a, Hv}}, H, &L.w_ba, m->ba_rows))) return fail(rc);
            if ((rc = fuse_rows(m, {{w.out_proj, H}}, m->value_dim, &L.w_out))) return fail(rc);
            if ((rc = small_f32(m, w.conv_w, (size_t)m->conv_dim * c.conv_k, &L.conv_w, same))) return fail(rc);
            if ((rc = small_f32(m, w.norm_w, c.lin_v_dim, &L.norm_w, same))) return fail(rc);
            if ((rc = small_f32(m, w.a_log, Hv, &L.base_g, negexp))) return fail(rc);
            if ((rc = small_f32(m, w.dt_bias, Hv, &L.dt_bias, same))) return fail(rc);
        } else {
            const int hd = c.head_dim;
            if ((rc = fuse_rows(m, {{w.q_proj, 2 * c.n_heads * hd}, {w.k_proj, c.n_kv_heads * hd}, {w.v_proj, c.n_kv_heads * hd}},
                                H, &L.w_qkv)))
                return fail(rc);
            if ((rc = fuse_rows(m, {{w.o_proj, H}}, c.n_heads * hd, &L.w_o))) return fail(rc);
            if ((rc = small_f32(m, w.q_norm, hd, &L.q_norm, eff))) return fail(rc);
            if ((rc = small_f32(m, w.k_norm, hd, &L.k_norm, eff))) return fail(rc);
        }
        m->layers.push_back(L);
    }
    if ((rc = fuse_rows(m, {{embed, c.vocab}}, H, &m->embed))) return fail(rc);
    if ((rc = small_f32(m, final_norm, H, &m->final_norm, eff))) return fail(rc);
    if (c.n_out > 0) {
        if ((rc = fuse_rows(m, {{head_w, c.n_out}}, H, &m->head_w))) return fail(rc);
        if (head_b) {
            std::vector<float> hb(c.n_out);
            if ((rc = hk_check_hip(ctx, hipMemcpy(hb.data(), head_b, c.n_out * 4, hipMemcpyDeviceToHost), "head bias")))
                return fail(rc);
            if ((rc = upload_f32(m, hb, &m->head_b))) return fail(rc);
        }
    }
    {
        const int half = c.rotary_dim / 2;
        std::vector<float> cs((size_t)c.max_context * half), sn((size_t)c.max_context * half);
        hk_rope_fill_table(c.rotary_dim, c.rope_theta, c.max_context, dtype, cs.data(), sn.data());
        if ((rc = upload_f32(m, cs, &m->rope_cos)) || (rc = upload_f32(m, sn, &m->rope_sin))) return fail(rc);
    }
    hipStreamSynchronize(nullptr);  // the weight copies, on the null stream, are complete before the
                                    // context's stream (non-blocking) uses them
    *out = m;
    return HK_OK;
}

namespace {

struct Workspace {
    size_t off = 0;
    char* base = nullptr;
    template <typename T>
    T* take(size_t count) {
        size_t bytes = (count * sizeof(T) + 255) & ~(size_t)255;
        T* p = (T*)(base ? base + off : nullptr);
        off += bytes;
        return p;
    }
    void* take_bytes(size_t bytes) {
        bytes = (bytes + 255) & ~(size_t)255;
        void* p = base ? base + off : nullptr;
        off += bytes;
        return p;
    }
};

struct Buffers {
    void *x, *h, *big, *ba, *q, *k, *v, *o, *act, *k_pool, *v_pool;
    float *g, *beta;
    int* ctx_lens;
    int* tok_sp;  // [n][2]: each token's sequence and absolute position
    size_t pool_bytes;
};

Buffers carve(const hk_kev_model* m, Workspace& ws, int n, int n_seqs, int num_pages) {
    const hk_kev_config& c = m->cfg;
    Buffers b{};
    const size_t e = m->esz;
    int big_cols = m->gdn_rows;
    if (m->attn_rows > big_cols) big_cols = m->attn_rows;
    if (2 * c.intermediate > big_cols) big_cols = 2 * c.intermediate;
    b.x = ws.take_bytes((size_t)n * c.hidden * (m->x_f32 ? 4 : e));
    b.h = ws.take_bytes((size_t)n * c.hidden * e);
    b.big = ws.take_bytes((size_t)n * big_cols * e);
    b.ba = ws.take_bytes((size_t)n * m->ba_rows * e);
    b.q = ws.take_bytes((size_t)n * m->key_dim * e);
    b.k = ws.take_bytes((size_t)n * m->key_dim * e);
    b.v = ws.take_bytes((size_t)n * m->value_dim * e);
    int o_cols = m->value_dim > c.n_heads * c.head_dim ? m->value_dim : c.n_heads * c.head_dim;
    b.o = ws.take_bytes((size_t)n * o_cols * e);
    b.act = ws.take_bytes((size_t)n * c.intermediate * e);
    b.g = ws.take<float>((size_t)n * c.lin_n_v_heads);
    b.beta = ws.take<float>((size_t)n * c.lin_n_v_heads);
    b.ctx_lens = ws.take<int>((size_t)n_seqs);
    b.tok_sp = ws.take<int>((size_t)2 * n);
    b.pool_bytes = (size_t)num_pages * c.n_kv_heads * c.page_size * c.head_dim * e;
    b.k_pool = ws.take_bytes(b.pool_bytes);
    b.v_pool = ws.take_bytes(b.pool_bytes);
    return b;
}

}  // namespace

size_t kev_workspace_bytes(const hk_kev_model* m, int n, int n_seqs, int num_pages) {
    Workspace ws;
    carve(m, ws, n, n_seqs, num_pages);
    return ws.off;
}

extern "C" int hk_kev_workspace_size(hk_kev_model* m, int n_tokens, int n_seqs, size_t* bytes_out) {
    if (!m || !bytes_out || n_tokens < 0 || n_seqs <= 0) return HK_ERR_INVALID;
    // pools sized for every sequence's pages; callers that share pages may pass fewer
    const int P = m->cfg.page_size;
    const int pages = (n_tokens + n_seqs * (P - 1)) / P + 1;
    Workspace ws;
    carve(m, ws, n_tokens, n_seqs, pages);
    *bytes_out = ws.off;
    return HK_OK;
}

// RMSNorm of the residual stream (fp32 rows when the model keeps it in fp32) into dtype rows.
static int norm_x(hk_kev_model* m, const void* x, const float* w, int n, void* y) {
    const int H = m->cfg.hidden;
    hk::NormArgs a{x, H, w, m->cfg.eps, n, H, y, H, m->x_f32 ? 1 : 0};
    return hk_launch_rms_norm(m->dtype, &a, m->ctx->stream) ? hk_fail(m->ctx, HK_ERR_DEVICE, "rms_norm launch") : HK_OK;
}

#define RUN(expr)                  \
    do {                           \
        int rc__ = (expr);         \
        if (rc__) return rc__;     \
    } while (0)

extern "C" int hk_kev_forward(hk_kev_model* m, const int32_t* ids, const int32_t* cu_dev, const int32_t* cu_host,
                              int n_seqs, const int32_t* bt, int bt_stride, int num_pages, void* workspace,
                              size_t workspace_bytes, float* logits, void* hidden_last) {
    if (!m) return HK_ERR_INVALID;
    if (m->cfg.n_out > 0 && !logits) return hk_fail(m->ctx, HK_ERR_INVALID, "logits output required");
    return kev_forward_impl(m, ids, cu_dev, cu_host, n_seqs, bt, bt_stride, num_pages, workspace, workspace_bytes,
                            logits, hidden_last, nullptr, nullptr);
}

extern "C" int hk_kev_forward_readout(hk_kev_model* m, const int32_t* ids, const int32_t* cu_dev,
                                      const int32_t* cu_host, int n_seqs, const int32_t* bt, int bt_stride,
                                      int num_pages, void* workspace, size_t workspace_bytes,
                                      const hk_kev_readout* readout, float* logits) {
    if (!m) return HK_ERR_INVALID;
    if (!readout) return hk_fail(m->ctx, HK_ERR_INVALID, "readout required");
    return kev_forward_impl(m, ids, cu_dev, cu_host, n_seqs, bt, bt_stride, num_pages, workspace, workspace_bytes,
                            logits, nullptr, nullptr, readout);
}

extern "C" int hk_kev_model_set_pointer_head(hk_kev_model* m, int head_dim, const float* q_w, const float* q_b,
                                             const float* k_w, const float* k_b) {
    if (!m) return HK_ERR_INVALID;
    hk_ctx* ctx = m->ctx;
    if (head_dim <= 0 || head_dim > 1024 || !q_w || !q_b || !k_w || !k_b)
        return hk_fail(ctx, HK_ERR_INVALID, "pointer head: head_dim in 1..1024 and all four tensors required");
    if (m->cfg.hidden + head_dim > 8190)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "pointer head: hidden + head_dim must be <= 8190");
    hipSetDevice(ctx->device);
    // the source tensors may still be written by work queued on the context's stream
    if (hipStreamSynchronize(ctx->stream) != hipSuccess)
        return hk_fail(ctx, HK_ERR_DEVICE, "pointer head: stream synchronisation failed");
    const size_t wb = (size_t)head_dim * m->cfg.hidden * 4, bb = (size_t)head_dim * 4;
    float *qw = nullptr, *qb = nullptr, *kw = nullptr, *kb = nullptr;
    bool ok = hipMalloc((void**)&qw, wb) == hipSuccess && hipMalloc((void**)&qb, bb) == hipSuccess &&
              hipMalloc((void**)&kw, wb) == hipSuccess && hipMalloc((void**)&kb, bb) == hipSuccess;
    ok = ok && hipMemcpy(qw, q_w, wb, hipMemcpyDeviceToDevice) == hipSuccess &&
         hipMemcpy(qb, q_b, bb, hipMemcpyDeviceToDevice) == hipSuccess &&
         hipMemcpy(kw, k_w, wb, hipMemcpyDeviceToDevice) == hipSuccess &&
         hipMemcpy(kb, k_b, bb, hipMemcpyDeviceToDevice) == hipSuccess;
    // the copies (null stream) are complete before the context's stream, which may be
    // non-blocking, reads the new head
    ok = ok && hipStreamSynchronize(nullptr) == hipSuccess;
    if (!ok) {
        for (float* p : {qw, qb, kw, kb})
            if (p) hipFree(p);
        return hk_fail(ctx, HK_ERR_NOMEM, "pointer head allocation or copy failed");
    }
    hipStreamSynchronize(ctx->stream);  // a previous head may still be in use by queued work
    for (float* p : {m->ptr_qw, m->ptr_qb, m->ptr_kw, m->ptr_kb})
        if (p) hipFree(p);
    m->ptr_qw = qw;
    m->ptr_qb = qb;
    m->ptr_kw = kw;
    m->ptr_kb = kb;
    m->ptr_hd = head_dim;
    return HK_OK;
}

int kev_validate_readout(hk_kev_model* m, const int32_t* cu_host, int n_seqs, const hk_kev_readout* r) {
    hk_ctx* ctx = m->ctx;
    if (!r->cu_positions_host || !r->cu_positions_dev || (!r->positions_host && r->cu_positions_host[n_seqs] > 0))
        return hk_fail(ctx, HK_ERR_INVALID, "readout: host and device position arrays are required");
    if (r->cu_positions_host[0] != 0) return hk_fail(ctx, HK_ERR_INVALID, "readout: cu_positions[0] must be 0");
    for (int s = 0; s < n_seqs; ++s) {
        const int a = r->cu_positions_host[s], b = r->cu_positions_host[s + 1];
        const int len = cu_host[s + 1] - cu_host[s];
        if (b < a) return hk_fail(ctx, HK_ERR_INVALID, "readout: cu_positions decreases at row %d", s);
        for (int i = a; i < b; ++i)
            if (r->positions_host[i] < 0 || r->positions_host[i] >= len)
                return hk_fail(ctx, HK_ERR_INVALID, "readout position %d is outside row %d's %d tokens",
                               r->positions_host[i], s, len);
    }
    const int np = r->cu_positions_host[n_seqs];
    if (np > 0 && !r->positions_dev) return hk_fail(ctx, HK_ERR_INVALID, "readout: positions_dev required");
    if (r->pointer_scores_dev && !m->ptr_qw)
        return hk_fail(ctx, HK_ERR_INVALID, "readout: pointer scores need a pointer head (hk_kev_model_set_pointer_head)");
    if (m->cfg.hidden + 4 > 8190) return hk_fail(ctx, HK_ERR_UNSUPPORTED, "readout: hidden too large");
    return HK_OK;
}

int kev_forward_impl(hk_kev_model* m, const int32_t* ids, const int32_t* cu_dev, const int32_t* cu_host, int n_seqs,
                     const int32_t* bt, int bt_stride, int num_pages, void* workspace, size_t workspace_bytes,
                     float* logits, void* hidden_last, const KevCacheView* view, const hk_kev_readout* readout) {
    if (!m) return HK_ERR_INVALID;
    hk_ctx* ctx = m->ctx;
    const hk_kev_config& c = m->cfg;
    if (!ids || !cu_dev || !cu_host || !bt || !workspace || n_seqs <= 0 || bt_stride <= 0 || num_pages <= 0)
        return hk_fail(ctx, HK_ERR_INVALID, "invalid forward arguments");
    // every buffer carved from the workspace starts at a multiple of 256 bytes from its base; the
    // vector kernels and the own GEMM need 16-byte aligned rows
    if ((uintptr_t)workspace & 15) return hk_fail(ctx, HK_ERR_INVALID, "workspace must be 16-byte aligned");
    // (callers check that the outputs they need are given; a null logits skips the head)
    if (cu_host[0] != 0) return hk_fail(ctx, HK_ERR_INVALID, "cu_seqlens[0] must be 0");
    int max_len = 0;
    for (int s = 0; s < n_seqs; ++s) {
        const int len = cu_host[s + 1] - cu_host[s];
        if (len <= 0) return hk_fail(ctx, HK_ERR_INVALID, "sequence %d is empty", s);
        if (len > c.max_context) return hk_fail(ctx, HK_ERR_INVALID, "sequence length %d exceeds max_context %d", len, c.max_context);
        if (!view && (len + c.page_size - 1) / c.page_size > bt_stride)
            return hk_fail(ctx, HK_ERR_INVALID, "sequence %d needs more pages than bt_stride", s);
        if (len > max_len) max_len = len;
    }
    if (readout)
        if (int rc = kev_validate_readout(m, cu_host, n_seqs, readout)) return rc;
    const int n = cu_host[n_seqs];
    Workspace ws;
    ws.base = (char*)workspace;
    Buffers b = carve(m, ws, n, n_seqs, view ? 0 : num_pages);
    if (ws.off > workspace_bytes) return hk_fail(ctx, HK_ERR_INVALID, "workspace too small: %zu < %zu", workspace_bytes, ws.off);
    hipSetDevice(ctx->device);
    const int dt = m->dtype;
    const size_t e = m->esz;
    const int H = c.hidden, I = c.intermediate, hd = c.head_dim;
    const int Hq = c.n_heads, Hkv = c.n_kv_heads, Hv = c.lin_n_v_heads, Hk = c.lin_n_k_heads;

    const int32_t* ctx_lens = view ? view->ctx_lens_dev : b.ctx_lens;
    if (view) {
        if (c.conv_k != 4) return hk_fail(ctx, HK_ERR_UNSUPPORTED, "cached continuation needs conv kernel 4");
        int n_attn = 0, n_gdn = 0;
        for (int l = 0; l < c.n_layers; ++l) (m->layers[l].type == 0 ? n_gdn : n_attn)++;
        if ((int)view->k_pools.size() != n_attn || (int)view->v_pools.size() != n_attn ||
            (int)view->init_rows.size() != n_gdn || (int)view->final_rows.size() != n_gdn ||
            (int)view->hist_rows.size() != n_gdn || (int)view->tail_rows.size() != n_gdn)
            return hk_fail(ctx, HK_ERR_INVALID, "cache view does not match the model's layers");
    } else {
        RUN(hk_launch_seq_lens(cu_dev, n_seqs, b.ctx_lens, ctx->stream) ? hk_fail(ctx, HK_ERR_DEVICE, "seq_lens") : 0);
    }
    // each token's sequence and position, once for all attention layers
    RUN(hk_launch_token_seq_pos(cu_dev, ctx_lens, n_seqs, n, b.tok_sp, ctx->fault_dev, ctx->stream)
            ? hk_fail(ctx, HK_ERR_DEVICE, "token_seq_pos launch")
            : 0);
    int ai = 0, gi = 0;  // attention / Gated DeltaNet layer ordinals
    const int xdt = m->x_f32 ? HK_F32 : dt;  // residual stream dtype
    RUN(hk_launch_embed(dt, m->x_f32, ids, n, m->embed, c.vocab, H, b.x, ctx->fault_dev, ctx->stream)
            ? hk_fail(ctx, HK_ERR_DEVICE, "embed launch")
            : 0);
    for (int l = 0; l < c.n_layers; ++l) {
        const Layer& L = m->layers[l];
        RUN(norm_x(m, b.x, L.in_norm, n, b.h));
        if (L.type == 0) {
            const int rows = m->gdn_rows;
            RUN(hk_gemm_xwt_pair(ctx, dt, n, H, b.h, H, rows, L.w_in, b.big, m->ba_rows, L.w_ba, b.ba));
            const int b_col = 0, a_col = Hv;
            const int dk = c.lin_key_dim, dv = c.lin_v_dim;
            if (dt != HK_F32 && c.conv_k == 4 && rows % 8 == 0 && dk == 128 && dv == 128) {
                // one kernel: conv + SiLU + l2norm + beta/g + chunked delta rule + gated RMSNorm
                RUN(hk_gdn_fused_rows(ctx, dt, b.big, rows, L.conv_w, c.conv_k, nullptr, nullptr, b.ba, m->ba_rows, b_col,
                                      a_col, L.base_g, L.dt_bias, (char*)b.big + (size_t)m->conv_dim * e, rows, L.norm_w,
                                      c.eps, cu_dev, n_seqs, n, Hv, Hk, nullptr, nullptr, b.o, (long)Hv * dv,
                                      view ? view->init_rows[gi] : nullptr, view ? view->final_rows[gi] : nullptr,
                                      view ? view->hist_rows[gi] : nullptr, view ? view->tail_rows[gi] : nullptr));
            } else {
                // the cache's per-sequence conv tails and states, as in the fused path
                RUN(hk_gdn_prep_rows(ctx, dt, b.big, rows, L.conv_w, c.conv_k, nullptr, b.ba, m->ba_rows, b_col, a_col,
                                     L.base_g, L.dt_bias, cu_dev, n_seqs, n, Hv, Hk, dk, dv, b.q, b.k, b.v, b.g, b.beta,
                                     nullptr, view ? view->hist_rows[gi] : nullptr,
                                     view ? view->tail_rows[gi] : nullptr));
                RUN(hk_gated_delta_chunked_rows(ctx, dt, b.q, (long)Hk * dk, b.k, (long)Hk * dk, b.v, (long)Hv * dv,
                                                b.g, b.beta, cu_dev, n_seqs, n, Hv, Hk, dk, dv, nullptr, nullptr, b.o,
                                                (long)Hv * dv, view ? view->init_rows[gi] : nullptr,
                                                view ? view->final_rows[gi] : nullptr));
                RUN(hk_gated_rms_norm(ctx, dt, b.o, (char*)b.big + (size_t)m->conv_dim * e, rows, Hv, L.norm_w, c.eps,
                                      n * Hv, dv, b.o));
            }
            RUN(hk_gemm_xwt_cd(ctx, dt, xdt, n, H, m->value_dim, b.o, m->value_dim, L.w_out, m->value_dim, b.x, H, b.x,
                               H, 1.0f, 1.0f));
            ++gi;
        } else {
            void* k_pool = view ? view->k_pools[ai] : b.k_pool;
            void* v_pool = view ? view->v_pools[ai] : b.v_pool;
            ++ai;
            const int rows = m->attn_rows;
            RUN(hk_gemm_xwt(ctx, dt, n, rows, H, b.h, H, L.w_qkv, H, b.big, rows, nullptr, 0, 1.0f, 0.0f));
            char* qg = (char*)b.big;
            char* kin = qg + (size_t)2 * Hq * hd * e;
            char* vin = kin + (size_t)Hkv * hd * e;
            RUN(hk_qk_norm_rope_kv_write_impl(ctx, dt, qg, rows, 2 * hd, kin, rows, vin, rows, L.q_norm, L.k_norm,
                                              c.eps, m->rope_cos, m->rope_sin, c.rotary_dim, c.max_context, cu_dev,
                                              ctx_lens, n_seqs, n, bt, bt_stride, num_pages, c.page_size, Hq, Hkv, hd,
                                              qg, rows, 2 * hd, k_pool, v_pool, b.tok_sp));
            RUN(hk_paged_prefill_attention_impl(ctx, dt, qg, rows, 2 * hd, k_pool, v_pool, num_pages, c.page_size, bt,
                                                bt_stride, cu_dev, ctx_lens, n_seqs, n, max_len, Hq, Hkv, hd,
                                                (float)(1.0 / sqrt((double)hd)), qg + (size_t)hd * e, rows, 2 * hd, b.o,
                                                (long)Hq * hd, hd, view ? view->max_ctx : max_len));
            RUN(hk_gemm_xwt_cd(ctx, dt, xdt, n, H, Hq * hd, b.o, Hq * hd, L.w_o, Hq * hd, b.x, H, b.x, H, 1.0f, 1.0f));
        }
        RUN(norm_x(m, b.x, L.post_norm, n, b.h));
        if (m->mlp_fused) {
            // gate|up GEMM with silu(gate) * up in its epilogue (Mlp::forward, qwen3_5.rs:1020-1031)
            RUN(hk_gemm_native(ctx, dt, hk::EPI_SWIGLU, n, 2 * I, H, b.h, H, L.w_gu, H, b.act, I, nullptr, 0));
        } else {
            RUN(hk_gemm_xwt(ctx, dt, n, 2 * I, H, b.h, H, L.w_gu, H, b.big, 2 * I, nullptr, 0, 1.0f, 0.0f));
            RUN(hk_swiglu(ctx, dt, b.big, 2 * I, I, n, I, b.act));
        }
        RUN(hk_gemm_xwt_cd(ctx, dt, xdt, n, H, I, b.act, I, L.w_down, I, b.x, H, b.x, H, 1.0f, 1.0f));
    }
    if ((c.n_out > 0 && logits) || hidden_last) {
        const int hrc = hk_launch_final_norm_head(dt, m->x_f32, b.x, H, cu_dev, n_seqs, m->final_norm, c.eps, H,
                                                  m->head_w, m->head_b, logits ? c.n_out : 0, logits, hidden_last,
                                                  ctx->stream);
        if (hrc) return hk_fail(ctx, hrc, hrc == HK_ERR_UNSUPPORTED ? "final head: hidden size too large" : "final head launch");
    }
    if (readout && (readout->hidden_dev || readout->pointer_scores_dev)) {
        hk::ReadoutArgs ra{};
        ra.x = b.x;
        ra.x_tok = H;
        ra.cu = cu_dev;
        ra.cu_pos = readout->cu_positions_dev;
        ra.positions = readout->positions_dev;
        ra.n_seqs = n_seqs;
        ra.n_positions = readout->cu_positions_host[n_seqs];
        ra.width = H;
        ra.w_eff = m->final_norm;
        ra.eps = c.eps;
        ra.hidden_out = readout->hidden_dev;
        ra.q_w = m->ptr_qw;
        ra.q_b = m->ptr_qb;
        ra.k_w = m->ptr_kw;
        ra.k_b = m->ptr_kb;
        ra.head_dim = m->ptr_hd;
        ra.scale = m->ptr_hd > 0 ? (float)(1.0 / sqrt((double)m->ptr_hd)) : 0.0f;
        ra.scores = readout->pointer_scores_dev;
        ra.fault = ctx->fault_dev;
        ra.x_f32 = m->x_f32 ? 1 : 0;
        RUN(hk_launch_readout(dt, &ra, ctx->stream) ? hk_fail(ctx, HK_ERR_DEVICE, "readout launch") : 0);
    }
    return HK_OK;
}

extern "C" int hk_lora_merge(hk_ctx* ctx, int dtype, void* w, int rows, int cols, const float* a, const float* b,
                             int rank, float scale) {
    if (!ctx) return HK_ERR_INVALID;
    if (dtype != HK_BF16 && dtype != HK_F16 && dtype != HK_F32) return hk_fail(ctx, HK_ERR_UNSUPPORTED, "dtype %d", dtype);
    if (!w || !a || !b || rows <= 0 || cols <= 0 || rank <= 0 || !std::isfinite(scale))
        return hk_fail(ctx, HK_ERR_INVALID, "lora merge: bad arguments (%d x %d, rank %d)", rows, cols, rank);
    if ((long)rows * cols > (long)UINT32_MAX * 256)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "lora merge: weight too large");
    hipSetDevice(ctx->device);
    return hk_launch_lora_merge(dtype, w, rows, cols, a, b, rank, scale, ctx->stream)
               ? hk_fail(ctx, HK_ERR_DEVICE, "lora merge launch")
               : HK_OK;
}

extern "C" int hk_kev_model_identity(hk_kev_model* m, char* buf, size_t len, size_t* needed) {
    if (!m) return HK_ERR_INVALID;
    const bool f32 = m->dtype == HK_F32;
    const char* dt = f32 ? "fp32" : m->dtype == HK_BF16 ? "bf16" : "fp16";
    char dev[96];
    snprintf(dev, sizeof dev, "rocm:%d (%s, %d CUs)", m->ctx->device, m->ctx->prop.gcnArchName,
             m->ctx->prop.multiProcessorCount);
    // shapes the MFMA kernels do not tile run on the general kernels, with their own numerics
    const hk_kev_config& c = m->cfg;
    const int group = c.n_heads / c.n_kv_heads;
    const bool attn_mfma = (c.head_dim == 128 || (c.head_dim == 256 && !f32)) &&
                           (group == 1 || group == 2 || group == 4 || group == 8);
    const bool gdn_mfma = c.lin_key_dim == 128 && c.lin_v_dim == 128;
    const char* attn_exec = !attn_mfma ? "rocm-paged-general-wave-per-row-v1"
                            : f32      ? "rocm-paged-flash-mfma-f32-v1"
                                       : "rocm-paged-flash-mfma-16bit-suffix-key-split-v2";
    const char* delta_exec = !gdn_mfma ? "rocm-recurrent-per-token-general-v1"
                             : f32     ? "rocm-chunked-c64-mfma-f32-few-rows-split-v2"
                                       : "rocm-chunked-c64-mfma-f16-operands-v1";
    return hk_write_identity(
        {{"device", dev},
         {"native_execution", "huncho-rocm-qwen35-v1"},
         {"device_path", "kev-rocm-gfx950-v1"},
         {"activation_dtype", dt},
         {"residual_stream_dtype", m->x_f32 ? "fp32" : dt},
         {"attention_compute_dtype", "fp32"},
         {"attention_execution", attn_exec},
         {"gqa_execution", "rocm-group-in-query-tile-v1"},
         {"paged_attention", "rocm-block-table-lds-gather-v1"},
         {"kv_storage", "rocm-pool-block-tables-v1"},
         {"kv_page_tokens", std::to_string(m->cfg.page_size)},
         {"delta_rule_execution", delta_exec},
         {"recurrent_state_dtype", "fp32"},
         {"causal_conv_execution", f32 || !gdn_mfma || c.conv_k != 4 ? "rocm-gdn-prep-v1" : "rocm-fused-gdn-layer-v1"},
         {"mlp_gate_execution", m->mlp_fused ? "rocm-gemm-swiglu-epilogue-v1" : "rocm-swiglu-v1"},
         {"projection_kernel", f32 ? "hipblaslt-pinned-or-heuristic-v1" : "rocm-gemm-few-rows-or-hipblaslt-v1"},
         {"pointer_head_dtype", "fp32"},
         {"library", hk_version()}},
        buf, len, needed);
}
