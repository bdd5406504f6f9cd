// blas.cpp - dense projections (candle Linear, qwen3_5.rs:306-515) on hipBLASLt.
//
// Row-major Y[n][out] = alpha * X[n][in] . W[out][in]^T + beta * C is the column-major
// product Y^T = W . X^T: m = out, n = n, k = in, op(A) = T on the weight, op(B) = N on the
// activations. bf16 or fp16 operands with fp32 accumulation (HIPBLAS_COMPUTE_32F), or fp32.
//
// Plans (descriptors + one algorithm per shape) are cached per shape. The algorithm is a
// deterministic function of the shape: the solution index pinned for it in kPinned (measured
// on MI355X with this hipBLASLt) when it supports the problem, else the heuristic's first
// choice. Building a plan allocates no device memory, times nothing and does not synchronise,
// so a forward stays stream-ordered on its first call for a batch shape. Timing every
// candidate is opt-in (hk_ctx_set_gemm_autotune): it allocates scratch, synchronises, and its
// choice then depends on the device's timing. The handle and the workspace belong to the
// context and are created by hk_blas_prepare (model creation), never inside a forward.
#include <hipblaslt/hipblaslt-ext.hpp>
#include <hipblaslt/hipblaslt.h>

#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "abi_internal.hpp"

namespace {

struct Plan {
    hipblasLtMatmulDesc_t desc = nullptr;
    hipblasLtMatrixLayout_t a = nullptr, b = nullptr, c = nullptr, d = nullptr;
    hipblasLtMatmulAlgo_t algo{};
    size_t ws = 0;
    int index = -1;      // hipBLASLt solution index
    const char* source = "";  // "pinned", "heuristic" or "timed"
};

// Solution indices pinned per (dtype, out, n, in, C operand) at the Kev-shaped 64 x 512 token
// batch and the ModernBERT-base-shaped 16-row batch (40,910 tokens), measured on MI355X (gfx950)
// with ROCm 7.2's hipBLASLt by timing every supported solution (hk_ctx_set_gemm_autotune) and
// keeping the fastest.
struct Pinned {
    int dtype, out, n, in, has_c, index;
    int cd = -1;  // C/D dtype; -1 = the operand dtype
};
const Pinned kPinned[] = {
    // bf16: [b | a] GDN columns, out_proj / o_proj (+ residual), down_proj (+ residual),
    // attention q|gate|k|v, MLP gate|up, GDN q|k|v|z
    {HK_BF16, 32, 32768, 1024, 0, 618524},   {HK_BF16, 1024, 32768, 2048, 1, 618612},
    {HK_BF16, 1024, 32768, 3584, 1, 618613}, {HK_BF16, 6144, 32768, 1024, 0, 618611},
    {HK_BF16, 7168, 32768, 1024, 0, 618611}, {HK_BF16, 8192, 32768, 1024, 0, 618611},
    // fp16, the same shapes
    {HK_F16, 32, 32768, 1024, 0, 625072},    {HK_F16, 1024, 32768, 2048, 1, 625107},
    {HK_F16, 1024, 32768, 3584, 1, 624960},  {HK_F16, 6144, 32768, 1024, 0, 625108},
    {HK_F16, 7168, 32768, 1024, 0, 625108},  {HK_F16, 8192, 32768, 1024, 0, 625108},
    // bf16 operands with an fp32 residual stream (C and D fp32): out_proj / o_proj, down_proj
    {HK_BF16, 1024, 32768, 2048, 1, 619295, HK_F32}, {HK_BF16, 1024, 32768, 3584, 1, 619295, HK_F32},
    // bf16 ModernBERT-base: Wqkv and Wi (GeGLU) 768 -> 2304, attention Wo (+ residual),
    // MLP Wo 1152 -> 768 (+ residual); 2.5 % of the encoder step over the heuristic's choices
    {HK_BF16, 2304, 40910, 768, 0, 618611},  {HK_BF16, 768, 40910, 768, 1, 618611},
    {HK_BF16, 768, 40910, 1152, 1, 618612},
};

typedef std::tuple<int, int, int, int, long, long, long, long, int, int> Key;  // ..., C/D dtype

}  // namespace

struct hk_blas {
    hipblasLtHandle_t handle = nullptr;
    void* workspace = nullptr;
    size_t ws_bytes = 0;
    bool autotune = false;
    std::map<Key, Plan> plans;
};

static const size_t kWorkspace = 128ull << 20;

void hk_blas_release(hk_ctx* ctx) {
    if (!ctx || !ctx->blas) return;
    hk_blas* b = ctx->blas;
    for (auto& kv : b->plans) {
        Plan& p = kv.second;
        if (p.a) hipblasLtMatrixLayoutDestroy(p.a);
        if (p.b) hipblasLtMatrixLayoutDestroy(p.b);
        if (p.c) hipblasLtMatrixLayoutDestroy(p.c);
        if (p.d) hipblasLtMatrixLayoutDestroy(p.d);
        if (p.desc) hipblasLtMatmulDescDestroy(p.desc);
    }
    if (b->workspace) hipFree(b->workspace);
    if (b->handle) hipblasLtDestroy(b->handle);
    delete b;
    ctx->blas = nullptr;
}

int hk_blas_prepare(hk_ctx* ctx) {
    if (ctx->blas) return HK_OK;
    hk_blas* b = new hk_blas();
    if (hipblasLtCreate(&b->handle) != HIPBLAS_STATUS_SUCCESS) {
        delete b;
        return hk_fail(ctx, HK_ERR_DEVICE, "hipblasLtCreate failed");
    }
    if (hipMalloc(&b->workspace, kWorkspace) != hipSuccess) {
        hipblasLtDestroy(b->handle);
        delete b;
        return hk_fail(ctx, HK_ERR_NOMEM, "GEMM workspace allocation failed");
    }
    b->ws_bytes = kWorkspace;
    ctx->blas = b;
    return HK_OK;
}

// Candidate algorithms for a plan: the heuristic's ranking first, then every other solution
// of the full list that supports the problem with the context's workspace.
static std::vector<std::pair<hipblasLtMatmulAlgo_t, size_t>> candidates(hk_ctx* ctx, Plan& p, hipDataType t,
                                                                          hipDataType tc,
                                                                          const hipblasLtMatmulHeuristicResult_t* res,
                                                                          int returned) {
    hk_blas* B = ctx->blas;
    std::vector<std::pair<hipblasLtMatmulAlgo_t, size_t>> out;
    std::vector<int> seen;
    for (int i = 0; i < returned; ++i) {
        if (res[i].state != HIPBLAS_STATUS_SUCCESS || res[i].workspaceSize > B->ws_bytes) continue;
        hipblasLtMatmulAlgo_t algo = res[i].algo;
        seen.push_back(hipblaslt_ext::getIndexFromAlgo(algo));
        out.emplace_back(algo, res[i].workspaceSize);
    }
    std::vector<hipblasLtMatmulHeuristicResult_t> all;
    if (hipblaslt_ext::getAllAlgos(B->handle, hipblaslt_ext::GemmType::HIPBLASLT_GEMM, HIPBLAS_OP_T, HIPBLAS_OP_N, t, t,
                                   tc, tc, HIPBLAS_COMPUTE_32F, all) != HIPBLAS_STATUS_SUCCESS)
        return out;
    const float one = 1.0f, zero = 0.0f;
    for (auto& r : all) {
        hipblasLtMatmulAlgo_t algo = r.algo;
        const int idx = hipblaslt_ext::getIndexFromAlgo(algo);
        if (std::find(seen.begin(), seen.end(), idx) != seen.end()) continue;
        size_t ws = 0;
        if (hipblaslt_ext::matmulIsAlgoSupported(B->handle, p.desc, &one, p.a, p.b, &zero, p.c, p.d, algo, ws) !=
                HIPBLAS_STATUS_SUCCESS ||
            ws > B->ws_bytes)
            continue;
        seen.push_back(idx);
        out.emplace_back(algo, ws);
    }
    return out;
}

// Times the candidates into a scratch output (the caller's buffers are untouched; with a C
// operand the scratch serves as C too, so the timed kernel reads C as the real call does):
// every candidate over 2 launches, then the best 8 in 3 interleaved rounds of 5 launches,
// keeping each one's fastest round. Returns the index of the fastest; 0 if timing fails.
static int pick_fastest(hk_ctx* ctx, Plan& p, std::vector<std::pair<hipblasLtMatmulAlgo_t, size_t>>& cands,
                        int cd_dtype, int n, const void* x, const void* w, long ldy, long ldc, bool has_c) {
    if (cands.size() <= 1) return 0;
    hk_blas* B = ctx->blas;
    void* scratch = nullptr;
    const size_t bytes = (size_t)std::max(ldy, ldc) * n * (cd_dtype == HK_F32 ? 4 : 2);
    if (hipMalloc(&scratch, bytes) != hipSuccess) return 0;
    hipEvent_t e0, e1;
    hipEventCreate(&e0);
    hipEventCreate(&e1);
    const float one = 1.0f, beta = has_c ? 1.0f : 0.0f;
    auto launch = [&](int i) {
        return hipblasLtMatmul(B->handle, p.desc, &one, w, p.a, x, p.b, &beta, scratch, p.c, scratch, p.d,
                               &cands[i].first, B->workspace, cands[i].second, ctx->stream) == HIPBLAS_STATUS_SUCCESS;
    };
    auto time_algo = [&](int i, int reps) -> float {
        bool ok = launch(i);
        hipEventRecord(e0, ctx->stream);
        for (int r = 0; ok && r < reps; ++r) ok = launch(i);
        hipEventRecord(e1, ctx->stream);
        float ms = 0.0f;
        if (!ok || hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess) return 1e30f;
        return ms / reps;
    };
    time_algo(0, 2);  // clocks up before the first measurement
    std::vector<std::pair<float, int>> t1;
    for (int i = 0; i < (int)cands.size(); ++i) t1.emplace_back(time_algo(i, 2), i);
    std::sort(t1.begin(), t1.end());
    int top = 0;
    while (top < (int)t1.size() && top < 8 && t1[top].first < 1e29f) ++top;
    std::vector<float> t2(top, 1e30f);
    for (int round = 0; round < 3; ++round)
        for (int k = 0; k < top; ++k) t2[k] = std::min(t2[k], time_algo(t1[k].second, 5));
    int best = t1[0].second;
    float best_ms = 1e30f;
    for (int k = 0; k < top; ++k)
        if (t2[k] < best_ms) {
            best_ms = t2[k];
            best = t1[k].second;
        }
    hipStreamSynchronize(ctx->stream);
    (void)hipGetLastError();
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    hipFree(scratch);
    return best;
}

int hk_gemm_xwt(hk_ctx* ctx, int dtype, int n, int out, int in, const void* x, long ldx, const void* w, long ldw,
                void* y, long ldy, const void* c, long ldc, float alpha, float beta) {
    return hk_gemm_xwt_cd(ctx, dtype, dtype, n, out, in, x, ldx, w, ldw, y, ldy, c, ldc, alpha, beta);
}

// The few-row kernel takes this product: 16-bit operands, whole K steps, 16-byte aligned rows and
// strides within its 32-bit copy offsets.
static bool few_rows_takes(int dtype, int epi, const hk::GemmArgs& a) {
    if (dtype != HK_BF16 && dtype != HK_F16) return false;
    const long ldc = a.c ? a.ldc : 0;
    const bool glu = epi == hk::EPI_SWIGLU || epi == hk::EPI_GEGLU;
    if (a.K <= 0 || a.K % 64 || a.N <= 0 || a.N % (glu ? 32 : 8) || a.N2 % 8 || a.ldx % 8 || a.ldw % 8 || a.ldy % 8 ||
        ldc % 8 || a.ldy2 % 8 || a.ldx >= 1 << 22 || a.ldw >= 1 << 22)
        return false;
    return (((uintptr_t)a.x | (uintptr_t)a.w | (uintptr_t)a.c | (uintptr_t)a.y | (uintptr_t)a.w2 | (uintptr_t)a.y2) & 15) == 0;
}

// Estimated times (us) of a product on the few-row kernel and on the library's.
static float few_rows_us(int epi, const hk::GemmArgs& a) {
    return 2.2f + (float)a.K / 1024.0f * hk_gemm_few_rows_cost(epi, &a);
}
static float library_us(const hk::GemmArgs& a) {
    return 5.0f + 2.2f * (float)a.K / 1024.0f + 0.9f * 2e-9f * (float)a.M * (float)a.N * (float)a.K;
}
// A model's projection takes the few-row kernel where its estimate is the lower one by 7 %. Measured beside the
// library's choice (bf16, weights from HBM): 8192 x 1024 at 169 rows 9.3 against 12.7, at 360 rows 14.3 and
// 13.8, at 512 rows 17.0 and 14.8, at 600 (library) 22 and 16.4; 1024 x 3584 + residual at 300 rows 12.3 against
// 17.2, at 1024 (library) 19.6 and 18.9, at 4096 (library) 46.1 and 36.6; 768 x 1152 + residual at 1700 rows 9.8 against
// 10.6, at 2704 (library) 14.6 and 12.7; 32 x 1024 at 16384 rows 5.4 against 10.1, at 32768 (library) 11.7 and 13.2.
// The few-row kernel's sums do not depend on the number of rows. The library's choice for the smallest batches
// adds in another order, and there the two differ by the rounding of their sums: up to 16 rows of 2304 to 8192
// columns, 31 of 768 x 768, 127 of 1024 columns + residual, and up to 160 and around 330 of 768 x 1152.
static bool few_rows_wins(int epi, const hk::GemmArgs& a) { return few_rows_us(epi, a) <= 0.93f * library_us(a); }
// The way such a projection takes, estimated
static float projection_us(const hk::GemmArgs& a) {
    return std::min(few_rows_us(hk::EPI_STORE, a), 0.93f * library_us(a));
}

int hk_gemm_xwt_pair(hk_ctx* ctx, int dtype, int n, int in, const void* x, long ldx, int out, const void* w, void* y,
                     int out2, const void* w2, void* y2) {
    const hk::GemmArgs a{x, w, nullptr, y, ldx, in, 0, out, n, out, in, w2, y2, out2, out2};
    const hk::GemmArgs a1{x, w, nullptr, y, ldx, in, 0, out, n, out, in, nullptr, nullptr, 0, 0},
        a2{x, w2, nullptr, y2, ldx, in, 0, out2, n, out2, in, nullptr, nullptr, 0, 0};
    // (one launch for both: 8192 and 32 columns x 1024 at 169 rows 10.7 us, two of this kernel 13.9; at 360 rows
    // 15.6 and 18.9; at 200 rows the columns of the second are a round of tiles of their own, 14.5 both ways)
    if (n > 0 && ctx->blas && !ctx->blas->autotune && few_rows_takes(dtype, hk::EPI_STORE, a) &&
        few_rows_us(hk::EPI_STORE, a) <= projection_us(a1) + projection_us(a2))
        return hk_launch_gemm_few_rows(dtype, hk::EPI_STORE, &a, ctx->stream) ? hk_fail(ctx, HK_ERR_DEVICE, "gemm launch failed")
                                                                           : HK_OK;
    if (int rc = hk_gemm_xwt(ctx, dtype, n, out, in, x, ldx, w, in, y, out, nullptr, 0, 1.0f, 0.0f)) return rc;
    return hk_gemm_xwt(ctx, dtype, n, out2, in, x, ldx, w2, in, y2, out2, nullptr, 0, 1.0f, 0.0f);
}

// The encoder's GeGLU in the projection's epilogue, one launch and one pass over 2 inter columns less (encoder of
// 22 layers, 653 rows: 1256 -> 1234 us; two runs of one side differ by 0.2 %): where the estimate is below that
// of the projection and a pass of 2.5 us. For many rows the pass on its own is the faster way (erf in
// the epilogue of large tiles leaves the matrix cores idle).
bool hk_gemm_geglu_few_rows(hk_ctx* ctx, int dtype, int n, int inter, int in, const void* x, const void* w, void* y, int* rc) {
    const hk::GemmArgs a{x, w, nullptr, y, in, in, 0, inter, n, 2 * inter, in, nullptr, nullptr, 0, 0};
    if (n <= 0 || !ctx->blas || ctx->blas->autotune || 4L * inter * in >= 1L << 31 || !few_rows_takes(dtype, hk::EPI_GEGLU, a) ||
        few_rows_us(hk::EPI_GEGLU, a) > projection_us(a) + 2.5f)
        return false;
    *rc = hk_launch_gemm_few_rows(dtype, hk::EPI_GEGLU, &a, ctx->stream) ? hk_fail(ctx, HK_ERR_DEVICE, "gemm launch failed")
                                                                         : HK_OK;
    return true;
}

int hk_gemm_xwt_cd(hk_ctx* ctx, int dtype, int cd_dtype, int n, int out, int in, const void* x, long ldx,
                   const void* w, long ldw, void* y, long ldy, const void* c, long ldc, float alpha, float beta) {
    if (n == 0 || out == 0) return HK_OK;
    if (!ctx->blas) return hk_fail(ctx, HK_ERR_INVALID, "GEMM state not prepared (hk_blas_prepare at model creation)");
    hk_blas* B = ctx->blas;
    const bool has_c = c != nullptr && beta != 0.0f;
    if (!B->autotune && alpha == 1.0f && (!has_c || beta == 1.0f) && (cd_dtype == dtype || (has_c && cd_dtype == HK_F32))) {
        const int epi = !has_c ? hk::EPI_STORE : cd_dtype == dtype ? hk::EPI_RESIDUAL : hk::EPI_RESIDUAL_F32;
        const hk::GemmArgs a{x, w, has_c ? c : nullptr, y, ldx, ldw, has_c ? ldc : 0, ldy, n, out, in, nullptr, nullptr, 0, 0};
        if (few_rows_takes(dtype, epi, a) && few_rows_wins(epi, a))
            return hk_launch_gemm_few_rows(dtype, epi, &a, ctx->stream) ? hk_fail(ctx, HK_ERR_DEVICE, "gemm launch failed")
                                                                     : HK_OK;
    }
    if (!has_c) {
        c = y;
        ldc = ldy;
    }
    Key key{dtype, out, n, in, ldw, ldx, ldy, ldc, has_c ? 1 : 0, cd_dtype};
    auto it = B->plans.find(key);
    if (it == B->plans.end()) {
        Plan p;
        auto hip_type = [](int d) { return d == HK_BF16 ? HIP_R_16BF : d == HK_F16 ? HIP_R_16F : HIP_R_32F; };
        const hipDataType t = hip_type(dtype), tc = hip_type(cd_dtype);
        bool ok = hipblasLtMatmulDescCreate(&p.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F) == HIPBLAS_STATUS_SUCCESS;
        hipblasOperation_t opT = HIPBLAS_OP_T, opN = HIPBLAS_OP_N;
        ok = ok && hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSA, &opT, sizeof(opT)) ==
                       HIPBLAS_STATUS_SUCCESS;
        ok = ok && hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSB, &opN, sizeof(opN)) ==
                       HIPBLAS_STATUS_SUCCESS;
        ok = ok && hipblasLtMatrixLayoutCreate(&p.a, t, in, out, ldw) == HIPBLAS_STATUS_SUCCESS;
        ok = ok && hipblasLtMatrixLayoutCreate(&p.b, t, in, n, ldx) == HIPBLAS_STATUS_SUCCESS;
        ok = ok && hipblasLtMatrixLayoutCreate(&p.c, tc, out, n, ldc) == HIPBLAS_STATUS_SUCCESS;
        ok = ok && hipblasLtMatrixLayoutCreate(&p.d, tc, out, n, ldy) == HIPBLAS_STATUS_SUCCESS;
        hipblasLtMatmulPreference_t pref = nullptr;
        ok = ok && hipblasLtMatmulPreferenceCreate(&pref) == HIPBLAS_STATUS_SUCCESS;
        uint64_t wsmax = B->ws_bytes;
        ok = ok && hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &wsmax,
                                                         sizeof(wsmax)) == HIPBLAS_STATUS_SUCCESS;
        hipblasLtMatmulHeuristicResult_t res[16];
        int returned = 0;
        ok = ok && hipblasLtMatmulAlgoGetHeuristic(B->handle, p.desc, p.a, p.b, p.c, p.d, pref, 16, res, &returned) ==
                       HIPBLAS_STATUS_SUCCESS;
        if (pref) hipblasLtMatmulPreferenceDestroy(pref);
        if (!ok || returned == 0) {
            if (p.a) hipblasLtMatrixLayoutDestroy(p.a);
            if (p.b) hipblasLtMatrixLayoutDestroy(p.b);
            if (p.c) hipblasLtMatrixLayoutDestroy(p.c);
            if (p.d) hipblasLtMatrixLayoutDestroy(p.d);
            if (p.desc) hipblasLtMatmulDescDestroy(p.desc);
            return hk_fail(ctx, HK_ERR_UNSUPPORTED, "no hipBLASLt algorithm for %dx%dx%d", out, n, in);
        }
        auto destroy = [&]() {
            hipblasLtMatrixLayoutDestroy(p.a);
            hipblasLtMatrixLayoutDestroy(p.b);
            hipblasLtMatrixLayoutDestroy(p.c);
            hipblasLtMatrixLayoutDestroy(p.d);
            hipblasLtMatmulDescDestroy(p.desc);
        };
        if (B->autotune) {
            auto cands = candidates(ctx, p, t, tc, res, returned);
            if (cands.empty()) {
                destroy();
                return hk_fail(ctx, HK_ERR_UNSUPPORTED, "no usable hipBLASLt algorithm for %dx%dx%d", out, n, in);
            }
            const int best = pick_fastest(ctx, p, cands, cd_dtype, n, x, w, ldy, ldc, has_c);
            p.algo = cands[best].first;
            p.ws = cands[best].second;
            p.source = "timed";
        } else {
            // the pinned solution when it supports this problem, else the heuristic's first
            // usable choice
            bool chosen = false;
            for (const Pinned& e : kPinned) {
                if (e.index < 0 || e.dtype != dtype || (e.cd < 0 ? e.dtype : e.cd) != cd_dtype || e.out != out || e.n != n || e.in != in ||
                    e.has_c != (has_c ? 1 : 0) || ldw != in || ldx != in || ldy != out || ldc != out)
                    continue;
                std::vector<int> idx{e.index};
                std::vector<hipblasLtMatmulHeuristicResult_t> got;
                if (hipblaslt_ext::getAlgosFromIndex(B->handle, idx, got) != HIPBLAS_STATUS_SUCCESS || got.empty())
                    break;
                const float one = 1.0f, zero = 0.0f;
                size_t ws = 0;
                if (hipblaslt_ext::matmulIsAlgoSupported(B->handle, p.desc, &one, p.a, p.b, &zero, p.c, p.d,
                                                         got[0].algo, ws) == HIPBLAS_STATUS_SUCCESS &&
                    ws <= B->ws_bytes) {
                    p.algo = got[0].algo;
                    p.ws = ws;
                    p.source = "pinned";
                    chosen = true;
                }
                break;
            }
            for (int i = 0; !chosen && i < returned; ++i) {
                if (res[i].state != HIPBLAS_STATUS_SUCCESS || res[i].workspaceSize > B->ws_bytes) continue;
                p.algo = res[i].algo;
                p.ws = res[i].workspaceSize;
                p.source = "heuristic";
                chosen = true;
            }
            if (!chosen) {
                destroy();
                return hk_fail(ctx, HK_ERR_UNSUPPORTED, "no usable hipBLASLt algorithm for %dx%dx%d", out, n, in);
            }
        }
        p.index = hipblaslt_ext::getIndexFromAlgo(p.algo);
        it = B->plans.emplace(key, p).first;
    }
    Plan& p = it->second;
    hipblasStatus_t st = hipblasLtMatmul(B->handle, p.desc, &alpha, w, p.a, x, p.b, &beta, c, p.c, y, p.d, &p.algo,
                                         B->workspace, p.ws, ctx->stream);
    if (st != HIPBLAS_STATUS_SUCCESS) return hk_fail(ctx, HK_ERR_DEVICE, "hipblasLtMatmul failed (%d)", (int)st);
    return HK_OK;
}

extern "C" int hk_ctx_set_gemm_autotune(hk_ctx* ctx, int enable) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = hk_blas_prepare(ctx)) return rc;
    ctx->blas->autotune = enable != 0;
    return HK_OK;
}

extern "C" int hk_ctx_gemm_plans(hk_ctx* ctx, char* buf, size_t len, size_t* needed) {
    if (!ctx) return HK_ERR_INVALID;
    std::string out;
    if (ctx->blas) {
        char line[160];
        for (auto& kv : ctx->blas->plans) {
            const Key& k = kv.first;
            snprintf(line, sizeof line,
                     "dtype=%d out=%d n=%d in=%d ldw=%ld ldx=%ld ldy=%ld ldc=%ld c=%d cd=%d index=%d %s\n",
                     std::get<0>(k), std::get<1>(k), std::get<2>(k), std::get<3>(k), std::get<4>(k), std::get<5>(k),
                     std::get<6>(k), std::get<7>(k), std::get<8>(k), std::get<9>(k), kv.second.index,
                     kv.second.source);
            out += line;
        }
    }
    if (needed) *needed = out.size() + 1;
    if (buf && len) {
        const size_t n = out.size() < len - 1 ? out.size() : len - 1;
        memcpy(buf, out.data(), n);
        buf[n] = 0;
    }
    return HK_OK;
}

// The library's own MFMA GEMM (gemm.hip) for 16-bit operands: N a multiple of 256, K of 64, rows
// 16-byte aligned. Returns HK_ERR_UNSUPPORTED (without an error message) for other shapes.
int hk_gemm_native(hk_ctx* ctx, int dtype, int epi, int n, int out, int in, const void* x, long ldx, const void* w,
                   long ldw, void* y, long ldy, const void* c, long ldc) {
    if (dtype != HK_BF16 && dtype != HK_F16) return HK_ERR_UNSUPPORTED;
    if (out % 256 || in % 64 || n < 0 || ldx % 8 || ldw % 8 || ldy % 8 || (epi == hk::EPI_RESIDUAL && ldc % 8) ||
        (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)(c ? c : y)) & 15))
        return HK_ERR_UNSUPPORTED;
    if (n == 0) return HK_OK;
    hk::GemmArgs a{x, w, epi == hk::EPI_RESIDUAL ? c : nullptr, y, ldx, ldw, ldc, ldy, n, out, in, nullptr, nullptr, 0, 0};
    // The 256 x 256 tiles of gemm.hip cost about 30 K / 1024 us per round of 256 workgroups, however few
    // the rows; the few-row kernel's tiles less while there are few of them (7168 x 1024 SwiGLU at 600
    // rows 21 against 33 us, at 1700 rows 39 and 37; 1024 x 3584 + residual at 4096 rows 46 against 99, at 8192 rows
    // 88 against 109, at 16384 rows 165 and 115).
    const int tiles = out / 256 * ((n + 255) / 256);
    if (few_rows_takes(dtype, epi, a) && hk_gemm_few_rows_cost(epi, &a) < 30.0f * (float)((tiles + 255) / 256))
        return hk_launch_gemm_few_rows(dtype, epi, &a, ctx->stream) ? hk_fail(ctx, HK_ERR_DEVICE, "gemm launch failed") : HK_OK;
    return hk_launch_gemm(dtype, epi, &a, ctx->stream) ? hk_fail(ctx, HK_ERR_DEVICE, "gemm launch failed") : HK_OK;
}

extern "C" int hk_linear(hk_ctx* ctx, int dtype, int epilogue, const void* x, long ldx, const void* w, long ldw,
                         int rows, int out, int in, const void* c, long ldc, void* y, long ldy) {
    if (!ctx) return HK_ERR_INVALID;
    if (!x || !w || !y || rows < 0 || out <= 0 || in <= 0 || epilogue < 0 || epilogue > 2 ||
        (epilogue == hk::EPI_RESIDUAL && !c))
        return hk_fail(ctx, HK_ERR_INVALID, "linear: bad arguments");
    const int y_cols = epilogue == hk::EPI_SWIGLU ? out / 2 : out;
    if (ldx < in || ldw < in || ldy < y_cols || (c && ldc < out))
        return hk_fail(ctx, HK_ERR_INVALID, "linear: row strides smaller than the rows");
    hipSetDevice(ctx->device);
    const int rc = hk_gemm_native(ctx, dtype, epilogue, rows, out, in, x, ldx, w, ldw, y, ldy, c, ldc);
    if (rc == HK_ERR_UNSUPPORTED)
        return hk_fail(ctx, rc, "linear: 16-bit dtype, out %% 256 == 0, in %% 64 == 0 and 16-byte aligned rows "
                                "are required (got out %d, in %d)", out, in);
    return rc;
}
