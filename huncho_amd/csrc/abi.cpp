// abi.cpp - host side of the libhuncho_rocm C ABI: context, error model, argument
// validation and launch of the gfx950 kernels. See include/huncho_rocm.h.
#include "abi_internal.hpp"

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>


// ---------------------------------------------------------------------------
// context and errors
// ---------------------------------------------------------------------------

int hk_fail(hk_ctx* ctx, int code, const char* fmt, ...) {
    if (ctx) {
        char buf[512];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(buf, sizeof(buf), fmt, ap);
        va_end(ap);
        ctx->last_error = buf;
    }
    return code;
}

int hk_check_hip(hk_ctx* ctx, hipError_t e, const char* what) {
    if (e == hipSuccess) return HK_OK;
    return hk_fail(ctx, HK_ERR_DEVICE, "%s: %s", what, hipGetErrorString(e));
}

extern "C" int hk_device_count(int* out) {
    if (!out) return HK_ERR_INVALID;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
    *out = n;
    return HK_OK;
}

extern "C" const char* hk_version(void) { return "huncho_rocm 0.1 (gfx950)"; }

// Blocks of split scratch. One per device is kept when its context is destroyed, for the next context, and freed
// with the device's last context.
namespace {
struct SplitPool {
    std::mutex lock;
    struct Device {
        int contexts = 0;
        void* spare = nullptr;
    };
    std::map<int, Device> devices;
};
SplitPool& split_pool() {
    static SplitPool* pool = new SplitPool();  // outlives contexts that are destroyed as the process ends
    return *pool;
}

// A block on the current device, or null
void* split_block_take(int device, int new_contexts) {
    void* p;
    {
        std::lock_guard<std::mutex> guard(split_pool().lock);
        SplitPool::Device& d = split_pool().devices[device];
        d.contexts += new_contexts;
        p = d.spare;
        d.spare = nullptr;
    }
    if (!p && hipMalloc(&p, kSplitScratch) != hipSuccess) {
        (void)hipGetLastError();
        p = nullptr;
    }
    return p;
}

// Work on the blocks has ended; the context is gone.
void split_blocks_give(int device, void* a, void* b) {
    void* drop[3] = {a, b, nullptr};
    {
        std::lock_guard<std::mutex> guard(split_pool().lock);
        SplitPool::Device& d = split_pool().devices[device];
        if (--d.contexts == 0) {
            drop[2] = d.spare;
            d.spare = nullptr;
        } else if (!d.spare) {
            d.spare = a;
            drop[0] = nullptr;
        }
    }
    for (void* p : drop)
        if (p) hipFree(p);
}
}  // namespace

extern "C" int hk_ctx_create(int device_ordinal, hk_ctx** out) {
    if (!out) return HK_ERR_INVALID;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return HK_ERR_UNSUPPORTED;
    if (device_ordinal < 0 || device_ordinal >= n) return HK_ERR_INVALID;
    if (hipSetDevice(device_ordinal) != hipSuccess) return HK_ERR_DEVICE;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device_ordinal) != hipSuccess) return HK_ERR_DEVICE;
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) return HK_ERR_UNSUPPORTED;
    hk_ctx* ctx = new hk_ctx();
    ctx->device = device_ordinal;
    ctx->prop = prop;
    if (hipStreamCreateWithFlags(&ctx->own_stream, hipStreamNonBlocking) != hipSuccess) {
        delete ctx;
        return HK_ERR_DEVICE;
    }
    ctx->stream = ctx->own_stream;
    if (hipMalloc(&ctx->fault_dev, 256) != hipSuccess) {
        hipStreamDestroy(ctx->own_stream);
        delete ctx;
        return HK_ERR_NOMEM;
    }
    if (hipMemset(ctx->fault_dev, 0, 256) != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
        hipFree(ctx->fault_dev);
        hipStreamDestroy(ctx->own_stream);
        delete ctx;
        return HK_ERR_DEVICE;
    }
    ctx->split_scratch = split_block_take(device_ordinal, 1);
    // the no-allocation entry point's scratch address on this device (retried on its first call
    // if this fails)
    hk_noalloc_scratch_init(device_ordinal);
    *out = ctx;
    return HK_OK;
}

extern "C" int hk_ctx_destroy(hk_ctx* ctx) {
    if (!ctx) return HK_ERR_INVALID;
    hipSetDevice(ctx->device);
    hipStreamSynchronize(ctx->stream);
    hk_noalloc_scratch_release(ctx);
    hk_blas_release(ctx);
    // the scratch's last use may be on a stream that the context has left
    if (ctx->split_used && (ctx->split_done || ctx->split_stream != ctx->stream)) hipDeviceSynchronize();
    split_blocks_give(ctx->device, ctx->split_scratch, ctx->split_first);
    if (ctx->split_done) hipEventDestroy(ctx->split_done);
    if (ctx->fault_dev) hipFree(ctx->fault_dev);
    if (ctx->own_stream) hipStreamDestroy(ctx->own_stream);
    delete ctx;
    return HK_OK;
}

extern "C" int hk_ctx_set_stream(hk_ctx* ctx, void* hip_stream) {
    if (!ctx) return HK_ERR_INVALID;
    ctx->stream = (hipStream_t)hip_stream;  // NULL is HIP's null stream
    return HK_OK;
}

size_t hk_gdn_split_bytes(int n_tokens, int n_seqs, int heads) {
    return (size_t)(n_tokens / 64 + n_seqs) * heads * hk::HK_GDN_SPLIT_SLOT;
}

// The scratch for a call on the context's stream, after its last use on another one; null: the call needs more
// than there is, or the stream is being captured (a graph may be replayed on any stream).
// An event per use costs 3 to 4 us (attention of 1 x 30 / 1030: 12.6 and 15.6), and an event on the stream that is
// left cannot be had later, when that stream may be gone. So a context that stays on one stream records none. From
// its first use on a second stream on it records one per use, and it leaves the block of the uses before,
// whose end nothing marks, alone until it is destroyed. (A stream that got the handle of a destroyed one
// counts as the same: hipStreamDestroy returns when the stream's work is done, measured with 42 ms of it.)
static void* split_scratch_for(hk_ctx* ctx, size_t bytes) {
    if (!ctx->split_scratch || bytes > kSplitScratch) return nullptr;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (ctx->split_used && ctx->split_stream != ctx->stream) {
        if (ctx->split_done) {
            if (hipStreamWaitEvent(ctx->stream, ctx->split_done, 0) != hipSuccess) {
                (void)hipGetLastError();
                return nullptr;
            }
        } else {
            if (hipEventCreateWithFlags(&ctx->split_done, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                ctx->split_done = nullptr;
                return nullptr;
            }
            ctx->split_first = ctx->split_scratch;
            ctx->split_scratch = split_block_take(ctx->device, 0);
            if (!ctx->split_scratch) return nullptr;
        }
    }
    return ctx->split_scratch;
}

// After the last launch of a use
static void split_scratch_done(hk_ctx* ctx) {
    ctx->split_used = true;
    ctx->split_stream = ctx->stream;
    if (!ctx->split_done || hipEventRecord(ctx->split_done, ctx->stream) == hipSuccess) return;
    (void)hipGetLastError();
    hipStreamSynchronize(ctx->stream);
}

extern "C" void* hk_ctx_own_stream(hk_ctx* ctx) { return ctx ? (void*)ctx->own_stream : nullptr; }

extern "C" void* hk_ctx_stream(hk_ctx* ctx) { return ctx ? (void*)ctx->stream : nullptr; }

extern "C" int hk_ctx_synchronize(hk_ctx* ctx) {
    if (!ctx) return HK_ERR_INVALID;
    hipSetDevice(ctx->device);
    return hk_check_hip(ctx, hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
}

extern "C" const char* hk_ctx_last_error(hk_ctx* ctx) { return ctx ? ctx->last_error.c_str() : "no context"; }

extern "C" int hk_ctx_device_info(hk_ctx* ctx, hk_device_info_t* out) {
    if (!ctx || !out) return HK_ERR_INVALID;
    memset(out, 0, sizeof(*out));
    snprintf(out->name, sizeof(out->name), "%s", ctx->prop.gcnArchName);
    out->compute_units = ctx->prop.multiProcessorCount;
    out->clock_khz = ctx->prop.clockRate;
    out->mem_clock_khz = ctx->prop.memoryClockRate;
    out->mem_bus_width = ctx->prop.memoryBusWidth;
    out->total_mem = ctx->prop.totalGlobalMem;
    out->lds_per_block = ctx->prop.sharedMemPerBlock;
    out->l2_bytes = ctx->prop.l2CacheSize;
    return HK_OK;
}

extern "C" int hk_ctx_take_faults(hk_ctx* ctx, int* faults_out) {
    if (!ctx || !faults_out) return HK_ERR_INVALID;
    hipSetDevice(ctx->device);
    int f = 0;
    int rc = hk_check_hip(ctx, hipMemcpyAsync(&f, ctx->fault_dev, sizeof(int), hipMemcpyDeviceToHost, ctx->stream),
                          "fault flag read");
    if (rc) return rc;
    rc = hk_check_hip(ctx, hipStreamSynchronize(ctx->stream), "fault flag sync");
    if (rc) return rc;
    *faults_out = f;
    if (f) {
        int zero = 0;
        rc = hk_check_hip(ctx, hipMemcpyAsync(ctx->fault_dev, &zero, sizeof(int), hipMemcpyHostToDevice, ctx->stream),
                          "fault flag clear");
        if (rc) return rc;
        rc = hk_check_hip(ctx, hipStreamSynchronize(ctx->stream), "fault flag clear sync");
    }
    return rc;
}

extern "C" int hk_buffer_alloc(hk_ctx* ctx, size_t bytes, void** dev_out) {
    if (!ctx || !dev_out) return HK_ERR_INVALID;
    *dev_out = nullptr;
    if (bytes == 0) return HK_OK;
    hipSetDevice(ctx->device);
    if (hipMalloc(dev_out, bytes) != hipSuccess) {
        (void)hipGetLastError();
        *dev_out = nullptr;
        return hk_fail(ctx, HK_ERR_NOMEM, "hipMalloc of %zu bytes failed", bytes);
    }
    return HK_OK;
}

extern "C" int hk_buffer_free(hk_ctx* ctx, void* dev) {
    if (!ctx) return HK_ERR_INVALID;
    if (!dev) return HK_OK;
    hipSetDevice(ctx->device);
    return hk_check_hip(ctx, hipFree(dev), "hipFree");
}

extern "C" int hk_memcpy_h2d(hk_ctx* ctx, void* dev_dst, const void* host_src, size_t bytes) {
    if (!ctx || ((!dev_dst || !host_src) && bytes)) return HK_ERR_INVALID;
    if (!bytes) return HK_OK;
    hipSetDevice(ctx->device);
    return hk_check_hip(ctx, hipMemcpyAsync(dev_dst, host_src, bytes, hipMemcpyHostToDevice, ctx->stream), "h2d copy");
}

extern "C" int hk_memcpy_d2h(hk_ctx* ctx, void* host_dst, const void* dev_src, size_t bytes) {
    if (!ctx || ((!host_dst || !dev_src) && bytes)) return HK_ERR_INVALID;
    if (!bytes) return HK_OK;
    hipSetDevice(ctx->device);
    int rc = hk_check_hip(ctx, hipMemcpyAsync(host_dst, dev_src, bytes, hipMemcpyDeviceToHost, ctx->stream), "d2h copy");
    return rc ? rc : hk_check_hip(ctx, hipStreamSynchronize(ctx->stream), "d2h sync");
}

// ---------------------------------------------------------------------------
// host helpers: rope table, calibration, synthetic inputs
// ---------------------------------------------------------------------------

static inline uint16_t f32_to_bf16_bits(float x) {
    uint32_t u;
    memcpy(&u, &x, 4);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return (uint16_t)((u >> 16) | 0x40u);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
static inline uint16_t f32_to_f16_bits(float x) {
    // round-to-nearest-even IEEE binary16 (finite inputs; overflow saturates to inf)
    uint32_t u;
    memcpy(&u, &x, 4);
    const uint32_t sign = (u >> 16) & 0x8000u;
    const uint32_t au = u & 0x7fffffffu;
    if (au >= 0x47800000u) return (uint16_t)(sign | (au > 0x7f800000u ? 0x7e00u : 0x7c00u));
    if (au < 0x38800000u) {  // subnormal half: quantum 2^-24
        float ax;
        memcpy(&ax, &au, 4);
        const uint32_t m = (uint32_t)nearbyintf(ax * 16777216.0f);
        return (uint16_t)(sign | m);
    }
    const uint32_t r = au + 0x0fffu + ((au >> 13) & 1u) - 0x38000000u;
    return (uint16_t)(sign | (r >> 13));
}
static inline float f16_bits_to_f32(uint16_t hbits) {
    const uint32_t sign = (uint32_t)(hbits & 0x8000u) << 16;
    const uint32_t e = (hbits >> 10) & 0x1fu, m = hbits & 0x3ffu;
    float v;
    if (e == 0) {
        v = (float)m * (1.0f / 16777216.0f);
    } else if (e == 31) {
        v = m ? NAN : INFINITY;
    } else {
        uint32_t u = ((e + 112u) << 23) | (m << 13);
        memcpy(&v, &u, 4);
    }
    uint32_t bits;
    memcpy(&bits, &v, 4);
    bits |= sign;
    memcpy(&v, &bits, 4);
    return v;
}
float hk_host_f16_to_f32(uint16_t b) { return f16_bits_to_f32(b); }
uint16_t hk_host_f32_to_f16(float x) { return f32_to_f16_bits(x); }

static inline float bf16_bits_to_f32(uint16_t b) {
    uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

extern "C" int hk_rope_fill_table(int rd, double theta, int max_pos, int round_dtype, float* cos_host, float* sin_host) {
    if (rd < 2 || (rd & 1) || max_pos < 0 || !cos_host || !sin_host || !(theta > 0)) return HK_ERR_INVALID;
    const int half = rd / 2;
    for (int p = 0; p < max_pos; ++p)
        for (int i = 0; i < half; ++i) {
            // qwen3_5.rs:229-244: inv_freq in f32, pos * inv_freq in f32, cos/sin in f32
            float inv = powf((float)theta, -(2.0f * (float)i) / (float)rd);
            float f = (float)p * inv;
            float c = cosf(f), s = sinf(f);
            if (round_dtype == HK_BF16) {
                c = bf16_bits_to_f32(f32_to_bf16_bits(c));
                s = bf16_bits_to_f32(f32_to_bf16_bits(s));
            } else if (round_dtype == HK_F16) {
                c = f16_bits_to_f32(f32_to_f16_bits(c));
                s = f16_bits_to_f32(f32_to_f16_bits(s));
            }
            cos_host[(size_t)p * half + i] = c;
            sin_host[(size_t)p * half + i] = s;
        }
    return HK_OK;
}

extern "C" int hk_calibrate(const float* logits, int n, float temperature, float* probs) {
    if (n < 0 || (n > 0 && (!logits || !probs))) return HK_ERR_INVALID;
    if (!(temperature > 0.0f) || !isfinite(temperature)) return HK_ERR_INVALID;
    for (int i = 0; i < n; ++i)
        if (!isfinite(logits[i])) return HK_ERR_INVALID;
    if (n == 0) return HK_OK;
    const float inv_t = 1.0f / temperature;
    float m = -INFINITY;
    for (int i = 0; i < n; ++i) m = logits[i] > m ? logits[i] : m;
    double sum = 0.0;
    for (int i = 0; i < n; ++i) {
        float e = expf((logits[i] - m) * inv_t);
        probs[i] = e;
        sum += (double)e;
    }
    for (int i = 0; i < n; ++i) {
        probs[i] = (float)((double)probs[i] / sum);
        if (!isfinite(probs[i])) return HK_ERR_INVALID;
    }
    return HK_OK;
}

static inline uint64_t splitmix64(uint64_t* s) {
    uint64_t z = (*s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
static inline uint64_t stream_state(uint64_t seed, uint64_t stream) { return seed ^ (stream * 0xD1B54A32D192ED03ull); }

template <typename F>
static void normal_stream(uint64_t seed, uint64_t stream, size_t n, float mean, float std, F&& put) {
    uint64_t s = stream_state(seed, stream);
    const double two_pi = 6.283185307179586476925286766559;
    for (size_t i = 0; i < n; i += 2) {
        uint64_t z = splitmix64(&s);
        double u1 = ((double)(z >> 40) + 0.5) * (1.0 / 16777216.0);
        double u2 = (double)((z >> 16) & 0xFFFFFFull) * (1.0 / 16777216.0);
        double r = sqrt(-2.0 * log(u1));
        put(i, (float)(mean + std * (r * cos(two_pi * u2))));
        if (i + 1 < n) put(i + 1, (float)(mean + std * (r * sin(two_pi * u2))));
    }
}

extern "C" int hk_synth_normal(uint64_t seed, uint64_t stream, float* out, size_t n, float mean, float std) {
    if (!out && n) return HK_ERR_INVALID;
    normal_stream(seed, stream, n, mean, std, [&](size_t i, float v) { out[i] = v; });
    return HK_OK;
}

extern "C" int hk_synth_normal_bf16(uint64_t seed, uint64_t stream, uint16_t* out, size_t n, float mean, float std) {
    if (!out && n) return HK_ERR_INVALID;
    normal_stream(seed, stream, n, mean, std, [&](size_t i, float v) { out[i] = f32_to_bf16_bits(v); });
    return HK_OK;
}

static uint64_t uniform_below(uint64_t* s, uint64_t range) {
    uint64_t limit = UINT64_MAX - (UINT64_MAX % range);
    uint64_t z;
    do {
        z = splitmix64(s);
    } while (z >= limit);
    return z % range;
}

extern "C" int hk_synth_uniform_int(uint64_t seed, uint64_t stream, int32_t* out, size_t n, int32_t lo, int32_t hi) {
    if ((!out && n) || hi < lo) return HK_ERR_INVALID;
    uint64_t s = stream_state(seed, stream);
    uint64_t range = (uint64_t)((int64_t)hi - (int64_t)lo + 1);
    for (size_t i = 0; i < n; ++i) out[i] = (int32_t)((int64_t)lo + (int64_t)uniform_below(&s, range));
    return HK_OK;
}

extern "C" int hk_synth_permutation(uint64_t seed, uint64_t stream, int32_t* out, int32_t n) {
    if (n < 0 || (!out && n)) return HK_ERR_INVALID;
    uint64_t s = stream_state(seed, stream);
    for (int32_t i = 0; i < n; ++i) out[i] = i;
    for (int32_t i = n - 1; i > 0; --i) {
        int32_t j = (int32_t)uniform_below(&s, (uint64_t)i + 1);
        int32_t t = out[i];
        out[i] = out[j];
        out[j] = t;
    }
    return HK_OK;
}

// ---------------------------------------------------------------------------
// validated ops
// ---------------------------------------------------------------------------

static int log2_exact(int v) {
    if (v <= 0 || (v & (v - 1))) return -1;
    int s = 0;
    while ((1 << s) < v) ++s;
    return s;
}

#define REQUIRE(cond, ...)                                              \
    do {                                                                \
        if (!(cond)) return hk_fail(ctx, HK_ERR_INVALID, __VA_ARGS__); \
    } while (0)

static int check_dtype(hk_ctx* ctx, int dtype) {
    if (dtype != HK_F32 && dtype != HK_BF16 && dtype != HK_F16)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "dtype %d is not supported", dtype);
    return HK_OK;
}

int hk_qk_norm_rope_kv_write_impl(hk_ctx* ctx, int dtype, const void* q_in, long q_in_tok, long q_in_head,
                                  const void* k_in, long k_in_tok, const void* v_in, long v_in_tok, const float* q_norm,
                                  const float* k_norm, float eps, const float* rope_cos, const float* rope_sin, int rd,
                                  int rope_max_pos, const int32_t* cu, const int32_t* ctxl, int n_seqs, int n_tokens,
                                  const int32_t* bt, int bt_stride, int num_pages, int page_size, int q_heads,
                                  int kv_heads, int head_dim, void* q_out, long q_out_tok, long q_out_head,
                                  void* k_pool, void* v_pool, const int32_t* tok_sp) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = check_dtype(ctx, dtype)) return rc;
    if (head_dim < 1 || head_dim > 256)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "head_dim %d: 1..256 are implemented", head_dim);
    const int shift = log2_exact(page_size);
    REQUIRE(shift >= 4 && shift <= 8, "page_size %d must be a power of two in 16..256", page_size);
    REQUIRE(n_seqs > 0 && n_tokens >= 0 && q_heads >= 0 && kv_heads > 0, "bad batch/head counts");
    REQUIRE(bt_stride > 0 && num_pages > 0, "bad block table geometry");
    REQUIRE(cu && ctxl && bt && k_in && v_in && k_pool && v_pool, "null pointer argument");
    REQUIRE(q_heads == 0 || (q_in && q_out), "null q pointer");
    REQUIRE(!rope_cos || (rope_sin && rd >= 2 && rd % 2 == 0 && rd <= head_dim && rope_max_pos > 0),
            "bad rope table arguments");
    REQUIRE(k_in_tok >= (long)kv_heads * head_dim && v_in_tok >= (long)kv_heads * head_dim, "k/v token stride too small");
    hipSetDevice(ctx->device);
    hk::KvArgs a{q_in, q_in_tok, q_in_head, k_in, k_in_tok, v_in, v_in_tok, q_norm, k_norm, eps, rope_cos, rope_sin,
                 rd, rope_max_pos, cu, ctxl, n_seqs, n_tokens, bt, bt_stride, num_pages, shift, q_heads, kv_heads,
                 q_out, q_out_tok, q_out_head, k_pool, v_pool, ctx->fault_dev, tok_sp};
    // 128- and 256-wide heads on the vectorised kernels (kv_ops.hip; 16-bit, 16-byte aligned rows;
    // otherwise 256-wide heads fall back to the general one), other widths on the general one
    int rc = head_dim == 128 || head_dim == 256 ? hk_launch_qk_norm_rope_kv_write(dtype, &a, head_dim, ctx->stream)
                                                : hk_launch_kv_write_gen(dtype, &a, head_dim, ctx->stream);
    return rc ? hk_fail(ctx, rc, "qk_norm_rope_kv_write launch failed") : HK_OK;
}

extern "C" int hk_qk_norm_rope_kv_write(hk_ctx* ctx, int dtype, const void* q_in, long q_in_tok, long q_in_head,
                                        const void* k_in, long k_in_tok, const void* v_in, long v_in_tok,
                                        const float* q_norm, const float* k_norm, float eps, const float* rope_cos,
                                        const float* rope_sin, int rd, int rope_max_pos, const int32_t* cu,
                                        const int32_t* ctxl, int n_seqs, int n_tokens, const int32_t* bt,
                                        int bt_stride, int num_pages, int page_size, int q_heads, int kv_heads,
                                        int head_dim, void* q_out, long q_out_tok, long q_out_head, void* k_pool,
                                        void* v_pool) {
    return hk_qk_norm_rope_kv_write_impl(ctx, dtype, q_in, q_in_tok, q_in_head, k_in, k_in_tok, v_in, v_in_tok, q_norm,
                                         k_norm, eps, rope_cos, rope_sin, rd, rope_max_pos, cu, ctxl, n_seqs, n_tokens,
                                         bt, bt_stride, num_pages, page_size, q_heads, kv_heads, head_dim, q_out,
                                         q_out_tok, q_out_head, k_pool, v_pool, nullptr);
}

extern "C" int hk_paged_kv_write(hk_ctx* ctx, int dtype, const void* k, const void* v, const int32_t* cu,
                                 const int32_t* ctxl, int n_seqs, int n_tokens, const int32_t* bt, int bt_stride,
                                 int num_pages, int page_size, int kv_heads, int head_dim, void* k_pool, void* v_pool) {
    return hk_qk_norm_rope_kv_write_impl(ctx, dtype, nullptr, 0, 0, k, (long)kv_heads * head_dim, v,
                                         (long)kv_heads * head_dim, nullptr, nullptr, 0.f, nullptr, nullptr, 0, 0, cu,
                                         ctxl, n_seqs, n_tokens, bt, bt_stride, num_pages, page_size, 0, kv_heads,
                                         head_dim, nullptr, 0, 0, k_pool, v_pool, nullptr);
}

// Ranges of a q-block of `tiles` key tiles in a batch that leaves most of the chip idle (1: not split): ranges
// of 4 tiles or more, at most kAttnParts workgroups and the 32 ranges that attn_combine takes. Where the
// estimates (us, 128-wide heads) favour it by 5 %: a pair of q-blocks runs its tiles at 1.2 us one after
// another; a range pays 1.25 us a tile (1.75 with two workgroups per CU), and its parts are written and
// read back. Measured, bf16, 16 / 8 heads, unsplit against split, rows x new tokens / context:
//   1 x 30 / 1030 25.6 12.8, / 2700 54.6 13.1; 5 x 30 / 2700 55.0 19.1; 12 x 24 / 2524 51.2 27.2; 16 x 30 /
//   1054 25.6 (not split), / 4096 78.0 43.6; 4 x 128 / 2048 87.4 26.8; 2 x 128 / 4128 168 26.7
static int attn_splits(long blocks, int tiles, int pair_tiles, bool paired) {
    const int n = std::min(std::min((tiles + 3) / 4, (int)(kAttnParts / blocks)), 32);
    const int per = (tiles + n - 1) / n;
    const float whole = 5.0f + 1.18f * pair_tiles + (paired ? 7.0f : 0.0f);
    const float split = 11.0f + per * (blocks * n > 256 ? 1.75f : 1.25f) + 0.0145f * (float)(blocks * n);
    return n > 1 && split < 0.95f * whole ? n : 1;
}
// The least number of key tiles from which a row of the batch is split (0: none is), and the most ranges of a
// row of max_tiles tiles. Only suffixes, contexts of 16 tiles (1,024 tokens) or more and at least four times
// as long as the row: the sums of split rows round differently, and a prefix computed alone keeps the bits
// that it has in a large batch. Which rows those are the kernel decides, row by row; a row's ranges depend on
// its own lengths, the number of rows and max_q_len, not on max_tiles.
static int attn_split_from(long blocks, long pairs, int n_qblocks, int pos_per_block, int max_tiles, int* n_split) {
    if (pairs >= 256 || blocks > kAttnParts / 2) return 0;
    for (int t = 16; t <= std::min(max_tiles, 64); ++t) {  // (past 64 tiles it no longer depends on them)
        // a pair's two blocks lie (n_qblocks - 1) x pos_per_block keys apart in all
        const int pair_tiles = n_qblocks == 1 ? t : 2 * t - (n_qblocks - 1) * pos_per_block / 64;
        if (attn_splits(blocks, t, pair_tiles, n_qblocks > 1) == 1) continue;
        *n_split = std::min(std::min((max_tiles + 3) / 4, (int)(kAttnParts / blocks)), 32);
        return t;
    }
    return 0;
}
static_assert((size_t)kAttnParts * 128 * (256 + 2) * sizeof(float) <= kSplitScratch, "every key-split launch fits");

int hk_paged_prefill_attention_impl(hk_ctx* ctx, int dtype, const void* q, long q_tok, long q_head, const void* k_pool,
                                    const void* v_pool, int num_pages, int page_size, const int32_t* bt, int bt_stride,
                                    const int32_t* cu, const int32_t* ctxl, int n_seqs, int n_tokens, int max_q_len,
                                    int q_heads, int kv_heads, int head_dim, float scale, const void* gate,
                                    long gate_tok, long gate_head, void* o, long o_tok, long o_head, int max_ctx) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = check_dtype(ctx, dtype)) return rc;
    if (head_dim < 1 || head_dim > 256)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "head_dim %d: 1..256 are implemented", head_dim);
    REQUIRE(kv_heads > 0 && q_heads > 0 && q_heads % kv_heads == 0, "q_heads %d not a multiple of kv_heads %d", q_heads,
            kv_heads);
    const int group = q_heads / kv_heads;
    // 128-wide heads (and 256-wide heads in 16-bit types) in groups of 1, 2, 4 or 8 run on the
    // MFMA kernels, every other shape on the general kernel (general.hip)
    const bool mfma = (head_dim == 128 || (head_dim == 256 && dtype != HK_F32)) &&
                      (group == 1 || group == 2 || group == 4 || group == 8);
    const int shift = log2_exact(page_size);
    REQUIRE(shift >= 4 && shift <= 8, "page_size %d must be a power of two in 16..256", page_size);
    REQUIRE(n_seqs > 0 && n_seqs <= 65535 && n_tokens >= 0 && max_q_len >= 0 && bt_stride > 0 && num_pages > 0,
            "bad batch geometry");
    REQUIRE(q && k_pool && v_pool && bt && cu && ctxl && o, "null pointer argument");
    REQUIRE(q_head >= head_dim && q_tok >= (long)q_heads * q_head - (q_head - head_dim), "q strides overlap heads");
    REQUIRE(o_head >= head_dim && o_tok >= (long)q_heads * o_head - (o_head - head_dim), "o strides overlap heads");
    REQUIRE(!gate || gate_head >= head_dim, "gate stride too small");
    REQUIRE(scale > 0 && isfinite(scale), "scale must be positive and finite");
    if (!mfma) {
        if (max_q_len == 0 || n_tokens == 0) return HK_OK;
        hipSetDevice(ctx->device);
        hk::AttnArgs a{q, q_tok, q_head, k_pool, v_pool, shift, bt, bt_stride, cu, ctxl, q_heads, kv_heads, group,
                       0, scale * 1.4426950408889634f, gate, gate_tok, gate_head, o, o_tok, o_head, num_pages,
                       n_tokens, ctx->fault_dev};
        int rc = hk_launch_attention_gen(dtype, &a, head_dim, n_seqs, ctx->stream);
        return rc ? hk_fail(ctx, rc, "attention launch failed") : HK_OK;
    }
    {  // vector widths of the kernels' loads and stores (elements): q rows, o / gate rows
        // 16-bit: 16-byte q loads, gate loads and O stores (8 elements); fp32: 8-byte q loads
        // and 16-byte O stores (4 elements; the gate is read per element)
        const long qv = dtype == HK_F32 ? 2 : 8, ov = dtype == HK_F32 ? 4 : 8, esz = dtype == HK_F32 ? 4 : 2;
        const uintptr_t qa = (uintptr_t)q, oa = (uintptr_t)o, ga = (uintptr_t)gate;
        REQUIRE(q_tok % qv == 0 && q_head % qv == 0 && qa % (qv * esz) == 0, "q rows must be %ld-element aligned", qv);
        REQUIRE(o_tok % ov == 0 && o_head % ov == 0 && oa % (ov * esz) == 0, "o rows must be %ld-element aligned", ov);
        REQUIRE(!gate || (gate_tok % ov == 0 && gate_head % ov == 0 && ga % (ov * esz) == 0),
                "gate rows must be %ld-element aligned", ov);
        REQUIRE((((uintptr_t)k_pool | (uintptr_t)v_pool) & 15) == 0, "K/V pools must be 16-byte aligned");
    }
    if (max_q_len == 0 || n_tokens == 0) return HK_OK;
    const int pos_per_block = 128 / group;
    const int n_qblocks = (max_q_len + pos_per_block - 1) / pos_per_block;
    REQUIRE(n_qblocks <= 65535, "max_q_len too large");
    hipSetDevice(ctx->device);
    hk::AttnArgs a{q, q_tok, q_head, k_pool, v_pool, shift, bt, bt_stride, cu, ctxl, q_heads, kv_heads, group,
                   pos_per_block, scale * 1.4426950408889634f, gate, gate_tok, gate_head, o, o_tok, o_head,
                   num_pages, n_tokens, ctx->fault_dev};
    if (dtype != HK_F32) {
        const long most = (long)bt_stride << shift, keys = max_ctx > 0 && max_ctx < most ? max_ctx : most;
        const int tiles = (int)((keys + 63) / 64 < (1 << 20) ? (keys + 63) / 64 : 1 << 20);
        const long rows = (long)kv_heads * n_seqs;
        int n = 1;
        const int from = keys / 4 < max_q_len ? 0
                                              : attn_split_from(rows * n_qblocks, rows * ((n_qblocks + 1) / 2), n_qblocks,
                                                                pos_per_block, tiles, &n);
        const size_t bytes = (size_t)(rows * n_qblocks * n) * 128 * (head_dim + 2) * sizeof(float);
        if (from) {
            if (void* scratch = split_scratch_for(ctx, bytes)) {
                a.n_split = n;
                a.split_from = from;
                a.n_qblocks = n_qblocks;
                a.part = (float*)scratch;
                a.part_ml = a.part + (size_t)(rows * n_qblocks * n) * 128 * head_dim;
                const int rc = hk_launch_paged_prefill_attention_split(dtype, &a, head_dim, n_seqs, ctx->stream);
                split_scratch_done(ctx);
                return rc ? hk_fail(ctx, rc, "attention launch failed") : HK_OK;
            }
        }
    }
    int rc = hk_launch_paged_prefill_attention(dtype, &a, head_dim, n_seqs, n_qblocks, ctx->stream);
    return rc ? hk_fail(ctx, rc, "attention launch failed") : HK_OK;
}

extern "C" int hk_paged_prefill_attention(hk_ctx* ctx, int dtype, const void* q, long q_tok, long q_head,
                                          const void* k_pool, const void* v_pool, int num_pages, int page_size,
                                          const int32_t* bt, int bt_stride, const int32_t* cu, const int32_t* ctxl,
                                          int n_seqs, int n_tokens, int max_q_len, int q_heads, int kv_heads,
                                          int head_dim, float scale, const void* gate, long gate_tok, long gate_head,
                                          void* o, long o_tok, long o_head) {
    return hk_paged_prefill_attention_impl(ctx, dtype, q, q_tok, q_head, k_pool, v_pool, num_pages, page_size, bt,
                                           bt_stride, cu, ctxl, n_seqs, n_tokens, max_q_len, q_heads, kv_heads, head_dim,
                                           scale, gate, gate_tok, gate_head, o, o_tok, o_head, 0);
}

// Whether the fp32 delta rule takes its three-kernel form (delta_rule_split.hip): few chains (pairs of a
// row and a head) of a chunk or more on average. Measured, 16 heads, us, one kernel against three, by rows
// x tokens: 1 x 64 37.6 26.6, x 512 256 54.3, x 2048 1055 153;  4 x 64 38.0 32.1, x 512 269 111;  8 x 64
// 39.9 47.7 (not split), x 128 73.4 64.3, x 1024 571 443
static bool delta_split_takes(int n_seqs, int n_tokens, int heads) {
    const long chains = (long)n_seqs * heads, chunks = n_tokens / 64;
    return chains <= 64 ? chunks >= n_seqs : chains <= 128 && chunks >= 2L * n_seqs;
}
size_t hk_delta_split_bytes(int n_tokens, int n_seqs, int heads) {
    return (size_t)(n_tokens / 64 + n_seqs) * heads * hk::HK_DELTA_SPLIT_SLOT;
}

int hk_gated_delta_chunked_rows(hk_ctx* ctx, int dtype, const void* q, long q_tok, const void* k, long k_tok,
                                const void* v, long v_tok, const float* g, const float* beta, const int32_t* cu,
                                int n_seqs, int n_tokens, int heads, int k_heads, int dk, int dv,
                                const float* initial_state, float* final_state, void* o, long o_tok,
                                const float* const* init_rows, float* const* final_rows) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = check_dtype(ctx, dtype)) return rc;
    // 128 x 128 states on the chunked MFMA kernels, others (each width in 1..256, at most 32768
    // state elements) on the general per-token recurrence (general.hip)
    const bool mfma = dk == 128 && dv == 128;
    if (dk < 1 || dv < 1 || dk > 256 || dv > 256 || dk * dv > 32768)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "dk=%d dv=%d: widths 1..256 with dk*dv <= 32768 are implemented", dk,
                       dv);
    REQUIRE(heads > 0 && k_heads > 0 && heads % k_heads == 0, "heads %d not a multiple of k_heads %d", heads, k_heads);
    REQUIRE(n_seqs > 0 && n_seqs <= 65535 && n_tokens >= 0, "bad batch geometry");
    REQUIRE(q && k && v && g && beta && cu && o, "null pointer argument");
    REQUIRE(q_tok >= (long)k_heads * dk && k_tok >= (long)k_heads * dk && v_tok >= (long)heads * dv &&
                o_tok >= (long)heads * dv,
            "token strides too small");
    if (mfma && dtype != HK_F32) {  // the 16-bit kernel moves rows in 16-byte vectors
        REQUIRE(q_tok % 8 == 0 && k_tok % 8 == 0 && v_tok % 8 == 0 && o_tok % 8 == 0 &&
                    (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) & 15) == 0,
                "16-bit q/k/v/o rows must be 16-byte aligned (token strides a multiple of 8)");
    }
    hipSetDevice(ctx->device);
    hk::GdnArgs a{q, k, v, q_tok, k_tok, v_tok, heads / k_heads, g, beta, (long)heads, cu, initial_state,
                  final_state, o, o_tok, heads, n_tokens, ctx->fault_dev, init_rows, final_rows};
    // (the split form reads q and k after it has written part of o: o in their place stays with one kernel)
    if (mfma && dtype == HK_F32 && delta_split_takes(n_seqs, n_tokens, heads) && o != q && o != k) {
        if (void* scratch = split_scratch_for(ctx, hk_delta_split_bytes(n_tokens, n_seqs, heads))) {
            const int rc = hk_launch_delta_split(&a, n_seqs, n_tokens / 64 + n_seqs, scratch, ctx->stream);
            split_scratch_done(ctx);
            return rc ? hk_fail(ctx, rc, "gated delta launch failed") : HK_OK;
        }
    }
    int rc = mfma ? hk_launch_gated_delta_chunked(dtype, &a, n_seqs, ctx->stream)
                  : hk_launch_delta_gen(dtype, &a, dk, dv, n_seqs, ctx->stream);
    return rc ? hk_fail(ctx, rc, "gated delta launch failed") : HK_OK;
}

extern "C" int hk_gated_delta_chunked(hk_ctx* ctx, int dtype, const void* q, long q_tok, const void* k, long k_tok,
                                      const void* v, long v_tok, const float* g, const float* beta, const int32_t* cu,
                                      int n_seqs, int n_tokens, int heads, int k_heads, int dk, int dv,
                                      const float* initial_state, float* final_state, void* o, long o_tok) {
    return hk_gated_delta_chunked_rows(ctx, dtype, q, q_tok, k, k_tok, v, v_tok, g, beta, cu, n_seqs, n_tokens, heads,
                                       k_heads, dk, dv, initial_state, final_state, o, o_tok, nullptr, nullptr);
}

int hk_gdn_prep_rows(hk_ctx* ctx, int dtype, const void* mixed, long mixed_tok, const float* conv_w, int conv_k,
                     const void* conv_hist, const void* ba, long ba_tok, int b_col, int a_col, const float* base_g,
                     const float* dt_bias, const int32_t* cu, int n_seqs, int n_tokens, int heads, int k_heads,
                     int dk, int dv, void* q_out, void* k_out, void* v_out, float* g_out, float* beta_out,
                     void* conv_tail_out, const void* const* hist_rows, void* const* tail_rows) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = check_dtype(ctx, dtype)) return rc;
    REQUIRE(heads > 0 && k_heads > 0 && heads % k_heads == 0, "heads %d not a multiple of k_heads %d", heads, k_heads);
    if (dk < 1 || dv < 1 || dk > 256 || dv > 256)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "dk=%d dv=%d: widths 1..256 are implemented", dk, dv);
    REQUIRE(conv_k >= 1 && conv_k <= 16, "conv kernel %d outside 1..16", conv_k);
    REQUIRE(n_seqs > 0 && n_tokens >= 0, "bad batch geometry");
    REQUIRE(mixed && conv_w && ba && base_g && dt_bias && cu && q_out && k_out && v_out && g_out && beta_out,
            "null pointer argument");
    const long conv_dim = 2L * k_heads * dk + (long)heads * dv;
    REQUIRE(mixed_tok >= conv_dim, "mixed token stride %ld < conv_dim %ld", mixed_tok, conv_dim);
    REQUIRE(b_col >= 0 && a_col >= 0 && b_col + heads <= ba_tok && a_col + heads <= ba_tok, "b/a columns outside a row");
    hipSetDevice(ctx->device);
    hk::PrepArgs a{mixed, mixed_tok, conv_w, conv_k, conv_hist, ba, ba_tok, b_col, a_col, base_g, dt_bias, cu, n_seqs,
                   n_tokens, k_heads, heads, (float)(1.0 / sqrt((double)dk)), q_out, k_out, v_out, g_out, beta_out,
                   ctx->fault_dev, hist_rows, tail_rows, dk, dv};
    int rc = hk_launch_gdn_prep(dtype, &a, conv_tail_out, ctx->stream);
    return rc ? hk_fail(ctx, rc, "gdn_prep launch failed") : HK_OK;
}

extern "C" int hk_gdn_prep(hk_ctx* ctx, int dtype, const void* mixed, long mixed_tok, const float* conv_w, int conv_k,
                           const void* conv_hist, const void* ba, long ba_tok, int b_col, int a_col, const float* base_g,
                           const float* dt_bias, const int32_t* cu, int n_seqs, int n_tokens, int heads, int k_heads,
                           void* q_out, void* k_out, void* v_out, float* g_out, float* beta_out, void* conv_tail_out) {
    return hk_gdn_prep_rows(ctx, dtype, mixed, mixed_tok, conv_w, conv_k, conv_hist, ba, ba_tok, b_col, a_col, base_g,
                            dt_bias, cu, n_seqs, n_tokens, heads, k_heads, 128, 128, q_out, k_out, v_out, g_out,
                            beta_out, conv_tail_out, nullptr, nullptr);
}

extern "C" int hk_rms_norm(hk_ctx* ctx, int dtype, const void* x, long x_tok, const float* w, float eps, int rows,
                           int width, void* y, long y_tok) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = check_dtype(ctx, dtype)) return rc;
    REQUIRE(x && w && y && rows >= 0 && width > 0 && x_tok >= width && y_tok >= width, "bad rms_norm arguments");
    hipSetDevice(ctx->device);
    hk::NormArgs a{x, x_tok, w, eps, rows, width, y, y_tok};
    int rc = hk_launch_rms_norm(dtype, &a, ctx->stream);
    return rc ? hk_fail(ctx, rc, "rms_norm launch failed") : HK_OK;
}

extern "C" int hk_gated_rms_norm(hk_ctx* ctx, int dtype, const void* x, const void* z, long z_tok, int heads,
                                 const float* w, float eps, int rows, int width, void* y) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = check_dtype(ctx, dtype)) return rc;
    REQUIRE(x && z && w && y && rows >= 0 && width > 0 && heads > 0 && rows % heads == 0 && z_tok >= (long)heads * width,
            "bad gated_rms_norm arguments");
    hipSetDevice(ctx->device);
    hk::GatedNormArgs a{x, z, z_tok, heads, w, eps, rows, width, y};
    int rc = hk_launch_gated_rms_norm(dtype, &a, ctx->stream);
    return rc ? hk_fail(ctx, rc, "gated_rms_norm launch failed") : HK_OK;
}

extern "C" int hk_swiglu(hk_ctx* ctx, int dtype, const void* gu, long gu_tok, long up_off, int rows, int width, void* y) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = check_dtype(ctx, dtype)) return rc;
    REQUIRE(gu && y && rows >= 0 && width > 0 && up_off >= width && gu_tok >= up_off + width, "bad swiglu arguments");
    hipSetDevice(ctx->device);
    hk::SwigluArgs a{gu, gu_tok, up_off, rows, width, y};
    int rc = hk_launch_swiglu(dtype, &a, ctx->stream);
    return rc ? hk_fail(ctx, rc, "swiglu launch failed") : HK_OK;
}

// Whether the batch takes the three-kernel form of the fused layer (gdn16_split.hip): few chains (pairs of
// a row and a head), whose rows are several chunks long on average. Measured, 16 heads, bf16, us, one
// kernel against three, by rows x tokens:
//   1 x 128 26.7 21.8, x 512 95.8 28.5, x 2048 386 66.6, x 4096 767 117;  4 x 128 26.7 23.6, x 512 99.3
//   45.3, x 2048 384 165;  6 x 128 26.8 29.4, x 256 50.3 42.8;  8 x 128 26.7 32.1, x 256 52.0 46.9, x 1024 197 161
static bool gdn_split_takes(int n_seqs, int n_tokens, int heads) {
    const long chains = (long)n_seqs * heads, chunks = n_tokens / 64;
    return chains <= 64 ? chunks >= 2L * n_seqs : chains <= 128 && chunks >= 4L * n_seqs;
}

// The fused layer with optional per-sequence row tables for the state and the conv history
// (device arrays of n_seqs pointers; used by the cached model forward).
int hk_gdn_fused_rows(hk_ctx* ctx, int dtype, const void* mixed, long mixed_tok, const float* conv_w, int conv_k,
                      const void* conv_hist, void* conv_tail_out, const void* ba, long ba_tok, int b_col, int a_col,
                      const float* base_g, const float* dt_bias, const void* z, long z_tok, const float* norm_w,
                      float eps, const int32_t* cu, int n_seqs, int n_tokens, int heads, int k_heads,
                      const float* initial_state, float* final_state, void* out, long out_tok,
                      const float* const* init_rows, float* const* final_rows, const void* const* hist_rows,
                      void* const* tail_rows) {
    if (!ctx) return HK_ERR_INVALID;
    if (dtype != HK_BF16 && dtype != HK_F16)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "fused Gated DeltaNet layer: 16-bit dtypes only (got %d)", dtype);
    if (conv_k != 4) return hk_fail(ctx, HK_ERR_UNSUPPORTED, "fused Gated DeltaNet layer: conv kernel 4 only");
    REQUIRE(heads > 0 && k_heads > 0 && heads % k_heads == 0, "heads %d not a multiple of k_heads %d", heads, k_heads);
    REQUIRE(n_seqs > 0 && n_seqs <= 65535 && n_tokens >= 0, "bad batch geometry");
    REQUIRE(mixed && conv_w && ba && base_g && dt_bias && z && norm_w && cu && out, "null pointer argument");
    {  // the kernel addresses a sequence's rows with 32-bit byte offsets (24-bit row strides)
        const long esz = dtype == HK_F32 ? 4 : 2, lim = 1L << 32;
        REQUIRE(n_tokens < (1 << 24) && mixed_tok * esz < (1 << 24) && z_tok * esz < (1 << 24) &&
                    out_tok * esz < (1 << 24) && n_tokens * mixed_tok * esz < lim && n_tokens * z_tok * esz < lim &&
                    n_tokens * out_tok * esz < lim,
                "fused Gated DeltaNet layer: token rows or the batch too large for 32-bit row offsets");
    }
    REQUIRE(((uintptr_t)conv_w & 15) == 0, "conv weights must be 16-byte aligned");
    const long conv_dim = (2L * k_heads + heads) * 128;
    REQUIRE(mixed_tok >= conv_dim && mixed_tok % 8 == 0 && ((uintptr_t)mixed & 15) == 0,
            "mixed rows must hold conv_dim channels with 16-byte aligned rows");
    REQUIRE(z_tok >= (long)heads * 128 && z_tok % 8 == 0 && ((uintptr_t)z & 15) == 0, "bad z rows");
    REQUIRE(out_tok >= (long)heads * 128 && out_tok % 8 == 0 && ((uintptr_t)out & 15) == 0, "bad output rows");
    REQUIRE(b_col >= 0 && a_col >= 0 && b_col + heads <= ba_tok && a_col + heads <= ba_tok, "b/a columns outside a row");
    hipSetDevice(ctx->device);
    hk::GdnArgs a{nullptr, nullptr, nullptr, 0, 0, 0, heads / k_heads, nullptr, nullptr, 0, cu, initial_state,
                  final_state, out, out_tok, heads, n_tokens, ctx->fault_dev, init_rows, final_rows};
    hk::GdnFusedArgs fa{mixed, mixed_tok, conv_w, (int)conv_dim, conv_hist, conv_tail_out, ba, ba_tok, b_col, a_col,
                        base_g, dt_bias, 1.0f / sqrtf(128.0f), k_heads, z, z_tok, norm_w, eps, hist_rows, tail_rows};
    if (gdn_split_takes(n_seqs, n_tokens, heads)) {
        if (void* scratch = split_scratch_for(ctx, hk_gdn_split_bytes(n_tokens, n_seqs, heads))) {
            const int rc = hk_launch_gdn16_split(dtype, &a, &fa, n_seqs, n_tokens / 64 + n_seqs, scratch, ctx->stream);
            split_scratch_done(ctx);
            return rc ? hk_fail(ctx, rc, "fused Gated DeltaNet launch failed") : HK_OK;
        }
    }
    int rc = hk_launch_gdn16(dtype, 1, &a, &fa, n_seqs, ctx->stream);
    return rc ? hk_fail(ctx, rc, "fused Gated DeltaNet launch failed") : HK_OK;
}

extern "C" int hk_gdn_fused(hk_ctx* ctx, int dtype, const void* mixed, long mixed_tok, const float* conv_w, int conv_k,
                            const void* conv_hist, void* conv_tail_out, const void* ba, long ba_tok, int b_col,
                            int a_col, const float* base_g, const float* dt_bias, const void* z, long z_tok,
                            const float* norm_w, float eps, const int32_t* cu, int n_seqs, int n_tokens, int heads,
                            int k_heads, const float* initial_state, float* final_state, void* out, long out_tok) {
    return hk_gdn_fused_rows(ctx, dtype, mixed, mixed_tok, conv_w, conv_k, conv_hist, conv_tail_out, ba, ba_tok, b_col,
                             a_col, base_g, dt_bias, z, z_tok, norm_w, eps, cu, n_seqs, n_tokens, heads, k_heads,
                             initial_state, final_state, out, out_tok, nullptr, nullptr, nullptr, nullptr);
}

// ---------------------------------------------------------------------------
// ModernBERT ops
// ---------------------------------------------------------------------------

extern "C" int hk_layer_norm(hk_ctx* ctx, int dtype, const void* x, long x_tok, const float* w, float eps, int rows,
                             int width, void* y, long y_tok) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = check_dtype(ctx, dtype)) return rc;
    REQUIRE(x && w && y, "null pointer argument");
    REQUIRE(rows >= 0 && width > 0 && width <= 2048, "width %d outside 1..2048", width);
    REQUIRE(x_tok >= width && y_tok >= width, "row strides too small");
    REQUIRE(eps > 0.0f, "eps must be positive");
    if (rows == 0) return HK_OK;
    hipSetDevice(ctx->device);
    hk::LayerNormArgs a{x, x_tok, w, eps, rows, width, y, y_tok};
    int rc = hk_launch_layer_norm(dtype, &a, ctx->stream);
    return rc ? hk_fail(ctx, rc, "layer_norm launch failed") : HK_OK;
}

extern "C" int hk_bidir_attention(hk_ctx* ctx, int dtype, const void* q, long q_tok, const void* k, long k_tok,
                                  const void* v, long v_tok, const int32_t* cu, int n_seqs, int n_tokens, int max_len,
                                  int heads, int head_dim, int half_window, float scale, void* o, long o_tok) {
    if (!ctx) return HK_ERR_INVALID;
    if (int rc = check_dtype(ctx, dtype)) return rc;
    // 64-wide heads on the MFMA / fp32 tile kernels (bert.hip), other widths up to 256 on the
    // general kernel (general.hip)
    if (head_dim < 1 || head_dim > 256)
        return hk_fail(ctx, HK_ERR_UNSUPPORTED, "head_dim %d: 1..256 are implemented", head_dim);
    REQUIRE(q && k && v && cu && o, "null pointer argument");
    REQUIRE(heads > 0 && n_seqs > 0 && n_seqs <= 65535 && n_tokens >= 0 && max_len >= 0, "bad batch geometry");
    const long hw = (long)heads * head_dim;
    REQUIRE(q_tok >= hw && k_tok >= hw && v_tok >= hw && o_tok >= hw, "token strides too small");
    REQUIRE(scale > 0 && isfinite(scale), "scale must be positive and finite");
    if (head_dim != 64) {
        if (max_len == 0 || n_tokens == 0) return HK_OK;
        hipSetDevice(ctx->device);
        hk::BertAttnArgs a{q, q_tok, k, k_tok, v, v_tok, o, o_tok, cu, n_seqs, n_tokens, heads, half_window,
                           scale * 1.4426950408889634f, ctx->fault_dev};
        int rc = hk_launch_bidir_gen(dtype, &a, head_dim, ctx->stream);
        return rc ? hk_fail(ctx, rc, "bidirectional attention launch failed") : HK_OK;
    }
    if (dtype != HK_F32) {  // 16-byte row loads, 8-byte output stores
        REQUIRE(q_tok % 8 == 0 && k_tok % 8 == 0 && v_tok % 8 == 0 && o_tok % 4 == 0 &&
                    (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15) == 0 && ((uintptr_t)o & 7) == 0,
                "16-bit q/k/v rows must be 16-byte aligned and o rows 8-byte aligned");
    }
    if (max_len == 0 || n_tokens == 0) return HK_OK;
    hipSetDevice(ctx->device);
    hk::BertAttnArgs a{q, q_tok, k, k_tok, v, v_tok, o, o_tok, cu, n_seqs, n_tokens, heads, half_window,
                       scale * 1.4426950408889634f, ctx->fault_dev};
    int rc = hk_launch_bidir_attention(dtype, &a, n_seqs, max_len, ctx->stream);
    return rc ? hk_fail(ctx, rc, "bidirectional attention launch failed") : HK_OK;
}

int hk_write_identity(std::vector<std::pair<std::string, std::string>> kv, char* buf, size_t len, size_t* needed) {
    std::sort(kv.begin(), kv.end());
    std::string out;
    for (auto& e : kv) out += e.first + "=" + e.second + "\n";
    if (needed) *needed = out.size() + 1;
    if (buf && len) {
        const size_t n = out.size() < len - 1 ? out.size() : len - 1;
        memcpy(buf, out.data(), n);
        buf[n] = 0;
    }
    return HK_OK;
}
