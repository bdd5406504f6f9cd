// kev_cache.cpp - device prefix cache for the Kev model: cached sequences ("handles") that
// continue with new tokens, fork into private branches and are released.
//
// Semantics follow the reference backend (crates/huncho-core/src/backend.rs:333-437,
// crates/huncho-backend/src/qwen3_5.rs:2655-2757, 2818-2847) and its paged KV cache
// (qwen3_5/kv_pages.rs:18-98, 307-341):
//   * a handle holds the K/V of its tokens in fixed-size pages of a shared pool, the Gated
//     DeltaNet recurrent state of every linear layer and the conv tail (last K-1 raw conv
//     inputs) of every linear layer;
//   * fork shares the parent's pages (reference counted) and copies its recurrent state and
//     conv tails; a page that is full is immutable, so only a shared, partially filled tail
//     page is copied before a branch appends to it (copy on write);
//   * a continuation commits only after the whole forward succeeded: new pages are taken
//     from the free list, the state is written to the handle's second state buffer, and the
//     token count, page list and active state buffer change only when the call returns OK;
//   * at most max_handles live handles (the reference allows 64, qwen3_5.rs:3257-3265);
//   * storage is allocated once, when the cache is created: the page pools, and one slab of
//     state slots (each slot two fp32 recurrent-state buffers and two conv-tail buffers) for
//     max_handles handles plus the retained snapshots. Open, fork and release hand slots and
//     pages out and take them back on the host; they allocate, free and synchronise nothing.
//     A released slot or page is reused by later work on the same stream, so stream order
//     keeps the earlier readers ahead of the new writers (a caller that moves the context to
//     another stream synchronises the old one first);
//   * exact-prefix retention under a charged-byte budget (prefill_cached, qwen3_5.rs:2850-2865,
//     2975-3031; PrefixSnapshots 1215-1234, FIFO eviction, at most 16 snapshots): a retained
//     prefix is an immutable snapshot (a private clone: shared pages, its own state) that a
//     later identical prefix clones instead of recomputing;
//   * resumable chunked prefill (begin / advance_resumable_prefill, qwen3_5.rs:2867-2934): a
//     pending handle advances one chunk per call, cannot be forked or continued until it is
//     complete, and is retained when it completes.
#include <string.h>

#include <algorithm>

#include <deque>
#include <map>
#include <unordered_map>
#include <vector>

#include "kev_internal.hpp"

namespace {

struct KevHandle {
    int tokens = 0;
    std::vector<int> pages;  // pool pages in sequence order
    int slot = -1;           // state slot: buffers 2 slot and 2 slot + 1 of the slabs
    int cur = 0;             // buffer of the slot holding the committed state
};

constexpr int kMaxSnapshots = 16;  // PrefixSnapshots::trim's count limit (qwen3_5.rs:1222-1233)

}  // namespace

namespace {

struct Pending {  // a resumable prefill in progress: its whole prefix and retention budget
    std::vector<int32_t> tokens;
    size_t max_bytes = 0;
};

struct Snapshot {  // a retained prefix
    KevHandle h;
    size_t bytes = 0;  // charged bytes
};

}  // namespace

struct hk_kev_cache {
    hk_kev_model* m = nullptr;
    int max_pages = 0, max_handles = 0, P = 0, n_attn = 0, n_gdn = 0, bt_stride = 0;
    size_t page_bytes = 0;                 // one page of one pool
    size_t state_layer = 0, conv_layer = 0;  // per layer (bytes) inside a state / conv buffer
    std::vector<void*> k_pools, v_pools;   // per attention layer [max_pages][Hkv][P][hd]
    // state slots: 2 buffers each of [n_gdn][H][dk][dv] fp32 and of [n_gdn][conv_dim][3]
    // (model dtype), allocated at creation for max_handles handles and the snapshots
    char* state_slab = nullptr;
    char* conv_slab = nullptr;
    std::vector<int> free_slots;
    std::vector<int> refs;                 // per page
    std::vector<int> free_list;
    std::unordered_map<uint64_t, KevHandle> handles;
    uint64_t next_id = 1;
    std::map<std::vector<int32_t>, Snapshot> prefixes;  // retained exact prefixes
    std::deque<std::vector<int32_t>> fifo;             // their insertion order
    size_t prefix_bytes = 0;
    std::unordered_map<uint64_t, Pending> pending;     // resumable prefills in progress
};

// Buffer j (0, 1) of h's slot: the recurrent state of every Gated DeltaNet layer, and the conv
// tails.
static float* state_buf(const hk_kev_cache* c, const KevHandle& h, int j) {
    return (float*)(c->state_slab + ((size_t)h.slot * 2 + j) * c->state_layer * c->n_gdn);
}
static void* conv_buf(const hk_kev_cache* c, const KevHandle& h, int j) {
    return c->conv_slab + ((size_t)h.slot * 2 + j) * c->conv_layer * c->n_gdn;
}

// Returns h's state slot to the free list (host bookkeeping only).
static void free_handle_buffers(hk_kev_cache* c, KevHandle& h) {
    if (h.slot >= 0) c->free_slots.push_back(h.slot);
    h.slot = -1;
}

// Takes a free state slot for h (host bookkeeping only; the slab is allocated at creation).
static int alloc_handle_buffers(hk_kev_cache* c, KevHandle& h) {
    if (c->free_slots.empty())
        return hk_fail(c->m->ctx, HK_ERR_NOMEM, "cache state slots exhausted (%d handles + %d snapshots)",
                       c->max_handles, kMaxSnapshots);
    h.slot = c->free_slots.back();
    c->free_slots.pop_back();
    h.cur = 0;
    return HK_OK;
}

static void free_storage(hk_kev_cache* c) {
    for (void* p : c->k_pools) hipFree(p);
    for (void* p : c->v_pools) hipFree(p);
    if (c->state_slab) hipFree(c->state_slab);
    if (c->conv_slab) hipFree(c->conv_slab);
}

extern "C" int hk_kev_cache_create(hk_kev_model* m, int max_pages, int max_handles, hk_kev_cache** out) {
    if (!m || !out) return HK_ERR_INVALID;
    hk_ctx* ctx = m->ctx;
    const hk_kev_config& cfg = m->cfg;
    if (cfg.conv_k != 4) return hk_fail(ctx, HK_ERR_UNSUPPORTED, "the prefix cache needs conv kernel 4");
    if (max_pages <= 0 || max_handles <= 0 || max_handles > 4096)
        return hk_fail(ctx, HK_ERR_INVALID, "max_pages %d / max_handles %d out of range", max_pages, max_handles);
    hk_kev_cache* c = new hk_kev_cache();
    c->m = m;
    c->max_pages = max_pages;
    c->max_handles = max_handles;
    c->P = cfg.page_size;
    c->bt_stride = (cfg.max_context + c->P - 1) / c->P;
    for (int l = 0; l < cfg.n_layers; ++l) (m->layers[l].type == 0 ? c->n_gdn : c->n_attn)++;
    c->page_bytes = (size_t)cfg.n_kv_heads * c->P * cfg.head_dim * m->esz;
    c->state_layer = (size_t)cfg.lin_n_v_heads * cfg.lin_key_dim * cfg.lin_v_dim * sizeof(float);
    c->conv_layer = (size_t)m->conv_dim * 3 * m->esz;
    hipSetDevice(ctx->device);
    for (int i = 0; i < c->n_attn; ++i) {
        void *k = nullptr, *v = nullptr;
        if (hipMalloc(&k, c->page_bytes * max_pages) != hipSuccess ||
            hipMalloc(&v, c->page_bytes * max_pages) != hipSuccess) {
            if (k) hipFree(k);
            free_storage(c);
            delete c;
            return hk_fail(ctx, HK_ERR_NOMEM, "page pool allocation failed");
        }
        c->k_pools.push_back(k);
        c->v_pools.push_back(v);
    }
    // one slot per live handle and per snapshot, plus one: a snapshot is cloned before the
    // oldest is evicted
    const int slots = max_handles + kMaxSnapshots + 1;
    const size_t state_bytes = (size_t)slots * 2 * c->state_layer * c->n_gdn;
    const size_t conv_bytes = (size_t)slots * 2 * c->conv_layer * c->n_gdn;
    if ((state_bytes && hipMalloc((void**)&c->state_slab, state_bytes) != hipSuccess) ||
        (conv_bytes && hipMalloc((void**)&c->conv_slab, conv_bytes) != hipSuccess)) {
        free_storage(c);
        delete c;
        return hk_fail(ctx, HK_ERR_NOMEM, "state slab allocation failed (%d slots, %zu bytes)", slots,
                       state_bytes + conv_bytes);
    }
    for (int i = slots - 1; i >= 0; --i) c->free_slots.push_back(i);
    c->refs.assign(max_pages, 0);
    for (int p = max_pages - 1; p >= 0; --p) c->free_list.push_back(p);
    *out = c;
    return HK_OK;
}

extern "C" int hk_kev_cache_destroy(hk_kev_cache* c) {
    if (!c) return HK_ERR_INVALID;
    hipSetDevice(c->m->ctx->device);
    hipStreamSynchronize(c->m->ctx->stream);
    free_storage(c);
    delete c;
    return HK_OK;
}

extern "C" int hk_kev_cache_open(hk_kev_cache* c, uint64_t* handle_out) {
    if (!c || !handle_out) return HK_ERR_INVALID;
    hk_ctx* ctx = c->m->ctx;
    if ((int)c->handles.size() >= c->max_handles)
        return hk_fail(ctx, HK_ERR_NOMEM, "cache holds its maximum of %d live handles", c->max_handles);
    KevHandle h;
    if (int rc = alloc_handle_buffers(c, h)) return rc;
    const uint64_t id = c->next_id++;
    c->handles.emplace(id, std::move(h));
    *handle_out = id;
    return HK_OK;
}

// A private clone of p into h (a free slot): p's pages (reference counted), a copy of its
// committed recurrent state and conv tails, queued on the context's stream.
static int clone_handle(hk_kev_cache* c, const KevHandle& p, KevHandle& h) {
    hk_ctx* ctx = c->m->ctx;
    hipSetDevice(ctx->device);
    if (int rc = alloc_handle_buffers(c, h)) return rc;
    h.tokens = p.tokens;
    h.pages = p.pages;
    if (p.tokens > 0 && c->n_gdn > 0) {
        if (hipMemcpyAsync(state_buf(c, h, 0), state_buf(c, p, p.cur), c->state_layer * c->n_gdn,
                           hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess ||
            hipMemcpyAsync(conv_buf(c, h, 0), conv_buf(c, p, p.cur), c->conv_layer * c->n_gdn, hipMemcpyDeviceToDevice,
                           ctx->stream) != hipSuccess) {
            free_handle_buffers(c, h);
            return hk_fail(ctx, HK_ERR_DEVICE, "fork state copy failed");
        }
    }
    for (int pg : h.pages) ++c->refs[pg];
    return HK_OK;
}

// Drops h's pages (returned to the pool when no other holder is left) and its state slot. Host
// bookkeeping only: work already queued that reads them runs before any later work that
// reuses them, on the same stream.
static void drop_handle(hk_kev_cache* c, KevHandle& h) {
    for (int pg : h.pages)
        if (--c->refs[pg] == 0) c->free_list.push_back(pg);
    h.pages.clear();
    free_handle_buffers(c, h);
}

extern "C" int hk_kev_cache_fork(hk_kev_cache* c, uint64_t parent, uint64_t* child_out) {
    if (!c || !child_out) return HK_ERR_INVALID;
    hk_ctx* ctx = c->m->ctx;
    auto it = c->handles.find(parent);
    if (it == c->handles.end()) return hk_fail(ctx, HK_ERR_INVALID, "unknown cache handle %llu", (unsigned long long)parent);
    if (c->pending.count(parent)) return hk_fail(ctx, HK_ERR_INVALID, "a partial prefill cannot be forked");
    if ((int)c->handles.size() >= c->max_handles)
        return hk_fail(ctx, HK_ERR_NOMEM, "cache holds its maximum of %d live handles", c->max_handles);
    KevHandle h;
    if (int rc = clone_handle(c, it->second, h)) return rc;
    const uint64_t id = c->next_id++;
    c->handles.emplace(id, std::move(h));
    *child_out = id;
    return HK_OK;
}

extern "C" int hk_kev_cache_release(hk_kev_cache* c, uint64_t handle) {
    if (!c) return HK_ERR_INVALID;
    hk_ctx* ctx = c->m->ctx;
    auto it = c->handles.find(handle);
    if (it == c->handles.end()) return hk_fail(ctx, HK_ERR_INVALID, "unknown cache handle %llu", (unsigned long long)handle);
    drop_handle(c, it->second);
    c->handles.erase(it);
    c->pending.erase(handle);
    return HK_OK;
}

extern "C" int hk_kev_cache_tokens(hk_kev_cache* c, uint64_t handle, int* tokens_out) {
    if (!c || !tokens_out) return HK_ERR_INVALID;
    auto it = c->handles.find(handle);
    if (it == c->handles.end())
        return hk_fail(c->m->ctx, HK_ERR_INVALID, "unknown cache handle %llu", (unsigned long long)handle);
    *tokens_out = it->second.tokens;
    return HK_OK;
}

extern "C" int hk_kev_cache_stats(hk_kev_cache* c, int* live_handles, int* free_pages) {
    if (!c || !live_handles || !free_pages) return HK_ERR_INVALID;
    *live_handles = (int)c->handles.size();
    *free_pages = (int)c->free_list.size();
    return HK_OK;
}

// Per-call tables after the model workspace: block tables, context lengths and the Gated
// DeltaNet row tables (4 per linear layer), then the prefill slot (one row's cu_seqlens for
// the library's own prefill chunks).
static size_t table_bytes(const hk_kev_cache* c, int n_seqs) {
    const size_t bt = (size_t)n_seqs * c->bt_stride * sizeof(int32_t);
    const size_t lens = (size_t)n_seqs * sizeof(int32_t);
    const size_t rows = (size_t)c->n_gdn * 4 * n_seqs * sizeof(void*);
    return ((bt + 255) & ~(size_t)255) + ((lens + 255) & ~(size_t)255) + ((rows + 255) & ~(size_t)255) + 256;
}

extern "C" int hk_kev_cache_workspace_size(hk_kev_cache* c, int n_tokens, int n_seqs, size_t* bytes_out) {
    if (!c || !bytes_out || n_tokens < 0 || n_seqs <= 0) return HK_ERR_INVALID;
    *bytes_out = ((kev_workspace_bytes(c->m, n_tokens, n_seqs, 0) + 255) & ~(size_t)255) + table_bytes(c, n_seqs);
    return HK_OK;
}

static int forward_cached(hk_kev_cache* c, const uint64_t* handles_host, int n_seqs, const int32_t* ids,
                          const int32_t* cu_dev, const int32_t* cu_host, void* workspace, size_t workspace_bytes,
                          float* logits, void* hidden_last, const hk_kev_readout* readout, bool prefill = false);

extern "C" int hk_kev_forward_cached(hk_kev_cache* c, const uint64_t* handles_host, int n_seqs, const int32_t* ids,
                                     const int32_t* cu_dev, const int32_t* cu_host, void* workspace,
                                     size_t workspace_bytes, float* logits, void* hidden_last) {
    return forward_cached(c, handles_host, n_seqs, ids, cu_dev, cu_host, workspace, workspace_bytes, logits,
                          hidden_last, nullptr);
}

extern "C" int hk_kev_forward_cached_readout(hk_kev_cache* c, const uint64_t* handles_host, int n_seqs,
                                             const int32_t* ids, const int32_t* cu_dev, const int32_t* cu_host,
                                             void* workspace, size_t workspace_bytes, const hk_kev_readout* readout,
                                             float* logits) {
    if (!c) return HK_ERR_INVALID;
    if (!readout) return hk_fail(c->m->ctx, HK_ERR_INVALID, "readout required");
    return forward_cached(c, handles_host, n_seqs, ids, cu_dev, cu_host, workspace, workspace_bytes, logits, nullptr,
                          readout);
}

// prefill: the library's own prefill chunk of a pending (or new) handle; no outputs are read
static int forward_cached(hk_kev_cache* c, const uint64_t* handles_host, int n_seqs, const int32_t* ids,
                          const int32_t* cu_dev, const int32_t* cu_host, void* workspace, size_t workspace_bytes,
                          float* logits, void* hidden_last, const hk_kev_readout* readout, bool prefill) {
    if (!c) return HK_ERR_INVALID;
    hk_kev_model* m = c->m;
    hk_ctx* ctx = m->ctx;
    const hk_kev_config& cfg = m->cfg;
    if (!handles_host || !ids || !cu_dev || !cu_host || !workspace || n_seqs <= 0 || n_seqs > 64)
        return hk_fail(ctx, HK_ERR_INVALID, "invalid cached forward arguments (1..64 rows)");
    if (!prefill && cfg.n_out > 0 && !logits && !readout) return hk_fail(ctx, HK_ERR_INVALID, "logits output required");
    if (cu_host[0] != 0) return hk_fail(ctx, HK_ERR_INVALID, "cu_seqlens[0] must be 0");
    // validate every row before any work (qwen3_5.rs:2656-2725)
    std::vector<KevHandle*> hs(n_seqs);
    for (int s = 0; s < n_seqs; ++s) {
        auto it = c->handles.find(handles_host[s]);
        if (it == c->handles.end())
            return hk_fail(ctx, HK_ERR_INVALID, "unknown cache handle %llu", (unsigned long long)handles_host[s]);
        for (int r = 0; r < s; ++r)
            if (handles_host[r] == handles_host[s]) return hk_fail(ctx, HK_ERR_INVALID, "row %d repeats a handle", s);
        if (!prefill && c->pending.count(handles_host[s]))
            return hk_fail(ctx, HK_ERR_INVALID, "handle %llu is a partial prefill: advance it to completion first",
                           (unsigned long long)handles_host[s]);
        hs[s] = &it->second;
        const int len = cu_host[s + 1] - cu_host[s];
        if (len <= 0) return hk_fail(ctx, HK_ERR_INVALID, "cached continuation requires nonempty tokens (row %d)", s);
        if (hs[s]->tokens + len > cfg.max_context)
            return hk_fail(ctx, HK_ERR_INVALID, "sequence length %d exceeds max_context %d", hs[s]->tokens + len,
                           cfg.max_context);
    }
    if (readout)
        if (int rc = kev_validate_readout(m, cu_host, n_seqs, readout)) return rc;
    const int n = cu_host[n_seqs];
    const size_t model_ws = (kev_workspace_bytes(m, n, n_seqs, 0) + 255) & ~(size_t)255;
    if (model_ws + table_bytes(c, n_seqs) > workspace_bytes)
        return hk_fail(ctx, HK_ERR_INVALID, "workspace too small: %zu < %zu", workspace_bytes,
                       model_ws + table_bytes(c, n_seqs));
    // page plan: a shared, partially filled tail page is replaced by a private copy; new pages
    // come from the free list; nothing changes in the cache until the forward succeeded
    std::vector<std::vector<int>> plan(n_seqs);
    std::vector<int> cow_src(n_seqs, -1), taken;
    int need = 0;
    for (int s = 0; s < n_seqs; ++s) {
        const KevHandle& h = *hs[s];
        const int total = h.tokens + (cu_host[s + 1] - cu_host[s]);
        const bool cow = h.tokens % c->P != 0 && c->refs[h.pages.back()] > 1;
        need += (total + c->P - 1) / c->P - (int)h.pages.size() + (cow ? 1 : 0);
    }
    if (need > (int)c->free_list.size())
        return hk_fail(ctx, HK_ERR_NOMEM, "page pool exhausted: %d pages needed, %zu free", need, c->free_list.size());
    hipSetDevice(ctx->device);
    for (int s = 0; s < n_seqs; ++s) {
        const KevHandle& h = *hs[s];
        const int total = h.tokens + (cu_host[s + 1] - cu_host[s]);
        plan[s] = h.pages;
        if (h.tokens % c->P != 0 && c->refs[h.pages.back()] > 1) {
            cow_src[s] = h.pages.back();
            plan[s].back() = c->free_list.back();
            c->free_list.pop_back();
            taken.push_back(plan[s].back());
        }
        while ((int)plan[s].size() < (total + c->P - 1) / c->P) {
            plan[s].push_back(c->free_list.back());
            c->free_list.pop_back();
            taken.push_back(plan[s].back());
        }
    }
    auto rollback = [&](int rc) {
        for (int pg : taken) c->free_list.push_back(pg);
        return rc;
    };
    for (int s = 0; s < n_seqs; ++s) {
        if (cow_src[s] < 0) continue;
        // the private copy replaces the handle's last page (new pages may follow it in the plan)
        const int copy = plan[s][hs[s]->pages.size() - 1];
        for (int l = 0; l < c->n_attn; ++l) {
            const size_t src = (size_t)cow_src[s] * c->page_bytes, dst = (size_t)copy * c->page_bytes;
            if (hipMemcpyAsync((char*)c->k_pools[l] + dst, (char*)c->k_pools[l] + src, c->page_bytes,
                               hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess ||
                hipMemcpyAsync((char*)c->v_pools[l] + dst, (char*)c->v_pools[l] + src, c->page_bytes,
                               hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess)
                return rollback(hk_fail(ctx, HK_ERR_DEVICE, "copy-on-write page copy failed"));
        }
    }
    // per-call tables: block tables, context lengths, row tables (state in: committed buffer,
    // or none for an empty handle; state out: the other buffer)
    std::vector<int32_t> bt((size_t)n_seqs * c->bt_stride, 0), lens(n_seqs);
    std::vector<const void*> rows((size_t)c->n_gdn * 4 * n_seqs);
    for (int s = 0; s < n_seqs; ++s) {
        const KevHandle& h = *hs[s];
        for (size_t i = 0; i < plan[s].size(); ++i) bt[(size_t)s * c->bt_stride + i] = plan[s][i];
        lens[s] = h.tokens + (cu_host[s + 1] - cu_host[s]);
        for (int g = 0; g < c->n_gdn; ++g) {
            const void** r = rows.data() + (size_t)g * 4 * n_seqs;
            r[s] = h.tokens > 0 ? (const char*)state_buf(c, h, h.cur) + g * c->state_layer : nullptr;
            r[n_seqs + s] = (const char*)state_buf(c, h, h.cur ^ 1) + g * c->state_layer;
            r[2 * n_seqs + s] = h.tokens > 0 ? (const char*)conv_buf(c, h, h.cur) + g * c->conv_layer : nullptr;
            r[3 * n_seqs + s] = (const char*)conv_buf(c, h, h.cur ^ 1) + g * c->conv_layer;
        }
    }
    char* tbase = (char*)workspace + model_ws;
    int32_t* bt_dev = (int32_t*)tbase;
    int32_t* lens_dev = (int32_t*)(tbase + ((bt.size() * 4 + 255) & ~(size_t)255));
    const void** rows_dev = (const void**)((char*)lens_dev + ((lens.size() * 4 + 255) & ~(size_t)255));
    if (hipMemcpyAsync(bt_dev, bt.data(), bt.size() * 4, hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
        hipMemcpyAsync(lens_dev, lens.data(), lens.size() * 4, hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
        hipMemcpyAsync(rows_dev, rows.data(), rows.size() * sizeof(void*), hipMemcpyHostToDevice, ctx->stream) !=
            hipSuccess)
        return rollback(hk_fail(ctx, HK_ERR_DEVICE, "cache table upload failed"));
    KevCacheView view;
    view.ctx_lens_dev = lens_dev;
    view.max_ctx = *std::max_element(lens.begin(), lens.end());
    view.k_pools = c->k_pools;
    view.v_pools = c->v_pools;
    for (int g = 0; g < c->n_gdn; ++g) {
        const void** r = rows_dev + (size_t)g * 4 * n_seqs;
        view.init_rows.push_back((const float* const*)r);
        view.final_rows.push_back((float* const*)(r + n_seqs));
        view.hist_rows.push_back((const void* const*)(r + 2 * n_seqs));
        view.tail_rows.push_back((void* const*)(r + 3 * n_seqs));
    }
    int rc = kev_forward_impl(m, ids, cu_dev, cu_host, n_seqs, bt_dev, c->bt_stride, c->max_pages, workspace, model_ws,
                              logits, hidden_last, &view, readout);
    if (rc) return rollback(rc);
    // commit only after the forward finished without device faults
    if (hipStreamSynchronize(ctx->stream) != hipSuccess)
        return rollback(hk_fail(ctx, HK_ERR_DEVICE, "cached forward failed on the device"));
    int faults = 0;
    if (hipMemcpy(&faults, ctx->fault_dev, sizeof(int), hipMemcpyDeviceToHost) != hipSuccess)
        return rollback(hk_fail(ctx, HK_ERR_DEVICE, "fault word read failed"));
    if (faults) {
        const int zero = 0;
        hipMemcpy(ctx->fault_dev, &zero, sizeof(int), hipMemcpyHostToDevice);
        return rollback(hk_fail(ctx, HK_ERR_DEVICE, "device faults 0x%x during the cached forward; nothing committed",
                                faults));
    }
    for (int s = 0; s < n_seqs; ++s) {
        KevHandle& h = *hs[s];
        // the replaced tail page loses this holder; when every holder continued in this call
        // (a parent and its fork together), each took a private copy and the page is free
        if (cow_src[s] >= 0 && --c->refs[cow_src[s]] == 0) c->free_list.push_back(cow_src[s]);
        for (size_t i = h.pages.size() - (cow_src[s] >= 0 ? 1 : 0); i < plan[s].size(); ++i) ++c->refs[plan[s][i]];
        h.pages = std::move(plan[s]);
        h.tokens = lens[s];
        h.cur ^= 1;
    }
    return HK_OK;
}

// ---------------------------------------------------------------------------
// exact-prefix retention and resumable chunked prefill
// ---------------------------------------------------------------------------

// Charged bytes of a retained prefix of `tokens` tokens, ModelCache::retention_bytes
// (qwen3_5.rs:1161-1185) on this cache's storage: 8 per token + 512, and per layer 512 plus
// the bytes it holds (attention: its K and V pages; Gated DeltaNet: the fp32 recurrent state
// and the conv tail).
static size_t retention_bytes(const hk_kev_cache* c, int tokens) {
    const size_t pages = (size_t)(tokens + c->P - 1) / c->P;
    return (size_t)tokens * 8 + 512 + (size_t)(c->n_attn + c->n_gdn) * 512 + (size_t)c->n_attn * pages * 2 * c->page_bytes +
           (size_t)c->n_gdn * (c->state_layer + c->conv_layer);
}

// PrefixSnapshots::trim (qwen3_5.rs:1222-1233): evict the oldest snapshots until the retained
// bytes fit max_bytes - incoming, and, when one is about to be added, until fewer than 16 remain.
static void trim_prefixes(hk_kev_cache* c, size_t max_bytes, size_t incoming) {
    const size_t cap = max_bytes > incoming ? max_bytes - incoming : 0;
    while (c->prefix_bytes > cap || (c->prefixes.size() >= (size_t)kMaxSnapshots && incoming > 0)) {
        if (c->fifo.empty()) break;
        auto it = c->prefixes.find(c->fifo.front());
        c->fifo.pop_front();
        if (it == c->prefixes.end()) continue;
        c->prefix_bytes -= it->second.bytes;
        drop_handle(c, it->second.h);
        c->prefixes.erase(it);
    }
}

// retain_prefix (qwen3_5.rs:3017-3041): keep one immutable snapshot of a completed prefix if its
// charged bytes fit the budget; a snapshot that cannot be made leaves the prefix uncached.
static void retain_prefix(hk_kev_cache* c, const KevHandle& h, const std::vector<int32_t>& key, size_t max_bytes) {
    if (c->prefixes.count(key)) return;
    const size_t bytes = retention_bytes(c, (int)key.size());
    if (bytes > max_bytes) return;
    Snapshot snap;
    if (clone_handle(c, h, snap.h) != HK_OK) return;
    trim_prefixes(c, max_bytes, bytes);
    snap.bytes = bytes;
    c->prefixes.emplace(key, std::move(snap));
    c->fifo.push_back(key);
    c->prefix_bytes += bytes;
}

// validate_prefix (qwen3_5.rs:3003-3015)
static int validate_prefix(hk_kev_cache* c, const int32_t* ids_host, int n) {
    const hk_kev_config& cfg = c->m->cfg;
    if (!ids_host || n <= 0 || n > cfg.max_context)
        return hk_fail(c->m->ctx, HK_ERR_INVALID, "prefill must be nonempty, contain valid token ids and fit max_context");
    for (int i = 0; i < n; ++i)
        if (ids_host[i] < 0 || ids_host[i] >= cfg.vocab)
            return hk_fail(c->m->ctx, HK_ERR_INVALID,
                           "prefill must be nonempty, contain valid token ids and fit max_context");
    return HK_OK;
}

// A new caller handle cloned from a retained snapshot.
static int clone_snapshot(hk_kev_cache* c, const Snapshot& snap, uint64_t* handle_out) {
    KevHandle h;
    if (int rc = clone_handle(c, snap.h, h)) return rc;
    const uint64_t id = c->next_id++;
    c->handles.emplace(id, std::move(h));
    *handle_out = id;
    return HK_OK;
}

// One prefill chunk ids_dev[0 .. len) appended to handle id (no outputs read).
static int run_chunk(hk_kev_cache* c, uint64_t id, const int32_t* ids_dev, int len, void* workspace,
                     size_t workspace_bytes) {
    const size_t model_ws = (kev_workspace_bytes(c->m, len, 1, 0) + 255) & ~(size_t)255;
    if (model_ws + table_bytes(c, 1) > workspace_bytes)
        return hk_fail(c->m->ctx, HK_ERR_INVALID, "workspace too small: %zu < %zu (hk_kev_cache_workspace_size of a chunk)",
                       workspace_bytes, model_ws + table_bytes(c, 1));
    int32_t* cu_dev = (int32_t*)((char*)workspace + model_ws + table_bytes(c, 1) - 256);
    const int32_t cu_host[2] = {0, len};
    hipSetDevice(c->m->ctx->device);
    // Work queued on the stream may still use this workspace, and cu_host lives on this stack
    // frame: wait for the stream, then copy synchronously (prefill is not a capture path, and
    // forward_cached synchronises at its end anyway), so no copy outlives the frame on any path.
    if (hipStreamSynchronize(c->m->ctx->stream) != hipSuccess ||
        hipMemcpy(cu_dev, cu_host, sizeof(cu_host), hipMemcpyHostToDevice) != hipSuccess)
        return hk_fail(c->m->ctx, HK_ERR_DEVICE, "prefill cu_seqlens upload failed");
    return forward_cached(c, &id, 1, ids_dev, cu_dev, cu_host, workspace, workspace_bytes, nullptr, nullptr, nullptr,
                          true);
}

static void count_chunk(hk_prefill_work* work, int len, bool second) {
    if (!work) return;
    work->forward_calls += 1;
    work->processed_tokens += (uint64_t)len;
    if (second) work->chunked_prefills += 1;
}

extern "C" int hk_kev_cache_prefill_cached(hk_kev_cache* c, const int32_t* ids_host, const int32_t* ids_dev,
                                           int n_tokens, size_t max_bytes, int chunk_tokens, void* workspace,
                                           size_t workspace_bytes, uint64_t* handle_out, int* hit_out,
                                           hk_prefill_work* work) {
    if (!c || !handle_out || !hit_out) return HK_ERR_INVALID;
    hk_ctx* ctx = c->m->ctx;
    if (int rc = validate_prefix(c, ids_host, n_tokens)) return rc;
    if (!ids_dev || !workspace || chunk_tokens < 0)
        return hk_fail(ctx, HK_ERR_INVALID, "invalid prefill arguments");
    trim_prefixes(c, max_bytes, 0);
    if ((int)c->handles.size() >= c->max_handles)
        return hk_fail(ctx, HK_ERR_NOMEM, "cache holds its maximum of %d live handles", c->max_handles);
    std::vector<int32_t> key(ids_host, ids_host + n_tokens);
    if (max_bytes > 0) {
        auto it = c->prefixes.find(key);
        if (it != c->prefixes.end()) {
            if (int rc = clone_snapshot(c, it->second, handle_out)) return rc;
            *hit_out = 1;
            return HK_OK;
        }
    }
    // compute_prefix (qwen3_5.rs:2937-2971): a new handle, the prefix in chunks of chunk_tokens
    // (0: one call)
    uint64_t id = 0;
    if (int rc = hk_kev_cache_open(c, &id)) return rc;
    const int step = chunk_tokens > 0 ? chunk_tokens : n_tokens;
    for (int off = 0, index = 0; off < n_tokens; off += step, ++index) {
        const int len = n_tokens - off < step ? n_tokens - off : step;
        count_chunk(work, len, index == 1);
        if (int rc = run_chunk(c, id, ids_dev + off, len, workspace, workspace_bytes)) {
            hk_kev_cache_release(c, id);
            return rc;
        }
    }
    retain_prefix(c, c->handles.at(id), key, max_bytes);
    *handle_out = id;
    *hit_out = 0;
    return HK_OK;
}

extern "C" int hk_kev_cache_begin_resumable(hk_kev_cache* c, const int32_t* ids_host, int n_tokens, size_t max_bytes,
                                            uint64_t* handle_out, int* hit_out) {
    if (!c || !handle_out || !hit_out) return HK_ERR_INVALID;
    hk_ctx* ctx = c->m->ctx;
    if (int rc = validate_prefix(c, ids_host, n_tokens)) return rc;
    if ((int)c->handles.size() >= c->max_handles)
        return hk_fail(ctx, HK_ERR_NOMEM, "cache holds its maximum of %d live handles", c->max_handles);
    trim_prefixes(c, max_bytes, 0);
    std::vector<int32_t> key(ids_host, ids_host + n_tokens);
    if (max_bytes > 0) {
        auto it = c->prefixes.find(key);
        if (it != c->prefixes.end()) {
            if (int rc = clone_snapshot(c, it->second, handle_out)) return rc;
            *hit_out = 1;
            return HK_OK;
        }
    }
    uint64_t id = 0;
    if (int rc = hk_kev_cache_open(c, &id)) return rc;
    Pending p;
    p.tokens = std::move(key);
    p.max_bytes = max_bytes;
    c->pending.emplace(id, std::move(p));
    *handle_out = id;
    *hit_out = 0;
    return HK_OK;
}

extern "C" int hk_kev_cache_advance_resumable(hk_kev_cache* c, uint64_t handle, const int32_t* ids_dev,
                                              int chunk_tokens, void* workspace, size_t workspace_bytes,
                                              hk_prefill_work* work, int* complete_out) {
    if (!c || !complete_out) return HK_ERR_INVALID;
    hk_ctx* ctx = c->m->ctx;
    auto pit = c->pending.find(handle);
    if (pit == c->pending.end()) return hk_fail(ctx, HK_ERR_INVALID, "unknown or completed resumable prefill handle");
    auto hit = c->handles.find(handle);
    if (hit == c->handles.end()) return hk_fail(ctx, HK_ERR_INVALID, "unknown resumable cache handle");
    if (!ids_dev || !workspace || chunk_tokens <= 0)
        return hk_fail(ctx, HK_ERR_INVALID, "resumable prefill needs the prefix ids and a chunk size > 0");
    const int n = (int)pit->second.tokens.size();
    const int off = hit->second.tokens;
    const int end = n < off + chunk_tokens ? n : off + chunk_tokens;
    // work counts every native attempt, failed ones included (backend.rs:413-425)
    count_chunk(work, end - off, off == chunk_tokens);
    if (int rc = run_chunk(c, handle, ids_dev + off, end - off, workspace, workspace_bytes)) return rc;
    const bool complete = end == n;
    if (complete) {
        Pending p = std::move(pit->second);
        c->pending.erase(pit);
        retain_prefix(c, c->handles.at(handle), p.tokens, p.max_bytes);
    }
    *complete_out = complete ? 1 : 0;
    return HK_OK;
}

extern "C" int hk_kev_cache_clear_prefixes(hk_kev_cache* c) {
    if (!c) return HK_ERR_INVALID;
    for (auto& kv : c->prefixes) drop_handle(c, kv.second.h);
    c->prefixes.clear();
    c->fifo.clear();
    c->prefix_bytes = 0;
    return HK_OK;
}

extern "C" int hk_kev_cache_prefix_stats(hk_kev_cache* c, int* count_out, size_t* bytes_out) {
    if (!c || !count_out || !bytes_out) return HK_ERR_INVALID;
    *count_out = (int)c->prefixes.size();
    *bytes_out = c->prefix_bytes;
    return HK_OK;
}
