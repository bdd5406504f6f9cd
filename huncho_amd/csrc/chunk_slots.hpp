// chunk_slots.hpp - the numbering of the 64-token chunks of a varlen batch, which the split forms of the delta rule
// (gdn16_split.hip, delta_rule_split.hip) give their scratch slots: chunk by chunk, row by row. Rows outside the
// batch (an inconsistent cu_seqlens) have none.
#pragma once
#include "common.hpp"
#include "kernel_args.hpp"

namespace hk {
namespace chunk_slots {

constexpr int TOKENS = 64;  // per chunk

// The rows of sequence s; false if cu_seqlens is inconsistent there
__device__ __forceinline__ bool seq_rows(const GdnArgs& a, int s, int& t0, int& Tn) {
    t0 = a.cu_seqlens[s];
    Tn = a.cu_seqlens[s + 1] - t0;
    return t0 >= 0 && Tn >= 0 && t0 + Tn <= a.n_tokens;
}
// First slot number of sequence s
__device__ __forceinline__ int first_chunk(const GdnArgs& a, int s) {
    int n = 0;
    for (int i = 0; i < s; ++i) {
        int t0, Tn;
        if (seq_rows(a, i, t0, Tn)) n += (Tn + TOKENS - 1) / TOKENS;
    }
    return n;
}
// Chunk number cid -> sequence and first token of the chunk in it; false past the last chunk
__device__ __forceinline__ bool find_chunk(const GdnArgs& a, int n_seqs, int cid, int& seq, int& c0, int& t0, int& Tn) {
    for (seq = 0; seq < n_seqs; ++seq) {
        if (!seq_rows(a, seq, t0, Tn)) continue;
        const int n = (Tn + TOKENS - 1) / TOKENS;
        if (cid < n) {
            c0 = cid * TOKENS;
            return true;
        }
        cid -= n;
    }
    return false;
}

}  // namespace chunk_slots
}  // namespace hk
