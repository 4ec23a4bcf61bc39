// Which keys a query of paged attention sees (the options are described in hybrid_attention.hip), for
// the kernels of hybrid_attention.hip and hybrid_prompts.hip.
#pragma once
#include "hybrid_merge.h"

namespace hyb {

struct KeyRule {
    int window;             // 0: every earlier key is visible
    int keep_first;
    const float* slopes;    // [H] or null
    int v_stride;           // elements from one (slot, KV head) value row to the next: E for a dense
                            // V cache, more when the value rows are the leading part of wider rows
                            // (values stored inside the key rows: v_cache then points into k_cache)
    const float* temps;     // [H] or null: multiplies the scaled score of head h
    float softcap;          // 0: none
    int pool;               // 0: no pooled blocks (needs window > 0 and keep_first == 0)
    int pool_rows;          // pooled rows per page
    long pool_base;         // first pooled row, in rows from the start of the K (and of the V) cache
    int chunk;              // 0: none (else keep_first == 0 and pool == 0)
    // the first key a query at position i sees besides kept first tokens and pooled rows; it never
    // falls as i grows
    __device__ __forceinline__ int first_key(int i) const {
        int lo = window > 0 ? max(0, i - window + 1) : 0;
        if (chunk > 0) lo = max(lo, i / chunk * chunk);
        return lo;
    }
    __device__ __forceinline__ float capped(float s) const {
        return softcap > 0.f ? softcap * tanhf(s / softcap) : s;
    }
    __device__ __forceinline__ float head_scale(float scale, int h) const {
        return temps ? scale * temps[h] : scale;
    }
    // pooled blocks a query that sees ctx keys without a window takes in
    __device__ __forceinline__ int pooled_for(int ctx) const {
        return (pool > 0 && ctx > window) ? (ctx - window) / pool : 0;
    }
    __device__ __forceinline__ long pooled_row(const int* table, int b) const {
        return pool_base + (long)table[b / pool_rows] * pool_rows + b % pool_rows;
    }
};

// The visible keys of a query that sees `ctx` keys without a window (its position is ctx - 1), as
// one run of virtual indices: [0, kept) are keys 0 .. kept-1, the rest the window's keys from `lo`.
struct VisibleKeys {
    int kept, lo, count;
    __device__ __forceinline__ VisibleKeys(int ctx, const KeyRule& r) {
        lo = r.first_key(ctx - 1);
        kept = r.pool > 0 ? r.pooled_for(ctx) : min(r.keep_first, lo);
        count = kept + ctx - lo;
    }
    __device__ __forceinline__ int key(int v) const { return v < kept ? v : lo + (v - kept); }
    // cache row of virtual key v (with pooled blocks the leading `kept` indices are pooled rows)
    __device__ __forceinline__ long row(int v, const int* table, int block_size, const KeyRule& r) const {
        if (r.pool > 0 && v < kept) return r.pooled_row(table, v);
        const int j = key(v);
        return (long)table[j / block_size] * block_size + j % block_size;
    }
};

inline bool chunk_rule_ok(const KeyRule& r) {
    return r.chunk == 0 || (r.chunk > 0 && r.keep_first == 0 && r.pool == 0);
}

// pooled blocks need a window, no kept first tokens, no distance penalty, and a place in the caches
inline bool pool_rule_ok(const KeyRule& r) {
    return r.pool == 0 || (r.pool > 0 && r.window > 0 && r.keep_first == 0 && !r.slopes &&
                           r.pool_rows > 0 && r.pool_base > 0);
}

// Output rows of a step that no sequence owns are zeros where the kernel is asked to see to it (end > 0): those of
// [first, end) ahead of its first sequence's and behind its last one's.  By the workgroups (head, sequence, part) of a grid.
struct RowSpan { long first, end; };
template <typename T>
__device__ __forceinline__ void clear_rest(T* out, const int* cu_q, const RowSpan& span, int h, int H, int E) {
    auto clear = [&](long from, long to) {
        for (long r = from + blockIdx.z; r < to; r += gridDim.z)
            for (int e = threadIdx.x; e < E; e += blockDim.x) out[(r * H + h) * E + e] = T(0);
    };
    if (blockIdx.y == 0) clear(span.first, cu_q[0]);
    if (blockIdx.y + 1 == gridDim.y) clear(cu_q[gridDim.y], span.end);
}

// hybrid_prompts.hip: prompt portions over bfloat16 and (_f32) float caches, operands as
// hyb_sink_attention_tiles; _ok: sizes in whole runs of eight numbers, 16-byte addresses, a grid that can
// be launched
bool prompt_attention_ok(const void* q, long q_row, long q_head, const void* k_cache, const void* v_cache,
                         const void* out, int nseq, int max_q, int D, int E, int v_stride, bool f32);
int prompt_attention(const void* q, long q_row, long q_head, const void* k_cache, const void* v_cache,
                     const void* block_tables, int max_blocks, int block_size, const void* cu_q,
                     const void* positions, const void* sink, const void* gate, long gate_row, void* out,
                     float scale, int nseq, int seq0, int max_q, int H, int G, int D, int E,
                     const KeyRule& rule, RowSpan clear, hipStream_t s);

int prompt_attention_f32(const void* q, long q_row, long q_head, const void* k_cache, const void* v_cache,
                         const void* block_tables, int max_blocks, int block_size, const void* cu_q,
                         const void* positions, const void* sink, const void* gate, long gate_row, void* out,
                         float scale, int nseq, int seq0, int max_q, int H, int G, int D, int E,
                         const KeyRule& rule, RowSpan clear, hipStream_t s);

// the same over formed keys and values of latent attention (hybrid_latent_form.hip, with the operands of
// hyb_latent_formed_prompts); _pages_ok: what the pages have to be
bool latent_prompts_pages_ok(int block_size, int max_blocks, int latent_row);
int latent_prompts(const void* q, long q_row, long q_head, const void* qr, long qr_row, const void* cache,
                   const void* block_tables, int max_blocks, int block_size, const void* cu_q, const void* positions,
                   const void* sink, const void* k, const void* v, long formed_rows, void* out, float scale, int nseq,
                   int max_q, int H, int D, int E, int R, int P, int window, hipStream_t s);

}  // namespace hyb
