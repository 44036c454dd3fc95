// tree.hip -- EAGLE3 draft-tree construction (gfx950).
//
// Restates on device memory the selection side of the reference's EAGLE3
// drafting (sima-neat/llima, paths relative to that repository):
//   topk<T>          sima_lmm/devkit/cpp/utils.hpp:216-281   heap top-k, its exact output order
//   logsoftmax<T>    sima_lmm/devkit/cpp/utils.hpp:283-301
//   topk_generate    sima_lmm/devkit/cpp/language_model_eagle3.cpp:808-1164
//   searchsorted     sima_lmm/devkit/cpp/eagle_helpers.hpp:197-214
// The draft model's forward passes between tree levels are the caller's.
//
// Heap top-k.  The reference keeps a min-heap of k values; its output order,
// and which of several values equal to the k-th it keeps, depend on the order
// of its insertions.  So the heap is replayed exactly: lane i of wavefront 0
// holds heap slot i, and each insertion and sift-down runs as the reference's
// does (uniform control flow, readlane/writelane).  What runs in parallel is
// finding the few values that can enter the heap.  Value j >= k enters iff it
// exceeds the root, which is then the k-th largest of values 0..j-1 (NaN never
// enters; a NaN among the first k values switches to replaying every value).
// The row is read in tiles of 16384 values; thread t of 1024 holds 16
// consecutive values of a tile.  The k-th largest of the 16 values of each
// earlier thread, and the root after the previous tile, are each at most that
// root, so a value not above their maximum cannot enter and is skipped.  The
// rest (a few hundred of a 32000-value row) are compacted in index order and
// replayed 64 at a time: a ballot finds the next one above the root.
//
// log-softmax.  The reference's float arithmetic (maximum, float sum of exp in
// index order, log(sum) + max, subtraction) with exp and log evaluated in
// double and rounded once to float: the correctly rounded values, which the C
// library's expf/logf return on all but a few arguments.
#include "common.hpp"
#include "../../include/llima_sampler.h"

namespace llima {

#define TK_WG 1024                        // threads of a top-k workgroup
#define TK_WAVES (TK_WG / 64)
#define TK_EPT 16                         // consecutive values per thread and tile
#define TK_TILE (TK_WG * TK_EPT)          // values per tile
#define TK_PAD(e) ((e) + ((e) >> 4))      // LDS slot of tile element e (conflict-free rows)
#define TK_CAP 4096                       // candidates of a tile held for the replay
#define TK_MAXK 32                        // the reference's limit on k
#define TK_PART_K 16                      // k at most for rows split into parts
#define TK_PART 4096                      // values of a part
#define TK_PARTS 64                       // parts of a row at most
#define TK_PSLOTS 256                     // a part's slots: the count, then its candidates
#define TK_PSTAGE 8                       // parts whose first candidates are staged together
#define TREE_WG 256
#define TREE_MAX_NODES 16384              // node scores the finish stages in LDS

// ------------------------------------------------------------------ tree state layout
// A caller-owned device buffer that persists from begin to finish: the current
// level's scores, the parent groups, every node's score and token, the draft
// attention mask, and the per-row top-k of the level being grown (total bytes);
// past them, in a buffer that has room, the candidates of rows split into parts.
struct TreeLayout {
    size_t score, parent, node_score, node_tok, mask, row_idx, row_val, cand, total;
};

__host__ __device__ inline size_t tree_take(size_t* o, size_t bytes) {
    const size_t r = *o;
    *o += (bytes + 255) & ~(size_t)255;
    return r;
}

__host__ __device__ inline TreeLayout tree_layout(int K, int depth) {
    TreeLayout L;
    size_t o = 0;
    const size_t nodes = (size_t)K + (size_t)(depth - 1) * K * K;
    L.score = tree_take(&o, 4 * (size_t)K);
    L.parent = tree_take(&o, 4 * (1 + (size_t)(depth - 1) * K));
    L.node_score = tree_take(&o, 4 * nodes);
    L.node_tok = tree_take(&o, 4 * nodes);
    L.mask = tree_take(&o, 4 * (size_t)K * K * depth);
    L.row_idx = tree_take(&o, 4 * (size_t)K * K);
    L.row_val = tree_take(&o, 4 * (size_t)K * K);
    L.total = L.cand = o;
    return L;
}

struct TreeParams {
    const void* x;           // top-k rows / level logits / root row
    int64_t row_stride;
    int32_t rows, cols, k;
    int32_t vec;             // rows 16-byte aligned: the fast top-k reads them with 16-byte loads
    int32_t* out_idx;        // [rows][k]
    float* out_val;          // [rows][k]
    const int32_t* d2t;
    char* state;
    int32_t K, depth, level, total, sample_token;
    int32_t* out_inputs;     // [K]
    int32_t* out_prow;       // [K]
    float* out_mask;         // [K][K * (level + 1)]
    int32_t* out_tokens;     // [N]
    float* out_tree_mask;    // [N][N]
    int32_t* out_pos;        // [N]
    int32_t* out_retrieve;   // [N][N]
    int32_t* out_dims;       // [2]
    int32_t parts;           // parts per row (0: rows not split)
    int32_t bf16;            // split rows: bf16 values
};

template <typename T>
__device__ __forceinline__ T* st(const TreeParams& P, size_t off) { return (T*)(P.state + off); }

// ------------------------------------------------------------------ helpers
template <typename TL>
__device__ __forceinline__ float tk_load(const TL* p, int64_t i);
template <>
__device__ __forceinline__ float tk_load<float>(const float* p, int64_t i) { return p[i]; }
template <>
__device__ __forceinline__ float tk_load<uint16_t>(const uint16_t* p, int64_t i) {
    return bf16_bits_to_f32(p[i]);
}

__device__ __forceinline__ float rdl_f(float v, int l) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), l));
}
// Lane l of v replaced by the uniform x (a compare and a select).
__device__ __forceinline__ float wrl_f(float v, float x, int l) {
    return (int)lane_id() == l ? x : v;
}
__device__ __forceinline__ int32_t rdl_i(int32_t v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ int32_t wrl_i(int32_t v, int32_t x, int l) {
    return (int)lane_id() == l ? x : v;
}

__device__ __forceinline__ float exp_cr(float x) { return (float)exp((double)x); }
__device__ __forceinline__ float log_cr(float x) { return (float)log((double)x); }

// Inclusive maximum over lanes 0..l (keys; 0 is the identity).
__device__ __forceinline__ uint32_t wave_incl_max_u32(uint32_t v) {
    auto mx = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
    v = mx(v, dpp32<DPP_ROW_SHR(1), 0xF, true>(0u, v));
    v = mx(v, dpp32<DPP_ROW_SHR(2), 0xF, true>(0u, v));
    v = mx(v, dpp32<DPP_ROW_SHR(4), 0xF, true>(0u, v));
    v = mx(v, dpp32<DPP_ROW_SHR(8), 0xF, true>(0u, v));
    v = mx(v, dpp32<DPP_ROW_BCAST15, 0xA, false>(0u, v));
    v = mx(v, dpp32<DPP_ROW_BCAST31, 0xC, false>(0u, v));
    return v;
}

// The k-th largest key (NaN: 0) of 16 values (k <= 16; 0 otherwise): a
// bitonic sorting network (descending) and a select.
__device__ __forceinline__ uint32_t kth_of_16(const float* vals, int k) {
    uint32_t v[TK_EPT];
#pragma unroll
    for (int i = 0; i < TK_EPT; ++i) v[i] = vals[i] == vals[i] ? f32_key(vals[i]) : 0u;
#pragma unroll
    for (int size = 2; size <= TK_EPT; size <<= 1) {
#pragma unroll
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
#pragma unroll
            for (int i = 0; i < TK_EPT; ++i) {
                const int j = i ^ stride;
                if (j > i) {
                    const bool desc = (i & size) == 0;
                    const uint32_t hi = v[i] > v[j] ? v[i] : v[j], lo = v[i] > v[j] ? v[j] : v[i];
                    v[i] = desc ? hi : lo;
                    v[j] = desc ? lo : hi;
                }
            }
        }
    }
    uint32_t r = 0;
#pragma unroll
    for (int i = 0; i < TK_EPT; ++i) r = i == k - 1 ? v[i] : r;
    return r;
}

struct TopkShared {
    float tile[TK_PAD(TK_TILE)];
    float cv[TK_CAP];
    int32_t ci[TK_CAP];
    uint32_t wpart[TK_WAVES + 1];          // + the fast path's heap root
    uint32_t init_k[TK_MAXK];
    uint32_t wcnt[TK_WAVES];
    float carry;             // the heap root after the previous tile
    uint32_t nan_init;       // a NaN among the first k values: replay every value
    float res_v[TK_MAXK];
    int32_t res_i[TK_MAXK];
};

template <typename TL>
__device__ __forceinline__ void tk_fetch(const TL* rowp, int base, int cols, float (&r)[TK_EPT]) {
#pragma unroll
    for (int i = 0; i < TK_EPT; ++i) {
        const int j = base + i * TK_WG + (int)threadIdx.x;
        r[i] = j < cols ? tk_load<TL>(rowp, j) : __builtin_nanf("");
    }
}

// Sift-down from slot `node` of the heap held by this wavefront (slot i in lane i).
__device__ __forceinline__ void heap_sift(float& hv, int32_t& hi, int node, int k) {
    for (;;) {
        int c = 2 * node + 1;
        if (c >= k) return;
        float vc = rdl_f(hv, c);
        if (c + 1 < k) {
            const float vr = rdl_f(hv, c + 1);
            if (vc > vr) { ++c; vc = vr; }
        }
        const float vn = rdl_f(hv, node);
        if (!(vn > vc)) return;
        const int32_t in_ = rdl_i(hi, node), ic = rdl_i(hi, c);
        hv = wrl_f(hv, vc, node);
        hv = wrl_f(hv, vn, c);
        hi = wrl_i(hi, ic, node);
        hi = wrl_i(hi, in_, c);
        node = c;
    }
}

// topk<T> of one row (utils.hpp:225-281) -> sh.res_v / sh.res_i [k], in the
// reference's output order, for any k <= 32 (readlane heap).  Every thread of
// the 1024 calls it.
template <typename TL>
__device__ __forceinline__ void topk_row_generic(const TL* rowp, int cols, int k, TopkShared& sh) {
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6;
    const int ntiles = (cols + TK_TILE - 1) / TK_TILE;
    if (t == 0) sh.nan_init = 0;
    __syncthreads();
    if (t < k) {
        const float v = tk_load<TL>(rowp, t);
        if (v != v) sh.nan_init = 1u;
    }
    float nxt[TK_EPT];
    tk_fetch<TL>(rowp, 0, cols, nxt);
    __syncthreads();
    const bool every = sh.nan_init != 0;
    float hv = 0.0f;                     // wavefront 0: heap slot `lane`
    int32_t hi = 0;
    for (int ti = 0; ti < ntiles; ++ti) {
        const int base = ti * TK_TILE;
#pragma unroll
        for (int i = 0; i < TK_EPT; ++i) sh.tile[TK_PAD(i * TK_WG + t)] = nxt[i];
        __syncthreads();
        if (ti + 1 < ntiles) tk_fetch<TL>(rowp, base + TK_TILE, cols, nxt);   // in flight meanwhile
        // ---- the candidates of this tile (thread t: values t*16 .. t*16+15, read
        //      from LDS each time they are needed, which keeps registers free)
        const float* seg = sh.tile + t * (TK_EPT + 1);                 // = TK_PAD(t * 16)
        uint32_t kk = kth_of_16(seg, k);
        uint32_t inc = wave_incl_max_u32(kk);
        uint32_t exc = (uint32_t)__shfl_up((int)inc, 1);
        exc = lane == 0 ? 0u : exc;
        if (lane == 63) sh.wpart[wave] = inc;
        __syncthreads();
        uint32_t lk = exc;
        for (int w = 0; w < wave; ++w) lk = sh.wpart[w] > lk ? sh.wpart[w] : lk;
        if (ti > 0) {
            const uint32_t ck = f32_key(sh.carry);
            lk = ck > lk ? ck : lk;
        }
        lk = lk > LLIMA_KEY_NEG_INF ? lk : LLIMA_KEY_NEG_INF;
        const float bound = key_f32(lk);
        uint32_t mine = 0;
#pragma unroll
        for (int q = 0; q < TK_EPT; ++q) {
            const int j = base + t * TK_EPT + q;
            mine += (j >= k && j < cols && seg[q] > bound) ? 1u : 0u;
        }
        const uint32_t winc = wave_incl_scan_u32(mine);
        if (lane == 63) sh.wcnt[wave] = winc;
        __syncthreads();
        uint32_t off = winc - mine, total = 0;
        for (int w = 0; w < TK_WAVES; ++w) {
            off += w < wave ? sh.wcnt[w] : 0u;
            total += sh.wcnt[w];
        }
        const bool all_values = every || total > TK_CAP;
        if (!all_values) {
#pragma unroll
            for (int q = 0; q < TK_EPT; ++q) {
                const int j = base + t * TK_EPT + q;
                if (j >= k && j < cols && seg[q] > bound) {
                    sh.cv[off] = seg[q];
                    sh.ci[off] = j;
                    ++off;
                }
            }
        }
        __syncthreads();
        // ---- the replay (wavefront 0)
        if (wave == 0) {
            if (ti == 0) {
                hv = lane < k ? sh.tile[TK_PAD(lane)] : 0.0f;
                hi = lane;
                for (int j = k / 2 - 1; j >= 0; --j) heap_sift(hv, hi, j, k);
            }
            const int n = all_values ? (cols - base < TK_TILE ? cols - base : TK_TILE) : (int)total;
            const int start = all_values && ti == 0 ? k : 0;
            float root = rdl_f(hv, 0);
            for (int g = start; g < n; g += 64) {
                const int e = g + lane;
                float x = __builtin_nanf("");
                int32_t xj = 0;
                if (e < n) {
                    x = all_values ? sh.tile[TK_PAD(e)] : sh.cv[e];
                    xj = all_values ? base + e : sh.ci[e];
                }
                uint64_t m = ballot(x > root);
                while (m) {
                    const int L = __builtin_ctzll(m);
                    const float xv = rdl_f(x, L);
                    hv = wrl_f(hv, xv, 0);
                    hi = wrl_i(hi, rdl_i(xj, L), 0);
                    heap_sift(hv, hi, 0, k);
                    root = rdl_f(hv, 0);
                    const uint64_t after = L == 63 ? 0ull : (~0ull << (L + 1));
                    m = ballot(x > root) & after;
                }
            }
            if (lane == 0) sh.carry = root;
        }
        __syncthreads();
    }
    // ---- output: the reference's selection sort over the heap slots
    if (wave == 0) {
        float rv = 0.0f;
        int32_t ri = 0;
        for (int a = 0; a < k; ++a) {
            int m = a;
            float vm = rdl_f(hv, a);
            for (int b = a + 1; b < k; ++b) {
                const float vb = rdl_f(hv, b);
                if (vb > vm) { m = b; vm = vb; }
            }
            rv = wrl_f(rv, vm, a);
            ri = wrl_i(ri, rdl_i(hi, m), a);
            hv = wrl_f(hv, rdl_f(hv, a), m);
            hi = wrl_i(hi, rdl_i(hi, a), m);
        }
        if (lane < k) { sh.res_v[lane] = rv; sh.res_i[lane] = ri; }
    }
    __syncthreads();
}

// ------------------------------------------------------------------ fast heap top-k (k <= 8)
// The same replay with the heap in registers: every lane of wavefront 0 holds
// the same copy (keys and ids, uniform control flow, uniform indices), so a
// sift-down step is a few register moves and compares instead of readlane
// round trips.  Keys compare as the floats do (order-preserving, -0 folded
// onto +0; no NaN is ever in the heap on this path).  Each thread's k-th
// largest key comes from a sorted list of its k largest (one max/min pair per
// list entry and value).  k from 9 on takes the generic heap here: the rows of
// a draft tree, whose k may be larger, are split into parts (further down).
#define TK_VPT 16
#define TK_FTILE (TK_WG * TK_VPT)

// Sift-down from slot NODE of a heap of KC keys: indices are compile-time
// constants, so the heap stays in registers.
template <int KC, int NODE>
__device__ __forceinline__ void uheap_sift(uint32_t (&hk)[KC], int32_t (&hi)[KC]) {
    constexpr int C = 2 * NODE + 1;
    if constexpr (C < KC) {
        bool right = false;
        uint32_t vc = hk[C];
        if constexpr (C + 1 < KC) {
            right = hk[C] > hk[C + 1];
            vc = right ? hk[C + 1] : vc;
        }
        const uint32_t vn = hk[NODE];
        if (vn > vc) {
            const int32_t in_ = hi[NODE];
            if constexpr (C + 1 < KC) {
                if (right) {
                    hk[NODE] = vc; hi[NODE] = hi[C + 1]; hk[C + 1] = vn; hi[C + 1] = in_;
                    uheap_sift<KC, C + 1>(hk, hi);
                    return;
                }
            }
            hk[NODE] = vc; hi[NODE] = hi[C]; hk[C] = vn; hi[C] = in_;
            uheap_sift<KC, C>(hk, hi);
        }
    }
}

// The reference's heapify of the first KC values: sift-down from KC/2 - 1 to 0.
template <int KC, int J>
__device__ __forceinline__ void uheap_build(uint32_t (&hk)[KC], int32_t (&hi)[KC]) {
    if constexpr (J >= 0) {
        uheap_sift<KC, J>(hk, hi);
        uheap_build<KC, J - 1>(hk, hi);
    }
}

// The raw bits of TK_VPT values from id i0 (ids at or past cols: a NaN
// pattern, which has no key), 16-byte loads when vec and the block lies in
// the row, else one value per load.
template <typename TL>
__device__ __forceinline__ void tk_raw(const TL* rowp, int i0, int cols, bool vec,
                                       llima_u32x4 (&q)[TK_VPT * sizeof(TL) / 16]) {
    constexpr int EPL = 16 / sizeof(TL);
    constexpr int NQ = TK_VPT / EPL;
    if (vec && i0 + TK_VPT <= cols) {
#pragma unroll
        for (int j = 0; j < NQ; ++j) q[j] = __builtin_nontemporal_load((const llima_u32x4*)(rowp + i0 + j * EPL));
    } else {
#pragma unroll
        for (int j = 0; j < NQ; ++j) {
            uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                const int i = i0 + j * EPL + e;
                uint32_t b;
                if constexpr (sizeof(TL) == 4) b = i < cols ? __float_as_uint(tk_load<TL>(rowp, i)) : 0x7FC00000u;
                else b = i < cols ? (uint32_t)((const uint16_t*)rowp)[i] : 0x7FC0u;
                if constexpr (sizeof(TL) == 4) w[e] = b;
                else w[e >> 1] |= b << ((e & 1) * 16);
            }
            q[j] = llima_u32x4{w[0], w[1], w[2], w[3]};
        }
    }
}

// The keys of a block's raw bits (a NaN: key 0, never a candidate).
template <typename TL>
__device__ __forceinline__ void tk_keys(const llima_u32x4 (&q)[TK_VPT * sizeof(TL) / 16],
                                        uint32_t (&kk)[TK_VPT]) {
    constexpr int EPL = 16 / sizeof(TL);
#pragma unroll
    for (int j = 0; j < TK_VPT / EPL; ++j) {
        const uint32_t w4[4] = {q[j].x, q[j].y, q[j].z, q[j].w};
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            const float f = sizeof(TL) == 4 ? __uint_as_float(w4[e])
                                            : __uint_as_float((e & 1) ? (w4[e >> 1] & 0xFFFF0000u)
                                                                      : (w4[e >> 1] << 16));
            kk[j * EPL + e] = f == f ? f32_key(f) : 0u;
        }
    }
}

// v into the descending list L[0, KC) of the KC largest keys (with multiplicity).
template <int KC>
__device__ __forceinline__ void tk_list_put(uint32_t (&L)[KC], uint32_t v) {
#pragma unroll
    for (int i = KC - 1; i > 0; --i) {
        const uint32_t lo = L[i - 1] < v ? L[i - 1] : v;
        L[i] = L[i] > lo ? L[i] : lo;
    }
    L[0] = L[0] > v ? L[0] : v;
}

// Rows are taken in tiles of TK_FTILE values; thread t holds the block of
// TK_VPT values at t TK_VPT.  A value after the first k is a candidate when it
// exceeds every earlier block's k-th largest key, the heap root after the
// earlier tiles, and the k-th largest key of its own block before it: each is
// at most the heap root when the value arrives.  The candidates, in id order,
// are replayed by wavefront 0.
template <typename TL, int KC>
__device__ __forceinline__ void topk_row_fast(const TL* rowp, int cols, bool vec, TopkShared& sh) {
    constexpr int k = KC;
    constexpr int NQ = TK_VPT * (int)sizeof(TL) / 16;
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6;
    uint32_t hk[KC];                // wavefront 0: the heap, every lane alike
    int32_t hi[KC];
#pragma unroll
    for (int i = 0; i < KC; ++i) { hk[i] = 0u; hi[i] = 0; }
    uint32_t carry = 0u;                   // the heap root after the earlier tiles
    for (int base = 0; base < cols; base += TK_FTILE) {
        const int ib = base + t * TK_VPT;
        llima_u32x4 q[NQ];
        tk_raw<TL>(rowp, ib, cols, vec, q);
        // ---- the block's k-th largest key, the bound from the earlier blocks
        uint32_t kth;
        {
            uint32_t kk[TK_VPT], L[KC];
            tk_keys<TL>(q, kk);
#pragma unroll
            for (int i = 0; i < KC; ++i) L[i] = 0u;
#pragma unroll
            for (int e = 0; e < TK_VPT; ++e) tk_list_put<KC>(L, kk[e]);
            kth = L[k - 1];
        }
        const uint32_t inc = wave_incl_max_u32(kth);
        uint32_t bound = (uint32_t)__shfl_up((int)inc, 1);
        bound = lane == 0 ? 0u : bound;
        bound = bound > carry ? bound : carry;
        if (lane == 63) sh.wpart[wave] = inc;
        __syncthreads();
        for (int w = 0; w < TK_WAVES; ++w) bound = w < wave && sh.wpart[w] > bound ? sh.wpart[w] : bound;
        // ---- candidates: above the bound and the block's own running k-th key
        uint32_t cmask = 0;
        {
            uint32_t kk[TK_VPT], L[KC];
            tk_keys<TL>(q, kk);
#pragma unroll
            for (int i = 0; i < KC; ++i) L[i] = 0u;
#pragma unroll
            for (int e = 0; e < TK_VPT; ++e) {
                const uint32_t thr = L[k - 1] > bound ? L[k - 1] : bound;
                cmask |= (ib + e >= k && kk[e] > thr) ? (1u << e) : 0u;
                tk_list_put<KC>(L, kk[e]);
            }
        }
        const uint32_t cnt = (uint32_t)__popc(cmask);
        const uint32_t ci = wave_incl_scan_u32(cnt);
        if (lane == 63) sh.wcnt[wave] = ci;
        if (base == 0 && t == 0) {                          // the first k values start the heap
            uint32_t kk[TK_VPT];
            tk_keys<TL>(q, kk);
#pragma unroll
            for (int e = 0; e < k; ++e) sh.init_k[e] = kk[e];
        }
        __syncthreads();
        uint32_t off = ci - cnt, total = 0;
        for (int w = 0; w < TK_WAVES; ++w) {
            off += w < wave ? sh.wcnt[w] : 0u;
            total += sh.wcnt[w];
        }
        if (wave == 0 && base == 0) {
            // readfirstlane: the heap is uniform, so the compiler keeps it in
            // scalar registers and sifts with scalar compares and branches
#pragma unroll
            for (int i = 0; i < k; ++i) {
                hk[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)sh.init_k[i]);
                hi[i] = i;
            }
            uheap_build<KC, KC / 2 - 1>(hk, hi);
        }
        // ---- rounds of TK_CAP candidates: staged in LDS, replayed by wavefront 0
        for (uint32_t r0 = 0; r0 < total; r0 += TK_CAP) {
            if (r0) __syncthreads();                        // wavefront 0 read the LDS
            {
                uint32_t kk[TK_VPT];
                tk_keys<TL>(q, kk);
                uint32_t o = off;
#pragma unroll
                for (int e = 0; e < TK_VPT; ++e) {
                    const bool c = (cmask >> e) & 1u;
                    if (c && o >= r0 && o < r0 + TK_CAP) {
                        sh.cv[o - r0] = __uint_as_float(kk[e]);    // the key's bits
                        sh.ci[o - r0] = ib + e;
                    }
                    o += c ? 1u : 0u;
                }
            }
            __syncthreads();
            if (wave == 0) {
                const uint32_t n = total - r0 < TK_CAP ? total - r0 : TK_CAP;
                uint32_t root = hk[0];
                for (uint32_t g = 0; g < n; g += 64) {
                    const uint32_t e = g + (uint32_t)lane;
                    const uint32_t x = e < n ? __float_as_uint(sh.cv[e]) : 0u;
                    const int32_t xj = e < n ? sh.ci[e] : 0;
                    uint64_t m = ballot(x > root);
                    while (m) {
                        const int Ln = __builtin_ctzll(m);
                        hk[0] = (uint32_t)__builtin_amdgcn_readlane((int)x, Ln);
                        hi[0] = __builtin_amdgcn_readlane(xj, Ln);
                        uheap_sift<KC, 0>(hk, hi);
                        root = hk[0];
                        const uint64_t after = Ln == 63 ? 0ull : (~0ull << (Ln + 1));
                        m = ballot(x > root) & after;
                    }
                }
            }
        }
        if (base + TK_FTILE < cols) {
            if (wave == 0 && lane == 0) sh.wpart[TK_WAVES] = hk[0];
            __syncthreads();
            carry = sh.wpart[TK_WAVES];                     // the k-th largest key so far
        }
    }
    // output: the reference's selection sort over the heap slots; the values
    // are the row's own (their bits, -0 included)
    if (wave == 0) {
        int32_t ri = 0;
#pragma unroll
        for (int a = 0; a < k; ++a) {
            // the first slot holding the largest of slots a .. k-1, then slot a's
            // entry moved into it (every index a select over the fixed slots)
            uint32_t vm = hk[a];
            int32_t im = hi[a];
            int m = a;
#pragma unroll
            for (int b = a + 1; b < k; ++b) {
                const bool gt = hk[b] > vm;
                vm = gt ? hk[b] : vm;
                im = gt ? hi[b] : im;
                m = gt ? b : m;
            }
            ri = lane == a ? im : ri;
#pragma unroll
            for (int b = a + 1; b < k; ++b) {
                hk[b] = m == b ? hk[a] : hk[b];
                hi[b] = m == b ? hi[a] : hi[b];
            }
        }
        if (lane < k) {
            sh.res_i[lane] = ri;
            sh.res_v[lane] = tk_load<TL>(rowp, ri);
        }
    }
    __syncthreads();
}

// topk<T> of one row (utils.hpp:225-281) -> sh.res_v / sh.res_i [k], in the
// reference's output order.  Every thread of the 1024 calls it.  k <= 8 with
// no NaN among the first k values takes the register heap.
template <typename TL>
__device__ __forceinline__ void topk_row(const TL* rowp, int cols, int k, bool vec, TopkShared& sh) {
    if (threadIdx.x == 0) sh.nan_init = 0;
    __syncthreads();
    if ((int)threadIdx.x < k) {
        const float v = tk_load<TL>(rowp, threadIdx.x);
        if (v != v) sh.nan_init = 1u;
    }
    __syncthreads();
    if (!sh.nan_init) {
        switch (k) {
            case 1: topk_row_fast<TL, 1>(rowp, cols, vec, sh); return;
            case 2: topk_row_fast<TL, 2>(rowp, cols, vec, sh); return;
            case 3: topk_row_fast<TL, 3>(rowp, cols, vec, sh); return;
            case 4: topk_row_fast<TL, 4>(rowp, cols, vec, sh); return;
            case 5: topk_row_fast<TL, 5>(rowp, cols, vec, sh); return;
            case 6: topk_row_fast<TL, 6>(rowp, cols, vec, sh); return;
            case 7: topk_row_fast<TL, 7>(rowp, cols, vec, sh); return;
            case 8: topk_row_fast<TL, 8>(rowp, cols, vec, sh); return;
            default: break;
        }
    }
    topk_row_generic<TL>(rowp, cols, k, sh);
}

// ------------------------------------------------------------------ kernels
template <typename TL>
__global__ __launch_bounds__(TK_WG) void topk_rows_kernel(TreeParams P) {
    __shared__ TopkShared sh;
    const int r = (int)blockIdx.x;
    topk_row<TL>((const TL*)P.x + (size_t)r * P.row_stride, P.cols, P.k, P.vec != 0, sh);
    if ((int)threadIdx.x < P.k) {
        P.out_idx[(size_t)r * P.k + threadIdx.x] = sh.res_i[threadIdx.x];
        P.out_val[(size_t)r * P.k + threadIdx.x] = sh.res_v[threadIdx.x];
    }
}

// topk<float> of n values in LDS by one thread (the reference's heap, in LDS
// slots hv/hi), into out_i / out_v.
__device__ void heap_topk_serial(const float* x, int n, int k, float* hv, int32_t* hi,
                                 int32_t* out_i, float* out_v) {
    for (int j = 0; j < k; ++j) { hv[j] = x[j]; hi[j] = j; }
    auto sift = [&](int node) {
        for (;;) {
            int c = 2 * node + 1;
            if (c >= k) return;
            if (c + 1 < k && hv[c] > hv[c + 1]) ++c;
            if (!(hv[node] > hv[c])) return;
            const float tv = hv[node]; hv[node] = hv[c]; hv[c] = tv;
            const int32_t ti = hi[node]; hi[node] = hi[c]; hi[c] = ti;
            node = c;
        }
    };
    for (int j = k / 2 - 1; j >= 0; --j) sift(j);
    for (int j = k; j < n; ++j)
        if (x[j] > hv[0]) { hv[0] = x[j]; hi[0] = j; sift(0); }
    for (int a = 0; a < k; ++a) {
        int m = a;
        for (int b = a + 1; b < k; ++b)
            if (hv[b] > hv[m]) m = b;
        out_v[a] = hv[m];
        out_i[a] = hi[m];
        hv[m] = hv[a];
        hi[m] = hi[a];
    }
}

// logsoftmax<float> of `rows` rows of n values in LDS (v, row-major) into out,
// by every thread of the workgroup: the row maximum (std::max order: a NaN
// never replaces it) and exp(v - max) per value in parallel, then per row the
// float sum of those terms in index order and log(sum) + max (one thread per
// row), then v - shift.  ex and shift are LDS scratch of rows * n and rows
// floats.  Contains two barriers; every thread calls it.
__device__ __forceinline__ void logsoftmax_rows(const float* v, int rows, int n, float* ex,
                                                float* shift, float* out) {
    const int t = (int)threadIdx.x;
    for (int q = t; q < rows * n; q += (int)blockDim.x) {
        const float* rv = v + (q / n) * n;
        float mx = -__builtin_inff();
        for (int i = 0; i < n; ++i) mx = mx < rv[i] ? rv[i] : mx;
        ex[q] = exp_cr(v[q] - mx);
    }
    __syncthreads();
    for (int r = t; r < rows; r += (int)blockDim.x) {
        const float* rv = v + r * n;
        float mx = -__builtin_inff(), sum = 0.0f;
        for (int i = 0; i < n; ++i) mx = mx < rv[i] ? rv[i] : mx;
        for (int i = 0; i < n; ++i) sum += ex[r * n + i];
        shift[r] = log_cr(sum) + mx;
    }
    __syncthreads();
    for (int q = t; q < rows * n; q += (int)blockDim.x) out[q] = v[q] - shift[q / n];
}

// topk<float> (the reference's heap) of n values in LDS, k = KC,
// by wavefront 0 (every lane alike) with the heap in scalar registers: the
// first KC values heapified, then every value above the root in index order
// (a ballot per 64 values finds them), then the selection sort.  Returns false
// (writing nothing) when a NaN is among the first KC values: the caller then
// takes heap_topk_serial.
template <int KC>
__device__ __forceinline__ bool heap_small(const float* x, int n, int32_t* out_i, float* out_v) {
    const int lane = (int)lane_id();
    uint32_t hk[KC];
    int32_t hi[KC];
    bool nan0 = false;
#pragma unroll
    for (int i = 0; i < KC; ++i) {
        const float f = x[i];
        nan0 = nan0 || f != f;
        hk[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)f32_key(f));
        hi[i] = i;
    }
    if (nan0) return false;
    uheap_build<KC, KC / 2 - 1>(hk, hi);
    uint32_t root = hk[0];
    for (int g = KC; g < n; g += 64) {
        const int e = g + lane;
        const float f = e < n ? x[e] : __builtin_nanf("");
        const uint32_t key = f == f ? f32_key(f) : 0u;         // a NaN never enters
        uint64_t m = ballot(key > root);
        while (m) {
            const int Ln = __builtin_ctzll(m);
            hk[0] = (uint32_t)__builtin_amdgcn_readlane((int)key, Ln);
            hi[0] = g + Ln;
            uheap_sift<KC, 0>(hk, hi);
            root = hk[0];
            const uint64_t after = Ln == 63 ? 0ull : (~0ull << (Ln + 1));
            m = ballot(key > root) & after;
        }
    }
    int32_t ri = 0;
#pragma unroll
    for (int a = 0; a < KC; ++a) {
        uint32_t vm = hk[a];
        int32_t im = hi[a];
        int m = a;
#pragma unroll
        for (int b = a + 1; b < KC; ++b) {
            const bool gt = hk[b] > vm;
            vm = gt ? hk[b] : vm;
            im = gt ? hi[b] : im;
            m = gt ? b : m;
        }
        ri = lane == a ? im : ri;
#pragma unroll
        for (int b = a + 1; b < KC; ++b) {
            hk[b] = m == b ? hk[a] : hk[b];
            hi[b] = m == b ? hi[a] : hi[b];
        }
    }
    if (lane < KC) {
        out_i[lane] = ri;
        out_v[lane] = x[ri];
    }
    return true;
}

// heap_small for a run-time k (wavefront 0); false when k > 8 or a NaN is
// among the first k values.
__device__ __forceinline__ bool heap_small_k(const float* x, int n, int k, int32_t* out_i,
                                             float* out_v) {
    switch (k) {
        case 1: return heap_small<1>(x, n, out_i, out_v);
        case 2: return heap_small<2>(x, n, out_i, out_v);
        case 3: return heap_small<3>(x, n, out_i, out_v);
        case 4: return heap_small<4>(x, n, out_i, out_v);
        case 5: return heap_small<5>(x, n, out_i, out_v);
        case 6: return heap_small<6>(x, n, out_i, out_v);
        case 7: return heap_small<7>(x, n, out_i, out_v);
        case 8: return heap_small<8>(x, n, out_i, out_v);
        default: return false;
    }
}

// The N largest keys of two descending lists (N a power of two) into a: the
// pairwise maxima of a and the reversed b are those N keys as a bitonic
// sequence, which log2 N exchanges sort.
template <int N>
__device__ __forceinline__ void tk_list_merge(uint32_t (&a)[N], const uint32_t (&b)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) a[i] = a[i] > b[N - 1 - i] ? a[i] : b[N - 1 - i];
#pragma unroll
    for (int s = N / 2; s > 0; s >>= 1)
#pragma unroll
        for (int i = 0; i < N; ++i)
            if ((i & s) == 0) {
                const uint32_t hi = a[i] > a[i + s] ? a[i] : a[i + s], lo = a[i] > a[i + s] ? a[i + s] : a[i];
                a[i] = hi;
                a[i + s] = lo;
            }
}

// ------------------------------------------------------------------ rows split into parts
// Measured for 5 rows of 32000 bf16 values, k 5: 5.0 us, and 12.3 us for the
// level kernel, where one workgroup per row took 17.9 and the combine 5.1; a
// tree of depth 4 131 -> 104 us per call.  Bound by latency: launches, the
// loads, the heap's ~45 dependent insertions.  k above 16 (the lists no longer
// fit the registers) and longer rows keep the kernels of one workgroup per row.
//
// A tree level's rows (k <= TK_PART_K, at most TK_PARTS parts): one 256-thread
// workgroup per 4096 values finds the values that can enter the row's heap,
// those that exceed the k-th largest value of the part before them (~40 of
// 4096), and writes them in id order to the part's slots; the level's last
// kernel replays each row's parts in order, a wavefront per row.  One
// workgroup per row instead runs ~900 vector instructions per thread on one
// CU.  A part with more of them than slots (ascending values) says so in its
// count, and its values are replayed one by one.
template <typename TL, int KC>
__global__ __launch_bounds__(TREE_WG) void eagle3_parts_kernel(TreeParams P) {
    constexpr int NQ = TK_VPT * (int)sizeof(TL) / 16;
    constexpr int N = KC <= 1 ? 1 : KC <= 2 ? 2 : KC <= 4 ? 4 : KC <= 8 ? 8 : 16;
    __shared__ uint32_t wlist[TREE_WG / 64][N], wcnt[TREE_WG / 64];
    const TreeLayout L = tree_layout(P.K, P.depth);
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6;
    const int row = (int)blockIdx.y, part = (int)blockIdx.x;
    const TL* rowp = (const TL*)P.x + (size_t)row * P.row_stride;
    const int ib = part * TK_PART + t * TK_VPT;
    llima_u32x4 q[NQ];
    tk_raw<TL>(rowp, ib, P.cols, P.vec != 0, q);
    uint32_t kk[TK_VPT], Lk[KC];
    tk_keys<TL>(q, kk);
#pragma unroll
    for (int i = 0; i < KC; ++i) Lk[i] = 0u;
#pragma unroll
    for (int e = 0; e < TK_VPT; ++e) tk_list_put<KC>(Lk, kk[e]);
    // the KC largest keys of all earlier threads: a scan over the lanes, then
    // the earlier waves' lists
    uint32_t A[N];
#pragma unroll
    for (int i = 0; i < N; ++i) A[i] = i < KC ? Lk[i < KC ? i : 0] : 0u;
    auto scan_step = [&](auto dpp) {
        uint32_t B[N];
#pragma unroll
        for (int i = 0; i < N; ++i) B[i] = dpp(A[i]);
        tk_list_merge<N>(A, B);
    };
    scan_step([](uint32_t v) { return dpp32<DPP_ROW_SHR(1), 0xF, true>(0u, v); });
    scan_step([](uint32_t v) { return dpp32<DPP_ROW_SHR(2), 0xF, true>(0u, v); });
    scan_step([](uint32_t v) { return dpp32<DPP_ROW_SHR(4), 0xF, true>(0u, v); });
    scan_step([](uint32_t v) { return dpp32<DPP_ROW_SHR(8), 0xF, true>(0u, v); });
    scan_step([](uint32_t v) { return dpp32<DPP_ROW_BCAST15, 0xA, false>(0u, v); });
    scan_step([](uint32_t v) { return dpp32<DPP_ROW_BCAST31, 0xC, false>(0u, v); });
    if (lane == 63) {
#pragma unroll
        for (int i = 0; i < N; ++i) wlist[wave][i] = A[i];
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const uint32_t v = (uint32_t)__shfl_up((int)A[i], 1);
        A[i] = lane == 0 ? 0u : v;
    }
    __syncthreads();
    for (int w = 0; w < wave; ++w) {
        uint32_t B[N];
#pragma unroll
        for (int i = 0; i < N; ++i) B[i] = wlist[w][i];
        tk_list_merge<N>(A, B);
    }
    // a value enters when it exceeds the k-th largest before it (ids below k
    // start the heap and are not written)
#pragma unroll
    for (int i = 0; i < KC; ++i) Lk[i] = A[i];
    uint32_t cmask = 0;
#pragma unroll
    for (int e = 0; e < TK_VPT; ++e) {
        cmask |= ib + e >= KC && kk[e] > Lk[KC - 1] ? 1u << e : 0u;
        tk_list_put<KC>(Lk, kk[e]);
    }
    const uint32_t cnt = (uint32_t)__popc(cmask);
    const uint32_t ci = wave_incl_scan_u32(cnt);
    if (lane == 63) wcnt[wave] = ci;
    __syncthreads();
    uint32_t off = ci - cnt, total = 0;
    for (int w = 0; w < TREE_WG / 64; ++w) {
        off += w < wave ? wcnt[w] : 0u;
        total += wcnt[w];
    }
    uint64_t* slots = st<uint64_t>(P, L.cand) + ((size_t)row * P.parts + part) * TK_PSLOTS;
#pragma unroll
    for (int e = 0; e < TK_VPT; ++e)
        if ((cmask >> e) & 1u) {
            if (off < TK_PSLOTS - 1) slots[1 + off] = ((uint64_t)kk[e] << 32) | (uint32_t)(ib + e);
            ++off;
        }
    if (t == 0) slots[0] = total;
}

// The heap of one row from its parts' candidates, by one wavefront (every lane
// alike), then the reference's selection sort: out_i / out_v [KC] (LDS).
template <int KC>
__device__ __forceinline__ void parts_replay(const TreeParams& P, const TreeLayout& L, int row,
                                             uint64_t (&stage)[TK_PSTAGE][64], int32_t* out_i,
                                             float* out_v) {
    const int lane = (int)lane_id();
    const int64_t r0 = (int64_t)row * P.row_stride;
    auto load = [&](int i) {                                // the row's value i
        return P.bf16 ? tk_load<uint16_t>((const uint16_t*)P.x + r0, i) : tk_load<float>((const float*)P.x + r0, i);
    };
    const uint64_t* slots = st<uint64_t>(P, L.cand) + (size_t)row * P.parts * TK_PSLOTS;
    // the first 64 candidates of TK_PSTAGE parts, requested together
    auto fetch = [&](int p0) {
        uint64_t c[TK_PSTAGE];
#pragma unroll
        for (int i = 0; i < TK_PSTAGE; ++i) {
            const int p = p0 + i < P.parts ? p0 + i : P.parts - 1;
            c[i] = slots[(size_t)p * TK_PSLOTS + 1 + lane];
        }
#pragma unroll
        for (int i = 0; i < TK_PSTAGE; ++i) stage[i][lane] = c[i];
    };
    const uint32_t pn = lane < P.parts ? (uint32_t)slots[(size_t)lane * TK_PSLOTS] : 0u;
    // The values that exceed the root's key, in id order: insert takes a key and
    // its id and returns the new root's key.  One copy of the loop per heap: the
    // code runs once per row, so its length is instruction fetch (unrolled over
    // the parts it took 113 us).
    auto replay = [&](uint32_t root, auto insert) {
#pragma unroll 1
        for (int p = 0; p < P.parts; ++p) {
            if (p % TK_PSTAGE == 0) fetch(p);
            const uint32_t stored = (uint32_t)__builtin_amdgcn_readlane((int)pn, p);
            const bool raw = stored > TK_PSLOTS - 1;        // not all stored: the part's values
            const int base = p * TK_PART;
            const int n = !raw ? (int)stored : P.cols - base < TK_PART ? P.cols - base : TK_PART;
#pragma unroll 1
            for (int g = 0; g < n; g += 64) {               // 64 values in id order (key 0: none)
                const int e = g + lane;
                uint32_t x = 0u;
                int32_t xj = base + e;
                if (raw) {
                    const float f = e < n ? load(base + e) : __builtin_nanf("");
                    x = xj >= KC && f == f ? f32_key(f) : 0u;
                } else {
                    const uint64_t v = g == 0 ? stage[p % TK_PSTAGE][lane]
                                              : slots[(size_t)p * TK_PSLOTS + 1 + (e < n ? e : g)];
                    x = e < n ? (uint32_t)(v >> 32) : 0u;
                    xj = (int32_t)(uint32_t)v;
                }
                uint64_t m = ballot(x > root);
                while (m) {
                    const int Ln = __builtin_ctzll(m);
                    root = insert((uint32_t)__builtin_amdgcn_readlane((int)x, Ln),
                                  __builtin_amdgcn_readlane(xj, Ln));
                    m = ballot(x > root) & (Ln == 63 ? 0ull : (~0ull << (Ln + 1)));
                }
            }
        }
    };
    const float f0 = lane < KC ? load(lane) : 0.0f;
    int32_t ri = 0;                                         // lane a: the id of place a
    if (ballot(f0 != f0)) {                                 // uniform: NaNs in the heap
        // Float compares, under which a NaN never moves and ends the sift above
        // it.  The slots the sift reaches from the root are a heap of their own
        // and the others hold at most the rest of the first k values, so at most
        // k - 1 values seen exceed the root: the values that do are candidates
        // here too.  A NaN root lets none in.
        float hv = f0;
        int32_t hi = lane;
        for (int j = KC / 2 - 1; j >= 0; --j) heap_sift(hv, hi, j, KC);
        auto top = [&]() {
            const float r = rdl_f(hv, 0);
            return r == r ? f32_key(r) : 0xFFFFFFFFu;
        };
        replay(top(), [&](uint32_t k, int32_t id) {
            hv = wrl_f(hv, key_f32(k), 0);
            hi = wrl_i(hi, id, 0);
            heap_sift(hv, hi, 0, KC);
            return top();
        });
        for (int a = 0; a < KC; ++a) {                      // the selection sort
            int m = a;
            float vm = rdl_f(hv, a);
            for (int b = a + 1; b < KC; ++b) {
                const float vb = rdl_f(hv, b);
                if (vb > vm) { m = b; vm = vb; }
            }
            const int32_t im = rdl_i(hi, m);
            ri = lane == a ? im : ri;
            hv = wrl_f(hv, rdl_f(hv, a), m);
            hi = wrl_i(hi, rdl_i(hi, a), m);
        }
    } else {
        uint32_t hk[KC];
        int32_t hi[KC];
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            hk[i] = (uint32_t)__builtin_amdgcn_readlane((int)f32_key(f0), i);
            hi[i] = i;
        }
        uheap_build<KC, KC / 2 - 1>(hk, hi);
        replay(hk[0], [&](uint32_t k, int32_t id) {
            hk[0] = k;
            hi[0] = id;
            uheap_sift<KC, 0>(hk, hi);
            return hk[0];
        });
#pragma unroll
        for (int a = 0; a < KC; ++a) {                      // the selection sort over the slots
            uint32_t vm = hk[a];
            int32_t im = hi[a];
            int m = a;
#pragma unroll
            for (int b = a + 1; b < KC; ++b) {
                const bool gt = hk[b] > vm;
                vm = gt ? hk[b] : vm;
                im = gt ? hi[b] : im;
                m = gt ? b : m;
            }
            ri = lane == a ? im : ri;
#pragma unroll
            for (int b = a + 1; b < KC; ++b) {
                hk[b] = m == b ? hk[a] : hk[b];
                hi[b] = m == b ? hi[a] : hi[b];
            }
        }
    }
    if (lane < KC) {
        out_i[lane] = ri;
        out_v[lane] = load(ri);                // the row's own bits (-0 included)
    }
}

// Level 0 from the root row's top K (res_i, res_v): their log-softmax as the
// scores, their mapped tokens; parent group 0; the draft mask starts as the
// K x K identity.
__device__ __forceinline__ void begin_level(const TreeParams& P, const TreeLayout& L,
                                            const int32_t* res_i, const float* res_v) {
    __shared__ float lp[TK_MAXK], ex[TK_MAXK], shift[1];
    const int K = P.K, t = (int)threadIdx.x;
    logsoftmax_rows(res_v, 1, K, ex, shift, lp);
    if (t < K) {
        const int32_t id = res_i[t];
        const int32_t tok = id + P.d2t[id];
        st<float>(P, L.score)[t] = lp[t];
        st<float>(P, L.node_score)[t] = lp[t];
        st<int32_t>(P, L.node_tok)[t] = tok;
        P.out_inputs[t] = tok;
    }
    if (t == 0) st<int32_t>(P, L.parent)[0] = 0;
    const int mc = K * P.depth;
    for (int e = t; e < K * mc; e += (int)blockDim.x)
        st<float>(P, L.mask)[e] = (e % mc) == e / mc ? 1.0f : 0.0f;
}

template <typename TL>
__global__ __launch_bounds__(TK_WG) void eagle3_begin_kernel(TreeParams P) {
    __shared__ TopkShared sh;
    topk_row<TL>((const TL*)P.x, P.cols, P.K, P.vec != 0, sh);
    begin_level(P, tree_layout(P.K, P.depth), sh.res_i, sh.res_v);
}

// The top K of each of the K rows of a level, into the state.
template <typename TL>
__global__ __launch_bounds__(TK_WG) void eagle3_rows_kernel(TreeParams P) {
    __shared__ TopkShared sh;
    const TreeLayout L = tree_layout(P.K, P.depth);
    const int K = P.K, r = (int)blockIdx.x;
    topk_row<TL>((const TL*)P.x + (size_t)r * P.row_stride, P.cols, K, P.vec != 0, sh);
    if ((int)threadIdx.x < K) {
        st<int32_t>(P, L.row_idx)[r * K + threadIdx.x] = sh.res_i[threadIdx.x];
        st<float>(P, L.row_val)[r * K + threadIdx.x] = sh.res_v[threadIdx.x];
    }
}

// Level `level` (1 .. depth-1) from the rows' top K (row_i, row_v, in LDS or in
// the state): cumulative scores, the best K of them, parent rows, next input
// ids, node lists, parent group, mask.
template <int KM>
__device__ __forceinline__ void combine_level(const TreeParams& P, const TreeLayout& L,
                                              const int32_t* row_i, const float* row_v) {
    __shared__ float cu[KM * KM];
    __shared__ int32_t tok[KM * KM];
    __shared__ float rv[KM * KM];
    __shared__ float score[KM], hv[KM], bestv[KM], shift[KM];
    __shared__ float ex[KM * KM];
    __shared__ int32_t hi[KM], best[KM];
    __shared__ uint32_t fast;
    __shared__ float oldm[KM * KM * 16];
    const int K = P.K, KK = K * K, t = (int)threadIdx.x, NT = (int)blockDim.x;
    const int i = P.level - 1;                    // the reference's loop counter
    const int mc = K * P.depth, acols = K * P.level;
    for (int q = t; q < KK; q += NT) {
        const int32_t id = row_i[q];
        tok[q] = id + P.d2t[id];
        rv[q] = row_v[q];
    }
    if (t < K) score[t] = st<float>(P, L.score)[t];
    for (int e = t; e < K * acols; e += NT)
        oldm[e] = st<float>(P, L.mask)[(e / acols) * mc + e % acols];
    __syncthreads();
    // each row's log-softmax plus the row's score (the reference's float steps)
    logsoftmax_rows(rv, K, K, ex, shift, cu);
    for (int q = t; q < KK; q += NT) cu[q] = cu[q] + score[q / K];
    __syncthreads();
    // the best K of the K*K cumulative scores (the reference's heap)
    if (t < 64) {
        bool ok;
        if constexpr (KM <= TK_PART_K) ok = heap_small<KM>(cu, KK, best, bestv);   // KM == K
        else ok = heap_small_k(cu, KK, K, best, bestv);
        if (t == 0) fast = ok ? 1u : 0u;
    }
    __syncthreads();
    if (!fast) {
        if (t == 0) heap_topk_serial(cu, KK, K, hv, hi, best, bestv);
        __syncthreads();
    }
    const size_t nbase = (size_t)K + (size_t)i * KK;
    for (int q = t; q < KK; q += NT) {
        st<float>(P, L.node_score)[nbase + q] = cu[q];
        st<int32_t>(P, L.node_tok)[nbase + q] = tok[q];
    }
    if (t < K) {
        const int32_t gbase = 1 + KK * (i - 1 > 0 ? i - 1 : 0) + (i > 0 ? K : 0);
        st<int32_t>(P, L.parent)[1 + i * K + t] = t + gbase;
        st<float>(P, L.score)[t] = bestv[t];
        P.out_inputs[t] = tok[best[t]];
        if (P.out_prow) P.out_prow[t] = best[t] / K;
    }
    // the mask: row r = old row of its parent, then an identity block
    const int ncols = acols + K;
    for (int e = t; e < K * ncols; e += NT) {
        const int r = e / ncols, c = e % ncols;
        const float v = c < acols ? oldm[(best[r] / K) * acols + c] : (c - acols == r ? 1.0f : 0.0f);
        st<float>(P, L.mask)[r * mc + c] = v;
        if (P.out_mask) P.out_mask[e] = v;
    }
}

__global__ __launch_bounds__(TREE_WG) void eagle3_combine_kernel(TreeParams P) {
    const TreeLayout L = tree_layout(P.K, P.depth);
    combine_level<TK_MAXK>(P, L, st<int32_t>(P, L.row_idx), st<float>(P, L.row_val));
}

// A level after eagle3_parts_kernel: wavefront r replays row r (K wavefronts,
// at least four; the root row alone at level 0), then the level's combine.
template <int KC>
__global__ __launch_bounds__(64 * (KC < 4 ? 4 : KC)) void eagle3_level_kernel(TreeParams P) {
    __shared__ int32_t row_i[KC * KC];
    __shared__ float row_v[KC * KC];
    __shared__ uint64_t stage[KC][TK_PSTAGE][64];
    const TreeLayout L = tree_layout(P.K, P.depth);
    const int w = (int)wave_id();
    if (w < (P.level == 0 ? 1 : KC)) parts_replay<KC>(P, L, w, stage[w], row_i + w * KC, row_v + w * KC);
    __syncthreads();
    if (P.level == 0) begin_level(P, L, row_i, row_v);
    else combine_level<KC>(P, L, row_i, row_v);
}

// The final tree: best `total` node scores, tokens, parents located among the
// survivors, tree mask, position ids, retrieve indices.  Only the set of the
// best `total` nodes matters (the reference sorts their positions), so it is
// found by ranking: node i is in when fewer than `total` nodes score above
// it; when the nodes equal to the boundary score are not all in, which of
// them the reference's heap keeps depends on its history, and one thread
// replays it (heap_topk_serial), as it does for NaN scores or more than
// TREE_RANK_MAX nodes.  The rest runs in parallel: positions by a scan of the
// membership flags, each survivor's parent by a binary search, each tree
// row's ancestors by walking up, leaves and their retrieve paths.
#define TREE_RANK_MAX 1024
__global__ __launch_bounds__(TREE_WG) void eagle3_finish_kernel(TreeParams P) {
    __shared__ float ns[TREE_MAX_NODES];
    __shared__ int32_t par[1 + TREE_MAX_NODES / TK_MAXK];
    __shared__ float hv[TK_MAXK], selv[TK_MAXK];
    __shared__ int32_t hi[TK_MAXK], sel[TK_MAXK], up[TK_MAXK];
    __shared__ uint64_t rowbits[TK_MAXK + 1];
    __shared__ uint32_t flag[TREE_RANK_MAX / 32];
    __shared__ uint32_t wsum[LLIMA_WAVES];
    __shared__ uint32_t slow, nan_any, bad_tie, parents_lo, parents_hi, maxpos_s;
    const TreeLayout L = tree_layout(P.K, P.depth);
    const int K = P.K, T = P.total, N = T + 1, t = (int)threadIdx.x;
    const int nodes = K + (P.depth - 1) * K * K, ngroups = 1 + (P.depth - 1) * K;
    const int rc = N;                        // a leaf path has at most N nodes
    if (t == 0) { nan_any = 0; bad_tie = 0; parents_lo = 0; parents_hi = 0; maxpos_s = 0; }
    for (int q = t; q < TREE_RANK_MAX / 32; q += TREE_WG) flag[q] = 0;
    for (int q = t; q < nodes; q += TREE_WG) ns[q] = st<float>(P, L.node_score)[q];
    for (int q = t; q < ngroups; q += TREE_WG) par[q] = st<int32_t>(P, L.parent)[q];
    for (int e = t; e < N * rc; e += TREE_WG) P.out_retrieve[e] = -1;
    __syncthreads();
    // ---- the set: rank every node against every node
    if (nodes <= TREE_RANK_MAX) {
        for (int i = t; i < nodes; i += TREE_WG) {
            const float v = ns[i];
            if (v != v) { nan_any = 1u; continue; }
            int gt = 0, eq = 0;
            for (int j = 0; j < nodes; ++j) {
                const float u = ns[j];
                gt += u > v ? 1 : 0;
                eq += u == v ? 1 : 0;
            }
            if (gt < T) {
                atomicOr(&flag[i >> 5], 1u << (i & 31));
                if (gt + eq > T) bad_tie = 1u;      // equal nodes straddle the boundary
            }
        }
    }
    __syncthreads();
    if (t == 0) slow = (nodes > TREE_RANK_MAX || nan_any || bad_tie) ? 1u : 0u;
    __syncthreads();
    if (slow) {
        if (t == 0) {
            heap_topk_serial(ns, nodes, T, hv, hi, sel, selv);
            for (int a = 1; a < T; ++a) {                       // ascending positions
                const int32_t v = sel[a];
                int b = a - 1;
                while (b >= 0 && sel[b] > v) { sel[b + 1] = sel[b]; --b; }
                sel[b + 1] = v;
            }
        }
    } else {
        // positions: a scan of the membership flags (thread t: nodes 4t .. 4t+3)
        const int i0 = 4 * t;
        uint32_t f4 = 0, c = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = i0 + e;
            const uint32_t b = i < nodes ? (flag[i >> 5] >> (i & 31)) & 1u : 0u;
            f4 |= b << e;
            c += b;
        }
        const uint32_t inc = wave_incl_scan_u32(c);
        if (lane_id() == 63) wsum[wave_id()] = inc;
        __syncthreads();
        uint32_t o = inc - c;
        for (uint32_t w = 0; w < wave_id(); ++w) o += wsum[w];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if ((f4 >> e) & 1u) sel[o++] = i0 + e;
    }
    __syncthreads();
    // ---- each survivor's parent: its group's entry minus 1 located among the
    //      sorted positions (eagle_helpers.hpp:197-214, lower bound), + 1
    if (t < T) {
        const int32_t pg = par[sel[t] / K];
        int lo = 0, hi2 = T;
        while (lo < hi2) {
            const int mid = (lo + hi2) >> 1;
            if (sel[mid] < pg - 1) lo = mid + 1; else hi2 = mid;
        }
        const int u = (pg == 0 ? -1 : lo) + 1;
        up[t] = u;
        if (u < 32) atomicOr(&parents_lo, 1u << u);
        else atomicOr(&parents_hi, 1u << (u - 32));
    }
    __syncthreads();
    // ---- tree rows: identity, column 0, and the ancestors (walk up)
    if (t < N) {
        uint64_t b = (1ull << t) | 1ull;
        int a = t;
        while (a > 0) {
            a = up[a - 1];
            b |= 1ull << a;
        }
        rowbits[t] = b;
        atomicMax(&maxpos_s, (uint32_t)(__popcll(b) - 1));
    }
    __syncthreads();
    const uint64_t parents = ((uint64_t)parents_hi << 32) | parents_lo;
    const int leaves = T - (__popcll(parents) - 1);
    // ---- retrieve: leaf r (the r-th node that is nobody's parent) walked
    //      back to the root
    if (t < N && !((parents >> t) & 1ull)) {
        const int row = t - __popcll(parents & ((1ull << t) - 1ull));   // nodes before t that are leaves
        if (row < leaves) {
            int at = t;
            for (int j = __popcll(rowbits[t]) - 1; j >= 0; --j) {
                P.out_retrieve[row * rc + j] = at;
                if (at > 0) at = up[at - 1];
            }
        }
    }
    for (int e = t; e < N * N; e += TREE_WG) {
        const int r = e / N, c = e % N;
        P.out_tree_mask[e] = (float)((rowbits[r] >> c) & 1ull);
    }
    if (t < N) {
        P.out_pos[t] = __popcll(rowbits[t]) - 1;
        P.out_tokens[t] = t == 0 ? P.sample_token : st<int32_t>(P, L.node_tok)[sel[t - 1]];
    }
    if (t == 0) {
        P.out_dims[0] = leaves;
        P.out_dims[1] = (int)maxpos_s + 1;
    }
}

}  // namespace llima

using namespace llima;

// Rows start on 16-byte boundaries (the row stride in bytes is a multiple of 16).
static int32_t rows_vec(const void* x, int64_t row_stride, int32_t dtype) {
    const int64_t esz = dtype == LLIMA_F32 ? 4 : 2;
    return ((uintptr_t)x % 16 == 0) && ((row_stride * esz) % 16 == 0) ? 1 : 0;
}

static bool tree_dims_ok(int32_t K, int32_t depth) {
    if (K < 1 || K > TK_MAXK || depth < 1 || depth > 16) return false;
    const int64_t nodes = (int64_t)K + (int64_t)(depth - 1) * K * K;
    return nodes <= TREE_MAX_NODES && (int64_t)K * K * (depth > 1 ? depth - 1 : 1) <= 16384;
}

// Parts per row when a level's rows can be split (0 when they cannot: k past
// the register heap, or more values than TK_PARTS parts hold), and the bytes of
// a state that holds the candidates of K such rows.
static int32_t tree_parts(int32_t K, int32_t Vd) {
    const int32_t n = Vd > 0 ? (Vd - 1) / TK_PART + 1 : 0;
    return K <= TK_PART_K && n <= TK_PARTS ? n : 0;
}

static size_t tree_split_bytes(int32_t K, int32_t depth, int32_t Vd) {
    return tree_layout(K, depth).total + sizeof(uint64_t) * (size_t)K * tree_parts(K, Vd) * TK_PSLOTS;
}

// Parts per row of a call: 0 also when the state has no room for the
// candidates, or is not aligned for their 8-byte slots (its own values are 4
// bytes wide), so that the state need not be larger than the tree.
static int32_t tree_call_parts(int32_t K, int32_t depth, int32_t Vd, const void* tree,
                               size_t tree_bytes) {
    return tree_bytes >= tree_split_bytes(K, depth, Vd) && (uintptr_t)tree % 8 == 0 ? tree_parts(K, Vd) : 0;
}

// A level's two kernels over split rows: the parts of `rows` rows, then the
// replay with the rest of the level (level 0 or a later one).
template <int KC>
static void launch_parts_k(const TreeParams& P, int rows, hipStream_t st) {
    const dim3 g(P.parts, rows);
    if (P.bf16) hipLaunchKernelGGL((eagle3_parts_kernel<uint16_t, KC>), g, dim3(TREE_WG), 0, st, P);
    else hipLaunchKernelGGL((eagle3_parts_kernel<float, KC>), g, dim3(TREE_WG), 0, st, P);
    hipLaunchKernelGGL(eagle3_level_kernel<KC>, dim3(1), dim3(64 * (KC < 4 ? 4 : KC)), 0, st, P);
}

static void launch_parts(const TreeParams& P, int rows, hipStream_t st) {
    switch (P.K) {
        case 1: launch_parts_k<1>(P, rows, st); break;
        case 2: launch_parts_k<2>(P, rows, st); break;
        case 3: launch_parts_k<3>(P, rows, st); break;
        case 4: launch_parts_k<4>(P, rows, st); break;
        case 5: launch_parts_k<5>(P, rows, st); break;
        case 6: launch_parts_k<6>(P, rows, st); break;
        case 7: launch_parts_k<7>(P, rows, st); break;
        case 8: launch_parts_k<8>(P, rows, st); break;
        case 9: launch_parts_k<9>(P, rows, st); break;
        case 10: launch_parts_k<10>(P, rows, st); break;
        case 11: launch_parts_k<11>(P, rows, st); break;
        case 12: launch_parts_k<12>(P, rows, st); break;
        case 13: launch_parts_k<13>(P, rows, st); break;
        case 14: launch_parts_k<14>(P, rows, st); break;
        case 15: launch_parts_k<15>(P, rows, st); break;
        case 16: launch_parts_k<16>(P, rows, st); break;
        default: break;
    }
}

extern "C" int llima_topk(const void* x, int32_t dtype, int32_t rows, int32_t cols,
                          int64_t row_stride, int32_t k, int32_t* out_idx, float* out_vals,
                          void* stream) {
    if (dtype != LLIMA_F32 && dtype != LLIMA_BF16) return LLIMA_E_INVAL;
    if (rows < 0 || k < 1 || k > TK_MAXK || cols < k || row_stride < cols) return LLIMA_E_INVAL;
    if (rows == 0) return LLIMA_OK;
    if (!x || !out_idx || !out_vals) return LLIMA_E_INVAL;
    TreeParams P = {};
    P.x = x; P.row_stride = row_stride; P.rows = rows; P.cols = cols; P.k = k;
    P.out_idx = out_idx; P.out_val = out_vals;
    P.vec = rows_vec(x, row_stride, dtype);
    hipStream_t st = (hipStream_t)stream;
    if (dtype == LLIMA_F32)
        hipLaunchKernelGGL(topk_rows_kernel<float>, dim3(rows), dim3(TK_WG), 0, st, P);
    else
        hipLaunchKernelGGL(topk_rows_kernel<uint16_t>, dim3(rows), dim3(TK_WG), 0, st, P);
    return hipGetLastError() == hipSuccess ? LLIMA_OK : LLIMA_E_HIP;
}

extern "C" size_t llima_eagle3_tree_bytes(int32_t K, int32_t depth) {
    if (!tree_dims_ok(K, depth)) return 0;
    return tree_layout(K, depth).total;
}

extern "C" size_t llima_eagle3_tree_split_bytes(int32_t K, int32_t depth, int32_t Vd) {
    if (!tree_dims_ok(K, depth)) return 0;
    return tree_split_bytes(K, depth, Vd);
}

extern "C" int llima_eagle3_tree_begin(const void* logits, int32_t dtype, int32_t Vd,
                                       const int32_t* d2t, int32_t K, int32_t depth, void* tree,
                                       size_t tree_bytes, int32_t* out_input_ids, void* stream) {
    if (dtype != LLIMA_F32 && dtype != LLIMA_BF16) return LLIMA_E_INVAL;
    if (!tree_dims_ok(K, depth) || Vd < K || !logits || !d2t || !out_input_ids) return LLIMA_E_INVAL;
    if (!tree || tree_bytes < tree_layout(K, depth).total) return LLIMA_E_WORKSPACE;
    TreeParams P = {};
    P.x = logits; P.cols = Vd; P.k = K; P.d2t = d2t; P.state = (char*)tree;
    P.K = K; P.depth = depth; P.out_inputs = out_input_ids;
    P.vec = rows_vec(logits, Vd, dtype);
    P.parts = tree_call_parts(K, depth, Vd, tree, tree_bytes);
    P.bf16 = dtype == LLIMA_BF16;
    hipStream_t st = (hipStream_t)stream;
    if (P.parts) launch_parts(P, 1, st);
    else if (dtype == LLIMA_F32)
        hipLaunchKernelGGL(eagle3_begin_kernel<float>, dim3(1), dim3(TK_WG), 0, st, P);
    else
        hipLaunchKernelGGL(eagle3_begin_kernel<uint16_t>, dim3(1), dim3(TK_WG), 0, st, P);
    return hipGetLastError() == hipSuccess ? LLIMA_OK : LLIMA_E_HIP;
}

extern "C" int llima_eagle3_tree_grow(const void* logits, int32_t dtype, int32_t Vd,
                                      int64_t row_stride, const int32_t* d2t, int32_t K,
                                      int32_t depth, int32_t level, void* tree, size_t tree_bytes,
                                      int32_t* out_input_ids, int32_t* out_parent_rows,
                                      float* out_mask, void* stream) {
    if (dtype != LLIMA_F32 && dtype != LLIMA_BF16) return LLIMA_E_INVAL;
    if (!tree_dims_ok(K, depth) || Vd < K || row_stride < Vd || level < 1 || level >= depth)
        return LLIMA_E_INVAL;
    if (!logits || !d2t || !out_input_ids) return LLIMA_E_INVAL;
    if (!tree || tree_bytes < tree_layout(K, depth).total) return LLIMA_E_WORKSPACE;
    TreeParams P = {};
    P.x = logits; P.row_stride = row_stride; P.cols = Vd; P.k = K; P.d2t = d2t;
    P.state = (char*)tree; P.K = K; P.depth = depth; P.level = level;
    P.out_inputs = out_input_ids; P.out_prow = out_parent_rows; P.out_mask = out_mask;
    P.vec = rows_vec(logits, row_stride, dtype);
    P.parts = tree_call_parts(K, depth, Vd, tree, tree_bytes);
    P.bf16 = dtype == LLIMA_BF16;
    hipStream_t st = (hipStream_t)stream;
    if (P.parts) {
        launch_parts(P, K, st);
        return hipGetLastError() == hipSuccess ? LLIMA_OK : LLIMA_E_HIP;
    }
    if (dtype == LLIMA_F32)
        hipLaunchKernelGGL(eagle3_rows_kernel<float>, dim3(K), dim3(TK_WG), 0, st, P);
    else
        hipLaunchKernelGGL(eagle3_rows_kernel<uint16_t>, dim3(K), dim3(TK_WG), 0, st, P);
    hipLaunchKernelGGL(eagle3_combine_kernel, dim3(1), dim3(TREE_WG), 0, st, P);
    return hipGetLastError() == hipSuccess ? LLIMA_OK : LLIMA_E_HIP;
}

extern "C" int llima_eagle3_tree_finish(void* tree, size_t tree_bytes, int32_t K, int32_t depth,
                                        int32_t total_tokens, int32_t sample_token,
                                        int32_t* out_tokens, float* out_tree_mask,
                                        int32_t* out_position_ids, int32_t* out_retrieve,
                                        int32_t* out_dims, void* stream) {
    if (!tree_dims_ok(K, depth) || total_tokens < 1 || total_tokens > TK_MAXK) return LLIMA_E_INVAL;
    if (total_tokens > K + (depth - 1) * K * K) return LLIMA_E_INVAL;
    if (!out_tokens || !out_tree_mask || !out_position_ids || !out_retrieve || !out_dims)
        return LLIMA_E_INVAL;
    if (!tree || tree_bytes < tree_layout(K, depth).total) return LLIMA_E_WORKSPACE;
    TreeParams P = {};
    P.state = (char*)tree; P.K = K; P.depth = depth; P.total = total_tokens;
    P.sample_token = sample_token;
    P.out_tokens = out_tokens; P.out_tree_mask = out_tree_mask; P.out_pos = out_position_ids;
    P.out_retrieve = out_retrieve; P.out_dims = out_dims;
    hipLaunchKernelGGL(eagle3_finish_kernel, dim3(1), dim3(TREE_WG), 0, (hipStream_t)stream, P);
    return hipGetLastError() == hipSuccess ? LLIMA_OK : LLIMA_E_HIP;
}
