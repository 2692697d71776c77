// Decode attention over the KV cache in place (attn::decode_attention,
// crates/tts-nn/src/attn.rs:18-73; the CPU path it is held to is Scores, softmax_last_dim and
// Weighted, attn.rs:85-126, 62, 189-226).
//
//   q     [b, n_kv, gqa, D] f32, any scale already folded in
//   cache [b, n_kv, cap, D] f16 or f32 (k and v)
//   out   [b, n_kv, gqa, D] f32
//   lane i attends to positions [window_start[i], span[i]); the reference's single span and
//   window start are the case where every lane has the same ones
//
// One workgroup per (lane, kv head): the cache rows of the span are read once, for all gqa query
// heads that share them. The span is split over groups of 16 lanes (4 per wave), each group
// taking every G-th position; a lane of a group owns D/16 dimensions: the score is a 16-lane
// shuffle reduction, and each group keeps a running softmax state (max m, sum l, weighted sum of
// v) updated position by position, or for f16 caches four positions at a time (online softmax).
// The groups' states are combined through LDS at the end: out = sum_k acc_k e^(m_k - M) /
// sum_k l_k e^(m_k - M), M the largest m_k (exponentials taken in base 2, below). This is the
// reference's exp(s - max) / sum weighting, regrouped; its K and V traffic is one pass.
// HBM-bound: 2 * D * (span - window_start) cache bytes per (lane, kv head).
//
// Long spans are split (flash-decoding): with a workspace, each workgroup takes kChunk positions
// of one (lane, kv head) and leaves its combined state (its max, its sum, its weighted v sum) in
// the workspace, and a second kernel merges a lane's chunks the same way. Without one, a
// workgroup takes the whole span.
#pragma once

#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "norm_rope.hpp"

namespace dtts {
namespace {

constexpr int kAttnMaxLanes = 256;

struct Spans {
    int32_t lo[kAttnMaxLanes];  // window start
    int32_t hi[kAttnMaxLanes];  // span (exclusive end)
};

// Where a lane's window [lo, hi) comes from: the kernel arguments (checked host arrays), or the
// device-resident position of the token being decoded (hi = pos + 1, the last `window`
// positions of it when a sliding window is set: Stack::forward's wstart, crates/qwen3tts/src/
// qwen3.rs:409-412), which keeps a captured graph valid from step to step.
struct HostSpans {
    Spans sp;
    __device__ __forceinline__ void get(int lane, int &lo, int &hi) const {
        lo = sp.lo[lane];
        hi = sp.hi[lane];
    }
};

struct DevSpans {
    const int32_t *pos;
    int window;  // 0: no window
    __device__ __forceinline__ void get(int lane, int &lo, int &hi) const {
        hi = pos[lane] + 1;
        lo = window > 0 && hi > window ? hi - window : 0;
    }
};

__device__ __forceinline__ void store_out(float *o, float v) { *o = v; }
__device__ __forceinline__ void store_out(half_t *o, float v) { *o = static_cast<half_t>(v); }

template <typename T>
struct CacheRow;  // D/16 consecutive elements of one cache row, as f32

template <>
struct CacheRow<half_t> {
    template <int E>
    __device__ __forceinline__ static void load(const half_t *p, float (&out)[E]) {
        static_assert(E == 8 || E == 4, "row slice");
        if constexpr (E == 8) {
            const half8_t v = *reinterpret_cast<const half8_t *>(p);
#pragma unroll
            for (int e = 0; e < 8; ++e) out[e] = static_cast<float>(v[e]);
        } else {
            const half4_t v = *reinterpret_cast<const half4_t *>(p);
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = static_cast<float>(v[e]);
        }
    }
};

template <>
struct CacheRow<float> {
    template <int E>
    __device__ __forceinline__ static void load(const float *p, float (&out)[E]) {
#pragma unroll
        for (int e = 0; e < E; e += 4) {
            const float4_t v = *reinterpret_cast<const float4_t *>(p + e);
            out[e] = v[0];
            out[e + 1] = v[1];
            out[e + 2] = v[2];
            out[e + 3] = v[3];
        }
    }
};

__device__ __forceinline__ float group16_sum(float v) {
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// The softmax runs in base 2: q is scaled by log2(e) as it is loaded, so scores, running maxima
// and the chunk states' m are log2 of the natural-base ones and every weight is one v_exp_f32
// (2^x; the library expf adds a range reduction and overflow checks, ~12 instructions). A weight
// 2^x with x below -126 is under 1e-38 of the running maximum's, whatever the unit rounds it to.
constexpr float kLog2e = 1.44269504088896340736f;
__device__ __forceinline__ float softmax_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Positions per workgroup when a span is split: kChunk at the entry points, whose workspace sizes
// are part of their interface. The stack step, which owns its workspace, halves it down to kChunkMin
// while the launch has few workgroups: a workgroup is a chain of dependent softmax updates, and few lanes
// leave most CUs without one (8 lanes, f32 caches of 1536 positions: 28.8 -> 15.3 us a layer, the merge
// 4.8 -> 5.3). Lines from 1 to 64 lanes and 64 to 4000 positions at 1, 2, 4 and 8 query heads per kv head:
// - fewer than kChunkFill workgroups (three per CU); 512 for f16 caches at 1 or 4 query heads, 320 at 8, whose
//   workgroups each combine 16 position groups of 8 heads (2 kv heads, D = 128, two layers: 64 lanes x 600
//   positions 14% faster at 384 workgroups than at 256; 16 lanes x 4000, the worst, 156 us at 256, 167 at 512, 225
//   at 1024);
// - at most 128 chunks x query heads, the rows that a merging workgroup reads;
// - a window that a merge costs more than it gives stays whole: 320 positions, 256 with f32 caches (32 lanes x 8 kv
//   heads x 300 positions, f16, one query head: 90.5 us whole, 94.5 in two chunks).
constexpr int kChunk = 512, kChunkMin = 128, kChunkFill = 768;

inline int attn_step_chunk(int64_t b, int64_t n_kv, int64_t gqa, bool f32, int64_t max_window) {
    if (max_window <= (f32 && gqa < 8 ? 256 : 320)) return kChunk;
    const int64_t fill = gqa >= 8 ? 320 : gqa == 2 || f32 ? kChunkFill : 512;
    auto chunks = [&](int c) { return (max_window + c - 1) / c; };
    int c = kChunk;
    while (c > kChunkMin && b * n_kv * chunks(c) < fill && chunks(c / 2) * gqa <= 128) c /= 2;
    return c;
}

// Chunks of a lane's window [lo, hi) when split; a chunk is a power of two.
__device__ __host__ inline int chunks_of(int lo, int hi, int chunk) {
    return (hi - lo + chunk - 1) >> (31 - __builtin_clz(static_cast<unsigned>(chunk)));
}

// The step's QK-norm, RoPE and cache append, done by the attention workgroups themselves (the same
// arithmetic as qk_rope_kernel): each makes its kv head's queries from the QKV projection's output,
// and the one whose chunk holds the new position also makes its k and v rows and writes the caches.
// Every chunk's workgroup repeats its GQA query rows of D values, which come from L2; the launch and its
// gap are gone (a predictor step at one lane 181 -> 169 us). With one or two query heads per kv head it is
// the faster way at every window up to kStepFuseMax (lane, kv head) pairs (two talker layers, f16 caches of
// 1536: 1 lane 111 -> 104.5 us, 16 lanes 140.3 -> 133.3), and beyond them while a window has at most two chunks (48
// lanes: 257 positions 142 -> 129 us, 800 6% to 12%, a predictor's 17 204 -> 191). With three chunks or more and
// more pairs it is between 14% faster and 2% slower (48 lanes of 1536: 200.3 -> 202.0), and qk_rope_kernel stays.
// Four query heads: from two chunks on (one: 2% to 6% slower). Eight, ten rows for four waves: 5% to 25%
// slower at most sizes, never.
constexpr int kStepFuseMax = 128;

inline bool step_fuses(int64_t pairs, int64_t gqa, int64_t chunks) {
    return gqa <= 4 && (gqa < 4 || chunks > 1) && (pairs <= kStepFuseMax || chunks <= 2);
}

struct QkvStep {
    const float *qkv;      // [b, (heads + 2 n_kv) D], or ys partials of it `stride` floats apart
    int ys;
    int64_t stride;
    bool round16;          // the summed output rounded to f16 first (candle's f16 matmul)
    const float *norms;    // [q | k] weights, or null
    const float *cos_t, *sin_t;
    float eps, q_scale;    // q_scale: on the roped q of layers without QK-norm
};
struct NoStep {};

// One row of D values by one wave: lane j holds dims j and j + D/2 (D = 64: lanes past 31 idle).
// w: the norm weights, or null for v (no norm, no RoPE).
template <int D>
__device__ __forceinline__ void step_row(const QkvStep &s, const float *src, const float *w, bool rope, const float *cos_r,
                                         const float *sin_r, int j, float &o1, float &o2) {
#pragma clang fp contract(off)
    constexpr int H = D / 2;
    auto ld = [&](const float *p) {  // the first eight partials requested together, summed in order
        float v8[8];
#pragma unroll
        for (int y = 0; y < 8; ++y)
            if (y < s.ys) v8[y] = p[y * s.stride];
        float v = v8[0];
#pragma unroll
        for (int y = 1; y < 8; ++y)
            if (y < s.ys) v += v8[y];
        for (int y = 8; y < s.ys; ++y) v += p[y * s.stride];
        return s.round16 ? static_cast<float>(static_cast<half_t>(v)) : v;
    };
    float x1 = 0.0f, x2 = 0.0f;
    if (j < H) {
        x1 = ld(src + j);
        x2 = ld(src + j + H);
    }
    o1 = x1;
    o2 = x2;
    if (!rope) return;
    const float ss = wave_sum(x1 * x1 + x2 * x2);
    if (w) {  // candle's rms_norm: (x / m) * w
        const float m = sqrtf(ss / static_cast<float>(D) + s.eps);
        if (j < H) {
            x1 = (x1 / m) * w[j];
            x2 = (x2 / m) * w[j + H];
        }
    }
    if (j < H) rope_pair(x1, x2, cos_r[j], sin_r[j], o1, o2);
}

// T: cache element type; D: head dim (64 or 128); GQA: query heads per kv head; NW: waves;
// Src: HostSpans or DevSpans; OutT: float, or half_t for a consumer that casts the result.
// part == nullptr: blockIdx.y is 0 and the workgroup writes out. Otherwise blockIdx.y is a chunk
// of `chunk` positions, and the workgroup writes its state to part (rows of D + 2 floats: the
// weighted v sum, the weight sum, the max score) at [(bh * max_chunks + chunk) * GQA + g].
// Step: QkvStep makes q and the new position here (q is unused; the caches are written at hi - 1), or
// NoStep reads q.
template <typename T, int D, int GQA, int NW, typename Src, typename OutT, typename Step>
__global__ __launch_bounds__(NW * 64, (std::is_same<Step, QkvStep>::value && GQA <= 2 ? 4 : 1)) void decode_attn_kernel(const float *q, T *kc, T *vc, OutT *out,
                                                              float *part, int max_chunks, int chunk, int n_kv, int cap,
                                                              Src sp, Step st) {
    constexpr bool STEP = std::is_same<Step, QkvStep>::value;
    constexpr int E = D / 16;     // dimensions per lane
    constexpr int G = NW * 4;     // position groups
    constexpr int UNROLL = 4;     // positions whose rows are in flight per group
    __shared__ float sm_m[G][GQA], sm_l[G][GQA];
    __shared__ __attribute__((aligned(16))) float sm_acc[G][GQA][D];
    float *sm_row = &sm_acc[0][0][0];  // STEP: the queries, k and v until the groups' states are written
    const int bh = blockIdx.x;  // lane * n_kv + kv head
    const int lane_idx = bh / n_kv;
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int grp = wave * 4 + ((tid & 63) >> 4);
    const int j = tid & 15;
    int lo, hi;
    sp.get(lane_idx, lo, hi);
    if (part && static_cast<int>(blockIdx.y) >= chunks_of(lo, hi, chunk)) return;  // the whole workgroup
    [[maybe_unused]] const int pos = hi - 1;  // the new position
    if (part) {
        lo += blockIdx.y * chunk;
        hi = hi < lo + chunk ? hi : lo + chunk;
    }
    [[maybe_unused]] const bool owns = STEP && hi == pos + 1;  // the chunk holds the new position
    float qv[GQA][E];
    if constexpr (STEP) {
        // the queries, then k and v of the new position, a row per wave in turn
        const int kh = bh - lane_idx * n_kv;
        const float *row = st.qkv + static_cast<int64_t>(lane_idx) * (GQA + 2) * n_kv * D;
        const float *cos_r = st.cos_t + static_cast<int64_t>(pos) * (D / 2), *sin_r = st.sin_t + static_cast<int64_t>(pos) * (D / 2);
        for (int task = wave; task < (owns ? GQA + 2 : GQA); task += NW) {
            const int lane = tid & 63;
            const bool is_q = task < GQA, is_v = task == GQA + 1;
            const int h = is_q ? kh * GQA + task : (is_v ? GQA + 1 : GQA) * n_kv + kh;
            float o1, o2;
            step_row<D>(st, row + static_cast<int64_t>(h) * D, st.norms ? st.norms + (is_q ? 0 : D) : nullptr, !is_v, cos_r,
                        sin_r, lane, o1, o2);
            if (is_q && st.q_scale != 1.0f) {
                o1 = o1 * st.q_scale;
                o2 = o2 * st.q_scale;
            }
            if (lane < D / 2) {
                if (!is_q) {  // as the cache holds them
                    T *dst = (is_v ? vc : kc) + (static_cast<int64_t>(bh) * cap + pos) * D;
                    const T c1 = static_cast<T>(o1), c2 = static_cast<T>(o2);
                    dst[lane] = c1;
                    dst[lane + D / 2] = c2;
                    o1 = static_cast<float>(c1);
                    o2 = static_cast<float>(c2);
                }
                float *r = sm_row + task * D;
                r[lane] = o1;
                r[lane + D / 2] = o2;
            }
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < GQA; ++g)
#pragma unroll
            for (int e = 0; e < E; ++e) qv[g][e] = sm_row[g * D + j * E + e] * kLog2e;
        if (owns) --hi;  // its row comes from LDS, below
    } else {
#pragma unroll
        for (int g = 0; g < GQA; ++g) {
            const float *qp = q + (static_cast<int64_t>(bh) * GQA + g) * D + j * E;
#pragma unroll
            for (int e = 0; e < E; ++e) qv[g][e] = qp[e] * kLog2e;
        }
    }
    float m[GQA], l[GQA], acc[GQA][E];
#pragma unroll
    for (int g = 0; g < GQA; ++g) {
        m[g] = -INFINITY;
        l[g] = 0.0f;
#pragma unroll
        for (int e = 0; e < E; ++e) acc[g][e] = 0.0f;
    }
    const T *kb = kc + static_cast<int64_t>(bh) * cap * D + j * E;
    const T *vb = vc + static_cast<int64_t>(bh) * cap * D + j * E;
    auto step = [&](const float (&kr)[E], const float (&vr)[E]) {
#pragma unroll
        for (int g = 0; g < GQA; ++g) {
            float s = 0.0f;
#pragma unroll
            for (int e = 0; e < E; ++e) s += qv[g][e] * kr[e];
            s = group16_sum(s);
            const float mn = fmaxf(m[g], s);
            const float c = softmax_exp2(m[g] - mn);  // 0 on the group's first position
            const float w = softmax_exp2(s - mn);
            l[g] = l[g] * c + w;
#pragma unroll
            for (int e = 0; e < E; ++e) acc[g][e] = acc[g][e] * c + w * vr[e];
            m[g] = mn;
        }
    };
    // UNROLL positions of the group at a time: their K and V rows are all requested before the
    // first is used (the group's 16 lanes read 16 * E contiguous elements per row). With f16
    // caches the online-softmax state moves once per UNROLL positions: one running maximum over
    // the block, one rescale of l and acc (one exponential for it), then the block's weighted rows
    // in order (decode attention 41.6 -> 39-40 us, the f16 talker step -2%). With f32 caches the
    // per-position update stays: held to four workgroups per CU (below), the block form measured
    // within +-2% there.
    auto step_block = [&](const float (&kr)[UNROLL][E], const float (&vr)[UNROLL][E]) {
#pragma unroll
        for (int g = 0; g < GQA; ++g) {
            float s[UNROLL];
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
                float d = 0.0f;
#pragma unroll
                for (int e = 0; e < E; ++e) d += qv[g][e] * kr[u][e];
                s[u] = group16_sum(d);
            }
            float mn = m[g];
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) mn = fmaxf(mn, s[u]);
            const float c = softmax_exp2(m[g] - mn);  // 0 on the group's first block
            float w[UNROLL];
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) w[u] = softmax_exp2(s[u] - mn);
            float lv = l[g] * c;
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) lv += w[u];
            l[g] = lv;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                float a = acc[g][e] * c;
#pragma unroll
                for (int u = 0; u < UNROLL; ++u) a += w[u] * vr[u][e];
                acc[g][e] = a;
            }
            m[g] = mn;
        }
    };
    int p = lo + grp;
    for (; p + (UNROLL - 1) * G < hi; p += UNROLL * G) {
        float kr[UNROLL][E], vr[UNROLL][E];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            CacheRow<T>::load(kb + static_cast<int64_t>(p + u * G) * D, kr[u]);
            CacheRow<T>::load(vb + static_cast<int64_t>(p + u * G) * D, vr[u]);
        }
        if constexpr (sizeof(T) == 2) {
            step_block(kr, vr);
        } else {
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) step(kr[u], vr[u]);
        }
    }
    for (; p < hi; p += G) {
        float kr[E], vr[E];
        CacheRow<T>::load(kb + static_cast<int64_t>(p) * D, kr);
        CacheRow<T>::load(vb + static_cast<int64_t>(p) * D, vr);
        step(kr, vr);
    }
    if constexpr (STEP) {
        if (owns && p == pos) {  // the group whose turn the new position is
            float kr[E], vr[E];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                kr[e] = sm_row[GQA * D + j * E + e];
                vr[e] = sm_row[(GQA + 1) * D + j * E + e];
            }
            step(kr, vr);
        }
        __syncthreads();  // the rows are read
    }

    // combine the groups' states
#pragma unroll
    for (int g = 0; g < GQA; ++g) {
#pragma unroll
        for (int e = 0; e < E; e += 4)
            *reinterpret_cast<float4_t *>(&sm_acc[grp][g][j * E + e]) =
                float4_t{acc[g][e], acc[g][e + 1], acc[g][e + 2], acc[g][e + 3]};
        if (j == 0) {
            sm_m[grp][g] = m[g];
            sm_l[grp][g] = l[g];
        }
    }
    __syncthreads();
    for (int t = tid; t < GQA * D; t += NW * 64) {
        const int g = t / D, d = t - (t / D) * D;
        float mx = -INFINITY;
#pragma unroll 4
        for (int k = 0; k < G; ++k) mx = fmaxf(mx, sm_m[k][g]);
        float den = 0.0f, num = 0.0f;
#pragma unroll 4
        for (int k = 0; k < G; ++k) {
            const float f = softmax_exp2(sm_m[k][g] - mx);  // 0 for groups that saw no position
            den += sm_l[k][g] * f;
            num += sm_acc[k][g][d] * f;
        }
        if (part) {
            float *pr = part + ((static_cast<int64_t>(bh) * max_chunks + blockIdx.y) * GQA + g) * (D + 2);
            pr[d] = num;
            if (d == 0) {
                pr[D] = den;
                pr[D + 1] = mx;
            }
        } else {
            store_out(out + (static_cast<int64_t>(bh) * GQA + g) * D + d, num / den);
        }
    }
}

// Merges the chunk states of each (lane, kv head): out = sum_c num_c e^(m_c - M) / sum_c den_c
// e^(m_c - M), M the largest m_c, chunks in order (m in log2 units, so 2^(m_c - M)).
// U: chunk states requested together (a loop would wait for each in turn).
template <int D, int GQA, int U, typename Src, typename OutT>
__global__ __launch_bounds__(256) void decode_attn_merge(const float *part, OutT *out, int max_chunks, int chunk,
                                                         int n_kv, Src sp) {
    const int bh = blockIdx.x;
    const int lane_idx = bh / n_kv;
    int lo, hi;
    sp.get(lane_idx, lo, hi);
    const int nch = chunks_of(lo, hi, chunk);
    for (int t = threadIdx.x; t < GQA * D; t += 256) {
        const int g = t / D, d = t - (t / D) * D;
        const float *pr = part + (static_cast<int64_t>(bh) * max_chunks * GQA + g) * (D + 2);
        const int64_t stride = static_cast<int64_t>(GQA) * (D + 2);
        float num = 0.0f, den = 0.0f, m = -INFINITY;
        for (int c0 = 0; c0 < nch; c0 += U) {
            float mc[U], nc[U], dc[U];
#pragma unroll
            for (int c = 0; c < U; ++c)
                if (c0 + c < nch) {
                    const float *pc = pr + (c0 + c) * stride;
                    mc[c] = pc[D + 1];
                    nc[c] = pc[d];
                    dc[c] = pc[D];
                }
            float mx = m;
#pragma unroll
            for (int c = 0; c < U; ++c)
                if (c0 + c < nch) mx = fmaxf(mx, mc[c]);
            if (c0 > 0) {  // the sums so far, at the new maximum
                const float f = softmax_exp2(m - mx);
                num *= f;
                den *= f;
            }
            m = mx;
#pragma unroll
            for (int c = 0; c < U; ++c)
                if (c0 + c < nch) {
                    const float f = softmax_exp2(mc[c] - mx);
                    num += nc[c] * f;
                    den += dc[c] * f;
                }
        }
        store_out(out + (static_cast<int64_t>(bh) * GQA + g) * D + d, num / den);
    }
}

// Unused dynamic LDS that holds decode attention to at most 5 workgroups per CU (f16 caches) or
// 4 (f32 caches), one wave per SIMD each: the kernel's registers would let 6 and 5 run, and more
// rows in flight than that measured slower (f32 caches: the F32 and Q8_0 talker steps 5.44 ->
// 5.85 ms at 5; f16 caches: attention 35.5 against 36.0 us at 6). 160 KB of LDS per CU.
template <typename T, int D, int GQA>
constexpr size_t attn_lds_pad() {
    constexpr size_t wg = sizeof(T) == 4 ? 4 : 5;
    constexpr size_t stat = sizeof(float) * (2 * 16 * GQA + 16 * GQA * D);  // the kernel's own LDS
    return stat < 160 * 1024 / wg ? (160 * 1024 / wg - stat) / 512 * 512 : 0;
}

template <typename T, int D, int GQA, typename Src, typename OutT, typename Step>
hipError_t launch_gqa(const float *q, T *kc, T *vc, OutT *out, float *part, int max_chunks, int chunk, int64_t b,
                      int64_t n_kv, int64_t cap, const Src &sp, const Step &st, hipStream_t stream) {
    const unsigned grid = static_cast<unsigned>(b * n_kv);
    constexpr size_t pad = attn_lds_pad<T, D, GQA>();
    if (!part) {
        decode_attn_kernel<T, D, GQA, 4, Src, OutT, Step><<<grid, 256, pad, stream>>>(
            q, kc, vc, out, nullptr, 0, 0, static_cast<int>(n_kv), static_cast<int>(cap), sp, st);
        return hipGetLastError();
    }
    decode_attn_kernel<T, D, GQA, 4, Src, OutT, Step><<<dim3(grid, max_chunks), 256, pad, stream>>>(
        q, kc, vc, out, part, max_chunks, chunk, static_cast<int>(n_kv), static_cast<int>(cap), sp, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (max_chunks <= 4)
        decode_attn_merge<D, GQA, 4, Src, OutT><<<grid, 256, 0, stream>>>(part, out, max_chunks, chunk, static_cast<int>(n_kv), sp);
    else
        decode_attn_merge<D, GQA, 16, Src, OutT><<<grid, 256, 0, stream>>>(part, out, max_chunks, chunk, static_cast<int>(n_kv), sp);
    return hipGetLastError();
}

// gqa in {1, 2, 4, 8} (8: NoStep only) and D in {64, 128}, checked by the caller.
template <typename T, typename Src, typename OutT, typename Step>
hipError_t launch_attention(const float *q, T *kc, T *vc, OutT *out, float *part, int max_window,
                            int chunk, int64_t b, int64_t n_kv, int64_t gqa, int64_t head_dim, int64_t cap, const Src &sp,
                            const Step &st, hipStream_t stream) {
    const int max_chunks = part ? (max_window + chunk - 1) / chunk : 0;
    if (head_dim == 128) {
        switch (gqa) {
            case 1: return launch_gqa<T, 128, 1>(q, kc, vc, out, part, max_chunks, chunk, b, n_kv, cap, sp, st, stream);
            case 2: return launch_gqa<T, 128, 2>(q, kc, vc, out, part, max_chunks, chunk, b, n_kv, cap, sp, st, stream);
            case 4: return launch_gqa<T, 128, 4>(q, kc, vc, out, part, max_chunks, chunk, b, n_kv, cap, sp, st, stream);
            default:
                if constexpr (std::is_same<Step, NoStep>::value)
                    return launch_gqa<T, 128, 8>(q, kc, vc, out, part, max_chunks, chunk, b, n_kv, cap, sp, st, stream);
                return hipErrorInvalidValue;
        }
    }
    switch (gqa) {
        case 1: return launch_gqa<T, 64, 1>(q, kc, vc, out, part, max_chunks, chunk, b, n_kv, cap, sp, st, stream);
        case 2: return launch_gqa<T, 64, 2>(q, kc, vc, out, part, max_chunks, chunk, b, n_kv, cap, sp, st, stream);
        case 4: return launch_gqa<T, 64, 4>(q, kc, vc, out, part, max_chunks, chunk, b, n_kv, cap, sp, st, stream);
        default:
            if constexpr (std::is_same<Step, NoStep>::value)
                return launch_gqa<T, 64, 8>(q, kc, vc, out, part, max_chunks, chunk, b, n_kv, cap, sp, st, stream);
            return hipErrorInvalidValue;
    }
}

// Workspace bytes for splitting windows of up to max_window positions into chunks of kChunk (0 when
// one chunk holds them).
inline size_t attn_workspace_bytes(int64_t b, int64_t n_kv, int64_t gqa, int64_t head_dim, int64_t max_window) {
    if (b <= 0 || n_kv <= 0 || gqa <= 0 || head_dim <= 0 || max_window <= kChunk) return 0;
    const int64_t chunks = (max_window + kChunk - 1) / kChunk;
    return static_cast<size_t>(b * n_kv * chunks * gqa * (head_dim + 2)) * sizeof(float);
}

// The stack step's workspace: room for every window up to max_window at any lane count up to b, so that
// one sized for the largest batch and capacity serves the smaller ones, whose chunks are shorter (a chunk
// below kChunk is taken only while twice its length gives under kChunkFill workgroups at most, so its chunks
// stay under twice the filling count). From kChunkFill lanes on the need only grows with the lanes.
inline size_t attn_step_workspace_bytes(int64_t b, int64_t n_kv, int64_t gqa, int64_t head_dim, int64_t max_window) {
    if (b <= 0 || n_kv <= 0 || gqa <= 0 || head_dim <= 0 || max_window <= 2 * kChunkMin) return 0;
    const int64_t shortest = (max_window + kChunkMin - 1) / kChunkMin, longest = (max_window + kChunk - 1) / kChunk;
    int64_t rows = 0;
    for (int64_t i = 1; i <= b && i <= kChunkFill; ++i) {
        const int64_t l = i < kChunkFill ? i : b;
        const int64_t fill = 2 * ((kChunkFill + l * n_kv - 1) / (l * n_kv));
        const int64_t most = shortest < fill ? shortest : (fill > longest ? fill : longest);
        rows = l * n_kv * most > rows ? l * n_kv * most : rows;
    }
    return static_cast<size_t>(rows * gqa * (head_dim + 2)) * sizeof(float);
}

}  // namespace
}  // namespace dtts
