// Attention with sinks for one decode token (GptOssModel::attention_from_cache,
// model.cpp:255-290), split over chunks of 64 cached positions.
//
//  partial: workgroup (chunk c, kv head h) scores the 8 query heads that share h
//           (GQA, head/8 = h) against positions of chunk c, and keeps per head the
//           chunk max m_c, sum l_c = sum exp(s - m_c) and o_c = sum exp(s - m_c) v.
//  combine: per query head, M = max(sink, max_c m_c),
//           den = exp(sink - M) + sum_c l_c exp(m_c - M),
//           out = sum_c o_c exp(m_c - M) / den -- the reference's softmax with the
//           sink in the max and the denominator only, regrouped by chunk.
// Even layers see the last 128 positions (the sliding window, one launch of
// attn_window_kernel), odd layers all (model.cpp:260).  The position is read from device memory, so one captured
// launch serves every decode step; chunks past the current length do nothing.
#include "ttl_internal.hpp"
#include "ttl_mfma.hpp"

#include <cmath>
#include <mutex>

namespace {

constexpr int kHead = 64, kQHeads = 64, kKvHeads = 8, kGroup = kQHeads / kKvHeads;
constexpr int kChunk = 64, kWindow = 128;
constexpr int kThreads = 256;

struct Span {
    uint32_t first, count;
};

__device__ inline Span span_of(uint32_t pos, uint32_t layer_index) {
    const uint32_t first = (layer_index % 2 == 0 && pos + 1 > uint32_t(kWindow)) ? pos + 1 - kWindow : 0;
    return {first, pos + 1 - first};
}

__device__ inline float wave_max(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        v = fmaxf(v, __shfl_xor(v, d));
    }
    return v;
}

__device__ inline float wave_sum(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        v += __shfl_xor(v, d);
    }
    return v;
}

// LDS row stride of the staged K/V chunk: 68 floats, so the 64 lanes of a score
// pass (one position each) read rows that start in different banks.
constexpr int kRowStride = kHead + 4;

__global__ __launch_bounds__(kThreads) void attn_partial_kernel(const float *__restrict__ q,
                                                                const float *__restrict__ k_cache,
                                                                const float *__restrict__ v_cache,
                                                                const int32_t *__restrict__ position,
                                                                uint32_t capacity, uint32_t layer_index,
                                                                uint32_t max_chunks, float *__restrict__ o_part,
                                                                float2 *__restrict__ ml_part) {
    __shared__ __attribute__((aligned(16))) float ks[kChunk * kRowStride];
    __shared__ __attribute__((aligned(16))) float vs[kChunk * kRowStride];
    // every thread stores its query float4 (t % 128) in a slot of its own, so the store
    // needs no branch (under one, the compiler places the K/V loads after it, and the
    // store waits for q alone); the scores read slots 0..127
    __shared__ float4 qs[kThreads];
    __shared__ float e[kGroup][kChunk];
    const uint32_t chunk = blockIdx.x, kvh = blockIdx.y, t = threadIdx.x;
    // Full-context layers only (their span starts at position 0), so the chunk's rows do
    // not depend on the position: the 8 query heads (every thread loads one of their 128
    // float4), the chunk's 64 K and V rows of head kvh (16 float4 per row; rows past
    // the capacity re-read the last) and the position are requested together, one
    // round trip.  Rows past the span's end are read but never used: their scores are
    // masked and the weighted sum stops at the span's end.
    // No early exit (the compiler would sink the loads below it): a workgroup past the
    // span, or of a position past the capacity, computes with a valid count and stores
    // nothing.
    const float4 qv = reinterpret_cast<const float4 *>(q + size_t(kvh) * kGroup * kHead)[t % (kGroup * kHead / 4)];
    constexpr int kPer = kChunk * (kHead / 4) / kThreads;  // 4 float4 of K and of V per thread
    float4 kr[kPer], vr[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t f = t + uint32_t(k) * kThreads, p = f / (kHead / 4), d4 = f % (kHead / 4);
        const size_t row = (size_t(min(chunk * kChunk + p, capacity - 1)) * kKvHeads + kvh) * kHead;
        kr[k] = reinterpret_cast<const float4 *>(k_cache + row)[d4];
        vr[k] = reinterpret_cast<const float4 *>(v_cache + row)[d4];
    }
    const uint32_t pos = uint32_t(*position);
    const Span sp = span_of(pos < capacity ? pos : 0u, layer_index);
    const bool live = pos < capacity && chunk * kChunk < sp.count;
    const uint32_t c0 = live ? chunk * kChunk : 0u;
    const uint32_t n = min(uint32_t(kChunk), sp.count - c0);
    qs[t] = qv;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t f = t + uint32_t(k) * kThreads, p = f / (kHead / 4), d4 = f % (kHead / 4);
        *reinterpret_cast<float4 *>(ks + p * kRowStride + 4 * d4) = kr[k];
        *reinterpret_cast<float4 *>(vs + p * kRowStride + 4 * d4) = vr[k];
    }
    __syncthreads();

    // scores: thread (p = t % 64, heads 2*(t/64), 2*(t/64)+1)
    {
        const uint32_t p = t % kChunk, g0 = 2 * (t / kChunk);
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int d = 0; d < kHead / 4; ++d) {
            const float4 kv = *reinterpret_cast<const float4 *>(ks + p * kRowStride + 4 * d);
            const float4 qa = qs[g0 * (kHead / 4) + d];
            const float4 qb = qs[(g0 + 1) * (kHead / 4) + d];
            a0 = fmaf(qa.x, kv.x, a0);
            a0 = fmaf(qa.y, kv.y, a0);
            a0 = fmaf(qa.z, kv.z, a0);
            a0 = fmaf(qa.w, kv.w, a0);
            a1 = fmaf(qb.x, kv.x, a1);
            a1 = fmaf(qb.y, kv.y, a1);
            a1 = fmaf(qb.z, kv.z, a1);
            a1 = fmaf(qb.w, kv.w, a1);
        }
        e[g0][p] = p < n ? a0 * 0.125f : -INFINITY;  // 1/sqrt(64), exact
        e[g0 + 1][p] = p < n ? a1 * 0.125f : -INFINITY;
    }
    __syncthreads();
    // per head: chunk max and exp sums (wave w handles heads 2w, 2w+1; lane = position)
    {
        const uint32_t w = t / 64, lane = t % 64;
        for (uint32_t g = 2 * w; g < 2 * w + 2; ++g) {
            const float s = e[g][lane];
            const float m = wave_max(s);
            const float x = lane < n ? expf(s - m) : 0.0f;
            const float l = wave_sum(x);
            e[g][lane] = x;
            if (lane == 0 && live) {
                ml_part[(size_t(kvh * kGroup + g)) * max_chunks + chunk] = make_float2(m, l);
            }
        }
    }
    __syncthreads();
    // o_c[g][d] = sum_p e[g][p] v[p][d]: thread (g = t/32, dims 2*(t%32), 2*(t%32)+1)
    {
        const uint32_t g = t / 32, d = 2 * (t % 32);
        float o0 = 0.0f, o1 = 0.0f;
        for (uint32_t p = 0; p < n; ++p) {
            const float2 v = *reinterpret_cast<const float2 *>(vs + p * kRowStride + d);
            const float x = e[g][p];
            o0 = fmaf(x, v.x, o0);
            o1 = fmaf(x, v.y, o1);
        }
        if (live) {
            float *dst = o_part + ((size_t(kvh * kGroup + g)) * max_chunks + chunk) * kHead + d;
            dst[0] = o0;
            dst[1] = o1;
        }
    }
}

// One workgroup per query head, one thread per dimension.  The chunk statistics
// are read once (a thread per chunk), the rescale factors shared through LDS.
constexpr int kMaxCombineChunks = 256;  // capacity up to 16384 positions

__global__ __launch_bounds__(kHead) void attn_combine_kernel(const float *__restrict__ o_part,
                                                             const float2 *__restrict__ ml_part,
                                                             const float *__restrict__ sinks,
                                                             const int32_t *__restrict__ position,
                                                             uint32_t capacity, uint32_t layer_index,
                                                             uint32_t max_chunks, float *__restrict__ out) {
    __shared__ float fs[kMaxCombineChunks];
    const uint32_t head = blockIdx.x, d = threadIdx.x;
    // The statistics and the first kEarly chunks' outputs are requested before the
    // position (the chunk count) is known: every address below max_chunks is inside
    // the partials, and chunks past the count are left out below by selection (their
    // stale contents never enter an arithmetic operation).
    constexpr int kPer = kMaxCombineChunks / kHead;
    float2 ml[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        ml[k] = ml_part[size_t(head) * max_chunks + min(d + uint32_t(k) * kHead, max_chunks - 1)];
    }
    constexpr int kEarly = 32;
    const float *op = o_part + size_t(head) * max_chunks * kHead + d;
    float early[kEarly];
#pragma unroll
    for (int c = 0; c < kEarly; ++c) {
        early[c] = op[size_t(min(uint32_t(c), max_chunks - 1)) * kHead];
    }
    __builtin_amdgcn_sched_barrier(0);  // all of them issued before the position is read
    const float sink = sinks[head];
    // no early exit (the compiler would sink the loads above below it): a position
    // past the capacity combines position 0's span and stores nothing
    const uint32_t pos = uint32_t(*position);
    const Span sp = span_of(pos < capacity ? pos : 0u, layer_index);
    const uint32_t chunks = (sp.count + kChunk - 1) / kChunk;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        if (d + uint32_t(k) * kHead >= chunks) {
            ml[k] = make_float2(-INFINITY, 0.0f);
        }
    }
    float m = sink;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        m = fmaxf(m, ml[k].x);
    }
    m = wave_max(m);
    float den = 0.0f;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t c = d + uint32_t(k) * kHead;
        const float f = c < chunks ? expf(ml[k].x - m) : 0.0f;
        den += ml[k].y * f;
        fs[c] = f;
    }
    den = wave_sum(den) + expf(sink - m);
    __syncthreads();
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < kEarly; ++c) {
        if (uint32_t(c) < chunks) {
            acc = fmaf(early[c], fs[c], acc);
        }
    }
#pragma unroll 8
    for (uint32_t c = kEarly; c < chunks; ++c) {
        acc = fmaf(op[size_t(c) * kHead], fs[c], acc);
    }
    if (pos < capacity) {
        out[head * kHead + d] = acc / den;
    }
}

// Sliding-window layers in one launch: workgroup = query head; the window (at most
// 128 positions of its kv head) sits in LDS, and the softmax with the sink is done
// in place -- no partials and no second kernel.  512 threads: each score is four
// 16-dimension partial dots added in LDS, each output dimension eight 16-position
// partial sums, so no thread's dependent chain is longer than 16 multiply-adds
// (5.54 -> 5.03 us per launch against 256 threads with 64- and 32-long chains).
constexpr int kWinThreads = 512;

__global__ __launch_bounds__(kWinThreads) void attn_window_kernel(const float *__restrict__ q,
                                                                  const float *__restrict__ k_cache,
                                                                  const float *__restrict__ v_cache,
                                                                  const float *__restrict__ sinks,
                                                                  const int32_t *__restrict__ position,
                                                                  uint32_t capacity, uint32_t layer_index,
                                                                  float *__restrict__ out) {
    __shared__ __attribute__((aligned(16))) float ks[kWindow * kRowStride];
    __shared__ __attribute__((aligned(16))) float vs[kWindow * kRowStride];
    __shared__ float4 qs[kWinThreads];  // thread t's copy of q float4 t % 16 (no branch)
    __shared__ float e[kWindow];
    __shared__ float sq[4][kWindow];
    __shared__ float stat[4];
    __shared__ float part[kWinThreads / kHead][kHead];
    // Workgroups are dealt to the 8 XCDs in turn (workgroup b to XCD b % 8), each XCD with
    // its own L2: workgroup b takes query head 8 (b % 8) + b / 8, so the 8 heads that read
    // one kv head's window run on one XCD and share its L2 (with head = b the window was
    // fetched once per XCD, 7.6 times its bytes).
    const uint32_t head = (blockIdx.x % kKvHeads) * kGroup + blockIdx.x / kKvHeads, kvh = head / kGroup;
    const uint32_t t = threadIdx.x;
    // q and the sink first (one of q's 16 float4 per thread), then the position, then the
    // window's K and V rows (positions past n re-read the last): two round trips
    const float4 qv = reinterpret_cast<const float4 *>(q + size_t(head) * kHead)[t % (kHead / 4)];
    const float sink = sinks[head];
    // no early exit (the compiler would sink the loads above below it): a position
    // past the capacity attends over position 0 and stores nothing
    const uint32_t pos = uint32_t(*position);
    const Span sp = span_of(pos < capacity ? pos : 0u, layer_index);
    const uint32_t n = sp.count;  // 1..128

    constexpr int kPer = kWindow * (kHead / 4) / kWinThreads;  // 4 float4 of K and of V per thread
    static_assert(kPer == 4, "the window of 128 positions over 512 threads");
    float4 kr[kPer], vr[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t f = t + uint32_t(k) * kWinThreads, p = f / (kHead / 4), d4 = f % (kHead / 4);
        const size_t row = (size_t(sp.first + (p < n ? p : n - 1)) * kKvHeads + kvh) * kHead;
        kr[k] = reinterpret_cast<const float4 *>(k_cache + row)[d4];
        vr[k] = reinterpret_cast<const float4 *>(v_cache + row)[d4];
    }
    qs[t] = qv;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t f = t + uint32_t(k) * kWinThreads, p = f / (kHead / 4), d4 = f % (kHead / 4);
        *reinterpret_cast<float4 *>(ks + p * kRowStride + 4 * d4) = kr[k];
        *reinterpret_cast<float4 *>(vs + p * kRowStride + 4 * d4) = vr[k];
    }
    __syncthreads();

    // scores: thread (position t % 128, dims 16 (t / 128) .. + 15), the quarters added in LDS
    const uint32_t w = t / 64, lane = t % 64;
    {
        const uint32_t p = t % kWindow, qd = t / kWindow;
        float a = 0.0f;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const float4 kv = *reinterpret_cast<const float4 *>(ks + p * kRowStride + 16 * qd + 4 * d);
            const float4 qq = qs[4 * qd + d];
            a = fmaf(qq.x, kv.x, a);
            a = fmaf(qq.y, kv.y, a);
            a = fmaf(qq.z, kv.z, a);
            a = fmaf(qq.w, kv.w, a);
        }
        sq[qd][p] = a;
    }
    __syncthreads();
    if (t < uint32_t(kWindow)) {
        const float a = ((sq[0][t] + sq[1][t]) + sq[2][t]) + sq[3][t];
        const float s = t < n ? a * 0.125f : -INFINITY;  // 1/sqrt(64), exact
        e[t] = s;
        const float m = wave_max(s);
        if (lane == 0) {
            stat[w] = m;
        }
    }
    __syncthreads();
    // model.cpp:270-281: the sink enters the max and the denominator only
    const float m = fmaxf(sink, fmaxf(stat[0], stat[1]));
    if (t < uint32_t(kWindow)) {
        const float x = t < n ? expf(e[t] - m) : 0.0f;
        e[t] = x;
        const float l = wave_sum(x);
        if (lane == 0) {
            stat[2 + w] = l;
        }
    }
    __syncthreads();
    const float den = expf(sink - m) + (stat[2] + stat[3]);
    // o[d] = sum_p e[p] v[p][d]: thread (eighth g = t / 64 of the positions, dim d)
    {
        const uint32_t g = t / kHead, d = t % kHead;
        float o = 0.0f;
        const uint32_t p0 = g * (kWindow / 8), p1 = min(p0 + kWindow / 8, n);
        for (uint32_t p = p0; p < p1; ++p) {
            o = fmaf(e[p], vs[p * kRowStride + d], o);
        }
        part[g][d] = o;
    }
    __syncthreads();
    if (t < uint32_t(kHead) && pos < capacity) {
        const float o = (((part[0][t] + part[1][t]) + (part[2][t] + part[3][t])) +
                         ((part[4][t] + part[5][t]) + (part[6][t] + part[7][t])));
        out[head * kHead + t] = o / den;
    }
}

// Prefill: attention of a run of tokens on bf16 MFMA, every f32 operand as three bf16
// planes.  One workgroup per (kv head, 16 consecutive tokens): the 8 query heads of the
// group times 16 tokens are 128 queries, in tiles of 16, two tiles per wave of a group of
// four waves.  Two such groups share the workgroup and take the chunks of 64 positions in
// turn (group 0 the first, third, ..., group 1 the others), each with an online softmax
// of its own.  Per chunk and query tile:
//  - S^T (positions x queries) = K Q^T, then an online softmax per query (a column of S^T:
//    the lane's 4 rows of each position tile and the 4 lanes of its column): m' = max(m,
//    scores), and l and O are rescaled by exp(m - m');
//  - O^T (dims x queries) += V^T P^T.
// At the end group 0 merges the two states and the sink, which takes part in the maximum
// and the denominator (model.cpp:270-281).  The output is O / l.
//
// v_mfma_f32_16x16x32_bf16 (D = A B + C): lane (n, g) = (l % 16, l / 16) holds 8 bf16 of
// A row n and of B column n for 8 of the 32 K indices, the same for A and B, and receives
// D rows 4g..4g+3 of column n.  In the first product lane group g takes dims 8g..8g+7 of
// each half of the head.  In the second, K step h covers position tiles 2h and 2h + 1, and
// lane group g takes positions 16 (2h) + 4g + i and 16 (2h + 1) + 4g + i, i = 0..3: the
// rows of the lane's own S^T tiles, so the probabilities never leave their registers; V is
// staged transposed, with the positions of a dim in that order.
//
// Numerics: x = x0 + x1 + x2, each plane the remainder rounded to bf16, holds every f32 of
// 2^-100 or more to its last bit or 2^-25 of it; the products x0 y0, x0 y1, x1 y0, x1 y1, x0 y2, x2 y0 are
// exact in f32 and the three left out are at most 2^-24 of |x y|, as much as f32 rounds
// the product itself.  Relative error against 64 bits, 512 tokens at 1536 (a sliding and a
// full layer): 3.9e-7 on f32 MFMA, 2.4e-7 this way.  The planes assume magnitudes whose
// sums stay finite: a chunk with a K of 2^60 or more, a V of 2^100 or more, an infinity or
// a NaN, and every chunk of a block with such a query, takes f32 MFMA (attn_chunk_f32).  So
// does a chunk with V that the planes run out of exponent for: eight V of one dim and parity
// of position below 2^-100 and not all zero.  (Of a smaller value among larger ones they
// hold 2^-134, of a probability the same: 2^-34 of the largest.  Small queries and keys
// need no more: their scores are next to zero.)
//
// What bounds it: on v_mfma_f32_16x16x4_f32 a chunk's two products of a wave take 256
// instructions of 32 cycles; six bf16 products take 192 of 16, and the second group puts a
// second wave on each SIMD, whose softmax and splitting partly overlap the other's MFMAs.
// Of the cycles of a full layer at 1536 the matrix cores are busy 46% and the VALU (splits,
// softmax, addresses) 45%, of a sliding layer's 24% and 40%.  512 tokens at 1536: 237 us for a
// sliding and a full layer on f32 MFMA with one group, 112 us now (on the way: planes 134,
// scores in units of log 2 125, LDS in fragment order and a barrier per group 113).
constexpr int kPfTokens = 16;
constexpr int kPfQueries = kPfTokens * kGroup;                   // 128
constexpr int kPfGroups = 2;                                     // groups of four waves
constexpr int kPfGroupThreads = 256;
constexpr int kPfThreads = kPfGroups * kPfGroupThreads;
constexpr int kPfTiles = kPfQueries / 16 / (kPfGroupThreads / 64);  // query tiles per wave: 2
constexpr int kPfPlanes = 3;
constexpr int kPfPlane = kChunk * kHead;  // bf16 of one staged plane, in fragment order [fragment][lane][8]

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ inline mf::f32x4 mfma_f32(float a, float b, const mf::f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Two f32 as three planes of two packed bf16 each (the first value in the low half).
__device__ __attribute__((always_inline)) inline void split3(float a, float b, uint32_t (&out)[kPfPlanes]) {
#pragma unroll
    for (int p = 0; p < kPfPlanes; ++p) {
        const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, mf::bf16x2));
        out[p] = w;
        a -= __uint_as_float(w << 16);
        b -= __uint_as_float(w & 0xffff0000u);
    }
}

// The planes of (a, b) x log2(e) / 8, the product carried past f32 into the last plane.
__device__ __attribute__((always_inline)) inline void split3_scaled(float a, float b, uint32_t (&out)[kPfPlanes]) {
#pragma clang fp contract(off)  // ah and bh are the rounded products
    constexpr float c = 0x1.715476p-3f, c_lo = 0x1.4ae0cp-29f;
    const float ah = a * c, bh = b * c;
    const float al = fmaf(a, c_lo, fmaf(a, c, -ah)), bl = fmaf(b, c_lo, fmaf(b, c, -bh));
    float ra = ah, rb = bh;
#pragma unroll
    for (int p = 0; p < kPfPlanes; ++p) {
        const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{ra, rb}, mf::bf16x2));
        out[p] = w;
        ra -= __uint_as_float(w << 16);
        rb -= __uint_as_float(w & 0xffff0000u);
        if (p == kPfPlanes - 2) {
            ra += al;
            rb += bl;
        }
    }
}

// The larger magnitudes of two packed pairs of bf16 (as bit patterns, so infinities and
// NaNs are the largest), and whether one of a pair, or each, is 2^E or more.
__device__ inline uint32_t pair_max(uint32_t acc, uint32_t w) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, acc),
                                                                  __builtin_bit_cast(u16x2, w & 0x7fff7fffu)));
}
template <int E>
__device__ inline bool at_least(uint32_t pair) {
    constexpr uint32_t bits = uint32_t(E + 127) << 7;
    return (pair & 0xffffu) >= bits || (pair >> 16) >= bits;
}
template <int E>
__device__ inline bool both_at_least(uint32_t pair) {
    constexpr uint32_t bits = uint32_t(E + 127) << 7;
    return (pair & 0xffffu) >= bits && (pair >> 16) >= bits;
}
constexpr int kPfKMax = 60, kPfVMax = 100;  // and 2^60 for the queries
constexpr int kPfVMin = -100;

// Scores and their maxima are kept in units of log 2 (times log2 e), so a probability is
// one v_exp_f32 (1 ulp); the factor goes into the queries, carried past f32.
constexpr float kLog2e = 0x1.715476p+0f, kLog2eLo = 0x1.4ae0cp-26f;  // log2 e = their sum

// A sink in units of log 2, as a value and what f32 rounds off it (of sinks small enough that
// it says something).  Scores are an f32 dot product / 8 and stay finite in these units; a
// sink of 2^127 may not, and the largest f32 outweighs every finite score as it does.
__device__ inline float sink_log2(float sink, float &lo) {
#pragma clang fp contract(off)
    const float hi = sink * kLog2e;
    lo = fabsf(sink) < 0x1p14f ? fmaf(sink, kLog2eLo, fmaf(sink, kLog2e, -hi)) : 0.0f;
    return isinf(hi) && !isinf(sink) ? copysignf(0x1.fffffep+127f, sink) : hi;
}

// The online softmax state of a wave's queries.
struct PfState {
    float m[kPfTiles], l[kPfTiles];
    mf::f32x4 o[kPfTiles][4];  // O^T tiles: dims 16M + 4g + i of the query
};

// The running maximum and rescaling of one query tile for a chunk whose largest score of
// the lane is cmax; returns what to subtract from the chunk's scores: the maximum, or zero
// while every score was masked (-infinity, whose exp2 is zero).
__device__ __attribute__((always_inline)) inline float pf_rescale(PfState &st, int qi, float cmax) {
    cmax = fmaxf(cmax, __shfl_xor(cmax, 16));
    cmax = fmaxf(cmax, __shfl_xor(cmax, 32));
    const float m2 = fmaxf(st.m[qi], cmax);
    const float base = m2 == -INFINITY ? 0.0f : m2;
    const float scale = __builtin_amdgcn_exp2f(st.m[qi] - base);
    st.l[qi] *= scale;
    st.m[qi] = m2;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            st.o[qi][mt][i] *= scale;
        }
    }
    return base;
}

// One chunk on f32 MFMA, operands straight from global memory: K step (s, j) of the scores
// covers dims 16s + 4k + j for lane group k; K step j of position tile p of the second
// product takes positions 16p + 4k + j.  A query's probabilities are zero outside its span,
// but zero times an infinite V is not: the second product runs once for each of the tile's
// two tokens, with that token's span of V rows, and a query keeps its own token's sums.
struct PfQueries {
    uint32_t row[kPfTiles], first[kPfTiles], pos[kPfTiles];
};
__device__ __attribute__((noinline)) void attn_chunk_f32(const float *q, const float *k_cache, const float *v_cache,
                                                         uint32_t kvh, uint32_t c0, uint32_t hi, const PfQueries &qs,
                                                         uint32_t n, uint32_t g, PfState &st) {
#pragma clang fp contract(off)  // s x log2 e rounded alike in the maximum and in the distance to it
    using mf::f32x4;
#pragma unroll 1
    for (int qi = 0; qi < kPfTiles; ++qi) {
        const float *qr = q + size_t(qs.row[qi]) * kHead;
        f32x4 sc[4];
        float cmax = -INFINITY;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            sc[p] = f32x4{0.f, 0.f, 0.f, 0.f};
            const size_t row = (size_t(min(c0 + 16 * p + n, hi)) * kKvHeads + kvh) * kHead;
            for (int s4 = 0; s4 < 4; ++s4) {
                const float4 a = *reinterpret_cast<const float4 *>(k_cache + row + 16 * s4 + 4 * g);
                const float4 b = *reinterpret_cast<const float4 *>(qr + 16 * s4 + 4 * g);
                sc[p] = mfma_f32(a.x, b.x, sc[p]);
                sc[p] = mfma_f32(a.y, b.y, sc[p]);
                sc[p] = mfma_f32(a.z, b.z, sc[p]);
                sc[p] = mfma_f32(a.w, b.w, sc[p]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t at = c0 + 16 * p + 4 * g + i;
                const float s = at >= qs.first[qi] && at <= qs.pos[qi] ? sc[p][i] * 0.125f : -INFINITY;
                sc[p][i] = s;
                cmax = fmaxf(cmax, s * kLog2e);
            }
        }
        const float m2 = pf_rescale(st, qi, cmax);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float s = sc[p][i];
                // the product's low part, for scores small enough that it says something
                const float hi2 = s * kLog2e, lo2 = fmaf(s, kLog2eLo, fmaf(s, kLog2e, -hi2));
                const float x = (hi2 - m2) + (fabsf(s) < 0x1p14f ? lo2 : 0.0f);
                sc[p][i] = s == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(x);
                st.l[qi] += sc[p][i];
            }
        }
        static_assert(kGroup == 8, "a tile's queries are two tokens' 8 heads");
        // (the tile's token u: query columns 8u..8u+7)
        const uint32_t first0 = __shfl(qs.first[qi], 0), pos0 = __shfl(qs.pos[qi], 0);
        const uint32_t first1 = __shfl(qs.first[qi], 8), pos1 = __shfl(qs.pos[qi], 8);
#pragma unroll 1
        for (int mt = 0; mt < 4; ++mt) {
            f32x4 o0 = st.o[qi][mt], o1 = o0;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t at = c0 + 16 * p + 4 * g + j;
                    const float v = v_cache[(size_t(min(at, hi)) * kKvHeads + kvh) * kHead + 16 * mt + n];
                    o0 = mfma_f32(at >= first0 && at <= pos0 ? v : 0.0f, sc[p][j], o0);
                    o1 = mfma_f32(at >= first1 && at <= pos1 ? v : 0.0f, sc[p][j], o1);
                }
            }
            st.o[qi][mt] = n < 8 ? o0 : o1;
        }
    }
}

// A barrier of one group's four waves (every wave of the group arrives, each time): a count
// in LDS that only grows, `target` its value once all have arrived.  LDS operations of a
// wave are done in order, so an arrival follows the wave's earlier LDS accesses.  With
// s_barrier the two groups ran in step, both on the matrix cores and then both on the VALU.
__device__ __attribute__((always_inline)) inline void group_sync(uint32_t *count, uint32_t target, uint32_t lane) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (lane == 0) {
        __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    while (uint32_t(__builtin_amdgcn_readfirstlane(
               __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))) < target) {
    }
    asm volatile("" ::: "memory");
}

__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2))) void attn_prefill_kernel(
    const float *__restrict__ q, const float *__restrict__ k_cache, const float *__restrict__ v_cache,
    const float *__restrict__ sinks, uint32_t first, uint32_t tokens, uint32_t layer_index,
    float *__restrict__ out) {
    using mf::bf16x8;
    using mf::f32x4;
    // per group: K planes in fragments (position tile, half of the head), V planes in
    // fragments (dim tile, K step)
    __shared__ __attribute__((aligned(16))) uint16_t kv[kPfGroups][2][kPfPlanes][kPfPlane];
    __shared__ uint32_t odd[kPfGroups][2];  // a chunk for the f32 path, by iteration parity
    __shared__ uint32_t odd_query;
    __shared__ uint32_t arrived[kPfGroups];
    const uint32_t t = threadIdx.x % kPfGroupThreads, grp = threadIdx.x / kPfGroupThreads;
    const uint32_t wave = t / 64, lane = t % 64, n = lane % 16, g = lane / 16;
    const uint32_t kvh = blockIdx.y, block0 = blockIdx.x * kPfTokens;
    const uint32_t last_local = min(block0 + kPfTokens, tokens) - 1;
    // the block's positions: from the first token's span start to the last token
    const uint32_t lo = span_of(first + block0, layer_index).first;
    const uint32_t hi = first + last_local;
    const uint32_t start = lo - lo % kChunk;
    const uint32_t chunks = (hi - start) / kChunk + 1;
    const uint32_t rounds = (chunks + kPfGroups - 1 - grp) / kPfGroups;  // this group's chunks

    // staging, so that the LDS stores spread over the banks as the fragment reads do: of K,
    // position n of each tile and dims 4 dq..+3; of V, dim `lane` of the wave's position tile
    const uint32_t dq = 4 * wave + g;
    float4 kr[4];
    float vr[16];
    auto request = [&](uint32_t round) __attribute__((always_inline)) {
        // positions past the block's last re-read it
        const uint32_t c0 = start + (round * kPfGroups + grp) * kChunk;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t kp = min(c0 + 16 * k + n, hi);
            kr[k] = *reinterpret_cast<const float4 *>(k_cache + (size_t(kp) * kKvHeads + kvh) * kHead + 4 * dq);
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const uint32_t vp = min(c0 + 16 * wave + k, hi);
            vr[k] = v_cache[(size_t(vp) * kKvHeads + kvh) * kHead + lane];
        }
    };
    request(0);

    // this lane's query (column n) of each of the wave's tiles, as B fragments of K step s
    uint32_t qp[kPfTiles][2][kPfPlanes][4];
    uint32_t qpos[kPfTiles], qfirst[kPfTiles], qrow[kPfTiles];
    float sink[kPfTiles];
    bool live[kPfTiles];
    PfState st;
    uint32_t bad_query = 0;
#pragma unroll
    for (int qi = 0; qi < kPfTiles; ++qi) {
        const uint32_t query = (wave * kPfTiles + qi) * 16 + n;
        const uint32_t local = block0 + query / kGroup, head = kvh * kGroup + query % kGroup;
        live[qi] = local < tokens;
        const uint32_t lc = min(local, last_local);  // past the last token: a stand-in, not written
        qpos[qi] = first + lc;
        qfirst[qi] = span_of(qpos[qi], layer_index).first;
        qrow[qi] = lc * kQHeads + head;
        const float4 *q4 = reinterpret_cast<const float4 *>(q + size_t(qrow[qi]) * kHead);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const float4 a = q4[8 * s + 2 * g], b = q4[8 * s + 2 * g + 1];
            const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t w[kPfPlanes];
                split3_scaled(v[2 * e], v[2 * e + 1], w);
                bad_query = pair_max(bad_query, w[0]);
#pragma unroll
                for (int p = 0; p < kPfPlanes; ++p) {
                    qp[qi][s][p][e] = w[p];
                }
            }
        }
        sink[qi] = sinks[head];
        st.m[qi] = -INFINITY;
        st.l[qi] = 0.0f;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            st.o[qi][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (threadIdx.x < 2 * kPfGroups) {
        (&odd[0][0])[threadIdx.x] = 0;
    }
    if (threadIdx.x < kPfGroups) {
        arrived[threadIdx.x] = 0;
    }
    if (threadIdx.x == 0) {
        odd_query = 0;
    }
    __syncthreads();
    if (at_least<kPfKMax>(bad_query)) {
        odd_query = 1;
    }
    __syncthreads();

    uint16_t *const ks = kv[grp][0][0], *const vs = kv[grp][1][0];
    const auto frag = [&](const uint16_t *base, int plane, int f) __attribute__((always_inline)) {
        return *reinterpret_cast<const bf16x8 *>(base + plane * kPfPlane + f * 512 + lane * 8);
    };
    const auto q_frag = [&](int qi, int s, int p) __attribute__((always_inline)) {
        return __builtin_bit_cast(bf16x8, mf::u32x4{qp[qi][s][p][0], qp[qi][s][p][1], qp[qi][s][p][2], qp[qi][s][p][3]});
    };
    // the six products, smallest first: planes (A, B)
    constexpr int kProducts = 6;
    constexpr int pa[kProducts] = {1, 2, 0, 1, 0, 0}, pb[kProducts] = {1, 0, 2, 0, 1, 0};

#pragma unroll 1
    for (uint32_t round = 0; round < rounds; ++round) {
        const uint32_t c0 = start + (round * kPfGroups + grp) * kChunk;
        group_sync(&arrived[grp], 8 * round + 4, lane);  // the previous chunk's reads are done
        {
            uint32_t bad_k = 0, bad_v = 0;
            // K: dims 4 dq..+3 are half dq % 2 of lane group (dq % 8) / 2 in fragment (tile, dq / 8)
            uint16_t *const kd = ks + (dq / 8) * 512 + (((dq % 8) / 2) * 16 + n) * 8 + (dq % 2) * 4;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t w0[kPfPlanes], w1[kPfPlanes];
                split3(kr[k].x, kr[k].y, w0);
                split3(kr[k].z, kr[k].w, w1);
                bad_k = pair_max(pair_max(bad_k, w0[0]), w1[0]);
#pragma unroll
                for (int p = 0; p < kPfPlanes; ++p) {
                    *reinterpret_cast<u32x2 *>(kd + p * kPfPlane + k * 1024) = u32x2{w0[p], w1[p]};
                }
            }
            // V: positions 4k..4k+3 of position tile `wave` are half wave % 2 of lane group k
            // in fragment (dim tile, wave / 2)
            uint16_t *const vd = vs + ((lane / 16) * 2 + wave / 2) * 512 + n * 8 + (wave % 2) * 4;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t w0[kPfPlanes], w1[kPfPlanes];
                split3(vr[4 * k], vr[4 * k + 1], w0);
                split3(vr[4 * k + 2], vr[4 * k + 3], w1);
                bad_v = pair_max(pair_max(bad_v, w0[0]), w1[0]);
#pragma unroll
                for (int p = 0; p < kPfPlanes; ++p) {
                    *reinterpret_cast<u32x2 *>(vd + p * kPfPlane + k * 128) = u32x2{w0[p], w1[p]};
                }
            }
            bool off = at_least<kPfKMax>(bad_k) || at_least<kPfVMax>(bad_v);
            if (!both_at_least<kPfVMin>(bad_v)) {  // the thread's V of a parity all small: zeros, or not?
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    off |= vr[k] != 0.0f && fabsf(vr[k]) < __builtin_ldexpf(1.0f, kPfVMin);
                }
            }
            if (off) {
                odd[grp][round % 2] = 1;
            }
        }
        group_sync(&arrived[grp], 8 * round + 8, lane);
        if (round + 1 < rounds) {
            request(round + 1);
        }
        const bool f32_chunk = (odd[grp][round % 2] | odd_query) != 0;
        if (t == 0) {
            odd[grp][(round + 1) % 2] = 0;  // set again only after the next two arrivals of this wave
        }
        if (f32_chunk) {
            // (copies: the state itself stays in registers)
            PfState s2 = st;
            const PfQueries qs = {{qrow[0], qrow[1]}, {qfirst[0], qfirst[1]}, {qpos[0], qpos[1]}};
            attn_chunk_f32(q, k_cache, v_cache, kvh, c0, hi, qs, n, g, s2);
            st = s2;
            // wait for the copies here: left to their first use, in the next chunk, the
            // compiler waited there for the K and V requests ahead of it, on every path
#pragma unroll
            for (int qi = 0; qi < kPfTiles; ++qi) {
                asm volatile("" : "+v"(st.m[qi]), "+v"(st.l[qi]), "+v"(st.o[qi][0]), "+v"(st.o[qi][1]),
                             "+v"(st.o[qi][2]), "+v"(st.o[qi][3]));
            }
            continue;
        }

        // S^T: [query tile][position tile], lane rows 4g..4g+3 = positions 16p + 4g + i
        f32x4 sc[kPfTiles][4];
#pragma unroll
        for (int p2 = 0; p2 < 4; p2 += 2) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                bf16x8 a[2][kPfPlanes];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
#pragma unroll
                    for (int p = 0; p < kPfPlanes; ++p) {
                        a[u][p] = frag(ks, p, 2 * (p2 + u) + s);
                    }
                }
#pragma unroll
                for (int x = 0; x < kProducts; ++x) {
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
#pragma unroll
                        for (int qi = 0; qi < kPfTiles; ++qi) {
                            sc[qi][p2 + u] = mf::mfma(a[u][pa[x]], q_frag(qi, s, pb[x]),
                                                      s == 0 && x == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sc[qi][p2 + u]);
                        }
                    }
                }
            }
        }
        // mask, online softmax; sc becomes P^T
        const bool whole = c0 + kChunk - 1 <= first + block0 && c0 >= span_of(hi, layer_index).first;
#pragma unroll
        for (int qi = 0; qi < kPfTiles; ++qi) {
            if (!whole) {  // (uniform) some position is outside some query's span
#pragma unroll
                for (int p = 0; p < 4; ++p) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t at = c0 + 16 * p + 4 * g + i;
                        sc[qi][p][i] = at >= qfirst[qi] && at <= qpos[qi] ? sc[qi][p][i] : -INFINITY;
                    }
                }
            }
            float cmax = sc[qi][0][0];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    cmax = fmaxf(cmax, sc[qi][p][i]);
                }
            }
            const float m2 = pf_rescale(st, qi, cmax);
            float lsum = 0.0f;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float x = __builtin_amdgcn_exp2f(sc[qi][p][i] - m2);
                    sc[qi][p][i] = x;
                    lsum += x;
                }
            }
            st.l[qi] += lsum;
        }
        // O^T += V^T P^T
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            mf::u32x4 pp[kPfTiles][kPfPlanes];
#pragma unroll
            for (int qi = 0; qi < kPfTiles; ++qi) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t w[kPfPlanes];
                    split3(sc[qi][2 * h + e / 2][2 * (e % 2)], sc[qi][2 * h + e / 2][2 * (e % 2) + 1], w);
#pragma unroll
                    for (int p = 0; p < kPfPlanes; ++p) {
                        pp[qi][p][e] = w[p];
                    }
                }
            }
#pragma unroll
            for (int m2 = 0; m2 < 4; m2 += 2) {
                bf16x8 a[2][kPfPlanes];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
#pragma unroll
                    for (int p = 0; p < kPfPlanes; ++p) {
                        a[u][p] = frag(vs, p, 2 * (m2 + u) + h);
                    }
                }
#pragma unroll
                for (int x = 0; x < kProducts; ++x) {
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
#pragma unroll
                        for (int qi = 0; qi < kPfTiles; ++qi) {
                            st.o[qi][m2 + u] = mf::mfma(a[u][pa[x]], mf::as_bf16x8v(pp[qi][pb[x]]), st.o[qi][m2 + u]);
                        }
                    }
                }
            }
        }
    }

    // group 1 hands its state to group 0's wave of the same queries through LDS
    constexpr int kState = 18;  // per lane and query tile: m, l and 16 of O
    float *const hand = reinterpret_cast<float *>(&kv[0][0][0][0]) + size_t(wave) * kPfTiles * kState * 64 + lane;
    static_assert(sizeof(float) * 4 * kPfTiles * kState * 64 <= sizeof(kv), "the handed state fits the staged planes");
    __syncthreads();
    if (grp == 1) {
#pragma unroll
        for (int qi = 0; qi < kPfTiles; ++qi) {
            float *d = hand + qi * kState * 64;
            d[0] = st.m[qi];
            d[64] = st.l[qi];
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    d[(2 + 4 * mt + i) * 64] = st.o[qi][mt][i];
                }
            }
        }
    }
    __syncthreads();
    if (grp == 1) {
        return;
    }
#pragma unroll
    for (int qi = 0; qi < kPfTiles; ++qi) {
        const float *d = hand + qi * kState * 64;
        const float m1 = d[0];
        float sink_lo;
        const float sink_hi = sink_log2(sink[qi], sink_lo);
        const float m = fmaxf(fmaxf(st.m[qi], m1), sink_hi);
        const float w0 = __builtin_amdgcn_exp2f(st.m[qi] - m), w1 = __builtin_amdgcn_exp2f(m1 - m);
        float den = st.l[qi] * w0 + d[64] * w1;
        den += __shfl_xor(den, 16);
        den += __shfl_xor(den, 32);
        den += __builtin_amdgcn_exp2f((sink_hi - m) + sink_lo);
        if (live[qi]) {
            float *dst = out + size_t(qrow[qi]) * kHead;
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = (st.o[qi][mt][i] * w0 + d[(2 + 4 * mt + i) * 64] * w1) / den;
                }
                *reinterpret_cast<float4 *>(dst + 16 * mt + 4 * g) = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
    }
}

}  // namespace

namespace ttl {
// Workspace floats needed by ttl_attention_decode for a given capacity.
size_t attention_partials_floats(uint32_t capacity) {
    const size_t chunks = (capacity + kChunk - 1) / kChunk;
    return size_t(kQHeads) * chunks * (kHead + 2);
}
}  // namespace ttl

namespace {

// Attention of the token at *position; max_chunks = the chunks the partials of
// one token hold (at least those of its span).
void launch_attention(ttl_ctx *ctx, const float *q, const float *k_cache, const float *v_cache, const float *sinks,
                      const int32_t *position, uint32_t capacity, uint32_t layer_index, uint32_t max_chunks,
                      float *workspace, float *out) {
    if (layer_index % 2 == 0) {
        // the sliding window fits one workgroup per query head
        attn_window_kernel<<<kQHeads, kWinThreads, 0, ctx->stream>>>(q, k_cache, v_cache, sinks, position, capacity,
                                                                     layer_index, out);
        return;
    }
    float *o_part = workspace;
    float2 *ml_part = reinterpret_cast<float2 *>(workspace + size_t(kQHeads) * max_chunks * kHead);
    attn_partial_kernel<<<dim3(max_chunks, kKvHeads), kThreads, 0, ctx->stream>>>(
        q, k_cache, v_cache, position, capacity, layer_index, max_chunks, o_part, ml_part);
    attn_combine_kernel<<<kQHeads, kHead, 0, ctx->stream>>>(o_part, ml_part, sinks, position, capacity, layer_index,
                                                            max_chunks, out);
}


// ---- ttl_attention_decode_noalloc: the partials in a static device array ------------
//
// For callers that cannot allocate (graph capture, serving loops): one array per GPU,
// sized for the largest capacity the kernels take (kMaxCombineChunks chunks of 64
// positions, 16384 positions: 64 x 256 x 66 floats = 4,325,376 bytes), which each GPU
// the library runs on holds until the process ends.  Host code never passes the
// array's name to a kernel: its device address is looked up once per device, with that
// device current, when a context opens (ttl::attention_scratch_init, from ttl_create).
constexpr size_t kScratchFloats = size_t(kQHeads) * kMaxCombineChunks * (kHead + 2);
static __device__ __align__(256) float scratch[kScratchFloats];

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mutex;
float *g_scratch_ptr[kMaxScratchDevices] = {};

float *scratch_for(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    return device >= 0 && device < kMaxScratchDevices ? g_scratch_ptr[device] : nullptr;
}

}  // namespace

namespace ttl {
int attention_scratch_init(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    TTL_REQUIRE(device >= 0 && device < kMaxScratchDevices, TTL_ERR_NO_DEVICE,
                "ttl_create: device ordinal %d above %d", device, kMaxScratchDevices - 1);
    if (g_scratch_ptr[device]) {
        return TTL_OK;
    }
    void *ptr = nullptr;
    TTL_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_scratch_ptr[device] = static_cast<float *>(ptr);
    return TTL_OK;
}
}  // namespace ttl

extern "C" {

size_t ttl_attention_workspace_bytes(uint32_t capacity) {
    return ttl::attention_partials_floats(capacity) * sizeof(float);
}

int ttl_attention_decode(ttl_ctx *ctx, const float *q_dev, const float *k_cache_dev, const float *v_cache_dev,
                         const float *sinks_dev, const int32_t *position_dev, uint32_t capacity, uint32_t layer_index,
                         float *workspace_dev, float *out_dev) {
    TTL_REQUIRE(ctx && q_dev && k_cache_dev && v_cache_dev && sinks_dev && position_dev && workspace_dev && out_dev,
                TTL_ERR_INVALID, "ttl_attention_decode: null argument");
    TTL_REQUIRE(capacity > 0 && capacity <= uint32_t(kMaxCombineChunks * kChunk), TTL_ERR_SHAPE,
                "ttl_attention_decode: capacity must be 1..%d", kMaxCombineChunks * kChunk);
    TTL_REQUIRE(((uintptr_t)q_dev & 15) == 0 && ((uintptr_t)k_cache_dev & 15) == 0 && ((uintptr_t)v_cache_dev & 15) == 0,
                TTL_ERR_INVALID, "ttl_attention_decode: q, k and v must be 16-byte aligned");
    launch_attention(ctx, q_dev, k_cache_dev, v_cache_dev, sinks_dev, position_dev, capacity, layer_index,
                     (capacity + kChunk - 1) / kChunk, workspace_dev, out_dev);
    TTL_LAUNCHED("attention kernels");
    return TTL_OK;
}


int ttl_attention_decode_noalloc(ttl_ctx *ctx, const float *q_dev, const float *k_cache_dev,
                                 const float *v_cache_dev, const float *sinks_dev, const int32_t *position_dev,
                                 uint32_t capacity, uint32_t layer_index, float *out_dev) {
    TTL_REQUIRE(ctx && q_dev && k_cache_dev && v_cache_dev && sinks_dev && position_dev && out_dev, TTL_ERR_INVALID,
                "ttl_attention_decode_noalloc: null argument");
    TTL_REQUIRE(capacity > 0 && capacity <= uint32_t(kMaxCombineChunks * kChunk), TTL_ERR_SHAPE,
                "ttl_attention_decode_noalloc: capacity must be 1..%d (the static partials hold %zu bytes)",
                kMaxCombineChunks * kChunk, kScratchFloats * sizeof(float));
    TTL_REQUIRE(((uintptr_t)q_dev & 15) == 0 && ((uintptr_t)k_cache_dev & 15) == 0 && ((uintptr_t)v_cache_dev & 15) == 0,
                TTL_ERR_INVALID, "ttl_attention_decode_noalloc: q, k and v must be 16-byte aligned");
    float *partials = scratch_for(ctx->device);
    TTL_REQUIRE(partials, TTL_ERR_INVALID, "ttl_attention_decode_noalloc: no static partials on device %d",
                ctx->device);
    const uint32_t chunks = (capacity + kChunk - 1) / kChunk;
    TTL_REQUIRE(ttl::attention_partials_floats(capacity) <= kScratchFloats, TTL_ERR_SHAPE,
                "ttl_attention_decode_noalloc: %u chunks exceed the static partials", chunks);
    launch_attention(ctx, q_dev, k_cache_dev, v_cache_dev, sinks_dev, position_dev, capacity, layer_index, chunks,
                     partials, out_dev);
    TTL_LAUNCHED("attention kernels");
    return TTL_OK;
}

int ttl_attention_prefill(ttl_ctx *ctx, const float *q_dev, const float *k_cache_dev, const float *v_cache_dev,
                          const float *sinks_dev, uint32_t first_position, uint32_t tokens, uint32_t capacity,
                          uint32_t layer_index, float *out_dev) {
    TTL_REQUIRE(ctx && q_dev && k_cache_dev && v_cache_dev && sinks_dev && out_dev, TTL_ERR_INVALID,
                "ttl_attention_prefill: null argument");
    TTL_REQUIRE(capacity > 0 && capacity <= uint32_t(kMaxCombineChunks * kChunk), TTL_ERR_SHAPE,
                "ttl_attention_prefill: capacity must be 1..%d", kMaxCombineChunks * kChunk);
    TTL_REQUIRE(tokens > 0 && tokens <= 65535 && size_t(first_position) + tokens <= capacity, TTL_ERR_SHAPE,
                "ttl_attention_prefill: positions %u..%u do not fit the capacity %u", first_position,
                first_position + tokens - 1, capacity);
    TTL_REQUIRE(((uintptr_t)q_dev & 15) == 0 && ((uintptr_t)k_cache_dev & 15) == 0 && ((uintptr_t)v_cache_dev & 15) == 0,
                TTL_ERR_INVALID, "ttl_attention_prefill: q, k and v must be 16-byte aligned");
    attn_prefill_kernel<<<dim3((tokens + kPfTokens - 1) / kPfTokens, kKvHeads), kPfThreads, 0, ctx->stream>>>(
        q_dev, k_cache_dev, v_cache_dev, sinks_dev, first_position, tokens, layer_index, out_dev);
    TTL_LAUNCHED("attn_prefill_kernel");
    return TTL_OK;
}

}  // extern "C"
