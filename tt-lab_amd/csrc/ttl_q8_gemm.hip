// Batched Q8_0 matmul on MFMA: matmul_add_q8_0 (tensor.cpp:529-566) for a batch of
// tokens, as GptOssModel::prefill runs the attention projections (model.cpp:493-498,
// 519-520).
//
// Operands of v_mfma_f32_16x16x32_f16 (D = A B + C; lane l holds 8 f16 of A row
// l%16 and of B column l%16 for the K offsets of lane group g = l/16, and receives D
// rows 4g..4g+3 of column l%16):
//  - one K step is one Q8_0 block of 32 columns; lane group g holds offsets 8g..8g+7;
//  - A is 16 tokens: token t's f32 activations times 2^k_t as two f16 planes
//    (mf::split_f16x2, k_t = mf::row_shift of the row's largest finite |x|);
//  - B is 16 weight rows: the int8 codes, exact in f16 (|q| <= 128 < 2^11);
//  - D[token][row]: a lane holds four tokens of one row, so the block's fp16 scale is
//    one value per lane, applied after the block: acc += d * (A0 B + A1 B).
// Every product q x is exact; the MFMA sums a block's products in f32 and d times that
// sum is added to the accumulator, all times 2^k_t, which the store takes back (powers
// of two: the same roundings as unscaled).  The two planes hold each activation to
// 2^-22 of itself (to 2^-39 of the row's largest below 2^-17 of it).  The reference sums
// the products sequentially from the bias (d q rounds to nothing: it has at most 19
// significant bits), so results agree to f32 rounding, not bit for bit.
//
// What bounds it: the projections are small (15 GFLOP at 512 tokens, 24 us of the card's
// library GEMM rate with both planes), so the split matters more than the inner loop.  One
// workgroup used to take all of K for 64 tokens x 4 row tiles: at 77 tokens 90 workgroups
// each ran a chain of 128 steps (46 us), and at 512 every wave read all token fragments
// from LDS for one row tile.  K now goes over the waves of a workgroup and the tile shape
// follows the call's size (launch_gemm_for).  Whole calls, 5120 x 2880 at 512 tokens: 62.5
// to 45.2 us; 2880 x 4096 at 512 tokens 83 to 49 us, at 77 tokens 51 to 22 us.
//
// Workspace: token fragments [16-token sub-tile][step][plane][lane][16 B] (steps past the
// last block -- K = 2880 has 90 blocks, padded to 92 -- hold zero tokens, and their row
// scales are zero), then the tokens' shifts k_t (int32), unless the caller passes them
// (ttl_matmul_q8_0_shifted).
#include "ttl_mfma.hpp"

#include <hip/hip_fp16.h>

namespace {

using mf::f16x8;
using mf::f32x4;

constexpr int kPlanes = 2;
constexpr int kSubTokens = 16;  // tokens of one fragment

template <int K>
struct Shape {
    static constexpr int blocks = K / 32;
    static constexpr int quads = (blocks + 3) / 4;
    static constexpr int steps = quads * 4;
    // one 16-token sub-tile: [step][plane] fragments
    static constexpr size_t sub_bytes = size_t(steps) * kPlanes * mf::frag_bytes;
};

// Token fragments, one wave per token: lane l requests the row's pieces of 8 values l, l + 64,
// ... at once, takes the largest finite |x| over the wave unless the shifts are given, and
// writes piece j = 4 step + g times 2^shift as two planes (16 bytes each, lane (t, g) of its
// sub-tile's fragment; the four tokens of a workgroup are neighbours there).  Tokens past
// the count and steps past the row are zero.  Replaces a launch for the shifts and one with
// a thread per piece: 4.6 + 5.2 us at 512 x 4096, one launch of 5.0 us.
constexpr int kGatherWaves = 4;
template <int K, bool SHIFTED>
__global__ __launch_bounds__(kGatherWaves * 64) void q8_gather_kernel(const float *__restrict__ x, uint32_t tokens,
                                                                      int32_t *__restrict__ shift,
                                                                      uint8_t *__restrict__ frags) {
    using S = Shape<K>;
    constexpr int pieces = K / 8, per = (S::steps * 4 + 63) / 64;
    const uint32_t token = blockIdx.x * kGatherWaves + threadIdx.x / 64, lane = threadIdx.x % 64;
    const bool live = token < tokens;
    const float4 *row = reinterpret_cast<const float4 *>(x + size_t(live ? token : 0) * K);
    float v[per][8];
#pragma unroll
    for (int i = 0; i < per; ++i) {
        const uint32_t j = min(lane + 64u * i, uint32_t(pieces - 1));
        const float4 lo = row[2 * j], hi = row[2 * j + 1];
        v[i][0] = lo.x;
        v[i][1] = lo.y;
        v[i][2] = lo.z;
        v[i][3] = lo.w;
        v[i][4] = hi.x;
        v[i][5] = hi.y;
        v[i][6] = hi.z;
        v[i][7] = hi.w;
    }
    int k;
    if constexpr (SHIFTED) {
        k = shift[live ? token : 0];
    } else {
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < per; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                m = mf::finite_max(m, v[i][e]);
            }
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            m = __builtin_fmaxf(m, __shfl_xor(m, d));
        }
        k = mf::row_shift(m);
        if (live && lane == 0) {
            shift[token] = k;
        }
    }
    uint8_t *dst = frags + size_t(token / kSubTokens) * S::sub_bytes + (token % kSubTokens) * 16;
#pragma unroll
    for (int i = 0; i < per; ++i) {
        const uint32_t j = lane + 64u * i;
        if (j >= uint32_t(S::steps * 4)) {
            continue;
        }
        uint4 out[kPlanes] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
        if (live && j < uint32_t(pieces)) {
            mf::split_f16x2(v[i], k, out);
        }
#pragma unroll
        for (int p = 0; p < kPlanes; ++p) {
            *reinterpret_cast<uint4 *>(dst + (size_t(j / 4) * kPlanes + p) * mf::frag_bytes + (j % 4) * 256) = out[p];
        }
    }
}

// 8 int8 codes (K order) as f16, exact: code q's byte with its top bit flipped is
// u = q + 128, and the f16 with bits 0x6400 | u is 1024 + u, so (1024 + u) - 1152 = q
// (an exact f16 subtraction).  Dword k holds codes 2k (low half) and 2k + 1.
__device__ inline f16x8 int8_f16(uint2 c) {
    typedef _Float16 f16x2v __attribute__((ext_vector_type(2)));
    const f16x2v bias = {_Float16(1152.0f), _Float16(1152.0f)};
    f16x8 r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t w = (k < 2 ? c.x : c.y) ^ 0x80808080u;
        // bytes (0x64, code 2k + 1, 0x64, code 2k): one byte permutation of (w, 0x64...)
        const uint32_t h = __builtin_amdgcn_perm(0x64646464u, w, k % 2 == 0 ? 0x04010400u : 0x04030402u);
        const f16x2v v = __builtin_bit_cast(f16x2v, h) - bias;
        r[2 * k] = v[0];
        r[2 * k + 1] = v[1];
    }
    return r;
}

struct GemmArgs {
    const uint8_t *codes;        // repacked [tiles][blocks][2 halves][16 rows][16 B]
    const uint16_t *row_scales;  // [rows][steps] fp16 (zero past the blocks, q8::row_scale_stride)
    const float *bias;           // [rows] or null
    const float *residual;       // [tokens][rows] or null
    float *out;                  // [tokens][rows]
    const uint8_t *frags;        // token fragments
    const int32_t *shift;        // [tokens] the tokens' k (fragments hold x 2^k)
    uint32_t rows, row_tiles, tokens;
};

// One workgroup: SUBS 16-token sub-tiles x TILES 16-row weight tiles, its KW waves each a
// range of the K quads over the whole of that (every fragment and code is requested once per
// workgroup, straight into registers: no LDS copy and no barrier in the loop), one step
// ahead.  The waves' sums are added in LDS in wave order, MS sub-tiles at a time.
template <int K, int SUBS, int TILES, int KW>
__global__ __launch_bounds__(KW * 64) __attribute__((amdgpu_waves_per_eu(2))) void q8_gemm_kernel(GemmArgs a) {
    using S = Shape<K>;
    constexpr int per = (S::quads + KW - 1) / KW;  // quads per wave
    constexpr int MS = SUBS < 2 || KW > 4 ? 1 : 2;
    constexpr int kRows = TILES * 16, kStride = kRows + 4;  // + 4: the lane groups' rows in other banks
    __shared__ float part[KW][MS * kSubTokens * kStride];
    // (the wave as a scalar: every address is a uniform base plus the lane's constant offset)
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t lane = threadIdx.x % 64, n = lane % 16, g = lane / 16;
    const uint32_t sub0 = blockIdx.y * SUBS, subs = (a.tokens + kSubTokens - 1) / kSubTokens;
    const uint32_t q0 = wave * per, q1 = min(q0 + per, uint32_t(S::quads));

    // sub-tiles past the tokens and row tiles past the matrix re-read the last (not written)
    const uint8_t *fp[SUBS];
#pragma unroll
    for (int m = 0; m < SUBS; ++m) {
        fp[m] = a.frags + size_t(min(sub0 + m, subs - 1)) * S::sub_bytes;
    }
    uint32_t rt[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        rt[t] = min(uint32_t(blockIdx.x * TILES + t), a.row_tiles - 1);
    }
    // bytes 8g..8g+7 of row n's block: half g / 2 (q8::code_offset), 8 (g % 2) into it
    const uint32_t code_at = (g / 2) * 32 + n * 2 + g % 2, scale_at = n * (S::steps / 4);  // in uint2

    f16x8 xf[2][SUBS][kPlanes];
    uint2 qc[2][TILES], qs[2][TILES];
    auto load_step = [&](uint32_t s, f16x8(&x)[SUBS][kPlanes], uint2(&c)[TILES]) __attribute__((always_inline)) {
        const uint32_t b = min(s, uint32_t(S::blocks - 1));
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            c[t] = reinterpret_cast<const uint2 *>(a.codes + (size_t(rt[t]) * S::blocks + b) * 512)[code_at];
        }
#pragma unroll
        for (int m = 0; m < SUBS; ++m) {
#pragma unroll
            for (int p = 0; p < kPlanes; ++p) {
                x[m][p] = reinterpret_cast<const f16x8 *>(fp[m] + (size_t(s) * kPlanes + p) * mf::frag_bytes)[lane];
            }
        }
    };
    auto load_scales = [&](uint32_t q, uint2(&d)[TILES]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            d[t] = reinterpret_cast<const uint2 *>(a.row_scales + size_t(rt[t]) * 16 * S::steps + 4 * q)[scale_at];
        }
    };

    f32x4 acc[SUBS][TILES];
#pragma unroll
    for (int m = 0; m < SUBS; ++m) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // One region per weight tile: the block's MFMAs of all sub-tiles, and between them, in
    // the 12 cycles that each leaves the VALU, the scaling of the tile before and the
    // decoding of the tile after (w, d: of the tile to multiply; pend, pend_d: products to scale).
    f16x8 w;
    float d = 0.0f, pend_d = 0.0f;
    f32x4 pend[SUBS];
#pragma unroll
    for (int m = 0; m < SUBS; ++m) {
        pend[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto scale_of = [&](int k, const uint2 &four) __attribute__((always_inline)) {
        return __half2float(__ushort_as_half(uint16_t((k < 2 ? four.x : four.y) >> (16 * (k % 2)))));
    };
    // step k of its quad; kn, cn, sn: the next step's place in its quad, first codes and scales
    auto step = [&](int k, const f16x8(&x)[SUBS][kPlanes], const uint2(&c)[TILES], const uint2(&s)[TILES], int kn,
                    const uint2 &cn, const uint2 &sn) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            f32x4 cur[SUBS];
#pragma unroll
            for (int m = 0; m < SUBS; ++m) {
                cur[m] = mf::mfma(x[m][0], w, f32x4{0.f, 0.f, 0.f, 0.f});
            }
#pragma unroll
            for (int m = 0; m < SUBS; ++m) {
                cur[m] = mf::mfma(x[m][1], w, cur[m]);
            }
            constexpr int last = TILES - 1;
#pragma unroll
            for (int m = 0; m < SUBS; ++m) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[m][t == 0 ? last : t - 1][e] = fmaf(pend_d, pend[m][e], acc[m][t == 0 ? last : t - 1][e]);
                }
            }
            const f16x8 wn = int8_f16(t < last ? c[t < last ? t + 1 : 0] : cn);
            const float dn = t < last ? scale_of(k, s[t < last ? t + 1 : 0]) : scale_of(kn, sn);
#pragma unroll
            for (int i = 0; i < SUBS * kPlanes; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA,
                __builtin_amdgcn_sched_group_barrier(0x002, SUBS == 4 ? 4 : (SUBS == 2 ? 6 : 9), 0);  // then VALU
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < SUBS; ++m) {
                // an empty statement that takes the sum in registers here: the compiler
                // otherwise sinks these updates and keeps every block product live
                asm volatile("" : "+v"(acc[m][t == 0 ? last : t - 1]));
                pend[m] = cur[m];
            }
            pend_d = d;
            w = wn;
            d = dn;
        }
    };

    if (q0 < q1) {
        load_scales(q0, qs[0]);
        load_step(4 * q0, xf[0], qc[0]);
        w = int8_f16(qc[0][0]);
        d = scale_of(0, qs[0][0]);
        // (requests past the range repeat its last quad or step)
        auto quad = [&](uint32_t q, const uint2(&s)[TILES], uint2(&next)[TILES]) __attribute__((always_inline)) {
            load_scales(min(q + 1, q1 - 1), next);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                load_step(min(4 * q + k + 1, 4 * q1 - 1), xf[(k + 1) % 2], qc[(k + 1) % 2]);
                __builtin_amdgcn_sched_barrier(0);
                step(k, xf[k % 2], qc[k % 2], s, (k + 1) % 4, qc[(k + 1) % 2][0], k < 3 ? s[0] : next[0]);
            }
        };
#pragma unroll 1
        for (uint32_t q = q0; q < q1; q += 2) {
            quad(q, qs[0], qs[1]);
            if (q + 1 < q1) {
                quad(q + 1, qs[1], qs[0]);
            }
        }
        // the last tile of the last step
#pragma unroll
        for (int m = 0; m < SUBS; ++m) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[m][TILES - 1][e] = fmaf(pend_d, pend[m][e], acc[m][TILES - 1][e]);
            }
        }
    }

    // D rows 4g..4g+3 of sub-tile m are tokens; the lane's column is weight row n
#pragma unroll
    for (int m0 = 0; m0 < SUBS; m0 += MS) {
        if (m0 > 0) {
            __syncthreads();
        }
#pragma unroll
        for (int m = 0; m < MS; ++m) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    part[wave][(m * kSubTokens + 4 * g + e) * kStride + t * 16 + n] = acc[m0 + m][t][e];
                }
            }
        }
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < uint32_t(MS * kSubTokens * kRows); i += KW * 64) {
            const uint32_t lt = i / kRows, lr = i % kRows;
            const uint32_t token = (sub0 + m0) * kSubTokens + lt, row = blockIdx.x * kRows + lr;
            if (token < a.tokens && row < a.rows) {
                float sum = part[0][lt * kStride + lr];
#pragma unroll
                for (int w = 1; w < KW; ++w) {
                    sum += part[w][lt * kStride + lr];
                }
                const size_t o = size_t(token) * a.rows + row;
                float v = __builtin_amdgcn_ldexpf(sum, -a.shift[token]);
                if (a.bias) {
                    v = a.bias[row] + v;
                }
                if (a.residual) {
                    v = a.residual[o] + v;
                }
                a.out[o] = v;
            }
        }
    }
}

// (room for whole groups of four sub-tiles)
constexpr uint32_t kRoomTokens = 4 * kSubTokens;
template <int K>
size_t frag_bytes_for(uint32_t tokens) {
    return (size_t((tokens + kRoomTokens - 1) / kRoomTokens) * 4 * Shape<K>::sub_bytes + 255) & ~size_t(255);
}

template <int K>
size_t workspace_for(uint32_t tokens) {
    return frag_bytes_for<K>(tokens) + size_t((tokens + kRoomTokens - 1) / kRoomTokens) * kRoomTokens * 4;
}

template <int K, int SUBS, int TILES, int KW>
void launch_gemm(const GemmArgs &a, hipStream_t stream) {
    const dim3 grid((a.row_tiles + TILES - 1) / TILES, (a.tokens + SUBS * kSubTokens - 1) / (SUBS * kSubTokens));
    q8_gemm_kernel<K, SUBS, TILES, KW><<<grid, KW * 64, 0, stream>>>(a);
}

// The split of a call: the tile shape with the least (rounds of one workgroup per CU) x
// (2 SUBS + 1) x (TILES + 1), the last two for what a workgroup's step costs (its products,
// and the loads of its fragments and codes), the smaller shape on a tie.  K goes over 8
// waves, or over 4 where the large shapes fill the CUs more than once (two workgroups of 4
// waves then share a CU).  Measured over 1 to 1024 tokens against every other shape, whole
// calls: 5120 x 2880 at 16 tokens 2 tiles of 1 sub-tile 11.7 us (2 x 2 12.5), at 77 2 x 2 18.7
// (4 x 5 24), at 128 2 x 5 19.5 (4 x 5 23.4), at 512 4 x 5 45.2 (4 x 3 58.8, 2 x 5 49.8); 2880 x
// 4096 at 16 tokens 1 x 1 13.7, at 128 2 x 3 21.6 (2 x 2 27.7), at 512 4 x 3 49.2 (4 x 5, whose 288
// workgroups are two rounds, 64.3).
template <int K>
void launch_gemm_for(const GemmArgs &a, uint32_t compute_units, hipStream_t stream) {
    constexpr struct {
        uint32_t subs, tiles;
    } shapes[] = {{1, 1}, {1, 2}, {2, 2}, {2, 3}, {2, 5}, {4, 3}, {4, 5}};
    const uint32_t subs = (a.tokens + kSubTokens - 1) / kSubTokens, cus = compute_units ? compute_units : 1;
    uint64_t best = ~0ull;
    uint32_t pick = 0, groups = 0;
    for (uint32_t i = 0; i < 7; ++i) {
        const uint32_t token_groups = (subs + shapes[i].subs - 1) / shapes[i].subs;
        const uint64_t w = uint64_t((a.row_tiles + shapes[i].tiles - 1) / shapes[i].tiles) * token_groups;
        const uint64_t cost = (w + cus - 1) / cus * (2 * shapes[i].subs + 1) * (shapes[i].tiles + 1);
        if (cost < best && token_groups <= 65535u) {  // (the grid's y)
            best = cost;
            pick = i;
            groups = w > cus ? 2 : 1;
        }
    }
    switch (pick) {
    case 0: launch_gemm<K, 1, 1, 8>(a, stream); break;
    case 1: launch_gemm<K, 1, 2, 8>(a, stream); break;
    case 2: launch_gemm<K, 2, 2, 8>(a, stream); break;
    case 3: launch_gemm<K, 2, 3, 8>(a, stream); break;
    case 4: groups > 1 ? launch_gemm<K, 2, 5, 4>(a, stream) : launch_gemm<K, 2, 5, 8>(a, stream); break;
    case 5: groups > 1 ? launch_gemm<K, 4, 3, 4>(a, stream) : launch_gemm<K, 4, 3, 8>(a, stream); break;
    default: groups > 1 ? launch_gemm<K, 4, 5, 4>(a, stream) : launch_gemm<K, 4, 5, 8>(a, stream); break;
    }
}

template <int K>
void launch_matmul(const GemmArgs &a, const float *x, bool shifted, int32_t *shift, uint8_t *frags,
                   uint32_t compute_units, hipStream_t stream) {
    const uint32_t gather = ((a.tokens + kSubTokens - 1) / kSubTokens) * (kSubTokens / kGatherWaves);
    if (shifted) {
        q8_gather_kernel<K, true><<<gather, kGatherWaves * 64, 0, stream>>>(x, a.tokens, shift, frags);
    } else {
        q8_gather_kernel<K, false><<<gather, kGatherWaves * 64, 0, stream>>>(x, a.tokens, shift, frags);
    }
    launch_gemm_for<K>(a, compute_units, stream);
}

int matmul_q8_0(ttl_ctx *ctx, const ttl_q8 *w, const float *bias_dev, const float *x_dev, const int32_t *shift_dev,
                uint32_t tokens, const float *residual_dev, float *out_dev, void *workspace_dev,
                size_t workspace_bytes, const char *who) {
    TTL_REQUIRE(ctx && w && w->codes && w->row_scales && x_dev && out_dev && workspace_dev, TTL_ERR_INVALID,
                "%s: null argument", who);
    TTL_REQUIRE(w->cols == 2880 || w->cols == 4096, TTL_ERR_SHAPE, "%s: cols must be 2880 or 4096", who);
    TTL_REQUIRE(tokens < (1u << 20), TTL_ERR_SHAPE, "%s: at most %u tokens per call", who, (1u << 20) - 1);
    const size_t need = ttl_matmul_q8_0_workspace_bytes(tokens, w->cols);
    TTL_REQUIRE(workspace_bytes >= need, TTL_ERR_SHAPE, "%s: workspace of %zu bytes, %zu needed", who,
                workspace_bytes, need);
    TTL_REQUIRE((reinterpret_cast<uintptr_t>(x_dev) & 15) == 0 && (reinterpret_cast<uintptr_t>(workspace_dev) & 15) == 0,
                TTL_ERR_INVALID, "%s: x and the workspace must be 16-byte aligned", who);
    if (tokens == 0) {
        return TTL_OK;
    }
    uint8_t *frags = static_cast<uint8_t *>(workspace_dev);
    int32_t *shift = shift_dev ? const_cast<int32_t *>(shift_dev)
                               : reinterpret_cast<int32_t *>(frags + (w->cols == 2880 ? frag_bytes_for<2880>(tokens)
                                                                                      : frag_bytes_for<4096>(tokens)));
    GemmArgs a;
    a.codes = w->codes;
    a.row_scales = w->row_scales;
    a.bias = bias_dev;
    a.residual = residual_dev;
    a.out = out_dev;
    a.frags = frags;
    a.shift = shift;
    a.rows = w->rows;
    a.row_tiles = w->tiles;
    a.tokens = tokens;
    if (w->cols == 2880) {
        launch_matmul<2880>(a, x_dev, shift_dev != nullptr, shift, frags, uint32_t(ctx->compute_units),
                            ctx->stream);
    } else {
        launch_matmul<4096>(a, x_dev, shift_dev != nullptr, shift, frags, uint32_t(ctx->compute_units),
                            ctx->stream);
    }
    TTL_LAUNCHED("q8 gemm kernels");
    return TTL_OK;
}

}  // namespace

extern "C" {

size_t ttl_matmul_q8_0_workspace_bytes(uint32_t tokens, uint32_t cols) {
    return cols == 4096 ? workspace_for<4096>(tokens) : workspace_for<2880>(tokens);
}

int ttl_matmul_q8_0(ttl_ctx *ctx, const ttl_q8 *w, const float *bias_dev, const float *x_dev, uint32_t tokens,
                    const float *residual_dev, float *out_dev, void *workspace_dev, size_t workspace_bytes) {
    return matmul_q8_0(ctx, w, bias_dev, x_dev, nullptr, tokens, residual_dev, out_dev, workspace_dev,
                       workspace_bytes, "ttl_matmul_q8_0");
}

int ttl_matmul_q8_0_shifted(ttl_ctx *ctx, const ttl_q8 *w, const float *bias_dev, const float *x_dev,
                            const int32_t *shift_dev, uint32_t tokens, const float *residual_dev, float *out_dev,
                            void *workspace_dev, size_t workspace_bytes) {
    TTL_REQUIRE(shift_dev, TTL_ERR_INVALID, "ttl_matmul_q8_0_shifted: null shifts");
    return matmul_q8_0(ctx, w, bias_dev, x_dev, shift_dev, tokens, residual_dev, out_dev, workspace_dev,
                       workspace_bytes, "ttl_matmul_q8_0_shifted");
}

}  // extern "C"
