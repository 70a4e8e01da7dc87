// Causal attention of a block of prompt tokens on the device (attn_rows.h), the operations
// of the host step (bnn-sw-v2/qwen3/qwen3.c:355-478) for every token of the block: products
// and quotients are formed elementwise, every sum runs in index or position order from +0
// with one rounding per addition, so each token's values are those of its own step, bit for
// bit.  Where a step of one token leaves the chip to a few serial chains, a block of tokens
// has thousands of independent ones: lanes own keys or head dims and walk
// the sums of several queries in order.
//
// Measured (28 layers of width 2048, 389 tokens in one call): 397 ms as 389 single-token
// steps, 6.3 ms as one block with attention tiles in LDS (scores 16.4 us, values 58 us per
// layer), 5.2 ms with the register-broadcast kernels below (scores and values 17 us each;
// the values' 4.8 GFLOP of separate multiplies and adds take ~7 us at the rate two waves per
// SIMD reach, the rest is the causal imbalance of the last rounds and the start).  Bound by
// vector issue.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <type_traits>

#include "attn_rows.h"

#define BNNE_EXPF_QUALIFIER static __device__ __forceinline__
#include "../csrc/libc_expf.h"

#pragma clang fp contract(off)

namespace bnne {
namespace {

constexpr uint32_t HD = kRowsHeadDim, half = HD / 2, hd4 = HD / 4;

__constant__ uint64_t kRowsExp2Table[32] = BNNE_EXP2_TABLE;

extern "C" __device__ float __ockl_wfred_max_f32(float);

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// +scale or -scale of the token's Q1_0 embedding row (qwen3.c:355-366), a workgroup per token
__global__ __launch_bounds__(256) void k_embed_rows(const int32_t* __restrict__ tokens, const uint8_t* __restrict__ bits,
                                                    const uint16_t* __restrict__ scales, uint32_t C,
                                                    float* __restrict__ x, int* __restrict__ err,
                                                    int* __restrict__ logit_bad) {
    const uint32_t r = blockIdx.x;
    const size_t token = (size_t)tokens[r];
    if (r == 0 && threadIdx.x == 0) {
        if (err)
            *err = 0;
        if (logit_bad)
            *logit_bad = 0;
    }
    for (uint32_t i = threadIdx.x; i < C; i += 256u) {
        const float s = __half2float(__ushort_as_half(scales[token * (C / 128u) + i / 128u]));
        const bool bit = (bits[token * (C / 8u) + i / 8u] >> (i & 7u)) & 1u;
        x[(size_t)r * C + i] = bit ? s : -s;
    }
}

// One wave per (token, head), query heads first, then key heads: RMSNorm over the head
// (qwen3.c:342-353), RoPE of the pairs (i, i + 64) (:368-376), in place for queries, into
// the cache row for keys, whose wave also stores the head's value row.  The in-order sum of
// the squares runs in every lane over LDS broadcasts (no exchange afterwards).
__global__ __launch_bounds__(256) void k_head_rows(AttnRows a) {
    __shared__ float4 sq4[4][hd4];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t h = blockIdx.y * 4u + wave, r = blockIdx.x, pos = a.pos0 + r;
    if (h >= a.heads + a.kv_heads)
        return;
    const bool is_q = h < a.heads;
    const size_t at = is_q ? (size_t)r * a.heads * HD + (size_t)h * HD
                           : (size_t)r * a.kv_dim + (size_t)(h - a.heads) * HD;
    const float* src = (is_q ? a.q : a.k) + at;
    const float* gain = is_q ? a.q_gain : a.k_gain;
    const float xa = src[lane], xb = src[lane + half];
    const float ga = gain[lane], gb = gain[lane + half];
    const float c = a.cosv[(size_t)pos * half + lane], s = a.sinv[(size_t)pos * half + lane];
    float va = 0.0f, vb = 0.0f;
    if (!is_q)
        va = a.v[at + lane], vb = a.v[at + lane + half];
    float* sq = reinterpret_cast<float*>(sq4[wave]);
    sq[lane] = xa * xa;
    sq[lane + half] = xb * xb;
    wave_lds_sync();
    float sum = 0.0f;
#pragma unroll 8
    for (uint32_t i = 0; i < hd4; ++i) {
        const float4 t = sq4[wave][i];
        sum = sum + t.x;
        sum = sum + t.y;
        sum = sum + t.z;
        sum = sum + t.w;
    }
    const float rms = sqrtf(sum / (float)HD + a.eps);
    if (!isfinite(rms) || rms == 0.0f) {
        if (lane == 0)
            *a.err = 1;
        return;
    }
    const float na = xa / rms * ga, nb = xb / rms * gb;
    const float ra = na * c - nb * s, rb = na * s + nb * c;
    if (is_q) {
        a.q[at + lane] = ra;
        a.q[at + lane + half] = rb;
    } else {
        const size_t row = (size_t)pos * a.kv_dim + (size_t)(h - a.heads) * HD;
        a.kc[row + lane] = ra;
        a.kc[row + lane + half] = rb;
        a.vc[row + lane] = va;
        a.vc[row + lane + half] = vb;
    }
}

// Value I of the lane's row of sixteen lanes, as the DPP operand of the multiply that uses it:
// sixteen values that every lane needs (a query's head dims against the lanes' keys, a
// query's probabilities against the lanes' head dims) sit in one register, repeated in the
// four rows of the wave, and reach the multiplies with no LDS read and no instruction of
// their own.
template <int I>
__device__ __forceinline__ float row_value(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + I, 0xf, 0xf, true));  // row_newbcast:I
}

// acc[q] += (value i of x[q]) * v[i] for i = 0 .. 15 in order, each product and sum rounded on
// its own.  The products run one step ahead of the additions, so that no instruction needs
// the result of the one before it (a dependent pair costs two issue slots); the scheduling
// barriers keep the compiler from pairing them up again.
template <int N, int I = 0>
__device__ __forceinline__ void add16(float (&acc)[N], const float (&x)[N], const float (&v)[16], float (&prod)[N]) {
    float next[N];
    if constexpr (I < 15) {
#pragma unroll
        for (int q = 0; q < N; ++q)
            next[q] = row_value<I + 1>(x[q]) * v[I + 1];
    }
#pragma unroll
    for (int q = 0; q < N; ++q)
        acc[q] = acc[q] + prod[q];
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (I < 15)
        add16<N, I + 1>(acc, x, v, next);
}
template <int N>
__device__ __forceinline__ void accumulate16(float (&acc)[N], const float (&x)[N], const float (&v)[16]) {
    float prod[N];
#pragma unroll
    for (int q = 0; q < N; ++q)
        prod[q] = row_value<0>(x[q]) * v[0];
    add16<N>(acc, x, v, prod);
}

// Scores of 4 Q queries x 64 keys of one head, Q per wave as independent chains: lane = key,
// sixteen head dims at a time in registers (from a tile that the workgroup loads into LDS,
// coalesced; rows padded to 132 floats), the queries' sixteen as one register each; every dot
// runs over head_dim in order (qwen3.c:441-452).  A wave whose keys lie past its queries does
// nothing.
constexpr uint32_t kScoreKeys = 64, kScoreWaves = 4, kPitch4 = hd4 + 1;

template <uint32_t Q>
__global__ __launch_bounds__(64 * kScoreWaves) void k_score_rows(AttnRows a) {
    __shared__ float4 ks[kScoreKeys * kPitch4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t h = blockIdx.x, k0 = blockIdx.y * kScoreKeys;
    const uint32_t w0 = blockIdx.z * kScoreWaves * Q;                       // the workgroup's first query
    const uint32_t last = a.pos0 + min(w0 + kScoreWaves * Q, a.rows) - 1u;  // and its last position
    if (k0 > last)
        return;
    const float* keys = a.kc + (size_t)(h / (a.heads / a.kv_heads)) * HD;
#pragma unroll
    for (uint32_t i = 0; i < kScoreKeys * hd4 / (64u * kScoreWaves); ++i) {
        const uint32_t at = tid + 64u * kScoreWaves * i, r = at / hd4, c = at % hd4;
        ks[r * kPitch4 + c] = reinterpret_cast<const float4*>(keys + (size_t)min(k0 + r, last) * a.kv_dim)[c];
    }
    const uint32_t q0 = w0 + wave * Q;
    const float* query = a.q + (size_t)h * HD + (lane & 15u);
    const size_t width = (size_t)a.heads * HD;
    float x[Q], next[Q], key[16], dot[Q] = {};
    const auto fetch = [&](float(&to)[Q], uint32_t c) {
#pragma unroll
        for (uint32_t i = 0; i < Q; ++i)
            to[i] = query[(size_t)min(q0 + i, a.rows - 1u) * width + 16u * c];
    };
    fetch(x, 0);
    __syncthreads();
    if (q0 >= a.rows || k0 > a.pos0 + min(q0 + Q, a.rows) - 1u)
        return;  // no query, or every key lies behind the last query's position
#pragma unroll 1
    for (uint32_t c = 0; c < HD / 16u; ++c) {
        // the next sixteen dims, in flight during these (the empty asm keeps the loads from
        // being moved behind the arithmetic)
        fetch(next, min(c + 1u, HD / 16u - 1u));
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            const float4 v = ks[lane * kPitch4 + 4u * c + i];
            key[4u * i] = v.x;
            key[4u * i + 1u] = v.y;
            key[4u * i + 2u] = v.z;
            key[4u * i + 3u] = v.w;
        }
        asm volatile("" ::: "memory");
        accumulate16<(int)Q>(dot, x, key);
#pragma unroll
        for (uint32_t i = 0; i < Q; ++i)
            x[i] = next[i];
    }
    const uint32_t t = k0 + lane;
    bool bad = false;
#pragma unroll
    for (uint32_t i = 0; i < Q; ++i) {
        const uint32_t r = q0 + i;
        const float score = dot[i] * a.scale;
        if (r < a.rows && t <= a.pos0 + r) {
            bad |= !isfinite(score);
            a.scores[((size_t)h * a.rows + r) * a.score_pitch + t] = score;
        }
    }
    if (bad)
        *a.err = 1;
}

// The probabilities of one (head, query) row in place (qwen3.c:453-465): the maximum
// (order-free: finite or flagged), expf(score - max), the sum in position order, the
// quotients.  One wave per row; the in-order sum runs in every lane over LDS broadcasts.
// Terms past the position are +0 up to a multiple of 64 (adding +0 to this sum of
// non-negative terms changes nothing), and are not stored.
constexpr uint32_t kSoftChunk = 1024;  // terms in LDS at a time

__global__ __launch_bounds__(64) void k_softmax_rows(AttnRows a) {
    __shared__ float4 p4[kSoftChunk / 4];
    __shared__ uint64_t exp_tab[32];
    float* p = reinterpret_cast<float*>(p4);
    const uint32_t lane = threadIdx.x, h = blockIdx.y, r = a.rows - 1u - blockIdx.x;
    const uint32_t n = a.pos0 + r + 1u, padded = (n + 63u) & ~63u;
    float* sc = a.scores + ((size_t)h * a.rows + r) * a.score_pitch;
    if (lane < 32u)
        exp_tab[lane] = kRowsExp2Table[lane];
    float mx = -INFINITY;
    for (uint32_t t0 = 0; t0 < n; t0 += 256u) {
        float x[4];
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c)
            x[c] = sc[min(t0 + 64u * c + lane, n - 1u)];
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c)
            mx = x[c] > mx ? x[c] : mx;
    }
    const float maximum = __ockl_wfred_max_f32(mx);
    wave_lds_sync();
    float sum = 0.0f;
    for (uint32_t t0 = 0; t0 < padded; t0 += kSoftChunk) {
        const uint32_t m = min(kSoftChunk, padded - t0);
        for (uint32_t t = lane; t < m; t += 64u) {
            const float e = t0 + t < n ? bnne_expf_libc(sc[t0 + t] - maximum, exp_tab) : 0.0f;
            p[t] = e;
            if (padded > kSoftChunk)
                sc[t0 + t] = e;
        }
        wave_lds_sync();
        for (uint32_t i = 0; i < m / 4u; i += 16u) {
            float4 v[16];
#pragma unroll
            for (uint32_t c = 0; c < 16u; ++c)
                v[c] = p4[i + c];
#pragma unroll
            for (uint32_t c = 0; c < 16u; ++c) {
                sum = sum + v[c].x;
                sum = sum + v[c].y;
                sum = sum + v[c].z;
                sum = sum + v[c].w;
            }
        }
        wave_lds_sync();
    }
    if (!(sum > 0.0f) || !isfinite(sum)) {
        if (lane == 0)
            *a.err = 1;
    }
    for (uint32_t t = lane; t < n; t += 64u)
        sc[t] = (padded > kSoftChunk ? sc[t] : p[t]) / sum;
}

// value[i] = sum over positions in order of p[t] * V[t][i] (qwen3.c:466-478): lane = head dim
// (64 of the 128 per workgroup), a wave takes Q queries of one head as independent chains, a
// workgroup 8 Q neighbouring ones; the V rows pass through LDS, 32 positions at a time (each
// wave reading them from the L2 had made the kernel L2-bound), and the probabilities come
// sixteen positions per register.  Positions up to a wave's first query's own are added for
// every query of the wave; of the few after it, those that a query does not see are selected
// away, so a value row of a later token never reaches an earlier one.
constexpr uint32_t kValueWaves = 8, kValueKeys = 32;

// accumulate16 where query i sees only the first n[i] of the sixteen (wave-uniform)
template <uint32_t Q, int I = 0>
__device__ __forceinline__ void values16_seen(float (&acc)[Q], const float (&p)[Q], const float (&v)[16],
                                              const int (&n)[Q]) {
#pragma unroll
    for (uint32_t i = 0; i < Q; ++i) {
        const float s = acc[i] + row_value<I>(p[i]) * v[I];
        acc[i] = I < n[i] ? s : acc[i];
    }
    if constexpr (I < 15)
        values16_seen<Q, I + 1>(acc, p, v, n);
}

template <uint32_t Q>
__global__ __launch_bounds__(64 * kValueWaves) void k_value_rows(AttnRows a) {
    __shared__ float4 vs4[2][kValueKeys * 64 / 4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t h = blockIdx.x, d0 = blockIdx.y * 64u;
    const uint32_t w0 = (gridDim.z - 1u - blockIdx.z) * kValueWaves * Q;  // the longest sums start first
    const uint32_t w_end = a.pos0 + min(w0 + kValueWaves * Q, a.rows);    // one past the workgroup's last position
    const uint32_t q0 = w0 + wave * Q;
    const bool live = q0 < a.rows;
    const uint32_t end = live ? a.pos0 + min(q0 + Q, a.rows) : 0u;  // one past the wave's last position
    const uint32_t whole = live ? a.pos0 + q0 + 1u : 0u;            // positions that all of its queries see
    const uint32_t top = (w_end - 1u) & ~15u;                       // the last sixteen of a row that are read
    const float4* v = reinterpret_cast<const float4*>(a.vc + (size_t)(h / (a.heads / a.kv_heads)) * HD + d0) + (tid & 15u);
    const float* p = a.scores + (size_t)h * a.rows * a.score_pitch + (lane & 15u);
    static_assert(kValueKeys * 16u == 64u * kValueWaves, "one 16-byte piece of a tile per thread");
    const auto fetch_v = [&](uint32_t t) { return v[(size_t)min(t + (tid >> 4), w_end - 1u) * (a.kv_dim / 4u)]; };
    const auto fetch_p = [&](float(&to)[2][Q], uint32_t t) {
#pragma unroll
        for (uint32_t f = 0; f < 2u; ++f)
#pragma unroll
            for (uint32_t i = 0; i < Q; ++i)
                to[f][i] = p[(size_t)min(q0 + i, a.rows - 1u) * a.score_pitch + min(t + 16u * f, top)];
    };
    float acc[Q] = {};
    float pp[2][Q], pn[2][Q];
    fetch_p(pp, 0);
    vs4[0][tid] = fetch_v(0);
    __syncthreads();
    uint32_t buf = 0;
    for (uint32_t t = 0; t < w_end; t += kValueKeys) {
        // the next tile's values, in flight during this one (the empty asm keeps the loads
        // from being moved behind the arithmetic)
        const float4 vn = fetch_v(t + kValueKeys);
        fetch_p(pn, t + kValueKeys);
        asm volatile("" ::: "memory");
        const float* vs = reinterpret_cast<const float*>(vs4[buf]) + lane;
#pragma unroll
        for (uint32_t f = 0; f < 2u; ++f) {
            const uint32_t t16 = t + 16u * f;
            if (t16 >= end)
                break;
            float vv[16];
#pragma unroll
            for (uint32_t u = 0; u < 16u; ++u)
                vv[u] = vs[(16u * f + u) * 64u];
            if (t16 + 16u <= whole) {
                accumulate16<(int)Q>(acc, pp[f], vv);
            } else {
                int n[Q];
#pragma unroll
                for (uint32_t i = 0; i < Q; ++i)
                    n[i] = (int)(a.pos0 + q0 + i + 1u) - (int)t16;
                values16_seen<Q>(acc, pp[f], vv, n);
            }
        }
        vs4[buf ^ 1u][tid] = vn;
#pragma unroll
        for (uint32_t f = 0; f < 2u; ++f)
#pragma unroll
            for (uint32_t i = 0; i < Q; ++i)
                pp[f][i] = pn[f][i];
        buf ^= 1u;
        __syncthreads();
    }
#pragma unroll
    for (uint32_t i = 0; i < Q; ++i)
        if (q0 + i < a.rows)
            a.y[(size_t)(q0 + i) * a.heads * HD + (size_t)h * HD + d0 + lane] = acc[i];
}

}  // namespace

void launch_embed_rows(hipStream_t stream, const int32_t* tokens, uint32_t rows, const uint8_t* bits,
                       const uint16_t* scales, uint32_t C, float* x, int* err, int* logit_bad) {
    hipLaunchKernelGGL(k_embed_rows, dim3(rows), dim3(256), 0, stream, tokens, bits, scales, C, x, err, logit_bad);
}

void launch_attn_rows(hipStream_t stream, const AttnRows& a) {
    const auto parts = [](uint32_t n, uint32_t per) { return (n + per - 1u) / per; };
    // queries per wave: 8 (fewest loads per value) where that still leaves about eight waves per
    // SIMD of 256 CUs, else 4 or 2 -- a SIMD issues a vector instruction per ~2.6 cycles from two
    // waves and more but one per ~6.5 from a single one (measured with chains like these).
    // Layers of 389 / 700 / 1024 tokens 188 / 330 / 408 us with a limit of two waves per SIMD,
    // 181 / 313 / 395 us with this one; up to 200 tokens the same.
    constexpr uint32_t kManyWaves = 8192;
    const uint32_t keys = a.pos0 + a.rows;
    const auto score_waves = [&](uint32_t q) { return a.heads * parts(keys, kScoreKeys) * parts(a.rows, q) / 2u; };
    const auto value_waves = [&](uint32_t q) { return a.heads * (HD / 64u) * parts(a.rows, q); };
    const auto score = [&](auto q) {
        constexpr uint32_t Q = decltype(q)::value;
        hipLaunchKernelGGL(k_score_rows<Q>, dim3(a.heads, parts(keys, kScoreKeys), parts(a.rows, Q * kScoreWaves)),
                           dim3(64 * kScoreWaves), 0, stream, a);
    };
    const auto value = [&](auto q) {
        constexpr uint32_t Q = decltype(q)::value;
        hipLaunchKernelGGL(k_value_rows<Q>, dim3(a.heads, HD / 64u, parts(a.rows, Q * kValueWaves)),
                           dim3(64 * kValueWaves), 0, stream, a);
    };
    using std::integral_constant;
    hipLaunchKernelGGL(k_head_rows, dim3(a.rows, parts(a.heads + a.kv_heads, 4u)), dim3(256), 0, stream, a);
    if (score_waves(8u) >= kManyWaves)
        score(integral_constant<uint32_t, 8>{});
    else if (score_waves(4u) >= kManyWaves)
        score(integral_constant<uint32_t, 4>{});
    else
        score(integral_constant<uint32_t, 2>{});
    hipLaunchKernelGGL(k_softmax_rows, dim3(a.rows, a.heads), dim3(64), 0, stream, a);
    if (value_waves(8u) >= kManyWaves)
        value(integral_constant<uint32_t, 8>{});
    else if (value_waves(4u) >= kManyWaves)
        value(integral_constant<uint32_t, 4>{});
    else
        value(integral_constant<uint32_t, 2>{});
}

}  // namespace bnne
