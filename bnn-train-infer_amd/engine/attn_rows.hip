// Causal attention of a block of prompt tokens on the device (attn_rows.h), the operations
// of the host step (bnn-sw-v2/qwen3/qwen3.c:355-478) for every token of the block: products
// and quotients are formed elementwise, every sum runs in index or position order from +0
// with one rounding per addition, so each token's values are those of its own step, bit for
// bit.  Where a step of one token leaves the chip to a few serial chains, a block of tokens
// has thousands of independent ones: lanes own (query, key) or (query, dim) pairs and walk
// the sums in order, as register tiles fed from LDS.
//
// Measured (28 layers of width 2048, 389 tokens in one call): 397 ms as 389 single-token
// steps, 6.3 ms as one block.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

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

// Scores of 64 queries x 64 keys of one head: each thread 4 x 4 pairs (queries ty + 16 i,
// keys tx + 16 j), every dot over head_dim in order (qwen3.c:441-452), 16-byte LDS reads of
// four head dims at a time (8 reads for 128 VALU instructions; rows padded to 132 floats, so
// the 16 rows a read touches fall into distinct bank groups).  Keys past a query's position
// are not stored.
constexpr uint32_t kTile = 64, kPitch4 = hd4 + 1;

__global__ __launch_bounds__(256) void k_score_rows(AttnRows a) {
    __shared__ float4 qs[kTile * kPitch4], ks[kTile * kPitch4];
    const uint32_t tid = threadIdx.x, tx = tid & 15u, ty = tid >> 4;
    const uint32_t h = blockIdx.y, q0 = blockIdx.z * kTile, k0 = blockIdx.x * kTile;
    const uint32_t last = a.pos0 + min(q0 + kTile, a.rows) - 1u;  // the tile's last position
    if (k0 > last)
        return;
    const uint32_t kv = h / (a.heads / a.kv_heads);
    for (uint32_t i = tid; i < kTile * hd4; i += 256u) {
        const uint32_t r = i / hd4, c = i % hd4;
        qs[r * kPitch4 + c] = reinterpret_cast<const float4*>(a.q + ((size_t)min(q0 + r, a.rows - 1u) * a.heads + h) * HD)[c];
        ks[r * kPitch4 + c] = reinterpret_cast<const float4*>(a.kc + (size_t)min(k0 + r, last) * a.kv_dim + (size_t)kv * HD)[c];
    }
    __syncthreads();
    float dot[4][4] = {};
#pragma unroll 2
    for (uint32_t c = 0; c < hd4; ++c) {
        float4 qv[4], kw[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            qv[i] = qs[(ty + 16u * i) * kPitch4 + c];
            kw[i] = ks[(tx + 16u * i) * kPitch4 + c];
        }
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) {
                dot[i][j] = dot[i][j] + qv[i].x * kw[j].x;
                dot[i][j] = dot[i][j] + qv[i].y * kw[j].y;
                dot[i][j] = dot[i][j] + qv[i].z * kw[j].z;
                dot[i][j] = dot[i][j] + qv[i].w * kw[j].w;
            }
    }
    bool bad = false;
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
        const uint32_t r = q0 + ty + 16u * i;
        if (r >= a.rows)
            continue;
        float* out = a.scores + ((size_t)h * a.rows + r) * a.score_pitch;
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) {
            const uint32_t t = k0 + tx + 16u * j;
            if (t <= a.pos0 + r) {
                const float score = dot[i][j] * a.scale;
                bad |= !isfinite(score);
                out[t] = score;
            }
        }
    }
    if (bad)
        *a.err = 1;
}

// The probabilities of one (head, query) row in place (qwen3.c:453-465): the maximum
// (order-free: finite or flagged), expf(score - max), the sum in position order, the
// quotients.  One wave per row; the in-order sum runs in every lane over LDS broadcasts.
// Terms past the position are +0 up to a multiple of 64 (adding +0 to this sum of
// non-negative terms changes nothing), and stay in the row as +0 probabilities up to the
// pitch's 64-value tile, which the value sums below read whole.
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
    for (uint32_t t = lane; t < padded; t += 64u) {
        const float e = padded > kSoftChunk ? sc[t] : p[t];
        sc[t] = t < n ? e / sum : 0.0f;
    }
}

// value[i] = sum over positions in order of p[t] * V[t][i] (qwen3.c:466-478): a workgroup
// takes 64 queries x 32 head dims of one head, each thread 2 queries x 4 dims; 32 positions
// of probabilities and V rows pass through LDS at a time.  Positions past a query's own are
// not added (their terms are selected away, so a value row of a later token never reaches an
// earlier one).
constexpr uint32_t kPvDims = 32, kPvKeys = 32;

__global__ __launch_bounds__(256) void k_value_rows(AttnRows a) {
    __shared__ float4 ps4[kTile * (kPvKeys / 4 + 1)];
    __shared__ float4 vs4[kPvKeys * kPvDims / 4];
    const uint32_t tid = threadIdx.x, dx = tid & 7u, qy = tid >> 3;
    const uint32_t h = blockIdx.y, d0 = blockIdx.z * kPvDims;
    const uint32_t qtiles = (a.rows + kTile - 1u) / kTile;
    const uint32_t q0 = (qtiles - 1u - blockIdx.x) * kTile;  // the longest sums start first
    const uint32_t last = a.pos0 + min(q0 + kTile, a.rows) - 1u;
    const uint32_t kv = h / (a.heads / a.kv_heads);
    const uint32_t r0 = q0 + qy, r1 = q0 + qy + 32u;
    const uint32_t n0 = r0 < a.rows ? a.pos0 + r0 + 1u : 0u, n1 = r1 < a.rows ? a.pos0 + r1 + 1u : 0u;
    float acc0[4] = {}, acc1[4] = {};
    for (uint32_t t0 = 0; t0 <= last; t0 += kPvKeys) {
        __syncthreads();
#pragma unroll
        for (uint32_t i = 0; i < kTile * kPvKeys / 4 / 256; ++i) {
            const uint32_t at = tid + 256u * i, r = at / (kPvKeys / 4u), c = at % (kPvKeys / 4u);
            const uint32_t row = min(q0 + r, a.rows - 1u);
            ps4[r * (kPvKeys / 4u + 1u) + c] =
                reinterpret_cast<const float4*>(a.scores + ((size_t)h * a.rows + row) * a.score_pitch + t0)[c];
        }
        {
            const uint32_t r = tid / (kPvDims / 4u), c = tid % (kPvDims / 4u);
            vs4[tid] = reinterpret_cast<const float4*>(a.vc + (size_t)min(t0 + r, last) * a.kv_dim + (size_t)kv * HD + d0)[c];
        }
        __syncthreads();
        const bool whole = t0 + kPvKeys <= a.pos0 + q0 + 1u && q0 + kTile <= a.rows;  // no masked pair in this step
#pragma unroll 2
        for (uint32_t c = 0; c < kPvKeys / 4u; ++c) {
            const float4 pa = ps4[qy * (kPvKeys / 4u + 1u) + c], pb = ps4[(qy + 32u) * (kPvKeys / 4u + 1u) + c];
            const float fa[4] = {pa.x, pa.y, pa.z, pa.w}, fb[4] = {pb.x, pb.y, pb.z, pb.w};
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                const float4 v = vs4[(4u * c + u) * (kPvDims / 4u) + dx];
                const float vv[4] = {v.x, v.y, v.z, v.w};
                const uint32_t t = t0 + 4u * c + u;
                if (whole) {
#pragma unroll
                    for (uint32_t d = 0; d < 4u; ++d) {
                        acc0[d] = acc0[d] + fa[u] * vv[d];
                        acc1[d] = acc1[d] + fb[u] * vv[d];
                    }
                } else {
#pragma unroll
                    for (uint32_t d = 0; d < 4u; ++d) {
                        const float s0 = acc0[d] + fa[u] * vv[d], s1 = acc1[d] + fb[u] * vv[d];
                        acc0[d] = t < n0 ? s0 : acc0[d];
                        acc1[d] = t < n1 ? s1 : acc1[d];
                    }
                }
            }
        }
    }
    const size_t width = (size_t)a.heads * HD, at = (size_t)h * HD + d0 + 4u * dx;
    if (n0)
        *reinterpret_cast<float4*>(a.y + r0 * width + at) = make_float4(acc0[0], acc0[1], acc0[2], acc0[3]);
    if (n1)
        *reinterpret_cast<float4*>(a.y + r1 * width + at) = make_float4(acc1[0], acc1[1], acc1[2], acc1[3]);
}

}  // namespace

void launch_embed_rows(hipStream_t stream, const int32_t* tokens, uint32_t rows, const uint8_t* bits,
                       const uint16_t* scales, uint32_t C, float* x, int* err, int* logit_bad) {
    hipLaunchKernelGGL(k_embed_rows, dim3(rows), dim3(256), 0, stream, tokens, bits, scales, C, x, err, logit_bad);
}

void launch_attn_rows(hipStream_t stream, const AttnRows& a) {
    const uint32_t qtiles = (a.rows + kTile - 1u) / kTile, ktiles = (a.pos0 + a.rows + kTile - 1u) / kTile;
    hipLaunchKernelGGL(k_head_rows, dim3(a.rows, (a.heads + a.kv_heads + 3u) / 4u), dim3(256), 0, stream, a);
    hipLaunchKernelGGL(k_score_rows, dim3(ktiles, a.heads, qtiles), dim3(256), 0, stream, a);
    hipLaunchKernelGGL(k_softmax_rows, dim3(a.rows, a.heads), dim3(64), 0, stream, a);
    hipLaunchKernelGGL(k_value_rows, dim3(qtiles, a.heads, HD / kPvDims), dim3(256), 0, stream, a);
}

}  // namespace bnne
