// The RMSNorm divisor of a row held in a workgroup's registers, with the sum of squares
// exactly as the reference's sequential loop rounds it (bnn-sw-v2/qwen3/qwen3.c:342-353).
// Shared by the fused kernels (bnn_fused.hip) and the multi-row row producer (bnn_rows.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bnn_bitplane.h"
#include "bnn_internal.h"

namespace bnnhip {
namespace {

extern "C" __device__ double __ockl_wfred_add_f64(double);

constexpr uint32_t kRowThreads = 1024;  // threads of a workgroup that holds a row
constexpr uint32_t kRowWaves = kRowThreads / 64;

// Element i of a thread of the row: half i % 2 of the 128-value group w + 16 (i / 2), w its
// wave (whole waves: K % 128 == 0), and whether that group exists.
__device__ __forceinline__ uint32_t row_elem(uint32_t wave, uint32_t lane, int i) {
    return (wave + kRowWaves * (uint32_t)(i >> 1)) * kGroup + 64u * (i & 1) + lane;
}

// The sum of the squares in index order, s_{i+1} = F32(s_i + t_i) from s_0 = +0,
// evaluated in segments of kSegment terms.  Segment j is run from kWindow candidate
// starts at once (one lane each): the binary32 values whose bit patterns lie around
// that of F32(E_j), E_j the sum of the earlier terms in binary64.  Afterwards one
// wave walks the segments in order: when the running sum is one of segment j's
// candidates, the lane that started from exactly that value has performed the same
// additions from the same value, and its end value is taken; otherwise the segment
// is added term by term.  Either way the result is bit-identical to the sequential
// loop; the walk costs one table lookup per segment in the usual case, where the
// accumulated rounding of the sequential sum stays within +-16 ulps of E_j.
constexpr uint32_t kSegment = 128;
constexpr uint32_t kWindow = 32;
constexpr uint32_t kSumChunk = 64;  // terms per binary64 partial sum (one wave's)

// s plus the n terms at p, one rounding per addition, in index order (n % 16 == 0)
__device__ __forceinline__ float add_in_order_lds(const float* p, uint32_t n, float s) {
    const float4* p4 = reinterpret_cast<const float4*>(p);
#pragma unroll 1
    for (uint32_t i = 0; i < n / 4u; i += 4u) {
        float4 v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
            v[c] = p4[i + c];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            s = s + v[c].x;
            s = s + v[c].y;
            s = s + v[c].z;
            s = s + v[c].w;
        }
    }
    return s;
}

// NC interleaved candidate chains of one wave over kSegment terms each
template <int NC>
__device__ __forceinline__ void run_chains(float (&c)[NC], const float4* const (&src)[NC]) {
#pragma unroll 2
    for (uint32_t i = 0; i < kSegment / 4u; i += 8u) {
        float4 v[NC][8];
#pragma unroll
        for (int r = 0; r < NC; ++r)
#pragma unroll
            for (int q = 0; q < 8; ++q)
                v[r][q] = src[r][i + q];
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int r = 0; r < NC; ++r) {
                c[r] = c[r] + v[r][q].x;
                c[r] = c[r] + v[r][q].y;
                c[r] = c[r] + v[r][q].z;
                c[r] = c[r] + v[r][q].w;
            }
    }
}

// LDS of the speculative sum for EPT row values per thread: binary64 sums of 64 terms, the
// candidates' end values (segments 2p and 2p + 1 in the two halves of row p), pair p's two
// segments composed per candidate of segment 2p, the segments' first candidate bit pattern,
// and the result.
template <int EPT>
struct RowSumLds {
    static constexpr uint32_t kRowMax = EPT * kRowThreads;
    static constexpr uint32_t kPairs = kRowMax / kSegment / 2u;
    double chunk_sum[kRowMax / kSumChunk];
    float seg_end[kPairs * 64u];
    float seg_comp[kPairs * 32u];
    int seg_base[kPairs * 2u];
    float rms;
};

// sqrtf(sum of x_i * x_i in index order / K + eps), the same value in every thread; `terms`
// (K floats of LDS, 16-byte aligned) is overwritten, and free again for every wave after the
// workgroup's next barrier.
template <int EPT>
__device__ __forceinline__ float row_rms(const float (&xv)[EPT], uint32_t K, float eps, float* terms,
                                         RowSumLds<EPT>& lds) {
    constexpr uint32_t kRowMax = RowSumLds<EPT>::kRowMax, kPairs = RowSumLds<EPT>::kPairs;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const auto elem = [&](int i) { return row_elem(wave, lane, i); };
    const auto live = [&](int i) { return wave + kRowWaves * (uint32_t)(i >> 1) < K / kGroup; };
    // the terms, and their binary64 sums per 64 (chunk k / 64)
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
        const uint32_t k = elem(i);
        const float sq = xv[i] * xv[i];
        if (live(i)) {
            terms[k] = sq;
            const double h = __ockl_wfred_add_f64((double)sq);
            if (lane == 0)
                lds.chunk_sum[k / kSumChunk] = h;
        }
    }
    lds_barrier();
    // candidate chains: wave w runs pairs w, w + 16, ... (segments 2p, 2p + 1)
    const uint32_t nseg = K / kSegment, npairs = (nseg + 1u) / 2u;
    const uint32_t half = lane >> 5, cand = lane & (kWindow - 1u);
    constexpr int kPairsPerWave = (kPairs + kRowWaves - 1) / kRowWaves;
    float c[kPairsPerWave];
    int bs[kPairsPerWave];
    const float4* src[kPairsPerWave];
#pragma unroll
    for (int r = 0; r < kPairsPerWave; ++r) {
        const uint32_t p = min(wave + kRowWaves * r, npairs - 1u);
        // E_{2p}: the chunks before segment 2p; E_{2p+1} adds segment 2p's two
        double e = 0.0;
#pragma unroll
        for (uint32_t cc = 0; cc < kRowMax / kSumChunk; cc += 64u)
            if (cc + lane < 4u * p)
                e += lds.chunk_sum[cc + lane];
        e = __ockl_wfred_add_f64(e);
        if (half)
            e = e + lds.chunk_sum[4u * p] + lds.chunk_sum[4u * p + 1u];
        const int base = __float_as_int((float)e) - (int)(kWindow / 2u);
        bs[r] = base;
        c[r] = __int_as_float(base + (int)cand);
        const uint32_t j = min(2u * p + half, nseg - 1u);
        src[r] = reinterpret_cast<const float4*>(terms + kSegment * j);
        if (cand == 0 && wave + kRowWaves * r < npairs && 2u * p + half < nseg)
            lds.seg_base[2u * p + half] = base;
    }
    if (kPairsPerWave > 1 && wave + kRowWaves < npairs) {
        run_chains<kPairsPerWave>(c, src);
    } else if (wave < npairs) {
        float c1[1] = {c[0]};
        const float4* const s1[1] = {src[0]};
        run_chains<1>(c1, s1);
        c[0] = c1[0];
    }
    // each pair's two segments composed in its own wave: candidate c of segment 2p ends at
    // a value whose offset in segment 2p + 1's window names the lane that continued from
    // it; an offset outside that window leaves the marker 0xffffffff (no candidate)
#pragma unroll
    for (int r = 0; r < kPairsPerWave; ++r) {
        const uint32_t pr = wave + kRowWaves * r;
        const uint32_t idx = (uint32_t)__float_as_int(c[r]) - (uint32_t)__builtin_amdgcn_readlane(bs[r], 32);
        const float nxt = __shfl(c[r], (int)(32u + (idx & (kWindow - 1u))));
        const float comp = 2u * pr + 1u >= nseg ? c[r] : idx < kWindow ? nxt : __int_as_float(-1);
        if (pr < npairs) {
            lds.seg_end[pr * 64u + lane] = c[r];
            if (lane < kWindow)
                lds.seg_comp[pr * kWindow + lane] = comp;
        }
    }
    lds_barrier();
    // the walk (wave 0) over the composed pairs: bits of the running sum, uniform across
    // the wave
    if (wave == 0) {
        float comps[kPairs];
#pragma unroll
        for (uint32_t m = 0; m < kPairs; ++m)
            comps[m] = lds.seg_comp[min(m, npairs - 1u) * kWindow + (lane & (kWindow - 1u))];
        const int bases = lds.seg_base[min(lane, nseg - 1u)];
        // branch-free lookups (a scalar branch per step costs more than the step); an
        // offset outside a window sets a bit above the window's in `any`, a composed miss
        // leaves the marker (caught by the next offset, or at the end), and either repeats
        // the walk below
        uint32_t v = 0, any = 0;
        if (npairs == kPairs) {
#pragma unroll
            for (uint32_t m = 0; m < kPairs; ++m) {
                const uint32_t idx = v - (uint32_t)__builtin_amdgcn_readlane(bases, 2u * m);
                any |= idx;
                v = (uint32_t)__builtin_amdgcn_readlane(__float_as_int(comps[m]), (int)(idx & (kWindow - 1u)));
            }
        } else {
#pragma unroll
            for (uint32_t m = 0; m < kPairs; ++m) {
                const uint32_t idx = v - (uint32_t)__builtin_amdgcn_readlane(bases, 2u * m);
                const uint32_t nv =
                    (uint32_t)__builtin_amdgcn_readlane(__float_as_int(comps[m]), (int)(idx & (kWindow - 1u)));
                const bool live = m < npairs;
                any |= live ? idx : 0u;
                v = live ? nv : v;
            }
        }
        const uint32_t miss = (any & ~(kWindow - 1u)) | (uint32_t)(v == 0xffffffffu);
        if (miss) {  // the walk with term-by-term additions where the running sum is no candidate
            v = 0;
            for (uint32_t j = 0; j < nseg; ++j) {
                const uint32_t idx = v - (uint32_t)lds.seg_base[j];
                if (idx < kWindow)
                    v = __float_as_uint(lds.seg_end[(j / 2u) * 64u + (j & 1u) * 32u + idx]);
                else
                    v = __float_as_uint(add_in_order_lds(terms + kSegment * j, kSegment, __uint_as_float(v)));
            }
        }
        if (lane == 0)
            lds.rms = sqrtf(__uint_as_float(v) / (float)K + eps);
    }
    lds_barrier();
    return lds.rms;
}

}  // namespace
}  // namespace bnnhip
