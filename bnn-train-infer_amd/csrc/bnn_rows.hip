// Multi-row pre-operations (BNNX_LaunchRows): the rows of a block of tokens produced on the
// device, checked and quantised for the matrix-core kernels, one 1024-thread workgroup per
// row (reference operation order: bnn-sw-v2/qwen3/qwen3.c:342-353 for RMSNorm with the
// residual add of :497-498/:510-511, :491-495 for SiLU(gate) * up; the check and the
// quantisation are soft-bnn-accelerator.c:175-211, :278-308).  The produced FP32 row never
// leaves the workgroup's registers.
//
// Bound by latency: two exchanges through LDS (the sum of squares, evaluated speculatively as
// in the fused kernels, and the absmax) around ~100 VALU instructions per value.  A workgroup
// per row puts two rows on a CU at a time.
#include <hip/hip_runtime.h>

#include "bnn_bitplane.h"
#include "bnn_internal.h"
#include "bnn_rowsum.h"

#define BNNE_EXPF_QUALIFIER static __device__ __forceinline__
#include "libc_expf.h"

#pragma clang fp contract(off)

namespace bnnhip {
namespace {

__constant__ uint64_t kRowsExp2Table[32] = BNNE_EXP2_TABLE;

template <int EPT, int KIND>
__global__ __launch_bounds__(kRowThreads) void k_rows(RowsArgs a, uint64_t seq, uint64_t* flag,
                                                      uint64_t* host_status) {
    constexpr uint32_t kRowMax = EPT * kRowThreads;
    __shared__ float4 terms4[KIND == PRE_RMSNORM ? kRowMax / 4 : 1];
    __shared__ RowSumLds<KIND == PRE_RMSNORM ? EPT : 2> sum_lds;
    __shared__ uint32_t amax_w[kRowWaves];
    __shared__ uint64_t exp_tab[32];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t K = a.width, G = K / kGroup;
    const size_t row = (size_t)blockIdx.x * K;
    const auto elem = [&](int i) { return row_elem(wave, lane, i); };
    const auto live = [&](int i) { return wave + kRowWaves * (uint32_t)(i >> 1) < G; };

    float xv[EPT], bv[EPT], gv[EPT];
#pragma unroll
    for (int i = 0; i < EPT; ++i)
        xv[i] = gload(a.a + row + min(elem(i), K - 1u));
    if (a.b) {
#pragma unroll
        for (int i = 0; i < EPT; ++i)
            bv[i] = gload(a.b + row + min(elem(i), K - 1u));
    }
    if constexpr (KIND == PRE_RMSNORM) {
#pragma unroll
        for (int i = 0; i < EPT; ++i)
            gv[i] = gload(a.gain + min(elem(i), K - 1u));
        if (a.b) {
#pragma unroll
            for (int i = 0; i < EPT; ++i)
                xv[i] = xv[i] + bv[i];
        }
        if (a.a_out) {
#pragma unroll
            for (int i = 0; i < EPT; ++i)
                if (live(i))
                    gstore(a.a_out + row + elem(i), xv[i]);
        }
        const float rms = row_rms<EPT>(xv, K, a.eps, reinterpret_cast<float*>(terms4), sum_lds);
        if (!__builtin_isfinite(rms) || rms == 0.0f) {
            if (tid == 0) {
                if (a.err)
                    atomicCAS(a.err, 0, a.err_code);
                raise_flag(seq, flag, host_status);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < EPT; ++i)
            xv[i] = xv[i] / rms * gv[i];
    } else {
        if (tid < 32u)
            exp_tab[tid] = kRowsExp2Table[tid];
        lds_barrier();
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
            const float silu = xv[i] / (1.0f + bnne_expf_libc(-xv[i], exp_tab));
            xv[i] = silu * bv[i];
        }
    }

    // the input check and the row scale in one exchange: a wave with a non-finite value posts
    // the all-ones word, above every finite |x| bit pattern
    uint32_t abits = 0;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
        if (live(i)) {
            const uint32_t v = __float_as_uint(xv[i]) & 0x7fffffffu;
            abits = max(abits, v >= 0x7f800000u ? 0xffffffffu : v);
        }
    }
    abits = __ockl_wfred_max_u32(abits);
    if (lane == 0)
        amax_w[wave] = abits;
    lds_barrier();
    abits = amax_w[0];
#pragma unroll
    for (uint32_t w = 1; w < kRowWaves; ++w)
        abits = max(abits, amax_w[w]);
    if (abits == 0xffffffffu) {
        if (tid == 0)
            raise_flag(seq, flag, host_status);
        return;
    }
    const float s = quant_row_scale(__uint_as_float(abits));
    const float rcp = quant_rcp(s);
    const bool exact = quant_exact(s);  // 1 / s may overflow
#pragma unroll
    for (int i = 0; i < EPT; ++i)
        if (live(i))
            *(__attribute__((address_space(1))) int8_t*)(a.q + row + elem(i)) =
                (int8_t)quantize_rcp(xv[i], s, rcp, exact);
    if (tid == 0)
        gstore(a.rscale + blockIdx.x, s);
}

template <int EPT>
void launch_rows_kind(hipStream_t stream, const RowsArgs& a, uint64_t seq, uint64_t* flag, uint64_t* host_status) {
    if (a.kind == PRE_RMSNORM)
        launch_kernel((k_rows<EPT, PRE_RMSNORM>), dim3(a.rows), dim3(kRowThreads), 0, stream, a, seq, flag,
                      host_status);
    else
        launch_kernel((k_rows<EPT, PRE_SILU_MUL>), dim3(a.rows), dim3(kRowThreads), 0, stream, a, seq, flag,
                      host_status);
}

}  // namespace

hipError_t launch_rows(hipStream_t stream, const RowsArgs& a, uint64_t seq, uint64_t* flag, uint64_t* host_status) {
    if (a.width <= 2u * kRowThreads)
        launch_rows_kind<2>(stream, a, seq, flag, host_status);
    else if (a.width <= 4u * kRowThreads)
        launch_rows_kind<4>(stream, a, seq, flag, host_status);
    else if (a.width <= 6u * kRowThreads)
        launch_rows_kind<6>(stream, a, seq, flag, host_status);
    else
        launch_rows_kind<8>(stream, a, seq, flag, host_status);
    return hipGetLastError();
}

}  // namespace bnnhip
