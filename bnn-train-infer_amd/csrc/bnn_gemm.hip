// Multi-row jobs (GEMM, GEMM_F32, DOT_GROUPS) on the gfx950 matrix cores
// (v_mfma_i32_16x16x64_i8), fed from the matrix's resident 1.125-bit layout: a byte table in
// LDS turns the sign bits of each 128-weight group into the MFMAs' +1/-1 operands.
//
// Numeric contract (reference bnn-accelerator.h:133-149, soft-bnn-accelerator.c:219-276),
// per 128-weight group g:
//   * two MFMAs per 16x16 output subtile accumulate D = sum_k Q[m][k] * W[n][k]
//     (exact) onto an accumulator initialised to 0x4B400000, so the integer result
//     is 0x4B400000 + D; read as a float that bit pattern is exactly 12582912 + D
//     (|D| <= 16256 < 2^22);
//   * fma(scale, 12582912 + D, -scale * 12582912) is the correctly rounded product
//     scale * D: the constant is exact in binary32 (11 + 2 significant bits), so the
//     fused operation rounds the exact value scale * D once;
//   * the product is added to the FP32 accumulator of (m, n) -- groups in
//     increasing order, one rounding per add.  A zero product comes out as +0
//     where the reference may form -0; the accumulator starts at +0 and never
//     becomes -0 (x + -x == +0 in round-to-nearest), so the sums agree bit for bit.
// DOT_GROUPS stores D itself as int16 (k_gemm_dots, k_gemm_dotf).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <utility>
#include <hip/hip_fp16.h>

#include "bnn_internal.h"

#pragma clang fp contract(off)

namespace bnnhip {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kMagicBits = 0x4B400000;  // bit pattern of 12582912.0f = 1.5 * 2^23
constexpr float kMagicValue = 12582912.0f;

// 4 sign bits -> 4 bytes of +1 (bit 1) or -1 (bit 0): the multiply places copies of
// the nibble at bit offsets 0, 7, 14, 21 (disjoint), the mask keeps bit i in byte i,
// then 1 -> ~0xFE = 0x01 and 0 -> ~0x00 = 0xFF per byte (no carries).
__device__ __forceinline__ uint32_t pm1_nibble(uint32_t nib) {
    return ~(((nib * 0x204081u) & 0x01010101u) * 0xFEu);
}

// A 128-byte LDS row holds 8 chunks of 16 bytes; chunk c of row r sits at
// r*128 + 16*(c ^ ((r >> 1) & 7)): the 16 lanes reading one MFMA fragment (16 rows,
// one chunk) hit 16 distinct 16-byte bank groups.
__device__ __forceinline__ uint32_t swz128(uint32_t r, uint32_t c) { return r * 128u + 16u * (c ^ ((r >> 1) & 7u)); }

// Output tiles in bands of `band` M tiles, M tile fastest within a band (the last
// band may be narrower), and workgroups remapped so that consecutive tiles run on one
// XCD: each XCD's share of the grid is then a rectangle of about band M tiles by
// (tiles / 8 / band) N tiles, whose rows and weights stay in that XCD's L2.  The host
// picks `band` so that the rows (re-read once per XCD that covers an M tile) and the
// weights (once per band) cost the least traffic.
struct TileRC {
    uint32_t mt, nt;
};
__device__ __forceinline__ TileRC gemm_tile_of_block(uint32_t b, uint32_t grid, uint32_t mtiles, uint32_t ntiles,
                                                     uint32_t band) {
    const uint32_t x = b % 8u, i = b / 8u, q = grid / 8u, r = grid % 8u;
    const uint32_t t = (x < r ? x * (q + 1u) : r * (q + 1u) + (x - r) * q) + i;
    const uint32_t bi = t / (band * ntiles), rest = t % (band * ntiles);
    const uint32_t width = min(band, mtiles - bi * band);
    return TileRC{bi * band + rest % width, rest / width};
}

// The tile's column tile within its part of the job, whose matrix and output `j` then
// describes (wave-uniform; as selects without the branch it measured the same or slower).
__device__ __forceinline__ uint32_t select_part(GemmJob& j, uint32_t nt) {
    uint32_t first = 0;
    if (j.extra != 0u) {
#pragma unroll
        for (uint32_t i = 0; i < kGemmParts - 1u; ++i) {
            if (i < j.extra && nt >= j.parts[i].first) {
                const GemmPart& p = j.parts[i];
                j.wbits = p.wbits;
                j.q = p.q;
                j.rscale = p.rscale;
                j.out = p.out;
                j.out_stride = p.out_stride;
                j.n = p.n;
                j.tiles = (p.n + kTile - 1u) / kTile;
                j.wscale = reinterpret_cast<const uint16_t*>(p.wbits + (size_t)j.tiles * j.groups * kTile);
                first = p.first;
            }
        }
    }
    return nt - first;
}

// 16 bytes per active lane from global memory into LDS at lds_addr + 16 * lane (the
// wave's LDS base goes in M0).  Inline assembly, so that the compiler's own wait
// insertion does not add a wait for every LDS DMA before each later LDS read: the
// kernel bounds the outstanding loads itself.  The s_nop covers the one wait state
// between writing M0 and the LDS DMA reading it.
__device__ __forceinline__ void dma16(const void* gptr, uint32_t lds_addr) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gptr), "{m0}"(lds_addr) : "memory");
}

// The same for the lanes of a constant mask only: the mask goes into exec inside the
// assembly (and exec is restored there), so that the caller needs no branch around
// the load -- a branch would split the loop body into blocks across which the
// compiler moves the arithmetic of one group into the next.
template <uint64_t LANES>
__device__ __forceinline__ void dma16_lanes(const void* gptr, uint32_t lds_addr) {
    if constexpr (LANES == ~0ull) {
        dma16(gptr, lds_addr);
    } else {
        uint64_t saved;
        asm volatile(
            "s_mov_b64 %0, exec\n\ts_mov_b64 exec, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
            "s_mov_b64 exec, %0"
            : "=&s"(saved)
            : "v"(gptr), "{m0}"(lds_addr), "s"(LANES)
            : "memory");
    }
}

// The same with the address as a wave-uniform base (SGPRs) plus a 32-bit per-lane
// offset: no 64-bit per-lane address arithmetic per DMA.
__device__ __forceinline__ void dma16_s(uint32_t voff, const void* sbase, uint32_t lds_addr) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(lds_addr) : "memory");
}

template <uint32_t N>
constexpr uint64_t lane_mask() {
    return N >= 64 ? ~0ull : (1ull << (N % 64u)) - 1ull;
}

__device__ __forceinline__ uint32_t lds_offset(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// A job's row scale through the global address space (a flat load would also count on the
// LDS counter that the kernels' LDS waits use).
__device__ __forceinline__ float row_scale(const GemmJob& j, uint32_t m) {
    return *(const __attribute__((address_space(1))) float*)(j.rscale + m);
}

// Output stores: nontemporal, or written through to memory (system-coherent, sc0 sc1) in a
// launch that signals its end itself (gemm_signal).
__device__ __forceinline__ void put(float* p, float v, bool through) {
    if (through)
        __hip_atomic_store((__attribute__((address_space(1))) float*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else
        __builtin_nontemporal_store(v, (__attribute__((address_space(1))) float*)p);
}
__device__ __forceinline__ void put4(void* p, v4i v, bool through) {
    if (through)
        asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
    else
        __builtin_nontemporal_store(v, (__attribute__((address_space(1))) v4i*)p);
}

__device__ __forceinline__ void put8(void* p, uint64_t v, bool through) {
    if (through)
        __hip_atomic_store((__attribute__((address_space(1))) uint64_t*)p, v, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    else
        *(__attribute__((address_space(1))) uint64_t*)p = v;
}
__device__ __forceinline__ void put2(void* p, uint16_t v, bool through) {
    if (through)
        asm volatile("global_store_short %0, %1, off sc0 sc1" ::"v"(p), "v"((uint32_t)v) : "memory");
    else
        *(__attribute__((address_space(1))) uint16_t*)p = v;
}
// two int16 at any even address
typedef uint32_t u32_at2 __attribute__((aligned(2)));
__device__ __forceinline__ void put2x2(void* p, uint32_t v, bool through) {
    if (through)
        asm volatile("global_store_dword %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
    else
        *(__attribute__((address_space(1))) u32_at2*)p = v;
}

// Workgroup barrier for data handed over in LDS: this wave's LDS accesses are done before it
// (s_barrier itself waits for none, and the compiler adds no wait on gfx950: another wave
// could read what is still on its way into LDS), and at most VM of its DMAs are in flight
// (63: any number).  The gfx9 encoding splits vmcnt into bits 3:0 and 15:14.
template <uint32_t VM = 63u>
__device__ __forceinline__ void lds_barrier() {
    static_assert(VM < 64u, "vmcnt field");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((int)((VM & 15u) | 0x0070u | ((VM >> 4) << 14)));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");  // no LDS access moves across it
}

// The end of a workgroup in a launch whose caller waits for it (GemmJob::done): once the
// stores of all its waves are complete (vmcnt), the workgroup stores seq into its own pinned
// host word; the host spins on those words instead of waiting for the end of the kernel, which
// the runtime reports several microseconds later (a call of 2048->6144 x 64 rows 20.6 -> 17.5
// us, 384->278 x 33 rows 19.0 -> 14.0).  Every thread of the workgroup comes here.
__device__ __forceinline__ void gemm_signal(const GemmJob& j, uint64_t seq) {
    if (j.done == nullptr)
        return;
    lds_barrier<0>();
    if (threadIdx.x == 0)
        __hip_atomic_store(j.done + blockIdx.x, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

uint32_t gemm_band(const GemmJob& job, uint32_t mtiles);
uint32_t gemm_ntiles(GemmJob& job, uint32_t tn);

// What every launcher passes on.
struct GemmLaunch {
    hipStream_t stream;
    uint64_t seq;
    const uint64_t* flag;
    uint32_t* signals;  // with job.done: receives the workgroups that signal
};

// One workgroup per tile.  Launches of more than kDoneWords workgroups, one per CU, do not
// signal.  Up to there it always paid (70 launches of 141..256 workgroups, 0.8 to 5.7 us a call:
// 1536->3000 x 160 rows, 235 workgroups, 21.7 -> 19.5 us); past it stores written through cost
// some launches more than the earlier word to the host saves (2048->8192 x 1500 rows, 768
// workgroups, 69.8 -> 70.2; 128->8000 x 700 dots, 693 of them, 23.1 -> 28.0), though not all
// (2048->8192 x 800 rows, 448 workgroups, 51.4 -> 49.6).
template <class Kernel>
hipError_t launch_tiles(const GemmLaunch& at, Kernel kernel, uint32_t threads, GemmJob& job, uint32_t mtiles,
                        uint32_t ntiles) {
    const uint32_t grid = mtiles * ntiles;
    if (grid > kDoneWords)
        job.done = nullptr;
    if (job.done)
        *at.signals = grid;
    launch_kernel(kernel, dim3(grid), dim3(threads), 0, at.stream, job, mtiles, ntiles, gemm_band(job, mtiles), at.seq,
                  at.flag);
    return hipGetLastError();
}


// k_gemm_ks: F32-accumulating jobs with too few tiles to give every CU a workgroup.
// Workgroup tile (16*TMS) x (16*TNS); the W waves split K instead of the tile: wave w
// computes groups w, w+W, w+2W, ... for the whole tile, its operands loaded from
// global memory straight into registers DEPTH-1 rounds ahead.  The K order inside a
// group is permuted so that a lane's share of a column's sign bits is 4 contiguous
// bytes: lane chunk c (lane / 16) covers weights 32c .. 32c+31, MFMA half h the 16
// starting at 32c + 16h, in the rows and the weights alike.  The bits of the next
// round become +1/-1 operands through the byte table while this round's MFMAs run.
// Per round each wave writes the exact products RN(scale * D) of its group to LDS;
// then every thread adds the W products of its outputs to its FP32 accumulators in
// group order -- the order of the sums is the reference's, only the integer work ran
// in parallel.
template <int TMS, int TNS>
struct KsOps {
    v4i a[TMS][2];
    uint32_t bits[TNS];
    uint16_t s[TNS];
    v4i b[TNS][2];  // the +1/-1 operands, from bits
};

__device__ __forceinline__ v4i gload_v4i(const void* p) {
    return *(const __attribute__((address_space(1))) v4i*)p;
}

template <int TMS, int TNS, int W, int DEPTH>
__global__ __launch_bounds__(64 * W) void k_gemm_ks(GemmJob j, uint32_t mtiles, uint32_t ntiles, uint32_t band,
    uint64_t seq,
                                                   const uint64_t* __restrict__ flag) {
    constexpr uint32_t TM = 16u * TMS, TN = 16u * TNS, SUBS = TMS * TNS, NT = 64u * W;
    constexpr uint32_t BLOCKS = SUBS * 64u;  // 16-byte blocks of products per wave
    constexpr uint32_t PER_THREAD = (BLOCKS + NT - 1u) / NT;
    static_assert(DEPTH >= 3, "the next round's bits loaded a round before their expansion");
    static_assert(TN <= 64, "a tile's columns lie in one 64-feature tile of the matrix layout");
    __shared__ __attribute__((aligned(16))) float prod[W][BLOCKS * 4u];  // [wave][subtile][lane][4]
    __shared__ uint2 lut[256];
    if (*flag == seq) {
        gemm_signal(j, seq);
        return;
    }
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    TileRC tile = gemm_tile_of_block(blockIdx.x, gridDim.x, mtiles, ntiles, band);
    tile.nt = select_part(j, tile.nt);
    const uint32_t mt = tile.mt, nt = tile.nt;
    const uint32_t m0 = mt * TM, n0 = nt * TN;
    // the row scales of this thread's outputs (F32 jobs), requested now (see k_gemm_kr)
    float rs[PER_THREAD][4];
#pragma unroll
    for (int i = 0; i < (int)PER_THREAD; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t m = m0 + 16u * ((W * i + wave) / TNS) + 4u * (lane >> 4) + r;
            rs[i][r] = j.mode == MODE_SUM_SCALED && W * i + wave < SUBS && m < j.rows ? row_scale(j, m) : 1.0f;
        }
    const uint32_t groups = j.groups;
    for (uint32_t i = tid; i < 256u; i += NT)
        lut[i] = make_uint2(pm1_nibble(i & 15u), pm1_nibble(i >> 4));

    // rows past the end are clamped (never stored); so is the matrix tile of columns
    // past the last tile
    const uint32_t chunk = lane >> 4;
    const uint8_t* a_ptr[TMS];
    const uint8_t* b_ptr[TNS];
    const uint16_t* s_ptr[TNS];
#pragma unroll
    for (int mi = 0; mi < TMS; ++mi) {
        const uint32_t m = min(m0 + 16u * mi + (lane & 15u), j.rows - 1u);
        a_ptr[mi] = reinterpret_cast<const uint8_t*>(j.q) + (size_t)m * j.k + 32u * chunk;
    }
#pragma unroll
    for (int ni = 0; ni < TNS; ++ni) {
        const uint32_t n = n0 + 16u * ni + (lane & 15u), st = min(n >> 6, j.tiles - 1u);
        b_ptr[ni] = reinterpret_cast<const uint8_t*>(j.wbits) + ((size_t)st * groups * kTile + (n & 63u)) * 16u +
                    4u * chunk;
        s_ptr[ni] = j.wscale + (size_t)st * groups * kTile + (n & 63u);
    }
    // loads are unconditional (group clamped into range) so that every path has the
    // same loads in flight
    auto load = [&](KsOps<TMS, TNS>& o, uint32_t round) {
        const uint32_t g = min(W * round + wave, groups - 1u);
#pragma unroll
        for (int mi = 0; mi < TMS; ++mi)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                o.a[mi][h] = gload_v4i(a_ptr[mi] + (size_t)g * kGroup + 16u * h);
#pragma unroll
        for (int ni = 0; ni < TNS; ++ni) {
            o.bits[ni] = *reinterpret_cast<const uint32_t*>(b_ptr[ni] + (size_t)g * kTile * 16u);
            o.s[ni] = s_ptr[ni][(size_t)g * kTile];
        }
    };
    auto expand = [&](KsOps<TMS, TNS>& o) {
#pragma unroll
        for (int ni = 0; ni < TNS; ++ni)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint2 lo = lut[(o.bits[ni] >> (16u * h)) & 0xffu];
                const uint2 hi = lut[(o.bits[ni] >> (16u * h + 8u)) & 0xffu];
                o.b[ni][h] = v4i{(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
            }
    };

    float acc[PER_THREAD][4];
#pragma unroll
    for (int i = 0; i < (int)PER_THREAD; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            acc[i][r] = 0.0f;
    const v4i c_init = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
    KsOps<TMS, TNS> o[DEPTH];

    // round r with its operands in o[d] (d = r % DEPTH)
    auto round = [&](int d, uint32_t r) {
        KsOps<TMS, TNS>& cur = o[d];
        load(o[(d + DEPTH - 1) % DEPTH], r + DEPTH - 1u);
        const uint32_t g = W * r + wave;
        float4 p[TMS][TNS];
        if (g < groups) {
#pragma unroll
            for (int ni = 0; ni < TNS; ++ni) {
                const float sc = __half2float(__ushort_as_half(cur.s[ni]));
                const float cneg = sc * -kMagicValue;  // exact
#pragma unroll
                for (int mi = 0; mi < TMS; ++mi) {
                    v4i dd = __builtin_amdgcn_mfma_i32_16x16x64_i8(cur.a[mi][0], cur.b[ni][0], c_init, 0, 0, 0);
                    dd = __builtin_amdgcn_mfma_i32_16x16x64_i8(cur.a[mi][1], cur.b[ni][1], dd, 0, 0, 0);
                    p[mi][ni].x = __builtin_fmaf(sc, __int_as_float(dd[0]), cneg);
                    p[mi][ni].y = __builtin_fmaf(sc, __int_as_float(dd[1]), cneg);
                    p[mi][ni].z = __builtin_fmaf(sc, __int_as_float(dd[2]), cneg);
                    p[mi][ni].w = __builtin_fmaf(sc, __int_as_float(dd[3]), cneg);
                }
            }
        }
        lds_barrier();               // the previous round's reads of prod are done
        expand(o[(d + 1) % DEPTH]);  // round r+1's operands, loaded one round ago
        if (g < groups) {
#pragma unroll
            for (int mi = 0; mi < TMS; ++mi)
#pragma unroll
                for (int ni = 0; ni < TNS; ++ni)
                    *reinterpret_cast<float4*>(&prod[wave][((mi * TNS + ni) * 64u + lane) * 4u]) = p[mi][ni];
        }
        lds_barrier();  // every wave's products are in LDS
#pragma unroll
        for (int w = 0; w < W; ++w) {
            if (W * r + w < groups) {
#pragma unroll
                for (int i = 0; i < (int)PER_THREAD; ++i) {
                    const uint32_t blk = NT * i + tid;
                    if (BLOCKS % NT == 0 || blk < BLOCKS) {
                        const float4 v = *reinterpret_cast<const float4*>(&prod[w][blk * 4u]);
                        acc[i][0] = acc[i][0] + v.x;
                        acc[i][1] = acc[i][1] + v.y;
                        acc[i][2] = acc[i][2] + v.z;
                        acc[i][3] = acc[i][3] + v.w;
                    }
                }
            }
        }
    };

#pragma unroll
    for (int d = 0; d + 1 < DEPTH; ++d)
        load(o[d], d);
    lds_barrier();  // the table is in LDS
    expand(o[0]);
    const uint32_t rounds = (groups + W - 1u) / W;
    // the round count is padded to a multiple of DEPTH with rounds of no groups
    for (uint32_t r = 0; r < rounds; r += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            round(d, r + d);
    }
    // stored in one of two forms, each without a branch per value
    const auto store = [&](auto through) {
        // block NT*i + tid is subtile W*i + wave, lane `lane`
#pragma unroll
        for (int i = 0; i < (int)PER_THREAD; ++i) {
            const uint32_t sub = W * i + wave;
            if (sub >= SUBS)
                continue;
            const uint32_t mi = sub / TNS, ni = sub % TNS;
            const uint32_t n = n0 + 16u * ni + (lane & 15u);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t m = m0 + 16u * mi + 4u * (lane >> 4) + r;
                if (m >= j.rows || n >= j.n)
                    continue;
                float* orow = reinterpret_cast<float*>(j.out + (size_t)m * j.out_stride);
                put(orow + n, j.mode == MODE_SUM_SCALED ? acc[i][r] * rs[i][r] : acc[i][r], through);
            }
        }
    };
    if (j.done)
        store(std::true_type{});
    else
        store(std::false_type{});
    gemm_signal(j, seq);
}

// k_gemm_wv: F32-accumulating jobs with few rows.  Every wave computes a (16*MS) x
// (16*NS) block of the output over the whole K on its own: its rows' quantised bytes,
// its columns' sign bits and scales come from global memory straight into a ring of
// DEPTH groups of registers; the bits become +1/-1 operands through the byte table
// (LDS, written once before the loop); no barrier or LDS exchange sits in the loop, so
// the waves of a CU run their chains independently and the latency of one group's
// loads is covered by the DEPTH-1 groups ahead of it.  The K order inside a group is
// that of k_gemm_ks (lane chunk c: weights 32c .. 32c+31, MFMA half h the 16 from
// 32c + 16h), so a lane's operands are 32 contiguous row bytes and 4 contiguous bytes
// of bits.  Group g's MFMAs write one of two D sets while group g-1's epilogue reads
// the other; each output element's products are added in group order by one thread.
// The group count is padded to a multiple of DEPTH with groups of scale 0 (the
// clamped last group's operands), whose products are +0 and leave the sums unchanged.
template <int MS, int NS>
struct WvOps {
    v4i a[MS][2];
    uint32_t bits[NS];
    uint32_t s[NS];
};

template <int MS, int NS, int WM, int WN, int DEPTH>
__global__ __launch_bounds__(64 * WM * WN) void k_gemm_wv(GemmJob j, uint32_t mtiles, uint32_t ntiles, uint32_t band,
                                                         uint64_t seq, const uint64_t* __restrict__ flag) {
    constexpr uint32_t TM = 16u * MS * WM, TN = 16u * NS * WN, NT = 64u * WM * WN;
    static_assert(DEPTH >= 2 && DEPTH % 2 == 0, "two D sets alternate with the ring slots");
    static_assert(16 * NS <= 64 && 64 % (16 * NS) == 0, "a wave's columns lie in one 64-feature tile");
    __shared__ uint2 lut[256];
    if (*flag == seq) {
        gemm_signal(j, seq);
        return;
    }
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave / WN, wn = wave % WN;
    TileRC tile = gemm_tile_of_block(blockIdx.x, gridDim.x, mtiles, ntiles, band);
    tile.nt = select_part(j, tile.nt);
    const uint32_t m0 = tile.mt * TM + 16u * MS * wm, n0 = tile.nt * TN + 16u * NS * wn;
    const uint32_t groups = j.groups;
    for (uint32_t i = tid; i < 256u; i += NT)
        lut[i] = make_uint2(pm1_nibble(i & 15u), pm1_nibble(i >> 4));

    // rows past the end are clamped (never stored); so is the matrix tile of columns
    // past the last tile
    const uint32_t chunk = lane >> 4;
    const uint8_t* a_ptr[MS];
    const uint8_t* b_ptr[NS];
    const uint16_t* s_ptr[NS];
#pragma unroll
    for (int mi = 0; mi < MS; ++mi) {
        const uint32_t m = min(m0 + 16u * mi + (lane & 15u), j.rows - 1u);
        a_ptr[mi] = reinterpret_cast<const uint8_t*>(j.q) + (size_t)m * j.k + 32u * chunk;
    }
#pragma unroll
    for (int ni = 0; ni < NS; ++ni) {
        const uint32_t n = n0 + 16u * ni + (lane & 15u), st = min(n >> 6, j.tiles - 1u);
        b_ptr[ni] = reinterpret_cast<const uint8_t*>(j.wbits) + ((size_t)st * groups * kTile + (n & 63u)) * 16u +
                    4u * chunk;
        s_ptr[ni] = j.wscale + (size_t)st * groups * kTile + (n & 63u);
    }
    // every load is unconditional (group clamped into range): the same loads are in
    // flight on every path
    auto load = [&](WvOps<MS, NS>& o, uint32_t g) {
        const uint32_t gc = min(g, groups - 1u);
#pragma unroll
        for (int mi = 0; mi < MS; ++mi)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                o.a[mi][h] = gload_v4i(a_ptr[mi] + (size_t)gc * kGroup + 16u * h);
#pragma unroll
        for (int ni = 0; ni < NS; ++ni) {
            o.bits[ni] = *reinterpret_cast<const uint32_t*>(b_ptr[ni] + (size_t)gc * kTile * 16u);
            o.s[ni] = s_ptr[ni][(size_t)gc * kTile];
        }
    };

    float acc[MS][NS][4];
    v4i dd[2][MS][NS];
    const v4i c_init = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
    float sc_prev[NS];
#pragma unroll
    for (int ni = 0; ni < NS; ++ni)
        sc_prev[ni] = 0.0f;  // the epilogue before group 0 adds +0
#pragma unroll
    for (int mi = 0; mi < MS; ++mi)
#pragma unroll
        for (int ni = 0; ni < NS; ++ni) {
            dd[1][mi][ni] = c_init;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[mi][ni][r] = 0.0f;
        }
    auto epilogue = [&](const v4i (&d)[MS][NS]) {
#pragma unroll
        for (int ni = 0; ni < NS; ++ni) {
            const float sc = sc_prev[ni];
            const float cneg = sc * -kMagicValue;  // exact
#pragma unroll
            for (int mi = 0; mi < MS; ++mi)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[mi][ni][r] = acc[mi][ni][r] + __builtin_fmaf(sc, __int_as_float(d[mi][ni][r]), cneg);
        }
    };

    WvOps<MS, NS> o[DEPTH];
#pragma unroll
    for (int d = 0; d + 1 < DEPTH; ++d)
        load(o[d], d);
    lds_barrier();  // the table is in LDS

    // group g = g0 + d from ring slot d: refill the slot emptied one group ago, expand
    // the bits, group g's MFMAs into D set d % 2, group g-1's epilogue from the other
    auto step = [&](int d, uint32_t g) {
        load(o[(d + DEPTH - 1) % DEPTH], g + DEPTH - 1u);
        const WvOps<MS, NS>& cur = o[d];
        v4i b[NS][2];
#pragma unroll
        for (int ni = 0; ni < NS; ++ni)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint2 lo = lut[(cur.bits[ni] >> (16u * h)) & 0xffu];
                const uint2 hi = lut[(cur.bits[ni] >> (16u * h + 8u)) & 0xffu];
                b[ni][h] = v4i{(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
            }
        v4i (&dn)[MS][NS] = dd[d & 1];
#pragma unroll
        for (int mi = 0; mi < MS; ++mi)
#pragma unroll
            for (int ni = 0; ni < NS; ++ni) {
                v4i x = __builtin_amdgcn_mfma_i32_16x16x64_i8(cur.a[mi][0], b[ni][0], c_init, 0, 0, 0);
                dn[mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(cur.a[mi][1], b[ni][1], x, 0, 0, 0);
            }
        epilogue(dd[(d & 1) ^ 1]);
#pragma unroll
        for (int ni = 0; ni < NS; ++ni)
            sc_prev[ni] = g < groups ? __half2float(__ushort_as_half((uint16_t)cur.s[ni])) : 0.0f;
    };
    for (uint32_t g0 = 0; g0 < groups; g0 += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            step(d, g0 + d);
    }
    epilogue(dd[(DEPTH - 1) & 1]);  // the last step's group

    // stored in one of two forms, each without a branch per value
    const auto store = [&](auto through) {
#pragma unroll
        for (int mi = 0; mi < MS; ++mi)
#pragma unroll
            for (int ni = 0; ni < NS; ++ni) {
                const uint32_t n = n0 + 16u * ni + (lane & 15u);
                if (n >= j.n)
                    continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t m = m0 + 16u * mi + 4u * (lane >> 4) + r;
                    if (m >= j.rows)
                        continue;
                    float* orow = reinterpret_cast<float*>(j.out + (size_t)m * j.out_stride);
                    put(orow + n, j.mode == MODE_SUM_SCALED ? acc[mi][ni][r] * j.rscale[m] : acc[mi][ni][r], through);
                }
            }
    };
    if (j.done)
        store(std::true_type{});
    else
        store(std::false_type{});
    gemm_signal(j, seq);
}

// k_gemm_dots<TNS, GB, WAVES>: DOT_GROUPS.  Every group's dots stand alone (no sum over groups), so a
// workgroup takes a 16 x (16 TNS) tile over the whole K, wave w the blocks of four
// groups w, w + WAVES, ... (at most GB blocks in all): a block's rows and sign bits are requested at
// once, straight into registers, expanded through the byte table, and each output's four dots
// go to LDS as 8 bytes.  A row's part of the tile, [column][group] int16, is one contiguous run
// of the output, so the tile leaves in 16- or 8-byte pieces of that run (4-byte ones at
// other alignments).  Bound by the launch for small jobs, by the stores for large ones; against
// the accumulating kernels' tiles storing 2 bytes per output and group from the loop: 896->1000
// x 37 rows 7.3 -> 5.3 us, 2048->2048 x 256 rows 27.7 -> 10.2, 8192->1000 x 64 rows 89.7 -> 11.3.
template <int TNS, int GB, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_gemm_dots(GemmJob j, uint32_t mtiles, uint32_t ntiles, uint32_t band,
                                                   uint64_t seq, const uint64_t* __restrict__ flag) {
    constexpr uint32_t TN = 16u * TNS, THREADS = 64u * WAVES;
    static_assert(THREADS >= 256u, "one thread per table entry");
    static_assert(64 % TN == 0, "the tile's columns lie in one 64-feature tile");
    // an output's dots: GB blocks of 8 bytes and 8 bytes that shift the next column's banks; for
    // group counts that are no multiple of 4, a row's run as it leaves instead (no gaps)
    constexpr uint32_t PITCH = 8u * GB + 8u, ROW = TN * PITCH;
    __shared__ __attribute__((aligned(16))) unsigned char dots[16u * ROW];
    __shared__ uint2 lut[256];
    if (*flag == seq) {
        gemm_signal(j, seq);
        return;
    }
    const uint32_t tid = threadIdx.x, lane = tid & 63u, chunk = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    TileRC tile = gemm_tile_of_block(blockIdx.x, gridDim.x, mtiles, ntiles, band);
    tile.nt = select_part(j, tile.nt);
    const bool through = j.done != nullptr;
    const uint32_t m0 = tile.mt * 16u, n0 = tile.nt * TN, groups = j.groups, blocks = (groups + 3u) / 4u;
    // rows past the end are clamped (never stored); so is the matrix tile of columns past the
    // last one.  The K order inside a group is that of k_gemm_ks / k_gemm_wv.
    const uint8_t* a_ptr = reinterpret_cast<const uint8_t*>(j.q) +
                           (size_t)min(m0 + (lane & 15u), j.rows - 1u) * j.k + 32u * chunk;
    const uint8_t* b_ptr[TNS];
#pragma unroll
    for (int ni = 0; ni < TNS; ++ni) {
        const uint32_t n = n0 + 16u * ni + (lane & 15u), st = min(n >> 6, j.tiles - 1u);
        b_ptr[ni] = reinterpret_cast<const uint8_t*>(j.wbits) + ((size_t)st * groups * kTile + (n & 63u)) * 16u +
                    4u * chunk;
    }
    v4i a[4][2];
    uint32_t bits[4][TNS];
    const auto load = [&](uint32_t b) {
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            const uint32_t g = min(4u * b + i, groups - 1u);
#pragma unroll
            for (int h = 0; h < 2; ++h)
                a[i][h] = gload_v4i(a_ptr + (size_t)g * kGroup + 16u * h);
#pragma unroll
            for (int ni = 0; ni < TNS; ++ni)
                bits[i][ni] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t*>(
                    (uintptr_t)(b_ptr[ni] + (size_t)g * kTile * 16u));
        }
    };
    load(min(wave, blocks - 1u));
    if (tid < 256u)
        lut[tid] = make_uint2(pm1_nibble(tid & 15u), pm1_nibble(tid >> 4));
    __syncthreads();
    const v4i zero = {0, 0, 0, 0};
    const bool gaps = groups % 4u == 0;
    for (uint32_t b = wave; b < blocks; b += WAVES) {
        v4i d[4][TNS];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
#pragma unroll
            for (int ni = 0; ni < TNS; ++ni) {
                const uint32_t w = bits[i][ni];
                const uint2 e0 = lut[w & 0xffu], e1 = lut[(w >> 8) & 0xffu], e2 = lut[(w >> 16) & 0xffu], e3 = lut[w >> 24];
                const v4i b0 = {(int)e0.x, (int)e0.y, (int)e1.x, (int)e1.y}, b1 = {(int)e2.x, (int)e2.y, (int)e3.x, (int)e3.y};
                const v4i x = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][0], b0, zero, 0, 0, 0);
                d[i][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][1], b1, x, 0, 0, 0);
            }
        if (b + WAVES < blocks)
            load(b + WAVES);  // the next block's operands, in flight during the stores
#pragma unroll
        for (int ni = 0; ni < TNS; ++ni)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t row = 4u * chunk + r, col = 16u * ni + (lane & 15u);
                if (gaps) {
                    uint2 v;
                    v.x = ((uint32_t)d[0][ni][r] & 0xffffu) | ((uint32_t)d[1][ni][r] << 16);
                    v.y = ((uint32_t)d[2][ni][r] & 0xffffu) | ((uint32_t)d[3][ni][r] << 16);
                    *reinterpret_cast<uint2*>(dots + row * ROW + col * PITCH + 8u * b) = v;
                } else {
                    uint16_t* run = reinterpret_cast<uint16_t*>(dots + row * ROW) + col * groups + 4u * b;
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i)
                        if (4u * b + i < groups)
                            run[i] = (uint16_t)d[i][ni][r];
                }
            }
    }
    __syncthreads();
    // the rows' runs: row r of the tile holds cols x groups int16 from out + r * stride + 2 n0 groups
    const uint32_t cols = min(TN, j.n - n0), rows = min(16u, j.rows - m0);
    unsigned char* const out = j.out + (size_t)m0 * j.out_stride + (size_t)n0 * groups * 2u;
    const uint64_t align = j.out_stride | (uint64_t)(uintptr_t)out;
    // piece p of the tile: elements of `per` groups each, `pieces` per row
    const auto each = [&](uint32_t pieces, auto&& store) {
        for (uint32_t i = tid; i < rows * pieces; i += THREADS) {
            const uint32_t row = i / pieces, p = i - row * pieces;
            store(row, p, out + (size_t)row * j.out_stride);
        }
    };
    if (groups % 8u == 0 && (align & 15u) == 0) {
        const uint32_t per = groups / 8u;
        each(cols * per, [&](uint32_t row, uint32_t p, unsigned char* run) {
            const uint32_t col = p / per, g = p - col * per;
            const uint2* src = reinterpret_cast<const uint2*>(dots + row * ROW + col * PITCH + 16u * g);
            const uint2 lo = src[0], hi = src[1];
            const v4i v = {(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
            put4(run + 16u * p, v, through);
        });
    } else if (groups % 4u == 0 && (align & 7u) == 0) {
        const uint32_t per = groups / 4u;
        each(cols * per, [&](uint32_t row, uint32_t p, unsigned char* run) {
            const uint32_t col = p / per, g = p - col * per;
            put8(run + 8u * p, *reinterpret_cast<const uint64_t*>(dots + row * ROW + col * PITCH + 8u * g), through);
        });
    } else if (!gaps && (align & 15u) == 0) {
        const uint32_t bytes = cols * groups * 2u;
        each((bytes + 15u) / 16u, [&](uint32_t row, uint32_t p, unsigned char* run) {
            const unsigned char* src = dots + row * ROW + 16u * p;
            if (16u * p + 16u <= bytes) {
                const v4i v = *reinterpret_cast<const v4i*>(src);
                put4(run + 16u * p, v, through);
            } else {
                for (uint32_t i = 16u * p; i < bytes; i += 2u)
                    put2(run + i, *reinterpret_cast<const uint16_t*>(dots + row * ROW + i), through);
            }
        });
    } else {  // any other alignment: two values at a time, the last of an odd number alone
        const uint32_t bytes = cols * groups * 2u, per = groups / 2u;
        each((bytes + 3u) / 4u, [&](uint32_t row, uint32_t p, unsigned char* run) {
            uint32_t at = 4u * p;
            if (gaps) {
                const uint32_t col = p / per;
                at = col * PITCH + 4u * (p - col * per);
            }
            const unsigned char* src = dots + row * ROW + at;
            if (4u * p + 4u <= bytes)
                put2x2(run + 4u * p, *reinterpret_cast<const uint32_t*>(src), through);
            else
                put2(run + 4u * p, *reinterpret_cast<const uint16_t*>(src), through);
        });
    }
    gemm_signal(j, seq);
}

// k_gemm_dotf<MS, NS, GC>: DOT_GROUPS of up to 8 groups.  With so few groups a tile over the
// whole K (k_gemm_dots) has next to nothing to compute, and its table, barriers and staging are
// most of a workgroup's time; here each of a workgroup's four waves takes a (16 MS) x (16 NS)
// block by itself, GC groups at a time: their rows and sign bits straight into registers, then
// each output's GC dots straight from the registers to memory, 2 GC contiguous bytes (two dots
// at a time and the last one alone where the group count is no multiple of GC).  Bound by the
// stores for large jobs; calls of 128->8000 x 700 rows 58.6 -> 22.1 us against k_gemm_dots,
// 256->2417 x 383 29.1 -> 17.5, 512->1001 x 200 22.4 -> 16.8, 896->6046 x 106 29.5 -> 24.8.
template <int MS, int NS, int GC>
__global__ __launch_bounds__(256) void k_gemm_dotf(GemmJob j, uint32_t mtiles, uint32_t ntiles, uint32_t band,
                                                   uint64_t seq, const uint64_t* __restrict__ flag) {
    static_assert(GC == 1 || GC == 2 || GC == 4, "dots per store");
    constexpr uint32_t TM = 32u * MS, TN = 32u * NS;
    __shared__ uint2 lut[256];
    const uint64_t failed_seq = *flag;  // checked before anything is stored
    const uint32_t tid = threadIdx.x, lane = tid & 63u, chunk = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    TileRC tile = gemm_tile_of_block(blockIdx.x, gridDim.x, mtiles, ntiles, band);
    tile.nt = select_part(j, tile.nt);
    const uint32_t m0 = tile.mt * TM + 16u * MS * (wave >> 1), n0 = tile.nt * TN + 16u * NS * (wave & 1u);
    const uint32_t groups = j.groups;
    // rows past the end are clamped (never stored); so is the matrix tile of columns past the
    // last one.  The K order inside a group is that of k_gemm_ks / k_gemm_wv.
    const uint8_t* a_ptr[MS];
    const uint8_t* b_ptr[NS];
#pragma unroll
    for (int mi = 0; mi < MS; ++mi)
        a_ptr[mi] = reinterpret_cast<const uint8_t*>(j.q) +
                    (size_t)min(m0 + 16u * mi + (lane & 15u), j.rows - 1u) * j.k + 32u * chunk;
#pragma unroll
    for (int ni = 0; ni < NS; ++ni) {
        const uint32_t n = n0 + 16u * ni + (lane & 15u), st = min(n >> 6, j.tiles - 1u);
        b_ptr[ni] = reinterpret_cast<const uint8_t*>(j.wbits) + ((size_t)st * groups * kTile + (n & 63u)) * 16u +
                    4u * chunk;
    }
    v4i a[GC][MS][2];
    uint32_t bits[GC][NS];
    const auto load = [&](uint32_t g0) {
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t)GC; ++i) {
            const uint32_t g = min(g0 + i, groups - 1u);
#pragma unroll
            for (int mi = 0; mi < MS; ++mi)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    a[i][mi][h] = gload_v4i(a_ptr[mi] + (size_t)g * kGroup + 16u * h);
#pragma unroll
            for (int ni = 0; ni < NS; ++ni)
                bits[i][ni] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t*>(
                    (uintptr_t)(b_ptr[ni] + (size_t)g * kTile * 16u));
        }
    };
    load(0);
    lut[tid] = make_uint2(pm1_nibble(tid & 15u), pm1_nibble(tid >> 4));
    lds_barrier();  // the table is in LDS
    if (failed_seq == seq) {
        gemm_signal(j, seq);
        return;
    }
    const v4i zero = {0, 0, 0, 0};
    const bool at8 = ((j.out_stride | (uint64_t)(uintptr_t)j.out) & 7u) == 0;  // and 8 bytes per 4 groups
    // in one of two forms, each without a branch per store
    const auto run = [&](auto through) {
        for (uint32_t g0 = 0; g0 < groups; g0 += GC) {
            v4i d[GC][MS][NS];
#pragma unroll
            for (int i = 0; i < GC; ++i)
#pragma unroll
                for (int ni = 0; ni < NS; ++ni) {
                    const uint32_t w = bits[i][ni];
                    const uint2 e0 = lut[w & 0xffu], e1 = lut[(w >> 8) & 0xffu], e2 = lut[(w >> 16) & 0xffu], e3 = lut[w >> 24];
                    const v4i b0 = {(int)e0.x, (int)e0.y, (int)e1.x, (int)e1.y}, b1 = {(int)e2.x, (int)e2.y, (int)e3.x, (int)e3.y};
#pragma unroll
                    for (int mi = 0; mi < MS; ++mi) {
                        const v4i x = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][mi][0], b0, zero, 0, 0, 0);
                        d[i][mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][mi][1], b1, x, 0, 0, 0);
                    }
                }
            if (g0 + GC < groups)
                load(g0 + GC);  // the next groups' operands, in flight during the stores
            const auto pair = [&](int i, int mi, int ni, int r) {
                return ((uint32_t)d[i][mi][ni][r] & 0xffffu) | ((uint32_t)d[(i + 1) % GC][mi][ni][r] << 16);
            };
#pragma unroll
            for (int mi = 0; mi < MS; ++mi)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t m = m0 + 16u * mi + 4u * chunk + r;
                    unsigned char* const row = j.out + (size_t)m * j.out_stride + 2u * g0;
#pragma unroll
                    for (int ni = 0; ni < NS; ++ni) {
                        const uint32_t n = n0 + 16u * ni + (lane & 15u);
                        if (m >= j.rows || n >= j.n)
                            continue;
                        unsigned char* const to = row + (size_t)n * groups * 2u;
                        if (GC == 1 || g0 + GC > groups) {  // one group, or the last of an odd number
                            put2(to, (uint16_t)d[0][mi][ni][r], through);
                        } else if (GC == 4 && at8) {
                            put8(to, pair(0, mi, ni, r) | ((uint64_t)pair(2 % GC, mi, ni, r) << 32), through);
                        } else {
#pragma unroll
                            for (int i = 0; i + 1 < GC; i += 2)
                                put2x2(to + 2u * i, pair(i, mi, ni, r), through);
                        }
                    }
                }
        }
    };
    if (j.done)
        run(std::true_type{});
    else
        run(std::false_type{});
    gemm_signal(j, seq);
}

// k_gemm_kr<TMS, TNS, W, R>: F32-accumulating jobs with few rows, whose tiles are too
// few to hide a chain of per-group steps.  Workgroup tile (16 TMS) x (16 TNS); the W
// waves split K (round r of wave w: group W r + w, at most R rounds), and each wave
// requests everything its own groups need -- the tile rows' quantised bytes, the
// columns' sign bits and scales -- into its own part of LDS by DMA before it computes
// anything: no registers are held while the loads are in flight, and no wave reads
// another wave's part, so a round waits for the wave's own loads (vmcnt) and for no
// barrier.  A round expands the bits through the byte table, runs the MFMAs and keeps
// the exact products RN(scale * D) in registers.  After the last round: one barrier,
// every wave's products into LDS by group, a second barrier, and each output's products
// added in group order by one thread -- the reference's order; only the integer work
// ran in parallel.  The K order inside a group is that of k_gemm_ks (lane chunk c:
// weights 32c .. 32c+31, MFMA half h the 16 from 32c + 16h).
template <int TMS, int TNS, int W, int R>
struct KrLayout {
    static constexpr uint32_t TM = 16u * TMS, TN = 16u * TNS, SUBS = TMS * TNS, NT = 64u * W;
    // a round's part: rows [TM][128] (chunks swizzled as swz128), the columns' 16-byte
    // sign-bit chunks [TN][16], their fp16 scales [TN]
    static constexpr uint32_t A_BYTES = TM * 128u, A_INS = A_BYTES / 1024u;
    static constexpr uint32_t BITS_BYTES = TN * 16u, SC_BYTES = TN * 2u, SC_LANES = SC_BYTES / 16u;
    static constexpr uint32_t ROUND_BYTES = A_BYTES + BITS_BYTES + SC_BYTES;
    static constexpr uint32_t DMA_PER_ROUND = A_INS + 2u;
    static constexpr uint32_t OPS_BYTES = W * R * ROUND_BYTES;
    static constexpr uint32_t PROD_BYTES = W * R * SUBS * 1024u;  // float4 [group][subtile][lane]
    // the byte table after the operands (copies of it, one per lane group, measured no
    // faster: the larger LDS footprint costs more than the bank conflicts); the products
    // reuse both once every wave is done with them
    static constexpr uint32_t OFF_LUT = OPS_BYTES;
    static constexpr uint32_t SMEM = OPS_BYTES + 2048u > PROD_BYTES ? OPS_BYTES + 2048u : PROD_BYTES;
    static_assert(A_BYTES % 1024u == 0, "whole 1 KiB row DMAs");
    static_assert(TN <= 64u && 64u % TN == 0, "a tile's columns lie in one 64-feature tile of the matrix layout");
    static_assert(SC_BYTES % 16u == 0, "whole 16-byte scale DMAs");
    static_assert(R * DMA_PER_ROUND < 64u, "vmcnt range");
    static_assert(SMEM <= 160u * 1024u, "LDS");
};

// One round's operands of a lane, read from LDS
template <int TMS, int TNS>
struct KrOps {
    v4i a[TMS][2];
    uint32_t bits[TNS];
    uint32_t s[TNS];
};

// f(std::integral_constant<uint32_t, i>) for i = 0 .. N-1, each i a constant expression
template <class F, uint32_t... I>
__device__ __forceinline__ void static_for_seq(F&& f, std::integer_sequence<uint32_t, I...>) {
    (f(std::integral_constant<uint32_t, I>{}), ...);
}
template <uint32_t N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_seq(f, std::make_integer_sequence<uint32_t, N>{});
}

// s_waitcnt vmcnt(N) alone (lgkmcnt and expcnt not waited for); the gfx9 encoding
// splits vmcnt into bits 3:0 and 15:14
template <uint32_t N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N < 64u, "vmcnt field");
    __builtin_amdgcn_s_waitcnt((int)((N & 15u) | 0x0F70u | ((N >> 4) << 14)));
}

// dma16_s for the lanes of a constant mask only (exec set inside the assembly)
template <uint64_t LANES>
__device__ __forceinline__ void dma16_s_lanes(uint32_t voff, const void* sbase, uint32_t lds_addr) {
    if constexpr (LANES == ~0ull) {
        dma16_s(voff, sbase, lds_addr);
    } else {
        uint64_t saved;
        asm volatile(
            "s_mov_b64 %0, exec\n\ts_mov_b64 exec, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\t"
            "s_mov_b64 exec, %0"
            : "=&s"(saved)
            : "v"(voff), "s"(sbase), "{m0}"(lds_addr), "s"(LANES)
            : "memory");
    }
}

template <int TMS, int TNS, int W, int R>
__global__ __launch_bounds__(64 * W) void k_gemm_kr(GemmJob j, uint32_t mtiles, uint32_t ntiles, uint32_t band,
                                                   uint64_t seq, const uint64_t* __restrict__ flag) {
    typedef KrLayout<TMS, TNS, W, R> T;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[T::SMEM];
    // the job's error flag is read now and checked before anything is stored: the DMAs
    // below read only memory of the job, so they need not wait for it
    const uint64_t failed_seq = *flag;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    TileRC tile = gemm_tile_of_block(blockIdx.x, gridDim.x, mtiles, ntiles, band);
    tile.nt = select_part(j, tile.nt);
    const uint32_t m0 = tile.mt * T::TM, n0 = tile.nt * T::TN;
    const uint32_t groups = j.groups;
    // the row scales of this thread's outputs (F32 jobs; the prep launch wrote them),
    // requested now: read at the store they had added a memory round trip after the sums
    constexpr uint32_t ELEMS = T::SUBS * 256u, ITEMS = (ELEMS + T::NT - 1u) / T::NT;
    float rs[ITEMS];
#pragma unroll
    for (uint32_t it = 0; it < ITEMS; ++it) {
        const uint32_t idx = T::NT * it + tid;
        const uint32_t blk = idx >> 2, e = idx & 3u, mi = (blk >> 6) / TNS;
        const uint32_t m = m0 + 16u * mi + 4u * ((blk & 63u) >> 4) + e;
        rs[it] = j.mode == MODE_SUM_SCALED && idx < ELEMS && m < j.rows ? row_scale(j, m) : 1.0f;
    }

    // 1. every round's DMAs.  Rows: position p = 64 i + lane of the 1 KiB DMA i holds
    // chunk (p & 7) ^ ((row >> 1) & 7) of row p >> 3, so that chunk c of row r sits at
    // swz128(r, c); rows past the end are clamped (never stored).  Columns: the tile's
    // TN 16-byte sign-bit chunks and TN scales are contiguous per group in the matrix
    // layout (one 64-feature tile; the tile past the last one is clamped).  Groups past
    // the last are clamped too, so that every path issues the same DMAs for the waits.
    const uint32_t part = lds_offset(smem) + wave * (R * T::ROUND_BYTES);
    uint32_t a_src[T::A_INS];
#pragma unroll
    for (uint32_t i = 0; i < T::A_INS; ++i) {
        const uint32_t p = 64u * i + lane, r = p >> 3;
        a_src[i] = min(m0 + r, j.rows - 1u) * j.k + 16u * ((p & 7u) ^ ((r >> 1) & 7u));
    }
    const uint32_t col0 = min(n0 >> 6, j.tiles - 1u) * groups * kTile + (n0 & 63u);
    const uint32_t bits_off = (col0 + min(lane, T::TN - 1u)) * 16u;
    const uint32_t sc_off = col0 * 2u + 16u * min(lane, T::SC_LANES - 1u);
    const uint32_t chunk = lane >> 4, lrow = lane & 15u;
#pragma unroll
    for (uint32_t r = 0; r < (uint32_t)R; ++r) {
        const uint32_t g = min(W * r + wave, groups - 1u);
        const uint32_t slot = part + r * T::ROUND_BYTES;
        const int8_t* qg = j.q + (size_t)g * kGroup;
#pragma unroll
        for (uint32_t i = 0; i < T::A_INS; ++i)
            dma16_s(a_src[i], qg, slot + 1024u * i);
        dma16_s_lanes<lane_mask<T::TN>()>(bits_off + g * (kTile * 16u), j.wbits, slot + T::A_BYTES);
        dma16_s_lanes<lane_mask<T::SC_LANES>()>(sc_off + g * (kTile * 2u), j.wscale,
                                                slot + T::A_BYTES + T::BITS_BYTES);
    }
    uint2* const lut = reinterpret_cast<uint2*>(smem + T::OFF_LUT);
    for (uint32_t i = tid; i < 256u; i += T::NT)
        lut[i] = make_uint2(pm1_nibble(i & 15u), pm1_nibble(i >> 4));
    lds_barrier();  // the table is in LDS

    // 2. the rounds, software-pipelined: iteration i reads round i's operands from LDS
    // (after waiting for this wave's DMAs of round i: at most (R - 1 - i) rounds of them
    // still in flight), expands round i-1's sign bits through the byte table, and runs
    // round i-2's MFMAs with the exact products RN(scale * D) kept in registers
    const unsigned char* const mine = smem + wave * (R * T::ROUND_BYTES);
    const v4i c_init = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
    v4f p[R][TMS][TNS];
    KrOps<TMS, TNS> raw[3];
    v4i b[2][TNS][2];
    const auto read = [&](auto rc) {
        constexpr uint32_t r = decltype(rc)::value;
        KrOps<TMS, TNS>& o = raw[r % 3u];
        const unsigned char* const slot = mine + r * T::ROUND_BYTES;
        wait_vm<((uint32_t)R - 1u - r) * T::DMA_PER_ROUND>();
#pragma unroll
        for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi)
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h)
                o.a[mi][h] = *reinterpret_cast<const v4i*>(slot + swz128(16u * mi + lrow, 2u * chunk + h));
#pragma unroll
        for (uint32_t ni = 0; ni < (uint32_t)TNS; ++ni) {
            const uint32_t f = 16u * ni + lrow;
            o.bits[ni] = *reinterpret_cast<const uint32_t*>(slot + T::A_BYTES + 16u * f + 4u * chunk);
            o.s[ni] = *reinterpret_cast<const uint16_t*>(slot + T::A_BYTES + T::BITS_BYTES + 2u * f);
        }
    };
    const auto expand = [&](auto rc) {
        constexpr uint32_t r = decltype(rc)::value;
        const KrOps<TMS, TNS>& o = raw[r % 3u];
#pragma unroll
        for (uint32_t ni = 0; ni < (uint32_t)TNS; ++ni)
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h) {
                const uint2 lo = lut[(o.bits[ni] >> (16u * h)) & 0xffu];
                const uint2 hi = lut[(o.bits[ni] >> (16u * h + 8u)) & 0xffu];
                b[r % 2u][ni][h] = v4i{(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
            }
    };
    const auto mma = [&](auto rc) {
        constexpr uint32_t r = decltype(rc)::value;
        const KrOps<TMS, TNS>& o = raw[r % 3u];
#pragma unroll
        for (uint32_t ni = 0; ni < (uint32_t)TNS; ++ni) {
            const float sc = __half2float(__ushort_as_half((uint16_t)o.s[ni]));
            const float cneg = sc * -kMagicValue;  // exact
#pragma unroll
            for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi) {
                v4i dd = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a[mi][0], b[r % 2u][ni][0], c_init, 0, 0, 0);
                dd = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a[mi][1], b[r % 2u][ni][1], dd, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    p[r][mi][ni][e] = __builtin_fmaf(sc, __int_as_float(dd[e]), cneg);
            }
        }
    };
    static_for<(uint32_t)R + 2u>([&](auto ic) {
        constexpr uint32_t i = decltype(ic)::value;
        if constexpr (i < (uint32_t)R)
            read(std::integral_constant<uint32_t, i>{});
        if constexpr (i >= 1u && i - 1u < (uint32_t)R)
            expand(std::integral_constant<uint32_t, i - 1u>{});
        if constexpr (i >= 2u)
            mma(std::integral_constant<uint32_t, i - 2u>{});
    });

    if (failed_seq == seq) {  // an illegal input row in this job: write nothing (the whole workgroup)
        gemm_signal(j, seq);
        return;
    }

    // 3. the products by group into LDS (over the operands: every wave has read its own
    // by the barrier), then the in-order sums
    __syncthreads();
    v4f* const prod = reinterpret_cast<v4f*>(smem);
#pragma unroll
    for (uint32_t r = 0; r < (uint32_t)R; ++r) {
        const uint32_t g = W * r + wave;
        if (g < groups) {
#pragma unroll
            for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi)
#pragma unroll
                for (uint32_t ni = 0; ni < (uint32_t)TNS; ++ni)
                    prod[(g * T::SUBS + mi * TNS + ni) * 64u + lane] = p[r][mi][ni];
        }
    }
    __syncthreads();
    // output elements tid, tid + NT, ... (element e of block (subtile, lane l) is
    // 4 (64 subtile + l) + e), their sums interleaved
    const bool scaled = j.mode == MODE_SUM_SCALED;
    const float* const prodf = reinterpret_cast<const float*>(smem) + tid;
    float acc[ITEMS];
#pragma unroll
    for (uint32_t it = 0; it < ITEMS; ++it)
        acc[it] = 0.0f;
    const auto add_group = [&](uint32_t g) {
        float v[ITEMS];
#pragma unroll
        for (uint32_t it = 0; it < ITEMS; ++it)
            v[it] = ELEMS % T::NT == 0 || T::NT * it + tid < ELEMS ? prodf[g * ELEMS + T::NT * it] : 0.0f;
#pragma unroll
        for (uint32_t it = 0; it < ITEMS; ++it)
            acc[it] = acc[it] + v[it];
    };
    uint32_t g = 0;
    for (; g + 4u <= groups; g += 4u) {
        add_group(g);
        add_group(g + 1u);
        add_group(g + 2u);
        add_group(g + 3u);
    }
    for (; g < groups; ++g)
        add_group(g);
    // stored in one of two forms, each without a branch per value
    const auto store = [&](auto through) {
#pragma unroll
        for (uint32_t it = 0; it < ITEMS; ++it) {
            const uint32_t idx = T::NT * it + tid;
            const uint32_t blk = idx >> 2, e = idx & 3u, sub = blk >> 6, l = blk & 63u;
            const uint32_t mi = sub / TNS, ni = sub % TNS;
            const uint32_t n = n0 + 16u * ni + (l & 15u), m = m0 + 16u * mi + 4u * (l >> 4) + e;
            if (idx >= ELEMS || n >= j.n || m >= j.rows)
                continue;
            float* orow = reinterpret_cast<float*>(j.out + (size_t)m * j.out_stride);
            put(orow + n, scaled ? acc[it] * rs[it] : acc[it], through);
        }
    };
    if (j.done)
        store(std::true_type{});
    else
        store(std::false_type{});
    gemm_signal(j, seq);
}

// k_gemm_kc<TMS, TNW, WN, KS, G>: F32-accumulating jobs with few rows and at most G
// groups, as k_gemm_kr but with contiguous K slices handing on an accumulator instead
// of exchanging every product.  Workgroup tile (16 TMS) x (16 TNW WN); wave w = s WN + nn
// computes the 16 TMS x 16 TNW block nn of the tile over K slice s (groups s G/KS ..
// (s+1) G/KS - 1).  All waves first bring every group's rows, sign bits and scales into
// LDS by DMA (wave w the groups w, w + W, ...), one barrier; then each wave computes its
// products RN(scale * D) in registers; slice 0 adds its products in group order from +0,
// and each later slice, after a barrier, takes the running sums through LDS and adds its
// own in group order -- the reference's order with only KS - 1 exchanges of one value
// per output.  The K order inside a group is that of k_gemm_ks.
template <int TMS, int TNW, int WN, int KS, int G>
struct KcLayout {
    static constexpr uint32_t W = WN * KS, NT = 64u * W, GS = G / KS;
    static constexpr uint32_t TM = 16u * TMS, TN = 16u * TNW * WN;
    static constexpr uint32_t A_BYTES = TM * 128u, A_INS = A_BYTES / 1024u;
    static constexpr uint32_t BITS_BYTES = TN * 16u, SC_BYTES = TN * 2u, SC_LANES = SC_BYTES / 16u;
    static constexpr uint32_t ROUND_BYTES = A_BYTES + BITS_BYTES + SC_BYTES;
    static constexpr uint32_t RD = (G + W - 1u) / W;  // DMA rounds per wave
    static constexpr uint32_t OPS_BYTES = G * ROUND_BYTES;
    static constexpr uint32_t OFF_LUT = OPS_BYTES, OFF_X = OFF_LUT + 2048u;
    static constexpr uint32_t SMEM = OFF_X + WN * TMS * TNW * 1024u;
    static_assert(G % KS == 0, "whole K slices");
    static_assert(A_BYTES % 1024u == 0, "whole 1 KiB row DMAs");
    static_assert(TN <= 64u && 64u % TN == 0, "a tile's columns lie in one 64-feature tile of the matrix layout");
    static_assert(SC_BYTES % 16u == 0, "whole 16-byte scale DMAs");
    static_assert(RD * (A_INS + 2u) < 64u, "vmcnt range");
    static_assert(SMEM <= 160u * 1024u, "LDS");
};

template <int TMS, int TNW, int WN, int KS, int G>
__global__ __launch_bounds__(64 * WN * KS) void k_gemm_kc(GemmJob j, uint32_t mtiles, uint32_t ntiles, uint32_t band,
                                                         uint64_t seq, const uint64_t* __restrict__ flag) {
    typedef KcLayout<TMS, TNW, WN, KS, G> T;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[T::SMEM];
    // the job's error flag, checked before anything is stored (the DMAs read only the job's
    // own memory, so they need not wait for it)
    const uint64_t failed_seq = *flag;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    TileRC tile = gemm_tile_of_block(blockIdx.x, gridDim.x, mtiles, ntiles, band);
    tile.nt = select_part(j, tile.nt);
    const uint32_t m0 = tile.mt * T::TM, n0 = tile.nt * T::TN;
    // the row scales of this thread's outputs (F32 jobs), requested now (see k_gemm_kr)
    float rs[TMS][4];
#pragma unroll
    for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi)
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) {
            const uint32_t m = m0 + 16u * mi + 4u * (lane >> 4) + e;
            rs[mi][e] = j.mode == MODE_SUM_SCALED && m < j.rows ? row_scale(j, m) : 1.0f;
        }
    const uint32_t groups = j.groups;

    // 1. the DMAs (the layout of a group as in k_gemm_kr; group g at g * ROUND_BYTES).
    // Groups past the last are clamped: the copies write the same bytes.
    uint32_t a_src[T::A_INS];
#pragma unroll
    for (uint32_t i = 0; i < T::A_INS; ++i) {
        const uint32_t p = 64u * i + lane, r = p >> 3;
        a_src[i] = min(m0 + r, j.rows - 1u) * j.k + 16u * ((p & 7u) ^ ((r >> 1) & 7u));
    }
    const uint32_t col0 = min(n0 >> 6, j.tiles - 1u) * groups * kTile + (n0 & 63u);
    const uint32_t bits_off = (col0 + min(lane, T::TN - 1u)) * 16u;
    const uint32_t sc_off = col0 * 2u + 16u * min(lane, T::SC_LANES - 1u);
    const uint32_t base = lds_offset(smem);
#pragma unroll
    for (uint32_t r = 0; r < T::RD; ++r) {
        const uint32_t g = min(T::W * r + wave, groups - 1u);
        const uint32_t slot = base + g * T::ROUND_BYTES;
        const int8_t* qg = j.q + (size_t)g * kGroup;
#pragma unroll
        for (uint32_t i = 0; i < T::A_INS; ++i)
            dma16_s(a_src[i], qg, slot + 1024u * i);
        dma16_s_lanes<lane_mask<T::TN>()>(bits_off + g * (kTile * 16u), j.wbits, slot + T::A_BYTES);
        dma16_s_lanes<lane_mask<T::SC_LANES>()>(sc_off + g * (kTile * 2u), j.wscale,
                                                slot + T::A_BYTES + T::BITS_BYTES);
    }
    uint2* const lut = reinterpret_cast<uint2*>(smem + T::OFF_LUT);
    for (uint32_t i = tid; i < 256u; i += T::NT)
        lut[i] = make_uint2(pm1_nibble(i & 15u), pm1_nibble(i >> 4));
    lds_barrier<0>();  // every wave's DMAs and the table are in LDS

    // 2. this wave's products over its K slice, software-pipelined as in k_gemm_kr
    const uint32_t nn = wave % WN, s = wave / WN, g0 = s * T::GS;
    const uint32_t chunk = lane >> 4, lrow = lane & 15u;
    const v4i c_init = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
    v4f p[T::GS][TMS][TNW];
    KrOps<TMS, TNW> raw[3];
    v4i b[2][TNW][2];
    const auto read = [&](auto ic) {
        constexpr uint32_t i = decltype(ic)::value;
        KrOps<TMS, TNW>& o = raw[i % 3u];
        const unsigned char* const slot = smem + min(g0 + i, groups - 1u) * T::ROUND_BYTES;
#pragma unroll
        for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi)
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h)
                o.a[mi][h] = *reinterpret_cast<const v4i*>(slot + swz128(16u * mi + lrow, 2u * chunk + h));
#pragma unroll
        for (uint32_t ni = 0; ni < (uint32_t)TNW; ++ni) {
            const uint32_t f = 16u * (nn * TNW + ni) + lrow;
            o.bits[ni] = *reinterpret_cast<const uint32_t*>(slot + T::A_BYTES + 16u * f + 4u * chunk);
            o.s[ni] = *reinterpret_cast<const uint16_t*>(slot + T::A_BYTES + T::BITS_BYTES + 2u * f);
        }
    };
    const auto expand = [&](auto ic) {
        constexpr uint32_t i = decltype(ic)::value;
        const KrOps<TMS, TNW>& o = raw[i % 3u];
#pragma unroll
        for (uint32_t ni = 0; ni < (uint32_t)TNW; ++ni)
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h) {
                const uint2 lo = lut[(o.bits[ni] >> (16u * h)) & 0xffu];
                const uint2 hi = lut[(o.bits[ni] >> (16u * h + 8u)) & 0xffu];
                b[i % 2u][ni][h] = v4i{(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
            }
    };
    const auto mma = [&](auto ic) {
        constexpr uint32_t i = decltype(ic)::value;
        const KrOps<TMS, TNW>& o = raw[i % 3u];
#pragma unroll
        for (uint32_t ni = 0; ni < (uint32_t)TNW; ++ni) {
            const float sc = __half2float(__ushort_as_half((uint16_t)o.s[ni]));
            const float cneg = sc * -kMagicValue;  // exact
#pragma unroll
            for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi) {
                v4i dd = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a[mi][0], b[i % 2u][ni][0], c_init, 0, 0, 0);
                dd = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a[mi][1], b[i % 2u][ni][1], dd, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    p[i][mi][ni][e] = __builtin_fmaf(sc, __int_as_float(dd[e]), cneg);
            }
        }
    };
    static_for<T::GS + 2u>([&](auto ic) {
        constexpr uint32_t i = decltype(ic)::value;
        if constexpr (i < T::GS)
            read(std::integral_constant<uint32_t, i>{});
        if constexpr (i >= 1u && i - 1u < T::GS)
            expand(std::integral_constant<uint32_t, i - 1u>{});
        if constexpr (i >= 2u)
            mma(std::integral_constant<uint32_t, i - 2u>{});
    });
    if (failed_seq == seq) {  // an illegal input row in this job: write nothing (the whole workgroup)
        gemm_signal(j, seq);
        return;
    }

    // 3. the running sums along the slices: slice 0 from +0, slice t after barrier t
    v4f acc[TMS][TNW];
    v4f* const xchg = reinterpret_cast<v4f*>(smem + T::OFF_X) + nn * (TMS * TNW * 64u) + lane;
    const auto add_slice = [&]() {
#pragma unroll
        for (uint32_t i = 0; i < T::GS; ++i) {
            if (g0 + i < groups) {
#pragma unroll
                for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi)
#pragma unroll
                    for (uint32_t ni = 0; ni < (uint32_t)TNW; ++ni)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            acc[mi][ni][e] = acc[mi][ni][e] + p[i][mi][ni][e];
            }
        }
    };
#pragma unroll
    for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi)
#pragma unroll
        for (uint32_t ni = 0; ni < (uint32_t)TNW; ++ni)
            acc[mi][ni] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    if (s == 0u)
        add_slice();
#pragma unroll
    for (uint32_t t = 1; t < (uint32_t)KS; ++t) {
        if (s == t - 1u) {
#pragma unroll
            for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi)
#pragma unroll
                for (uint32_t ni = 0; ni < (uint32_t)TNW; ++ni)
                    xchg[(mi * TNW + ni) * 64u] = acc[mi][ni];
        }
        lds_barrier();
        if (s == t) {
#pragma unroll
            for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi)
#pragma unroll
                for (uint32_t ni = 0; ni < (uint32_t)TNW; ++ni)
                    acc[mi][ni] = xchg[(mi * TNW + ni) * 64u];
            add_slice();
        }
    }
    // stored in one of two forms, each without a branch per value
    const auto store = [&](auto through) {
        const bool scaled = j.mode == MODE_SUM_SCALED;
#pragma unroll
        for (uint32_t mi = 0; mi < (uint32_t)TMS; ++mi)
#pragma unroll
            for (uint32_t ni = 0; ni < (uint32_t)TNW; ++ni) {
                const uint32_t n = n0 + 16u * (nn * TNW + ni) + lrow;
                if (n >= j.n || s != (uint32_t)KS - 1u)  // the last slice holds the sums
                    continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t m = m0 + 16u * mi + 4u * chunk + e;
                    if (m >= j.rows)
                        continue;
                    float* orow = reinterpret_cast<float*>(j.out + (size_t)m * j.out_stride);
                    put(orow + n, scaled ? acc[mi][ni][e] * rs[mi][e] : acc[mi][ni][e], through);
                }
            }
    };
    if (j.done)
        store(std::true_type{});
    else
        store(std::false_type{});
    gemm_signal(j, seq);
}

// k_gemm_mx<TM, TN, WGM, WGN>: GEMM / GEMM_F32 with a chip's worth of TM x TN tiles,
// one workgroup of WGM x WGN waves per CU (two waves per SIMD for 8 waves).  Per
// 128-weight group g:
//   * the TM rows' quantised bytes and the TN columns' sign bits and scales reach LDS by
//     DMA, DEPTH groups ahead, in a ring of DEPTH + 1 slots: A_INS + 1 DMA instructions
//     per wave and group (one barrier per group: every wave has read slot g-1 before the
//     DMAs of group g+DEPTH reuse it);
//   * every wave expands its own columns' sign bits (4 bytes per lane) straight into
//     +1/-1 MFMA operands through the byte table -- no +1/-1 tile in LDS;
//   * group g-1's exact epilogue on each 16 x 16 subtile (the other D set) comes before
//     group g's first-half MFMA on it; the second halves follow, each accumulating onto
//     a first half issued MS * NS MFMAs earlier.
// The K order inside a group is that of k_gemm_ks / k_gemm_wv (lane chunk c: weights
// 32c .. 32c+31, MFMA half h the 16 from 32c + 16h).  The tile leaves through LDS as
// 16-byte row-contiguous stores where the output view allows (stored straight from the
// registers, 64 bytes per row and instruction, it ran as fast but wrote 1.3-1.45x the
// output's bytes).
template <int TM, int TN, int WGM, int WGN>
struct MxTiling {
    static constexpr uint32_t WAVES = WGM * WGN, THREADS = 64u * WAVES;
    static constexpr uint32_t WTM = TM / WGM, WTN = TN / WGN, MS = WTM / 16u, NS = WTN / 16u;
    static constexpr uint32_t DEPTH = 3, SLOTS = DEPTH + 1;
    static constexpr uint32_t A_INS = TM * 8u / THREADS;  // 16-byte row chunks per thread and group
    // a slot: rows [TM][128] (chunks swizzled), then the columns' 16-byte sign-bit chunks
    // [TN][16], then their fp16 scales [TN]; the column part as TN + TN / 8 chunks of 16
    // bytes, CPW per wave
    static constexpr uint32_t A_BYTES = TM * 128u, COL_CHUNKS = TN + TN / 8u, CPW = COL_CHUNKS / WAVES;
    static constexpr uint32_t SLOT_BYTES = A_BYTES + 16u * COL_CHUNKS;
    // vector-memory operations a wave issues per group (row DMAs, one column DMA)
    static constexpr uint32_t VM_PER_GROUP = A_INS + 1u;
    // the byte table in 32 copies, entry e of copy c at (32 e + c) * 8 bytes: lane l reads
    // copy l % 32, i.e. only its own pair of the 64 banks, so that the lanes' lookups of
    // arbitrary entries never conflict
    static constexpr uint32_t LUT_COPIES = 32;
    static constexpr uint32_t OFF_LUT = SLOTS * SLOT_BYTES, LOOP_BYTES = OFF_LUT + 256u * LUT_COPIES * 8u;
    static constexpr uint32_t OUT_STRIDE = TN + 4u;  // floats per staged output row
    static constexpr uint32_t OUT_BYTES = TM * OUT_STRIDE * 4u;
    static constexpr uint32_t SMEM = LOOP_BYTES > OUT_BYTES ? LOOP_BYTES : OUT_BYTES;
    static_assert(TM % (16 * WGM) == 0 && TN % (16 * WGN) == 0, "wave tiles of 16 x 16 subtiles");
    static_assert(TN % 64 == 0, "whole 64-feature tiles of the matrix layout");
    static_assert(TM * 8u % THREADS == 0 && A_INS >= 1u, "whole row DMAs per thread");
    static_assert(COL_CHUNKS % WAVES == 0 && CPW <= 64u, "column DMA chunks per wave");
    static_assert(SLOT_BYTES % 16u == 0 && OFF_LUT % 16u == 0, "16-byte DMA destinations");
    static_assert((DEPTH - 1u) * VM_PER_GROUP < 64u, "vmcnt range");
    static_assert(SMEM <= 160u * 1024u, "LDS");
    static_assert(TM * TN / 4u % THREADS == 0, "output chunks per thread");
};

template <int TM, int TN, int WGM, int WGN>
__global__ __launch_bounds__(64 * WGM * WGN) void k_gemm_mx(GemmJob j, uint32_t mtiles, uint32_t ntiles,
                                                            uint32_t band, uint64_t seq,
                                                            const uint64_t* __restrict__ flag) {
    using T = MxTiling<TM, TN, WGM, WGN>;
    constexpr uint32_t MS = T::MS, NS = T::NS, THREADS = T::THREADS, DEPTH = T::DEPTH;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[T::SMEM];
    if (*flag == seq) {
        gemm_signal(j, seq);
        return;
    }
    const uint32_t tid = threadIdx.x, lane = tid & 63u, chunk = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave / WGN, wn = wave % WGN;
    TileRC tile = gemm_tile_of_block(blockIdx.x, gridDim.x, mtiles, ntiles, band);
    tile.nt = select_part(j, tile.nt);
    const uint32_t m0 = tile.mt * TM, n0 = tile.nt * TN;
    const uint32_t groups = j.groups;
    uint2* const lut_all = reinterpret_cast<uint2*>(smem + T::OFF_LUT);
    for (uint32_t i = tid; i < 256u * T::LUT_COPIES; i += THREADS) {
        const uint32_t e = i / T::LUT_COPIES;
        lut_all[i] = make_uint2(pm1_nibble(e & 15u), pm1_nibble(e >> 4));
    }
    const uint2* const lut = lut_all + (lane % T::LUT_COPIES);  // entry e at lut[32 e]

    // the rows' DMA: instruction i of wave w fills LDS chunks p = 64 (A_INS w + i) + lane
    // of a slot's rows, as a wave-uniform base plus a 32-bit per-lane offset (the rows of
    // one launch chunk are far below 4 GiB); rows past the end are clamped (never stored)
    uint32_t a_src[T::A_INS];
#pragma unroll
    for (uint32_t i = 0; i < T::A_INS; ++i) {
        const uint32_t p = 64u * (T::A_INS * wave + i) + lane, r = p >> 3;
        const uint32_t c = (p & 7u) ^ ((r >> 1) & 7u);
        a_src[i] = min(m0 + r, j.rows - 1u) * j.k + 16u * c;
    }
    // the columns' DMA: chunk k = CPW w + lane of wave w (lanes past CPW inactive): chunk
    // k < TN is the 16 bytes of sign bits of column n0 + k, chunk TN + c the scales of
    // columns n0 + 8c .. +7; per group the bits advance 1 KiB (one 64-feature tile) and
    // the scales 128 bytes.  The matrix tile of columns past the last one is clamped
    // (never stored).
    const unsigned char* col_src;
    uint32_t col_step;
    {
        const uint32_t k = T::CPW * wave + min(lane, T::CPW - 1u);
        const uint32_t col = k < (uint32_t)TN ? k : 8u * (k - TN);
        const size_t t = min((n0 + col) >> 6, j.tiles - 1u);
        if (k < (uint32_t)TN) {
            col_src = reinterpret_cast<const unsigned char*>(j.wbits) + (t * groups * kTile + (col & 63u)) * 16u;
            col_step = kTile * 16u;
        } else {
            col_src = reinterpret_cast<const unsigned char*>(j.wscale) + (t * groups * kTile + (col & 63u)) * 2u;
            col_step = kTile * 2u;
        }
    }
    const uint32_t la0 = lds_offset(smem);
    auto issue_group = [&](uint32_t g) {
        const uint32_t gg = min(g, groups - 1u);
        const uint8_t* base = reinterpret_cast<const uint8_t*>(j.q) + (size_t)gg * kGroup;
        const uint32_t slot = la0 + (g % T::SLOTS) * T::SLOT_BYTES;
#pragma unroll
        for (uint32_t i = 0; i < T::A_INS; ++i)
            dma16_s(a_src[i], base, slot + 1024u * (T::A_INS * wave + i));
        dma16_lanes<lane_mask<T::CPW>()>(col_src + (size_t)gg * col_step, slot + T::A_BYTES + 16u * T::CPW * wave);
    };
    // A operand rows of this wave in a slot: row r = wm * WTM + 16 mi + (lane & 15)
    uint32_t a_off[MS][2];
#pragma unroll
    for (uint32_t mi = 0; mi < MS; ++mi)
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h)
            a_off[mi][h] = swz128(wm * T::WTM + 16u * mi + (lane & 15u), 2u * chunk + h);
    // this lane's columns in a slot: 4 bytes of sign bits (chunk c of the 16) and the scale
    const uint32_t col0 = wn * T::WTN + (lane & 15u);

    v4i dd[2][MS][NS];
    float acc[MS][NS][4];
#pragma unroll
    for (uint32_t mi = 0; mi < MS; ++mi)
#pragma unroll
        for (uint32_t ni = 0; ni < NS; ++ni)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[mi][ni][r] = 0.0f;
    float sc_prev[NS], cneg_prev[NS];
    const v4i c_init = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};

    // group g (D set e = g % 2): its MFMAs into dd[e]; with `epi`, group g-1's epilogue
    // from dd[e ^ 1] (scales sc_prev)
    auto step = [&](uint32_t g, uint32_t e, bool epi) {
        // this wave's DMAs of group g have landed (those of groups g+1 .. g+DEPTH-1 are
        // newer); then every wave's have, and every wave has read the slot that group
        // g+DEPTH takes
        lds_barrier<(DEPTH - 1u) * T::VM_PER_GROUP>();
        const unsigned char* slot = smem + (g % T::SLOTS) * T::SLOT_BYTES;
        uint32_t bits[NS];
        uint16_t sraw[NS];
#pragma unroll
        for (uint32_t ni = 0; ni < NS; ++ni) {
            bits[ni] = *reinterpret_cast<const uint32_t*>(slot + T::A_BYTES + (col0 + 16u * ni) * 16u + 4u * chunk);
            sraw[ni] = *reinterpret_cast<const uint16_t*>(slot + T::A_BYTES + 16u * TN + (col0 + 16u * ni) * 2u);
        }
        v4i a[MS][2], b[NS][2];
#pragma unroll
        for (uint32_t mi = 0; mi < MS; ++mi)
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h)
                a[mi][h] = *reinterpret_cast<const v4i*>(slot + a_off[mi][h]);
#pragma unroll
        for (uint32_t ni = 0; ni < NS; ++ni)
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                const uint2 lo = lut[T::LUT_COPIES * ((bits[ni] >> (16u * h)) & 0xffu)];
                const uint2 hi = lut[T::LUT_COPIES * ((bits[ni] >> (16u * h + 8u)) & 0xffu)];
                b[ni][h] = v4i{(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
            }
        float sc[NS], cneg[NS];
#pragma unroll
        for (uint32_t ni = 0; ni < NS; ++ni) {
            sc[ni] = __half2float(__ushort_as_half(sraw[ni]));
            // the converted scale as a register operand of the epilogue's FMAs (folded into
            // them, the conversion would make each a mixed-precision FMA)
            asm volatile("" : "+v"(sc[ni]));
            cneg[ni] = sc[ni] * -kMagicValue;  // exact
        }
        issue_group(g + DEPTH);
        // the first halves of all subtiles (independent MFMAs, each after group g-1's
        // epilogue on that subtile), then the second halves, each accumulating onto a first
        // half issued MS * NS MFMAs earlier (a dependent MFMA right behind its source waits
        // for that one's result)
#pragma unroll
        for (uint32_t mi = 0; mi < MS; ++mi)
#pragma unroll
            for (uint32_t ni = 0; ni < NS; ++ni) {
                if (epi) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        acc[mi][ni][r] = acc[mi][ni][r] + __builtin_fmaf(sc_prev[ni],
                                                                         __int_as_float(dd[e ^ 1u][mi][ni][r]),
                                                                         cneg_prev[ni]);
                }
                dd[e][mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[mi][0], b[ni][0], c_init, 0, 0, 0);
            }
#pragma unroll
        for (uint32_t mi = 0; mi < MS; ++mi)
#pragma unroll
            for (uint32_t ni = 0; ni < NS; ++ni)
                dd[e][mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[mi][1], b[ni][1], dd[e][mi][ni], 0, 0, 0);
#pragma unroll
        for (uint32_t ni = 0; ni < NS; ++ni) {
            sc_prev[ni] = sc[ni];
            cneg_prev[ni] = cneg[ni];
        }
    };

    // prologue: groups 0 .. DEPTH-1 (the order the waits of step() count on)
#pragma unroll
    for (uint32_t g = 0; g < DEPTH; ++g)
        issue_group(g);
    step(0, 0, false);
    uint32_t g = 1;
    for (; g + 1u < groups; g += 2u) {
        step(g, 1, true);
        step(g + 1u, 0, true);
    }
    const bool last_in_d1 = g < groups;
    if (last_in_d1)
        step(g, 1, true);
    // epilogue of the last group
#pragma unroll
    for (uint32_t mi = 0; mi < MS; ++mi)
#pragma unroll
        for (uint32_t ni = 0; ni < NS; ++ni)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[mi][ni][r] = acc[mi][ni][r] + __builtin_fmaf(sc_prev[ni],
                                                                 __int_as_float(last_in_d1 ? dd[1][mi][ni][r]
                                                                                           : dd[0][mi][ni][r]),
                                                                 cneg_prev[ni]);
    // no DMA may still be writing LDS when it is reused for the staged tile
    lds_barrier<0>();
    float* const so = reinterpret_cast<float*>(smem);
#pragma unroll
    for (uint32_t mi = 0; mi < MS; ++mi)
#pragma unroll
        for (uint32_t ni = 0; ni < NS; ++ni)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
                so[(wm * T::WTM + 16u * mi + 4u * chunk + r) * T::OUT_STRIDE + wn * T::WTN + 16u * ni + (lane & 15u)] =
                    acc[mi][ni][r];
    lds_barrier();
    // stored in one of two forms, each without a branch per value
    const auto store = [&](auto through) {
        const bool vec = ((j.out_stride | (uint64_t)(uintptr_t)j.out) & 15u) == 0;
        const bool scaled = j.mode == MODE_SUM_SCALED;
#pragma unroll
        for (uint32_t c0 = 0; c0 < TM * TN / 4u; c0 += THREADS) {
            const uint32_t c = c0 + tid, row = c / (TN / 4u), col = 4u * (c % (TN / 4u));
            const uint32_t m = m0 + row, n = n0 + col;
            if (m >= j.rows || n >= j.n)
                continue;
            float4 v = *reinterpret_cast<const float4*>(so + row * T::OUT_STRIDE + col);
            if (scaled) {
                const float s = row_scale(j, m);
                v.x = v.x * s;
                v.y = v.y * s;
                v.z = v.z * s;
                v.w = v.w * s;
            }
            float* dst = reinterpret_cast<float*>(j.out + (size_t)m * j.out_stride) + n;
            if (vec && n + 4u <= j.n) {
                put4(dst, v4i{__float_as_int(v.x), __float_as_int(v.y), __float_as_int(v.z), __float_as_int(v.w)}, through);
            } else {
                put(dst, v.x, through);
                if (n + 1u < j.n)
                    put(dst + 1, v.y, through);
                if (n + 2u < j.n)
                    put(dst + 2, v.z, through);
                if (n + 3u < j.n)
                    put(dst + 3, v.w, through);
            }
        }
    };
    if (j.done)
        store(std::true_type{});
    else
        store(std::false_type{});
    gemm_signal(j, seq);
}

// The band width (in M tiles) of gemm_tile_of_block: an XCD covering band M tiles of
// mtiles and (tiles / 8 / band) N tiles makes the rows (rows * k bytes) be fetched
// into about 8 * band / mtiles L2s and the weights (1.125 bits each) into
// mtiles / band of them; the band minimising the sum.
uint32_t gemm_band(const GemmJob& job, uint32_t mtiles) {
    double n = job.n;
    for (uint32_t i = 0; i < job.extra; ++i)
        n += job.parts[i].n;
    const double a = (double)job.rows * job.k, b = n * job.k * 0.140625;
    uint32_t best = 1;
    double best_cost = 0.0;
    for (uint32_t band = 1; band <= mtiles; ++band) {
        const double xcds_per_mtile = std::min(8.0, 8.0 * band / mtiles);
        const double cost = a * std::max(1.0, xcds_per_mtile) + b * ((mtiles + band - 1u) / band);
        if (band == 1 || cost < best_cost)
            best = band, best_cost = cost;
    }
    return best;
}

// Column tiles of `tn` columns of every part of the job, whose first tiles it fills in.
uint32_t gemm_ntiles(GemmJob& job, uint32_t tn) {
    uint32_t t = (job.n + tn - 1u) / tn;
    for (uint32_t i = 0; i < job.extra; ++i) {
        job.parts[i].first = t;
        t += (job.parts[i].n + tn - 1u) / tn;
    }
    return t;
}

template <int TMS, int TNS, int W, int DEPTH>
hipError_t launch_ks(const GemmLaunch& at, GemmJob job) {
    const uint32_t mtiles = (job.rows + 16u * TMS - 1u) / (16u * TMS);
    const uint32_t ntiles = gemm_ntiles(job, 16u * TNS);
    return launch_tiles(at, k_gemm_ks<TMS, TNS, W, DEPTH>, 64 * W, job, mtiles, ntiles);
}

template <int TMS, int TNS, int W, int R>
hipError_t launch_kr(const GemmLaunch& at, GemmJob job) {
    if (job.groups > (uint32_t)(W * R) || job.mode == MODE_DOT_I16)
        return hipErrorInvalidValue;  // the selection below never asks for this
    const uint32_t mtiles = (job.rows + 16u * TMS - 1u) / (16u * TMS);
    const uint32_t ntiles = gemm_ntiles(job, 16u * TNS);
    return launch_tiles(at, k_gemm_kr<TMS, TNS, W, R>, 64 * W, job, mtiles, ntiles);
}

template <int TMS, int TNW, int WN, int KS, int G>
hipError_t launch_kc(const GemmLaunch& at, GemmJob job) {
    if (job.groups > (uint32_t)G || job.mode == MODE_DOT_I16)
        return hipErrorInvalidValue;  // the selection below never asks for this
    const uint32_t mtiles = (job.rows + 16u * TMS - 1u) / (16u * TMS);
    const uint32_t ntiles = gemm_ntiles(job, 16u * TNW * WN);
    return launch_tiles(at, k_gemm_kc<TMS, TNW, WN, KS, G>, 64 * WN * KS, job, mtiles, ntiles);
}

template <int TM, int TN, int WGM, int WGN>
hipError_t launch_mx(const GemmLaunch& at, GemmJob job) {
    const uint32_t mtiles = (job.rows + TM - 1u) / TM, ntiles = gemm_ntiles(job, TN);
    return launch_tiles(at, k_gemm_mx<TM, TN, WGM, WGN>, 64 * WGM * WGN, job, mtiles, ntiles);
}

template <int MS, int NS, int WM, int WN, int DEPTH>
hipError_t launch_wv(const GemmLaunch& at, GemmJob job) {
    constexpr uint32_t TM = 16u * MS * WM, TN = 16u * NS * WN;
    const uint32_t mtiles = (job.rows + TM - 1u) / TM, ntiles = gemm_ntiles(job, TN);
    return launch_tiles(at, k_gemm_wv<MS, NS, WM, WN, DEPTH>, 64 * WM * WN, job, mtiles, ntiles);
}

template <int TNS, int GB, int WAVES>
hipError_t launch_dots(const GemmLaunch& at, GemmJob job) {
    if (job.groups > 4u * GB || job.mode != MODE_DOT_I16)
        return hipErrorInvalidValue;  // the selection below never asks for this
    const uint32_t mtiles = (job.rows + 15u) / 16u, ntiles = gemm_ntiles(job, 16u * TNS);
    return launch_tiles(at, k_gemm_dots<TNS, GB, WAVES>, 64 * WAVES, job, mtiles, ntiles);
}

template <int MS, int NS, int GC>
hipError_t launch_dotf(const GemmLaunch& at, GemmJob job) {
    if (job.groups > 8u || job.groups % (GC == 4 ? 4u : 1u) != 0 || job.mode != MODE_DOT_I16)
        return hipErrorInvalidValue;  // the selection below never asks for this
    const uint32_t mtiles = (job.rows + 32u * MS - 1u) / (32u * MS), ntiles = gemm_ntiles(job, 32u * NS);
    return launch_tiles(at, k_gemm_dotf<MS, NS, GC>, 256, job, mtiles, ntiles);
}

}  // namespace

// Workgroups of tm x tn tiles over every part of the job.
static uint64_t gemm_blocks(const GemmJob& job, uint32_t tm, uint32_t tn) {
    uint64_t cols = (job.n + tn - 1u) / tn;
    for (uint32_t i = 0; i < job.extra; ++i)
        cols += (job.parts[i].n + tn - 1u) / tn;
    return (uint64_t)((job.rows + tm - 1u) / tm) * cols;
}

// The tiles of k_gemm_mx and the time of the job in the one whose rounds of workgroups take
// the least.  A round takes ~2.5 us and, per group, the step that a sweep gave for each tile
// (17 shapes of K = 384..8192 and N = 1000..8192 x 14 row counts from 48 to 1024, all outputs
// bit-identical; the choice was within 4% of the best tile for every one).
enum MxTile { MX_64x64, MX_64x128, MX_64x192, MX_128x128, MX_128x192, MX_TILES };
static MxTile mx_tile(const GemmJob& job, uint64_t cus, double* us) {
    static const struct {
        uint32_t tm, tn;
        double step;
    } tiles[MX_TILES] = {{64, 64, 0.34}, {64, 128, 0.45}, {64, 192, 0.60}, {128, 128, 0.72}, {128, 192, 0.88}};
    MxTile best = MX_64x64;
    for (int t = 0; t < MX_TILES; ++t) {
        const uint64_t rounds = (gemm_blocks(job, tiles[t].tm, tiles[t].tn) + cus - 1u) / cus;
        const double time = (double)rounds * (2.5 + tiles[t].step * job.groups);
        if (t == 0 || time < *us)
            best = (MxTile)t, *us = time;
    }
    return best;
}

double gemm_launch_us(const GemmJob& job, uint32_t cu_count) {
    const uint64_t cus = cu_count ? cu_count : 256u;
    const uint32_t g = job.groups;
    double us = 0.0;
    if (job.mode == MODE_DOT_I16) {
        double columns = job.n;
        for (uint32_t i = 0; i < job.extra; ++i)
            columns += job.parts[i].n;
        us = 2.9 + 0.07 * g + 0.45e-6 * (columns * g * 2.0 * job.rows);
    } else if (gemm_blocks(job, 16, 32) <= cus || (g <= 16u && gemm_blocks(job, 32, 64) <= cus)) {
        us = 1.3 + 0.12 * g;
    } else if (g > 16u && gemm_blocks(job, 32, 64) <= cus) {
        us = 3.0 + 0.30 * g;
    } else {
        (void)mx_tile(job, cus, &us);
        us += 1.0;
    }
    return std::max(us, 4.4);
}

// launch_gemm's rules: the K-split kernels for few rows, then a wave per block, then the tile
// of k_gemm_mx whose rounds of workgroups take the least time.
hipError_t launch_gemm(hipStream_t stream, const GemmJob& job, uint32_t cu_count, uint64_t seq,
                       const uint64_t* flag, uint32_t* signals) {
    const GemmLaunch at{stream, seq, flag, signals};
    const uint64_t cus = cu_count ? cu_count : 256u;
    const auto blocks = [&](uint32_t tm, uint32_t tn) { return gemm_blocks(job, tm, tn); };
    if (job.mode == MODE_DOT_I16) {
        const uint32_t g = job.groups;
        // Up to 4 groups, and up to 8 past a round of k_gemm_dots' smallest tiles, the blocks of
        // k_gemm_dotf, 64 x 64 per workgroup up to one per CU (those signal), then 64 x 128: a
        // sweep of 100 shapes of up to 8 groups, N = 64..8192 and 17..1024 rows, both kernels, e.g.
        // 640->5065 x 27 rows 23.9 -> 19.2 us, 640->1226 x 72, less than a round, 18.8 and 19.2.
        if (g <= 4u || (g <= 8u && blocks(16, 32) > cus)) {
            if (blocks(64, 64) <= cus)
                return g == 1u       ? launch_dotf<2, 2, 1>(at, job)
                       : g % 4u == 0 ? launch_dotf<2, 2, 4>(at, job)
                                     : launch_dotf<2, 2, 2>(at, job);
            return g == 1u       ? launch_dotf<2, 4, 1>(at, job)
                   : g % 4u == 0 ? launch_dotf<2, 4, 4>(at, job)
                                 : launch_dotf<2, 4, 2>(at, job);
        }
        // 32-column tiles up to two per CU, and past 16 groups, whose tiles of 64 columns would
        // not fit two workgroups' LDS
        if (g > 16u)
            return launch_dots<2, 16, 8>(at, job);
        return blocks(16, 32) <= 2u * cus ? launch_dots<2, 4, 4>(at, job)
                                          : launch_dots<4, 4, 4>(at, job);
    }
    // Few rows: K split over the waves of a workgroup, every wave's operands brought into
    // LDS by DMA before anything is computed (k_gemm_kr, k_gemm_kc).  The rules follow a
    // forced-choice sweep over K = 1024..8192, N = 1024..8192 and 8..256 rows (all outputs
    // bit-identical); against the kernels below, e.g. 2048->6144 x 64 rows 9.6 -> 5.8 us,
    // 6144->2048 x 64 rows 9.6 -> 6.4 us, 2048->2048 x 128 rows 7.7 -> 4.6 us, 4096->2048 x
    // 256 rows 14.5 -> 12.2 us, 6144->2048 x 128 rows 13.3 -> 9.6 us, 8192->2048 x 32 rows
    // 9.2 -> 7.0 us.  Up to 16 groups: 16 x 32 tiles (up to 16 rows) or 32 x 32 tiles while they
    // fit one per CU, then 32 x 64 tiles while those do (16 waves of one group each above 8
    // groups), then, above 8 groups, 32 x 32 tiles up to two per CU; 17..32 groups: 16 x 32
    // tiles, then 32 x 32; 33..48 groups: 16 x 32 tiles, then 16 x 64 tiles with the slices'
    // running sums handed on (k_gemm_kc); 49..64 groups: 16 x 16 tiles; each one per CU.  Past
    // those bounds k_gemm_mx wins (2048->2048 x 320 rows a call of 25.0 us against 23.0, x 256
    // 20.0 against 22.6; 4096->2048 x 180 27.9 against 26.3, x 100 21.9 against 24.1).
    {
        const uint32_t g = job.groups;
        if (g <= 16u) {
            if (job.rows <= 16u && blocks(16, 32) <= cus)
                return launch_kr<1, 2, 4, 4>(at, job);
            if (blocks(32, 32) <= cus)
                return launch_kr<2, 2, 8, 2>(at, job);
            if (blocks(32, 64) <= cus && g > 8u)
                return launch_kr<2, 4, 16, 1>(at, job);  // 2048->6144 x 64 rows 6.2 -> 5.7 us
            if (blocks(32, 64) <= cus)
                return launch_kr<2, 4, 8, 2>(at, job);
            if (g > 8u && blocks(32, 32) <= 2u * cus)
                return launch_kr<2, 2, 8, 2>(at, job);
        } else if (g <= 32u) {
            if (blocks(16, 32) <= cus)
                return launch_kr<1, 2, 8, 4>(at, job);
            if (blocks(32, 32) <= cus)
                return launch_kr<2, 2, 8, 4>(at, job);
        } else if (g <= 48u) {
            if (blocks(16, 32) <= cus)
                return launch_kr<1, 2, 8, 6>(at, job);
            if (blocks(16, 64) <= cus)
                return launch_kc<1, 1, 4, 2, 48>(at, job);
        } else if (g <= 64u) {
            if (blocks(16, 16) <= cus)
                return launch_kc<1, 1, 1, 8, 64>(at, job);
        }
    }
    // few rows past the rules above (more than 48 groups and more than a round of 16 x 16
    // tiles): one wave per 16 x 16 output block with its operands straight in registers,
    // while that makes at most three waves per CU (the blocks of 16 columns each load their
    // rows, and more of them outrun the loads a CU keeps in flight)
    if (job.rows <= 64u && (job.rows <= 32u || job.groups <= 16u) &&
        blocks(16, 16) <= 3u * cus)
        return launch_wv<1, 1, 1, 1, 8>(at, job);
    // too few tiles for the CUs (jobs of more than 48 groups get here): K split across eight
    // waves of a workgroup with 32 x 32 tiles between three quarters of a round and one round
    // of them, or across four waves with 32 x 16 tiles in one round (8192->1000 x 180 rows a
    // call of 31.1 us against 34.6 with k_gemm_mx, x 100 28.3 against 31.9)
    if (blocks(32, 32) <= cus) {
        if (blocks(32, 32) >= cus * 3u / 4u)
            return launch_ks<2, 2, 8, 3>(at, job);
        if (blocks(32, 16) <= cus)
            return launch_ks<2, 1, 4, 3>(at, job);
    }
    // past 16 groups in one round of 32 x 64 tiles: a step of the smallest tile is the
    // shortest (6144->2048 x 180 rows 32.1 -> 31.0 us a call against a K split over the waves
    // of 32 x 64 tiles, 8192->1000 x 130 40.7 -> 32.9, 5120->2048 x 130 30.7 -> 27.5,
    // 4096->8192 x 64 27.8 -> 24.7); up to 16 groups 64 x 64 tiles are as fast
    if (job.groups > 16u && blocks(32, 64) <= cus)
        return launch_mx<32, 64, 1, 4>(at, job);
    // Everything else: k_gemm_mx, one workgroup per CU (mx_tile).  With tiles of 128 x 192 and 64
    // x 128 only, other kernels had filled the gaps, a call of 6144->2048 x 389 rows 42.8 -> 34.1
    // us, x 640 56.4 -> 41.5, 4096->4096 x 389 43.4 -> 33.2, 2048->2048 x 640 32.5 -> 25.3,
    // 2048->4096 x 256 27.0 -> 23.1, 8192->4096 x 768 85 -> 69.
    double us = 0.0;
    switch (mx_tile(job, cus, &us)) {
    case MX_64x64:
        return launch_mx<64, 64, 2, 4>(at, job);
    case MX_64x128:
        return launch_mx<64, 128, 2, 4>(at, job);
    case MX_64x192:
        return launch_mx<64, 192, 2, 4>(at, job);
    case MX_128x128:
        return launch_mx<128, 128, 2, 4>(at, job);
    default:
        return launch_mx<128, 192, 2, 4>(at, job);
    }
}

}  // namespace bnnhip
