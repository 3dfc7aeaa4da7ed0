// gemm_common.hpp -- what the bf16 product kernels (gemm.hip, gemm_ring.hpp)
// share: types and conversions, the LDS layouts of staged operands, the order of
// the tiles over the XCDs, the epilogue and the description of one product.
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <atomic>

#include "agk_rmsnorm.h"

namespace agk_gemm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int BK = 64;            // k per staged tile
constexpr int kStride = BK;       // bf16 per LDS row of a k-contiguous operand (128 bytes)

// LDS position of k-chunk c (8 bf16 = 16 bytes) of row `row`: chunks are
// XOR-swizzled by the row's low bits, so the 8 lanes of a 16-byte fragment
// read (8 consecutive rows, one chunk) and the 8-byte writes of the
// transposing stager (rows 8 apart) land on different banks.
__device__ __forceinline__ int lds_off(int row, int c) {
    return row * kStride + ((c ^ (row & 7) ^ ((row >> 3) & 7)) << 3);
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// fp32 -> bf16, round to nearest even (v_cvt_pk_bf16_f32: NaN stays NaN).
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
    return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}
// lo16(a) | lo16(b) << 16 and hi16(a) | hi16(b) << 16 (v_perm_b32)
__device__ __forceinline__ uint32_t lo_pair(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_perm(b, a, 0x05040100u);
}
__device__ __forceinline__ uint32_t hi_pair(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

__device__ __forceinline__ bf16x8 lds_frag(const uint16_t* lds, int row, int k) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(lds + lds_off(row, k >> 3)));
}

// ---- LDS layout of a stage half of ROWS rows (A) or columns (B) ------------------
// k-contiguous: lds_off, rows of 64 k.  k-strided: 64 k-rows of ROWS elements,
// whose 64-byte groups are XOR-swizzled so that the four k-rows a transposing
// read touches start on four different 64-byte quarters of the 64 banks.
template <int ROWS>
__device__ __forceinline__ int tr_swz(int k) {
    if constexpr (ROWS % 128 == 0) return k & 3;        // rows start on the same bank
    else if constexpr (ROWS % 64 == 0) return (k >> 1) & 1;  // rows alternate 128 bytes
    else return 0;                                      // 64-byte rows: already distinct
}

template <int ROWS>
__device__ __forceinline__ int tr_stage_off(int k, int col) {
    return k * ROWS + (((col >> 3) ^ (tr_swz<ROWS>(k) << 2)) << 3) + (col & 7);
}

// The last K % 64 k of an operand, staged through registers with zeros past K
// (a load to LDS could not zero them): the same LDS layout.
template <bool TR, int ROWS>
__device__ __forceinline__ void stage_k_tail(uint16_t* lds, const uint16_t* __restrict__ src,
                                             int64_t ld, int rows, int k0, int K) {
    const int tid = threadIdx.x;
    u32x4 v[ROWS / 32];
#pragma unroll
    for (int j = 0; j < ROWS / 32; ++j) {
        const int q = j * 256 + tid;
        int k, r;
        if constexpr (!TR) {
            r = q >> 3;
            k = k0 + (((q & 7) ^ (r & 7) ^ ((r >> 3) & 7)) << 3);
            r = r < rows ? r : rows - 1;
        } else {
            constexpr int kChunks = ROWS / 8;
            k = k0 + q / kChunks;
            r = ((q % kChunks) ^ (tr_swz<ROWS>(q / kChunks) << 2)) * 8;
            r = r < rows ? r : rows - 8;
        }
        const int kc = k < K ? k : k0;  // an address inside the operand; zeroed below
        const int64_t at = TR ? static_cast<int64_t>(kc) * ld + r
                              : static_cast<int64_t>(r) * ld + kc;
        v[j] = *reinterpret_cast<const u32x4*>(src + at);
        if (k >= K) v[j] = u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int j = 0; j < ROWS / 32; ++j)
        *reinterpret_cast<u32x4*>(lds + (j * 256 + tid) * 8) = v[j];
}

// This wave's loads but the newest N have landed and its LDS reads and writes
// are done; then every wave's.
template <int N>
__device__ __forceinline__ void stage_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// ---- tile order ----------------------------------------------------------------
// Workgroups are dispatched round-robin over the 8 XCDs (workgroup L runs on
// XCD L % 8), each XCD with its own L2.  The tile order below gives each XCD
// a contiguous chunk of a grouped ordering (group_m m-tiles x all n-tiles,
// column by column), so the ~32 workgroups resident on one XCD at a time
// cover about group_m x 32 / group_m tiles and share their A row-panels and B
// column-panels in that XCD's L2, instead of every neighbouring tile landing
// on a different XCD.  group_m = 4 (kGroupM) for every product: over 15 sizes of 4096
// to 16384 rows by 2048 to 28672 columns in three layouts on MI355X it came within
// 0.8 % of each one's best on average (1: 5.4 %, 2: 1.8, 3: 1.2, 6: 1.0, 8: 1.6, 16:
// 4.7).  Single sizes gain up to 4 % from another (8192 x 4096 x 11008 with B^T 533 -> 512
// us at 8), by no rule that was found (16384 x 4096 x 11008 1137 -> 1164 at 8).
constexpr int kXcds = 8;
constexpr int kGroupM = 4;

__device__ __forceinline__ void tile_of(int L, int tiles_m, int tiles_n, int group_m, int& tm,
                                        int& tn) {
    const int T = tiles_m * tiles_n;
    const int x = L % kXcds, s = L / kXcds;
    const int q = T / kXcds, r = T % kXcds;  // XCDs below r get q + 1 tiles
    const int g = x < r ? x * (q + 1) + s : r * (q + 1) + (x - r) * q + s;
    const int per_group = group_m * tiles_n;
    const int group = g / per_group;
    const int gm0 = group * group_m;
    const int gsize = tiles_m - gm0 < group_m ? tiles_m - gm0 : group_m;
    const int in = g - group * per_group;
    tm = gm0 + in % gsize;
    tn = in / gsize;
}

// The product rounded to bf16, plus a bf16 bias term (then rounded again when
// stored): `matmul(X, W^T) + b` with its two roundings, as a bf16 product and
// a bf16 sum give them.
__device__ __forceinline__ float with_bias(float v, uint16_t b) {
    v = __uint_as_float(f32_to_bf16_bits(v) << 16);
    return v + __uint_as_float(static_cast<uint32_t>(b) << 16);
}

// What a store applies to the product: nothing, a column bias (bf16 output
// only), or any of rowscale, bias and accumulate, tested per element.
enum class Epi { kPlain, kBias, kAny };

// CHECK: rows past M and columns past N skipped.  store_block picks the variant
// once per call (uniform values), so the plain and the biased interior stores
// have no per-element branches.  kBias loads the lane's TNW bias values once; in
// kAny each element waits for a load of its own, up to 256 in a row, which is
// what bounded a biased product.  y = x w^T + b, kAny -> kBias: 1032 x 4096 x 4096
// 62.7 -> 42.4 us, 3288 x 3568 x 136 75 -> 21.6, 2480 x 2064 x 1152 34.4 -> 25.3,
// 3000 x 800 x 2624 32 -> 25.3; the same bits.
template <bool OUT_F32, Epi EPI, bool CHECK, int TMW, int TNW>
__device__ __forceinline__ void store_c_impl(const f32x16 (&acc)[TMW][TNW], void* __restrict__ C,
                                             int64_t ldc, int M, int N, int row0, int col0,
                                             int lane, const float* __restrict__ rowscale,
                                             const uint16_t* __restrict__ colbias,
                                             int accumulate) {
    const int col_l = lane & 31;
    const int row_l = 4 * (lane >> 5);
    uint16_t bias[TNW] = {};
    if constexpr (EPI == Epi::kBias) {
#pragma unroll
        for (int j = 0; j < TNW; ++j) {
            const int col = col0 + j * 32 + col_l;
            if (!CHECK || col < N) bias[j] = colbias[col];
        }
    }
#pragma unroll
    for (int i = 0; i < TMW; ++i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int row = row0 + i * 32 + 8 * (e >> 2) + row_l + (e & 3);
            if (CHECK && row >= M) continue;
            float rs = 1.0f;
            if constexpr (EPI == Epi::kAny) rs = rowscale ? rowscale[row] : 1.0f;
#pragma unroll
            for (int j = 0; j < TNW; ++j) {
                const int col = col0 + j * 32 + col_l;
                if (CHECK && col >= N) continue;
                float v = acc[i][j][e];
                if constexpr (EPI == Epi::kAny) {
                    v *= rs;
                    // accumulation rounds the product first (no fused multiply-add)
                    asm volatile("" : "+v"(v));
                }
                if constexpr (OUT_F32) {
                    float* p = static_cast<float*>(C) + static_cast<int64_t>(row) * ldc + col;
                    if constexpr (EPI == Epi::kAny) {
                        *p = accumulate ? *p + v : v;
                    } else {
                        // Plain fp32 stores are whole 128-byte lines per 32 lanes:
                        // non-temporal, so a round's C tiles (64 MB) do not evict
                        // the operand panels from L2 and stream out as they come.
                        // Measured on dW at c5 (4096 x 11008 x 8192, one box, three
                        // alternations): 557-561 -> 528-529 us.  bf16 outputs keep
                        // ordinary stores: no gain there, and the RMSNorm backward
                        // reads dh from the caches right after its product.
                        __builtin_nontemporal_store(v, p);
                    }
                } else {
                    uint16_t* p = static_cast<uint16_t*>(C) + static_cast<int64_t>(row) * ldc + col;
                    if constexpr (EPI == Epi::kAny) {
                        if (accumulate) v = __uint_as_float(static_cast<uint32_t>(*p) << 16) + v;
                        if (colbias) v = with_bias(v, colbias[col]);
                    } else if constexpr (EPI == Epi::kBias) {
                        v = with_bias(v, bias[j]);
                    }
                    *p = static_cast<uint16_t>(f32_to_bf16_bits(v));
                }
            }
        }
    }
}

// The stores a kernel holds.  kBiasOnly: a bias, nothing else.  kNoBias: the plain
// ones, and kAny for the rest (a bias too).  kAll: kNoBias with the biased ones.
// The 256 x 256 kernel, whose unrolled stores are four times the others', is built
// as kNoBias and as kBiasOnly: holding all of them in one kernel costs its plain
// product 0.7 % in a training pass, where each kernel's code is fetched afresh
// (8192 x 11008 x 4096: 600 -> 604 us; equal when it repeats alone).
enum class Stores { kAll, kNoBias, kBiasOnly };

// Stores a wave's block of TMW x TNW accumulators whose first element is
// C[row0][col0]; which variant runs is uniform over the wave.
template <bool OUT_F32, Stores S, int TMW, int TNW>
__device__ __forceinline__ void store_block(const f32x16 (&acc)[TMW][TNW], void* __restrict__ C,
                                            int64_t ldc, int M, int N, int row0, int col0,
                                            int lane, const float* __restrict__ rowscale,
                                            const uint16_t* __restrict__ colbias,
                                            int accumulate) {
    const bool inner = row0 + TMW * 32 <= M && col0 + TNW * 32 <= N;
    const bool scaled = rowscale != nullptr || accumulate;
    if constexpr (!OUT_F32 && S != Stores::kNoBias) {
        if (S == Stores::kBiasOnly || (!scaled && colbias != nullptr)) {
            if (inner)
                store_c_impl<OUT_F32, Epi::kBias, false>(acc, C, ldc, M, N, row0, col0, lane,
                                                         nullptr, colbias, 0);
            else
                store_c_impl<OUT_F32, Epi::kBias, true>(acc, C, ldc, M, N, row0, col0, lane,
                                                        nullptr, colbias, 0);
            return;
        }
    }
    if constexpr (S != Stores::kBiasOnly) {
        if (scaled || colbias != nullptr) {
            store_c_impl<OUT_F32, Epi::kAny, true>(acc, C, ldc, M, N, row0, col0, lane, rowscale,
                                                   colbias, accumulate);
        } else if (inner) {
            store_c_impl<OUT_F32, Epi::kPlain, false>(acc, C, ldc, M, N, row0, col0, lane,
                                                      nullptr, nullptr, 0);
        } else {
            store_c_impl<OUT_F32, Epi::kPlain, true>(acc, C, ldc, M, N, row0, col0, lane, nullptr,
                                                     nullptr, 0);
        }
    }
}

// Compute units of the current device (looked up once per device; 256 on
// MI355X), for the choice of a tile shape and the direct kernel's last-round split.
inline int device_cus() {
    constexpr int kMaxDev = 64;
    static std::atomic<int> cached[kMaxDev];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) return 256;
    int v = cached[dev].load(std::memory_order_relaxed);
    if (v > 0) return v;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        v <= 0)
        v = 256;
    cached[dev].store(v, std::memory_order_relaxed);
    return v;
}

// One product's arguments, for the direct and ring launches.
struct GemmCall {
    const uint16_t* A;
    int64_t lda;
    const uint16_t* B;
    int64_t ldb;
    void* C;
    int64_t ldc;
    int M, N, K;
    const float* rowscale;
    const uint16_t* colbias;
    int accumulate;
    hipStream_t st;
};

}  // namespace agk_gemm
