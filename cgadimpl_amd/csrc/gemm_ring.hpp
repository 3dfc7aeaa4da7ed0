// gemm_ring.hpp -- the bf16 product for shapes whose 256 x 256 tiles would
// leave CUs idle (the same operands, layouts, epilogue and k order as gemm.hip's
// direct-to-LDS kernel).  Included by gemm.hip for the declarations, and by
// gemm_ring_n.hip / gemm_ring_t.hip, which instantiate the kernels for A
// k-contiguous / k-strided (AGK_RING_KERNELS).
//
// Tile: BM x BN per workgroup of 4 waves (WVM along M), each wave TM x TN
// accumulators of v_mfma_f32_32x32x16_bf16.  K is walked in 64-deep tiles
// through a ring of NST LDS stages filled by `buffer_load_dwordx4 ... lds`:
// while tile t is multiplied the loads of tiles t + 1 .. t + NST - 1 are in
// flight.  With tiles this small a k-step's MFMAs (0.1-0.3 us) are far shorter
// than a load's latency (1-2 us); the deeper ring, or two workgroups per CU, keeps
// the bytes in flight that cover it.  Measured on MI355X: 1032 x 4096 x 4096 in 192 x
// 128 tiles, the waves wait for 16 % of their cycles and the matrix cores of the 192
// CUs with a tile are busy 44 % of the time at 2.4 GHz (the idle CUs and the lower
// clock are the rest); 16 x 11008 x 4096 in 64 x 64 tiles, 57 % waiting, the weights read
// at 5.2 TB/s.
//
// Step t: the fragments run one 16-deep substep ahead of the MFMAs, across the
// barrier, as in the direct kernel.  At the end of the step each wave waits
// until only the loads of tiles t + 2 .. are outstanding (its share of tile
// t + 1 has landed) and for its own fragment reads, then the barrier; after it
// tile t's stage is free and the next step loads tile t + NST into it.  Steps
// past the last tile issue the same loads through a zero-byte resource (no
// memory traffic), so the outstanding count is the same in every step.
// One __shared__ array per stage: the compiler proves the loads of one stage
// disjoint from the fragment reads of another only per array.
#pragma once

#include "gemm_common.hpp"

namespace agk_gemm {

// The kernel's shapes: id, tile rows and columns, waves along M, stages.
#define AGK_RING_SHAPES(X)                                                              \
    X(1, 256, 128, 2, 3) X(2, 192, 128, 2, 3) X(3, 128, 192, 2, 3) X(4, 128, 256, 2, 3) \
    X(5, 128, 128, 2, 3) X(6, 128, 64, 2, 3) X(7, 64, 128, 2, 3) X(8, 64, 64, 2, 4)
constexpr int kRingSmallK = 8;   // fewer than 64 k: one tail tile, nothing to stream
constexpr int kRingLargest = 1;  // the same where 64 x 64 tiles are too many for a grid

template <int BM_, int BN_, int WVM, int NST>
struct RingShape {
    static constexpr int kBM = BM_, kBN = BN_, kWvm = WVM, kWvn = 4 / WVM, kStages = NST;
    static constexpr int kTm = BM_ / WVM / 32, kTn = BN_ / (4 / WVM) / 32;
    static constexpr int kElems = (BM_ + BN_) * BK;
    static constexpr int kLoads = (BM_ + BN_) / 32;  // per wave and k-tile
    // workgroups per CU that the LDS allows, capped at two (waves per SIMD)
    static constexpr int kPerCu = 2 * NST * kElems * 2 <= 160 * 1024 ? 2 : 1;
};

// Microseconds of a 64-deep k-step of one round, measured (pick_shape): few
// workgroups / every CU's slots full.  id 0: the direct kernel.
struct RingCost {
    int id, bm, bn, per_cu;
    double light, full;
};
constexpr RingCost kRingCosts[] = {
    {0, 256, 256, 1, 0.90, 1.55}, {1, 256, 128, 1, 0.66, 0.91}, {2, 192, 128, 1, 0.52, 0.66},
    {3, 128, 192, 1, 0.51, 0.67}, {4, 128, 256, 1, 0.59, 0.88}, {5, 128, 128, 1, 0.39, 0.53},
    {6, 128, 64, 2, 0.30, 0.65},  {7, 64, 128, 2, 0.32, 0.65},  {8, 64, 64, 2, 0.29, 0.46},
};

template <bool A_TR, bool B_TR>
int launch_ring(int shape, bool f32, const GemmCall& c);

}  // namespace agk_gemm

#ifdef AGK_RING_KERNELS

namespace agk_gemm {

// Byte offsets of a wave's ROWS / 32 loads of one operand (load j fills the
// kilobyte wave * ROWS / 32 + j of the operand's half of a stage).
template <bool TR, int ROWS>
__device__ __forceinline__ void ring_offsets(uint32_t (&o)[ROWS / 32], int wave, int lane,
                                             int rows, int64_t ld) {
#pragma unroll
    for (int j = 0; j < ROWS / 32; ++j) {
        const int q = (wave * (ROWS / 32) + j) * 64 + lane;  // 16-byte chunk of the half
        if constexpr (!TR) {
            const int row = q >> 3;
            const int c = (q & 7) ^ (row & 7) ^ ((row >> 3) & 7);
            const int r = row < rows ? row : rows - 1;  // rows past M or N: the last valid row
            o[j] = (static_cast<uint32_t>(r) * static_cast<uint32_t>(ld) + c * 8) * 2;
        } else {
            constexpr int kChunks = ROWS / 8;
            const int k = q / kChunks;
            const int c = (q % kChunks) ^ (tr_swz<ROWS>(k) << 2);
            const int col = c * 8 < rows ? c * 8 : rows - 8;  // columns past M or N: the last 8
            o[j] = (static_cast<uint32_t>(k) * static_cast<uint32_t>(ld) + col) * 2;
        }
    }
}

// ---- fragments -------------------------------------------------------------------

template <int TMW, int TNW>
struct RingFrags {
    bf16x8 a[TMW], b[TNW];
};

template <bool TR, int ROWS>
__device__ __forceinline__ bf16x8 ring_frag(const uint16_t* half, int c0, int s, int lane) {
    if constexpr (!TR) {
        return lds_frag(half, c0 + (lane & 31), s * 16 + (lane >> 5) * 8);
    } else {
        const int g = lane >> 4, sl = lane & 15;
        const int k = s * 16 + (g >> 1) * 8 + (sl >> 2);
        const int col = c0 + (g & 1) * 16 + 4 * (sl & 3);
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4_t)(half + tr_stage_off<ROWS>(k, col)));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4_t)(half + tr_stage_off<ROWS>(k + 4, col)));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
}

template <bool A_TR, bool B_TR, class SH>
__device__ __forceinline__ void ring_read(RingFrags<SH::kTm, SH::kTn>& f, const uint16_t* stage,
                                          int s, int wm, int wn, int lane) {
#pragma unroll
    for (int i = 0; i < SH::kTm; ++i)
        f.a[i] = ring_frag<A_TR, SH::kBM>(stage, (wm * SH::kTm + i) * 32, s, lane);
#pragma unroll
    for (int j = 0; j < SH::kTn; ++j)
        f.b[j] = ring_frag<B_TR, SH::kBN>(stage + SH::kBM * BK, (wn * SH::kTn + j) * 32, s, lane);
}

template <int TMW, int TNW>
__device__ __forceinline__ void ring_mfma(const RingFrags<TMW, TNW>& f, f32x16 (&acc)[TMW][TNW]) {
#pragma unroll
    for (int i = 0; i < TMW; ++i)
#pragma unroll
        for (int j = 0; j < TNW; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
}

template <class SH>
struct RingOffsets {
    uint32_t a[SH::kBM / 32], b[SH::kBN / 32];  // ring_offsets of each operand
};

struct RingOperands {
    const void *a, *b;
    int bytes_a, bytes_b;  // what the tile's loads can address
    int step_a, step_b;    // bytes from one k-tile to the next
    int nk;                // whole 64-deep k-tiles
};

struct RingRsrc {
    __amdgpu_buffer_rsrc_t a, b;
};
__device__ __forceinline__ RingRsrc ring_rsrc(const RingOperands& r, bool in) {
    RingRsrc q;
    q.a = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(r.a), static_cast<short>(0),
                                            in ? r.bytes_a : 0, 0x00020000);
    q.b = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(r.b), static_cast<short>(0),
                                            in ? r.bytes_b : 0, 0x00020000);
    return q;
}
__device__ __forceinline__ void ring_load_a(const RingRsrc& q, uint16_t* lds, uint32_t off,
                                            int at) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(q.a, (lds_ptr_t)lds, 16, off, at, 0, 0);
}
__device__ __forceinline__ void ring_load_b(const RingRsrc& q, uint16_t* lds, uint32_t off,
                                            int at) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(q.b, (lds_ptr_t)lds, 16, off, at, 0, 0);
}

// Loads one operand of k-tile t (nothing past the last one: a zero-byte
// resource).
template <class SH>
__device__ __forceinline__ void ring_issue_a(const RingOperands& r, const RingOffsets<SH>& o,
                                             uint16_t* stage, int t, int wave) {
    const bool in = t < r.nk;
    const RingRsrc q = ring_rsrc(r, in);
#pragma unroll
    for (int j = 0; j < SH::kBM / 32; ++j)
        ring_load_a(q, stage + (wave * (SH::kBM / 32) + j) * 512, o.a[j], in ? t * r.step_a : 0);
}
template <class SH>
__device__ __forceinline__ void ring_issue_b(const RingOperands& r, const RingOffsets<SH>& o,
                                             uint16_t* stage, int t, int wave) {
    const bool in = t < r.nk;
    const RingRsrc q = ring_rsrc(r, in);
#pragma unroll
    for (int j = 0; j < SH::kBN / 32; ++j)
        ring_load_b(q, stage + SH::kBM * BK + (wave * (SH::kBN / 32) + j) * 512, o.b[j],
                    in ? t * r.step_b : 0);
}
template <class SH>
__device__ __forceinline__ void ring_issue(const RingOperands& r, const RingOffsets<SH>& o,
                                           uint16_t* stage, int t, int wave) {
    ring_issue_a<SH>(r, o, stage, t, wave);
    ring_issue_b<SH>(r, o, stage, t, wave);
}

// Scheduling groups of a substep: one load (if LOADS), READS fragment reads,
// one MFMA, N times.
template <int N, int READS, bool LOADS>
__device__ __forceinline__ void ring_sched() {
    if constexpr (N > 0) {
        if constexpr (LOADS) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        ring_sched<N - 1, READS, LOADS>();
    }
}

// One k-tile out of `cur`, loading tile `ahead` into `into` (the stage the
// previous step read).  FIRST: no straddling substep to multiply.
template <bool FIRST, bool A_TR, bool B_TR, class SH>
__device__ __forceinline__ void ring_step(const RingOperands& r,
                                          const RingOffsets<SH>& o, const uint16_t* cur,
                                          uint16_t* into, int ahead,
                                          f32x16 (&acc)[SH::kTm][SH::kTn],
                                          RingFrags<SH::kTm, SH::kTn>& f0,
                                          RingFrags<SH::kTm, SH::kTn>& f1, int wm, int wn,
                                          int lane, int wave) {
    constexpr int kMfma = SH::kTm * SH::kTn;
    constexpr int kReads = SH::kTm * (A_TR ? 2 : 1) + SH::kTn * (B_TR ? 2 : 1);
    constexpr int kPer = (kReads + kMfma - 1) / kMfma;
    ring_issue_a<SH>(r, o, into, ahead, wave);
    ring_read<A_TR, B_TR, SH>(f0, cur, 0, wm, wn, lane);
    if constexpr (!FIRST) {
        ring_mfma(f1, acc);
        ring_sched<kMfma, kPer, true>();
    }
    __builtin_amdgcn_sched_barrier(0);
    ring_issue_b<SH>(r, o, into, ahead, wave);
    ring_read<A_TR, B_TR, SH>(f1, cur, 1, wm, wn, lane);
    ring_mfma(f0, acc);
    ring_sched<kMfma, kPer, true>();
    __builtin_amdgcn_sched_barrier(0);
    ring_read<A_TR, B_TR, SH>(f0, cur, 2, wm, wn, lane);
    ring_mfma(f1, acc);
    ring_sched<kMfma, kPer, false>();
    __builtin_amdgcn_sched_barrier(0);
    ring_read<A_TR, B_TR, SH>(f1, cur, 3, wm, wn, lane);
    ring_mfma(f0, acc);
    ring_sched<kMfma, kPer, false>();
    stage_barrier<(SH::kStages - 2) * SH::kLoads>();
}

// The K % 64 tail out of `stage` (zeros past K), all four substeps.
template <bool A_TR, bool B_TR, class SH>
__device__ __forceinline__ void ring_tail(const uint16_t* stage, int k_left,
                                          f32x16 (&acc)[SH::kTm][SH::kTn], int wm, int wn,
                                          int lane) {
    for (int s = 0; s * 16 < k_left; ++s) {
        RingFrags<SH::kTm, SH::kTn> f;
        ring_read<A_TR, B_TR, SH>(f, stage, s, wm, wn, lane);
        ring_mfma(f, acc);
    }
}

template <bool OUT_F32, bool A_TR, bool B_TR, class SH>
__global__ __launch_bounds__(256, SH::kPerCu) void gemm_ring_kernel(
    const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ B, int64_t ldb,
    void* __restrict__ C, int64_t ldc, int M, int N, int K, const float* __restrict__ rowscale,
    const uint16_t* __restrict__ colbias, int accumulate, int tiles_m, int tiles_n, int group_m) {
    constexpr int NST = SH::kStages;
    __shared__ __attribute__((aligned(16))) uint16_t st0[SH::kElems];
    __shared__ __attribute__((aligned(16))) uint16_t st1[SH::kElems];
    __shared__ __attribute__((aligned(16))) uint16_t st2[SH::kElems];
    __shared__ __attribute__((aligned(16))) uint16_t st3[NST > 3 ? SH::kElems : 8];
    static_assert(NST == 3 || NST == 4, "ring of three or four stages");

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / SH::kWvn;
    const int wn = wave % SH::kWvn;
    int tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, group_m, tm, tn);
    const int m0 = tm * SH::kBM;
    const int n0 = tn * SH::kBN;
    const int rows_a = M - m0 < SH::kBM ? M - m0 : SH::kBM;
    const int rows_b = N - n0 < SH::kBN ? N - n0 : SH::kBN;
    const uint16_t* a0 = A_TR ? A + m0 : A + static_cast<int64_t>(m0) * lda;
    const uint16_t* b0 = B_TR ? B + n0 : B + static_cast<int64_t>(n0) * ldb;

    RingOperands r;
    r.a = a0;
    r.b = b0;
    r.bytes_a = static_cast<int>(A_TR ? ((K - 1) * lda + rows_a) * 2 : ((rows_a - 1) * lda + K) * 2);
    r.bytes_b = static_cast<int>(B_TR ? ((K - 1) * ldb + rows_b) * 2 : ((rows_b - 1) * ldb + K) * 2);
    r.step_a = A_TR ? static_cast<int>(BK * lda * 2) : BK * 2;
    r.step_b = B_TR ? static_cast<int>(BK * ldb * 2) : BK * 2;
    r.nk = K / BK;
    RingOffsets<SH> o;
    ring_offsets<A_TR, SH::kBM>(o.a, wave, lane, rows_a, lda);
    ring_offsets<B_TR, SH::kBN>(o.b, wave, lane, rows_b, ldb);

    f32x16 acc[SH::kTm][SH::kTn];
#pragma unroll
    for (int i = 0; i < SH::kTm; ++i)
#pragma unroll
        for (int j = 0; j < SH::kTn; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // The K % 64 tail goes first, through the last stage, whose own loads are
    // issued by step 0.
    uint16_t* const last = NST == 3 ? st2 : st3;
    const int k_left = K - r.nk * BK;
    if (k_left) {
        stage_k_tail<A_TR, SH::kBM>(last, a0, lda, rows_a, r.nk * BK, K);
        stage_k_tail<B_TR, SH::kBN>(last + SH::kBM * BK, b0, ldb, rows_b, r.nk * BK, K);
    }
    ring_issue<SH>(r, o, st0, 0, wave);
    ring_issue<SH>(r, o, st1, 1, wave);
    if constexpr (NST > 3) ring_issue<SH>(r, o, st2, 2, wave);
    if (k_left) {
        stage_barrier<(NST - 1) * SH::kLoads>();  // the tail's LDS writes, every wave
        ring_tail<A_TR, B_TR, SH>(last, k_left, acc, wm, wn, lane);
    }
    stage_barrier<(NST - 2) * SH::kLoads>();  // tile 0 has landed; the tail's reads are done

    if (r.nk > 0) {
        RingFrags<SH::kTm, SH::kTn> f0, f1;
#define AGK_RING(FIRST, CUR, INTO, t)                                                           \
    ring_step<FIRST, A_TR, B_TR, SH>(r, o, CUR, INTO, (t) + NST - 1, acc, f0, f1, wm, wn, lane, \
                                     wave)
        AGK_RING(true, st0, last, 0);
        int t = 1;
        if constexpr (NST == 3) {
            for (; t + 2 < r.nk; t += 3) {
                AGK_RING(false, st1, st0, t);
                AGK_RING(false, st2, st1, t + 1);
                AGK_RING(false, st0, st2, t + 2);
            }
            if (t < r.nk) {
                AGK_RING(false, st1, st0, t);
                if (t + 1 < r.nk) AGK_RING(false, st2, st1, t + 1);
            }
        } else {
            for (; t + 3 < r.nk; t += 4) {
                AGK_RING(false, st1, st0, t);
                AGK_RING(false, st2, st1, t + 1);
                AGK_RING(false, st3, st2, t + 2);
                AGK_RING(false, st0, st3, t + 3);
            }
            if (t < r.nk) {
                AGK_RING(false, st1, st0, t);
                if (t + 1 < r.nk) {
                    AGK_RING(false, st2, st1, t + 1);
                    if (t + 2 < r.nk) AGK_RING(false, st3, st2, t + 2);
                }
            }
        }
#undef AGK_RING
        ring_mfma(f1, acc);  // substep 3 of the last tile
    }
    // the empty loads of the last steps still name this workgroup's LDS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    store_block<OUT_F32, Stores::kAll>(acc, C, ldc, M, N, m0 + wm * SH::kTm * 32,
                                       n0 + wn * SH::kTn * 32, lane, rowscale, colbias,
                                       accumulate);
}

template <bool A_TR, bool B_TR>
int launch_ring(int shape, bool f32, const GemmCall& c) {
#define AGK_RING_LAUNCH(F32)                                                                    \
    hipLaunchKernelGGL((gemm_ring_kernel<F32, A_TR, B_TR, SH>), dim3(tiles_m * tiles_n),        \
                       dim3(256), 0, c.st, c.A, c.lda, c.B, c.ldb, c.C, c.ldc, c.M, c.N, c.K,   \
                       c.rowscale, c.colbias, c.accumulate, tiles_m, tiles_n, kGroupM)
#define AGK_RING_CASE(ID, BM_, BN_, WVM, NST)                                                   \
    case ID: {                                                                                  \
        using SH = RingShape<BM_, BN_, WVM, NST>;                                               \
        const int tiles_m = (c.M + BM_ - 1) / BM_, tiles_n = (c.N + BN_ - 1) / BN_;             \
        if (f32) AGK_RING_LAUNCH(true);                                                         \
        else AGK_RING_LAUNCH(false);                                                            \
        break;                                                                                  \
    }
    switch (shape) { AGK_RING_SHAPES(AGK_RING_CASE) }
#undef AGK_RING_CASE
#undef AGK_RING_LAUNCH
    return hipGetLastError() == hipSuccess ? AGK_OK : AGK_EHIP;
}

}  // namespace agk_gemm

#endif  // AGK_RING_KERNELS
