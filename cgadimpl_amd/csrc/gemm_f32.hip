// gemm_f32.hip -- fp32 GEMM for the graph layer's matmul on float32 tensors
// (cgadimpl/src/ops/linalg.cpp:12-20 and its VJP's products,
// cgadimpl/src/autodiff/autodiff_vjp_ops.cpp:258-263), on CDNA4's fp32
// matrix instruction v_mfma_f32_32x32x2_f32.  Not on the RMSNorm layer's
// measured path (its products are bf16, gemm.hip): a general kernel for any
// sizes, leading dimensions, layouts and alignment.
//
//   C[M][ldc] (+)= op(A) op(B)
//
// Tiled kernel.  A workgroup of 256 lanes (4 waves, 2 x 2) computes a BM x BN
// tile of C; each wave owns a quarter of it as 32 x 32 MFMA accumulators.  K
// is walked in steps of 32 through two LDS stages: the loads of step t + 2 are
// issued while step t is multiplied and step t + 1's values, loaded a step
// earlier, are written to the other stage (one barrier per step).  An fp32
// MFMA takes 64 cycles, so a step's MFMAs (0.4 us per wave and 32 x 32 block)
// outlast everything else once a step's loads have two steps to arrive; with
// one step of 16 k to arrive in, as before, the wait for them set the pace.
//
// Operands.  Each operand is staged as a logical [rows][K] matrix (A: M rows,
// B: N rows) into LDS rows of 32 k (128 bytes, 16-byte chunks XOR-swizzled by
// the row), whatever its memory layout:
//  - k contiguous in memory (A as [M][K], B given as B^T [N][K]): 8 lanes load a
//    row's 128 bytes and store them as they are;
//  - rows contiguous (A given as A^T [K][M], B as [K][N]): a lane loads four
//    rows at each of BM / 32 consecutive k and stores BM / 32 k of each row.
// Every load is four consecutive floats, which needs only 4-byte alignment.
// Rows past the matrix repeat valid ones (their products are not stored); k
// past K are staged as zeros.
// An MFMA multiplies two k; which two is free as long as A and B agree, so a
// lane takes four consecutive k of its row as one 16-byte LDS read (lanes 0-31
// k 8 s .. + 3 of substep s, lanes 32-63 k 8 s + 4 .. + 7) and spends them on
// four MFMAs.
//
// Split kernel.  A product with too few tiles for the CUs runs one 32 x 32
// tile per workgroup, its four waves taking the 32-deep steps of K in turn
// (no LDS staging: operands go from memory to the MFMA's registers), their
// sums added in wave order through LDS.
//
// MFMA lane layout (the 32 x 32 block instructions' layout, as in gemm.hip):
// A operand lane l holds row l % 32, k = l / 32; B operand lane l holds
// column l % 32, the same k; accumulator element e of lane l is
// C[8 * (e / 4) + 4 * (l / 32) + e % 4][l % 32].
//
// Determinism: every output element is summed in an order fixed by the sizes
// (no atomics), so results are bit-identical run to run.
// Rounding: fp32 products and sums in the matrix core; the bound is that of
// fp32 summation, |C - exact| <= (K + 1) 2^-24 (|A| |B|).

#include <hip/hip_runtime.h>

#include <stdint.h>

#include "agk_rmsnorm.h"
#include "gemm_common.hpp"
#include "rowcommon.hpp"

namespace agk_sgemm {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));  // in memory, at any float

constexpr int BK = 32;

// Float offset of 16-byte chunk c (0..7) of LDS row `row`: two rows share 256
// bytes (all 64 banks), whose 16 chunks are XOR-swizzled by the row pair.  The
// 16 lanes a 16-byte access serves at a time (rows 0-7 and 24-31 of one chunk,
// or 8 row quads of two chunks) then touch every bank once.
__device__ __forceinline__ int chunk_off(int row, int c) {
    return (row >> 1) * (2 * BK) + (((((row & 1) << 3) | c) ^ ((row >> 1) & 15)) << 2);
}

// One operand's 32-deep step of ROWS rows, as a lane holds it between its
// loads and its LDS writes: ROWS / 32 quads.
template <int ROWS>
struct Step {
    f32x4 v[ROWS / 32];
};

// What lane t of 256 loads of the operand whose rows r0 .. start at p, fixed for
// all steps.  KC: quad i holds k (t % 8) * 4 .. + 3 of row t / 8 + 32 i.
// Otherwise quad i holds four rows at k + i; 8 lanes cover 32 rows (128 bytes).
template <bool KC, int ROWS>
struct Place {
    const float* p;    // the quad's address at k = 0, quad 0
    int64_t ld;
    int rows;          // valid rows of the tile
    int r, k;          // first row and first k of the lane's quads, as staged
    int from;          // !KC: the first row loaded (below r by `shift` at the matrix's edge)
    int shift;
    bool edge;         // !KC: some lane of the workgroup has a shift
};

template <bool KC, int ROWS>
__device__ __forceinline__ Place<KC, ROWS> place(const float* __restrict__ src, int64_t ld, int r0,
                                                 int rows_total, int t) {
    Place<KC, ROWS> q;
    q.ld = ld;
    q.rows = rows_total - r0 < ROWS ? rows_total - r0 : ROWS;
    q.shift = 0;
    q.edge = false;
    if constexpr (KC) {
        q.r = q.from = t >> 3;
        q.k = (t & 7) * 4;
        q.p = src + static_cast<int64_t>(r0) * ld;
    } else {
        constexpr int kKb = 32 / (ROWS / 32);  // k groups of a step
        q.r = ((t & 7) + 8 * ((t >> 3) / kKb)) * 4;
        q.k = ((t >> 3) % kKb) * (ROWS / 32);
        q.p = src + r0;
        // rows_total >= 4: the quad stays inside the matrix (perhaps in the
        // tile before this one)
        q.from = q.r <= q.rows - 4 ? q.r : q.rows - 4;
        q.shift = q.r - q.from < 4 ? q.r - q.from : 0;
        q.edge = (q.rows & 3) != 0;
    }
    return q;
}

// Loads the whole step at k0 (k0 + 32 <= K).
template <bool KC, int ROWS>
__device__ __forceinline__ void load_step(Step<ROWS>& s, const Place<KC, ROWS>& q, int k0) {
#pragma unroll
    for (int i = 0; i < ROWS / 32; ++i) {
        if constexpr (KC) {
            const int row = q.r + 32 * i < q.rows ? q.r + 32 * i : q.rows - 1;
            s.v[i] = *reinterpret_cast<const f32x4_a4*>(q.p + static_cast<int64_t>(row) * q.ld + k0 +
                                                        q.k);
        } else {
            s.v[i] = *reinterpret_cast<const f32x4_a4*>(
                q.p + static_cast<int64_t>(k0 + q.k + i) * q.ld + q.from);
        }
    }
}

// The last K % 32 k, at k0: element by element, zeros past K.
template <bool KC, int ROWS>
__device__ __forceinline__ void load_tail(Step<ROWS>& s, const Place<KC, ROWS>& q, int k0, int K) {
#pragma unroll
    for (int i = 0; i < ROWS / 32; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = k0 + q.k + (KC ? e : i);
            int row = KC ? q.r + 32 * i : q.from + e;
            row = row < q.rows ? row : q.rows - 1;
            s.v[i][e] = k >= K ? 0.0f
                               : KC ? q.p[static_cast<int64_t>(row) * q.ld + k]
                                    : q.p[static_cast<int64_t>(k) * q.ld + row];
        }
}

template <bool KC, int ROWS>
__device__ __forceinline__ void store_step(const Step<ROWS>& s, const Place<KC, ROWS>& q,
                                           float* lds) {
    if constexpr (KC) {
#pragma unroll
        for (int i = 0; i < ROWS / 32; ++i)
            *reinterpret_cast<f32x4*>(lds + chunk_off(q.r + 32 * i, q.k >> 2)) = s.v[i];
    } else {
        Step<ROWS> w = s;
        if (q.edge) {  // a quad moved down by `shift` rows holds row r + e at e + shift
#pragma unroll
            for (int i = 0; i < ROWS / 32; ++i)
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                    float x = s.v[i][e];
                    x = q.shift == 1 ? s.v[i][e + 1] : x;
                    x = q.shift == 2 ? s.v[i][e + 2 < 4 ? e + 2 : 3] : x;
                    x = q.shift == 3 ? s.v[i][3] : x;
                    w.v[i][e] = x;
                }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float* at = lds + chunk_off(q.r + e, q.k >> 2) + (q.k & 3);
            if constexpr (ROWS == 64)
                *reinterpret_cast<f32x2*>(at) = f32x2{w.v[0][e], w.v[1][e]};
            else
                *reinterpret_cast<f32x4*>(at) =
                    f32x4{w.v[0][e], w.v[1][e], w.v[2][e], w.v[3][e]};
        }
    }
}

template <int NT>
struct Quads {
    f32x4 v[NT];
};

// The quads of substep s for NT blocks of 32 rows from row0.
template <int NT>
__device__ __forceinline__ void read_quads(Quads<NT>& f, const float* lds, int row0, int s,
                                           int lane) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
        f.v[i] = *reinterpret_cast<const f32x4*>(
            lds + chunk_off(row0 + i * 32 + (lane & 31), 2 * s + (lane >> 5)));
}

template <int TM, int TN>
__device__ __forceinline__ void mfma_quads(const Quads<TM>& a, const Quads<TN>& b,
                                           f32x16 (&acc)[TM][TN]) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[i][e], b.v[j][e], acc[i][j],
                                                                 0, 0, 0);
}

// A_KC: A is [M][lda] (k contiguous), else A^T [K][lda]; B_KC: B is given as
// B^T [N][ldb] (k contiguous), else B [K][ldb].
template <int BM, int BN, bool A_KC, bool B_KC>
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
    float* __restrict__ C, int64_t ldc, int M, int N, int K, int accumulate, int tiles_m,
    int tiles_n) {
    constexpr int kStage = (BM + BN) * BK;
    __shared__ __attribute__((aligned(16))) float l0[kStage];
    __shared__ __attribute__((aligned(16))) float l1[kStage];

    constexpr int TM = BM / 64, TN = BN / 64;  // 32 x 32 MFMA blocks per wave
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    int tm, tn;
    agk_gemm::tile_of(blockIdx.x, tiles_m, tiles_n, agk_gemm::kGroupM, tm, tn);
    const int m0 = tm * BM;
    const int n0 = tn * BN;

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    const Place<A_KC, BM> pa = place<A_KC, BM>(A, lda, m0, M, tid);
    const Place<B_KC, BN> pb = place<B_KC, BN>(B, ldb, n0, N, tid);
    const int nk = K / BK;  // whole steps
    Quads<TM> fa[2];
    Quads<TN> fb[2];
    auto read = [&](int f, const float* stage, int s) {
        read_quads(fa[f], stage, wm * (BM / 2), s, lane);
        read_quads(fb[f], stage + BM * BK, wn * (BN / 2), s, lane);
    };
    if (K % BK) {  // the ragged end of K first
        Step<BM> ta;
        Step<BN> tb;
        load_tail(ta, pa, nk * BK, K);
        load_tail(tb, pb, nk * BK, K);
        store_step(ta, pa, l1);
        store_step(tb, pb, l1 + BM * BK);
        __syncthreads();
        for (int s = 0; s * 8 < K % BK; ++s) {
            read(0, l1, s);
            mfma_quads(fa[0], fb[0], acc);
        }
    }
    if (nk > 0) {
        Step<BM> a0, a1;
        Step<BN> b0, b1;
        // step u, or the last one again: the loop below loads and stores
        // without conditions, so that the compiler can count the loads in
        // flight (behind a condition it waited for all of them each step)
        auto load = [&](Step<BM>& a, Step<BN>& b, int u) {
            const int k0 = (u < nk ? u : nk - 1) * BK;
            load_step(a, pa, k0);
            load_step(b, pb, k0);
        };
        auto store = [&](const Step<BM>& a, const Step<BN>& b, float* stage) {
            store_step(a, pa, stage);
            store_step(b, pb, stage + BM * BK);
        };
        load(a0, b0, 0);
        load(a1, b1, 1);
        store(a0, b0, l0);
        __syncthreads();
        // Step t out of `cur`.  (na, nb) are free and take step t + 2; (wa, wb)
        // hold step t + 1, for `nxt`.  The fragments run one substep ahead of
        // the MFMAs, across the barrier.
#define AGK_F32_STEP(FIRST, t, cur, nxt, na, nb, wa, wb) \
    load(na, nb, (t) + 2);                               \
    read(0, cur, 0);                                     \
    if (!FIRST) mfma_quads(fa[1], fb[1], acc);           \
    read(1, cur, 1);                                     \
    mfma_quads(fa[0], fb[0], acc);                       \
    read(0, cur, 2);                                     \
    mfma_quads(fa[1], fb[1], acc);                       \
    read(1, cur, 3);                                     \
    store(wa, wb, nxt);                                  \
    mfma_quads(fa[0], fb[0], acc);                       \
    __syncthreads();
        AGK_F32_STEP(true, 0, l0, l1, a0, b0, a1, b1)
        int t = 1;
        for (; t + 1 < nk; t += 2) {
            AGK_F32_STEP(false, t, l1, l0, a1, b1, a0, b0)
            AGK_F32_STEP(false, t + 1, l0, l1, a0, b0, a1, b1)
        }
        if (t < nk) {
            AGK_F32_STEP(false, t, l1, l0, a1, b1, a0, b0)
        }
#undef AGK_F32_STEP
        mfma_quads(fa[1], fb[1], acc);  // the last step's substep 3
    }

    const int col_l = lane & 31;
    const int row_l = 4 * (lane >> 5);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int row = m0 + wm * (BM / 2) + i * 32 + 8 * (e >> 2) + row_l + (e & 3);
            if (row >= M) continue;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int col = n0 + wn * (BN / 2) + j * 32 + col_l;
                if (col >= N) continue;
                float* p = C + static_cast<int64_t>(row) * ldc + col;
                const float v = acc[i][j][e];
                *p = accumulate ? agk::acc_add(*p, v) : v;
            }
        }
    }
}

// ---- split kernel --------------------------------------------------------------------
constexpr int kSplitWaves = 4;

// An operand's values for a 32-deep step, in MFMA order: v[s][e] is k
// 8 s + 4 (lane / 32) + e of the lane's row.
struct DirectStep {
    f32x4 v[4];
};

// p: the lane's row at k = 4 (lane / 32) of the step's first k.
template <bool KC>
__device__ __forceinline__ void direct_step(DirectStep& d, const float* __restrict__ p,
                                            int64_t ld) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if constexpr (KC) {
            d.v[s] = *reinterpret_cast<const f32x4_a4*>(p + 8 * s);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) d.v[s][e] = p[(8 * s + e) * ld];
        }
    }
}

// The ragged last step: `left` k remain from the lane's first; zeros past them.
template <bool KC>
__device__ __forceinline__ void direct_tail(DirectStep& d, const float* __restrict__ p, int64_t ld,
                                            int left) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            d.v[s][e] = 8 * s + e >= left ? 0.0f : KC ? p[8 * s + e] : p[(8 * s + e) * ld];
}

__device__ __forceinline__ void direct_mfma(const DirectStep& a, const DirectStep& b,
                                            f32x16& acc) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[s][e], b.v[s][e], acc, 0, 0, 0);
}

template <bool A_KC, bool B_KC>
__global__ __launch_bounds__(kSplitWaves * 64, 2) void gemm_f32_split_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
    float* __restrict__ C, int64_t ldc, int M, int N, int K, int accumulate, int tiles,
    int tiles_n) {
    __shared__ float part[kSplitWaves][16][64];  // [wave][accumulator element][lane]

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int half = lane >> 5;
    const int tile = static_cast<int>(blockIdx.y * gridDim.x + blockIdx.x);
    if (tile >= tiles) return;  // workgroup-uniform, before any barrier
    const int m0 = (tile / tiles_n) * 32;
    const int n0 = (tile % tiles_n) * 32;
    const int64_t ra = m0 + (lane & 31) < M ? m0 + (lane & 31) : M - 1;
    const int64_t rb = n0 + (lane & 31) < N ? n0 + (lane & 31) : N - 1;
    // the lane's row at k = 32 wave + 4 half, and what 32 kSplitWaves k further on are
    const int64_t k1 = 32 * wave + 4 * half;
    const float* pa = A_KC ? A + ra * lda + k1 : A + k1 * lda + ra;
    const float* pb = B_KC ? B + rb * ldb + k1 : B + k1 * ldb + rb;
    const int64_t da = 32 * kSplitWaves * (A_KC ? 1 : lda), db = 32 * kSplitWaves * (B_KC ? 1 : ldb);

    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    // this wave's steps: wave, wave + kSplitWaves, ...; the next one's loads are in
    // flight while one is multiplied
    const int whole = K / BK;
    DirectStep a0, b0, a1, b1;
    int t = wave;
    if (t < whole) {
        direct_step<A_KC>(a0, pa, lda);
        direct_step<B_KC>(b0, pb, ldb);
    }
    for (; t + kSplitWaves < whole; t += 2 * kSplitWaves) {
        pa += da;
        pb += db;
        direct_step<A_KC>(a1, pa, lda);
        direct_step<B_KC>(b1, pb, ldb);
        direct_mfma(a0, b0, acc);
        pa += da;
        pb += db;
        if (t + 2 * kSplitWaves < whole) {
            direct_step<A_KC>(a0, pa, lda);
            direct_step<B_KC>(b0, pb, ldb);
        }
        direct_mfma(a1, b1, acc);
    }
    if (t < whole) {
        direct_mfma(a0, b0, acc);
        t += kSplitWaves;
        pa += da;
        pb += db;
    }
    if (t * BK < K) {  // the ragged step falls to the wave whose turn it is
        const int left = K - t * BK - 4 * half;
        direct_tail<A_KC>(a0, pa, lda, left);
        direct_tail<B_KC>(b0, pb, ldb, left);
        direct_mfma(a0, b0, acc);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) part[wave][e][lane] = acc[e];
    __syncthreads();
    // wave w adds and stores elements 16 w / kSplitWaves ..
#pragma unroll
    for (int i = 0; i < 16 / kSplitWaves; ++i) {
        const int e = wave * (16 / kSplitWaves) + i;
        float v = part[0][e][lane];
#pragma unroll
        for (int w = 1; w < kSplitWaves; ++w) v += part[w][e][lane];
        const int row = m0 + 8 * (e >> 2) + 4 * half + (e & 3);
        const int col = n0 + (lane & 31);
        if (row < M && col < N) {
            float* p = C + static_cast<int64_t>(row) * ldc + col;
            *p = accumulate ? agk::acc_add(*p, v) : v;
        }
    }
}

// C = 0 over M rows of N columns (ldc apart): the empty sum (K == 0).  A
// kernel, not a memset, so that the call can be captured.
__global__ __launch_bounds__(256) void zero_rows_kernel(float* __restrict__ C, int64_t ldc,
                                                        int N) {
    float* r = C + static_cast<int64_t>(blockIdx.x) * ldc;
    for (int c = threadIdx.x; c < N; c += 256) r[c] = 0.0f;
}

// 2: 128 x 128 tiles, 1: 64 x 64 tiles, 0: 32 x 32 tiles with K split over the
// waves.  The cheapest by the microseconds a CU spends per 32-deep step: its
// share of the tiles times a tile's time, measured on MI355X.  A tile's MFMAs
// take 1.7 / 0.43 / 0.11 us; what it costs beyond them is staging and, alone
// on its CU, waiting:
//               alone   with others   measured (us; K-contiguous operands)
//   128 x 128    2.1       1.95       4096^3: 1000 (64 x 64: 1022, split: 1803)
//   64 x 64      0.6       0.53       1024^3: 24 (128 x 128: 71, split: 34)
//   split        0.25      0.25       300 x 500 x 4095: 33 (64 x 64: 77)
// The kernel this replaced: 1024^3 42 us, 300 x 500 x 4095 143 us,
// 4096^3 1138-1333 us (by layout; now 1000-1049).
inline int pick_f32(int64_t M, int64_t N, int cus) {
    auto per_cu = [&](int64_t t) {
        return static_cast<double>((((M + t - 1) / t) * ((N + t - 1) / t) + cus - 1) / cus);
    };
    const double c32 = per_cu(32), c64 = per_cu(64), c128 = per_cu(128);
    const double split = 0.25 * c32;
    const double small = c64 > 1 ? 0.53 * c64 : 0.6;
    const double large = c128 > 1 ? 1.95 * c128 : 2.1;
    if (split < small && split < large) return 0;
    return small < large ? 1 : 2;
}

struct F32Plan {
    int shape, tile;  // pick_f32's, and its tile's rows and columns
    int64_t tiles_m, tiles_n;
    int64_t grid_x, grid_y;  // the split kernel's tiles may need a second dimension
};

// a_kc: A k-contiguous (not given transposed); b_kc: B k-contiguous (given as B^T).
inline F32Plan plan_f32(int64_t M, int64_t N, bool a_kc, bool b_kc, int cus) {
    F32Plan p;
    p.shape = pick_f32(M, N, cus);
    // the tiled kernel loads four rows at a time of an operand whose rows are
    // contiguous: it needs four of them
    if ((!a_kc && M < 4) || (!b_kc && N < 4)) p.shape = 0;
    auto set = [&](int shape) {
        p.shape = shape;
        p.tile = shape == 2 ? 128 : shape == 1 ? 64 : 32;
        p.tiles_m = (M + p.tile - 1) / p.tile;
        p.tiles_n = (N + p.tile - 1) / p.tile;
    };
    set(p.shape);
    p.grid_x = p.tiles_m * p.tiles_n;
    p.grid_y = 1;
    if (p.shape == 1 && !agk::grid_fits(p.grid_x, 256)) {
        set(2);
        p.grid_x = p.tiles_m * p.tiles_n;
    } else if (p.shape == 0 && !agk::grid_fits(p.grid_x, 256)) {
        constexpr int64_t kRow = 1 << 20;
        p.grid_y = (p.grid_x + kRow - 1) / kRow;
        p.grid_x = kRow;
    }
    return p;
}

}  // namespace agk_sgemm

extern "C" int agk_gemm_f32_launch_plan(int64_t M, int64_t N, int a_trans, int b_trans, int cus,
                                        int64_t* plan) {
    using namespace agk_sgemm;
    constexpr int64_t kMax = 0x7fffffffLL;
    if (!plan || M < 1 || N < 1 || M > kMax || N > kMax) return AGK_EINVAL;
    const F32Plan p = plan_f32(M, N, a_trans == 0, b_trans != 0,
                               cus > 0 ? cus : agk_gemm::device_cus());
    plan[0] = p.shape;
    plan[1] = plan[2] = p.tile;
    plan[3] = p.grid_x;
    plan[4] = p.grid_y;
    return AGK_OK;
}

extern "C" int agk_gemm_f32(const float* A, int64_t lda, int a_trans, const float* B, int64_t ldb,
                            int b_trans, float* C, int64_t ldc, int64_t M, int64_t N, int64_t K,
                            int accumulate, agk_stream_t stream) {
    using namespace agk_sgemm;
    constexpr int64_t kMax = 0x7fffffffLL;
    if (M < 0 || N < 0 || K < 0 || M > kMax || N > kMax || K > kMax) return AGK_EINVAL;
    if (M == 0 || N == 0) return AGK_OK;
    if (!C || ldc < N) return AGK_EINVAL;
    if (K > 0) {
        if (!A || !B) return AGK_EINVAL;
        if (lda < (a_trans ? M : K) || ldb < (b_trans ? K : N)) return AGK_EINVAL;
    }
    agk::clear_pending_error();
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
    if (K == 0) {  // the empty sum: zeros, or C as it was
        if (accumulate) return AGK_OK;
        hipLaunchKernelGGL(zero_rows_kernel, dim3(static_cast<unsigned>(m)), dim3(256), 0, st, C,
                           ldc, n);
        return agk::check_launch();
    }
    const bool a_kc = a_trans == 0, b_kc = b_trans != 0;
    const F32Plan p = plan_f32(M, N, a_kc, b_kc, agk_gemm::device_cus());
    if (p.tiles_m * p.tiles_n > kMax) return AGK_EINVAL;
    const dim3 grid(static_cast<unsigned>(p.grid_x), static_cast<unsigned>(p.grid_y));
    const int acc = accumulate != 0;
    const int tm = static_cast<int>(p.tiles_m), tn = static_cast<int>(p.tiles_n);
#define AGK_F32(AK, BKC)                                                                      \
    switch (p.shape) {                                                                        \
        case 2:                                                                               \
            hipLaunchKernelGGL((gemm_f32_kernel<128, 128, AK, BKC>), grid, dim3(256), 0, st,  \
                               A, lda, B, ldb, C, ldc, m, n, k, acc, tm, tn);                 \
            break;                                                                            \
        case 1:                                                                               \
            hipLaunchKernelGGL((gemm_f32_kernel<64, 64, AK, BKC>), grid, dim3(256), 0, st, A, \
                               lda, B, ldb, C, ldc, m, n, k, acc, tm, tn);                    \
            break;                                                                            \
        default:                                                                              \
            hipLaunchKernelGGL((gemm_f32_split_kernel<AK, BKC>), grid, dim3(kSplitWaves * 64), \
                               0, st, A, lda, B, ldb, C, ldc, m, n, k, acc, tm * tn, tn);     \
    }
    if (a_kc && b_kc) AGK_F32(true, true)
    else if (a_kc) AGK_F32(true, false)
    else if (b_kc) AGK_F32(false, true)
    else AGK_F32(false, false)
#undef AGK_F32
    return agk::check_launch();
}
