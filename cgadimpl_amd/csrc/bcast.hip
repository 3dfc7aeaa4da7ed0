// bcast.hip -- element-wise multiply under numpy broadcasting and its VJP:
// mul_nodeops for operands of any broadcast-compatible shapes
// (cgadimpl/src/ops/arithmetic.cpp:31-39, `a->value * b->value`) and vjp_Mul
// (cgadimpl/src/autodiff/autodiff_vjp_ops.cpp:54-59) with reduce_for_broadcast
// (:15-35): the gradient of an operand is gy * other, summed over the axes on
// which that operand was broadcast (axes it lacks, or where its extent is 1
// and the output's is not).
//
// The hot broadcast of the RMSNorm layer (a row vector over the rows) has its
// own kernels in rowops.hip; this file covers every other shape pair, e.g.
// [B, T, D] * [B, 1, D], [R, 1] * [1, C], a scalar times a tensor.
//
// Layout: all operands contiguous, row-major.  Shapes align at the trailing
// axis; after alignment each axis of an operand has the output's extent or 1.
// The host merges adjacent axes that both operands walk contiguously (and
// drops extent-1 output axes), so a launch sees at most 8 axes, usually 2-3.
//
// The broadcasts that training code writes most -- a full operand times a vector
// per group of rows ([B, T, D] * [B, 1, D], [B, T, D] * [T, D]) or a scalar per row
// ([B, T, D] * [B, T, 1]) -- have kernels of their own over a rows x cols view of
// the full operand (RowsView): 16-byte accesses at any element alignment
// (rowcommon.hpp, ragged rows), and a backward that reads gy and the full operand
// once for both gradients.  The general kernels take every other pair, products that
// they are faster for (rows_mul_fits) and outputs that lie over the operands:
//
// Forward / full-shape gradient (y (+)= a * b): one workgroup row per run of
// the innermost output axis; its base offsets into a and b are decomposed once
// per run, the lanes walk the run, 16 bytes at a time when the innermost axis
// is contiguous or broadcast in both operands and aligned (element by element
// otherwise).  HBM-bound: reads a and b (b often from cache), writes y.
//
// Reduced gradient (d[j] (+)= sum over the broadcast positions of gy * other),
// accumulating exact products in fp64 and rounding to fp32 once, in an order
// fixed by the shapes (results identical run to run):
//  - the output keeps the innermost axis ([B, T, D] -> [B, 1, D]): a lane per
//    output element, 64 consecutive ones per workgroup, each of its four waves
//    summing a contiguous quarter of the reduced positions (loads contiguous
//    across the lanes); the quarters are added in order;
//  - otherwise (the innermost axis is reduced: [R, C] -> [R, 1]): one wave
//    (short sums) or one 256-lane workgroup (long sums) per output element;
//    lane l takes positions l, l + lanes, ... of the reduced index space in
//    row-major order, and the lanes' partials meet in a fixed tree in LDS.

#include <hip/hip_runtime.h>

#include <stdint.h>

#include "agk_rmsnorm.h"
#include "rowcommon.hpp"

namespace agk {

constexpr int kBcastMaxDims = 8;
constexpr int kBcastBlock = 256;

// Output axes (outermost first) with each operand's element stride (0 where it
// is broadcast).
struct BcastGeom {
    int nd;
    int64_t size[kBcastMaxDims];
    int64_t sa[kBcastMaxDims];
    int64_t sb[kBcastMaxDims];
};

// A gradient reduction: the kept axes (extent > 1 in the target, in order,
// so the target's own offset is the row-major index over them) and the
// reduced axes; strides into gy (the output layout) and into the other
// operand for each.
struct BcastRed {
    int nk, nr;
    int64_t ksize[kBcastMaxDims], kgy[kBcastMaxDims], ko[kBcastMaxDims];
    int64_t rsize[kBcastMaxDims], rgy[kBcastMaxDims], ro[kBcastMaxDims];
    int64_t rtotal;  // product of rsize
};

// y[o] (+)= a[.] * b[.] over the output; each block row handles runs of the
// innermost axis (grid-stride over runs).  The product is rounded to storage
// before an accumulating add, as `grad += g` rounds g first.
template <class S>
__global__ __launch_bounds__(kBcastBlock) void bcast_mul_kernel(const typename S::T* __restrict__ a,
                                                               const typename S::T* __restrict__ b,
                                                               typename S::T* __restrict__ y,
                                                               const BcastGeom g, int64_t runs,
                                                               int accumulate) {
    const int last = g.nd - 1;
    const int64_t inner = g.size[last];
    for (int64_t run = blockIdx.y; run < runs; run += gridDim.y) {
        int64_t oa = 0, ob = 0, rem = run;
        for (int d = last - 1; d >= 0; --d) {
            const int64_t c = rem % g.size[d];
            rem /= g.size[d];
            oa += c * g.sa[d];
            ob += c * g.sb[d];
        }
        typename S::T* yr = y + run * inner;
        for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBcastBlock + threadIdx.x; i < inner;
             i += static_cast<int64_t>(gridDim.x) * kBcastBlock) {
            const float p = S::get(a + oa + i * g.sa[last]) * S::get(b + ob + i * g.sb[last]);
            if (accumulate)
                S::put(yr + i, acc_add(S::get(yr + i), S::stored(p)));
            else
                S::put(yr + i, p);
        }
    }
}

// d[j] (+)= sum over reduced positions of gy * other, fp64, fixed order.
// LANES lanes per element of d (64: one wave; 256: the whole workgroup).
template <class S, int LANES>
__global__ __launch_bounds__(kBcastBlock) void bcast_reduce_kernel(
    const typename S::T* __restrict__ gy, const typename S::T* __restrict__ other,
    float* __restrict__ d, const BcastRed r, int64_t n_out, int accumulate) {
    constexpr int kPer = kBcastBlock / LANES;  // elements of d per workgroup
    __shared__ double part[kBcastBlock];
    const int lane = threadIdx.x % LANES;
    const int slot = threadIdx.x / LANES;
    for (int64_t base = static_cast<int64_t>(blockIdx.x) * kPer; base < n_out;
         base += static_cast<int64_t>(gridDim.x) * kPer) {
        const int64_t j = base + slot;
        double acc = 0.0;
        if (j < n_out) {
            int64_t og = 0, oo = 0, rem = j;
            for (int k = r.nk - 1; k >= 0; --k) {
                const int64_t c = rem % r.ksize[k];
                rem /= r.ksize[k];
                og += c * r.kgy[k];
                oo += c * r.ko[k];
            }
            // position q = oq * inner_r + i (oq over the outer reduced axes, i
            // along the innermost one); q steps by LANES, and the outer offsets
            // are re-derived only when i leaves the innermost axis
            const int ia = r.nr - 1;
            const int64_t inner_r = r.rsize[ia], sg = r.rgy[ia], so = r.ro[ia];
            auto outer = [&](int64_t oq, int64_t& bg, int64_t& bo) {
                bg = og;
                bo = oo;
                for (int k = ia - 1; k >= 0; --k) {
                    const int64_t c = oq % r.rsize[k];
                    oq /= r.rsize[k];
                    bg += c * r.rgy[k];
                    bo += c * r.ro[k];
                }
            };
            int64_t oq = lane / inner_r, i = lane - oq * inner_r, bg, bo;
            outer(oq, bg, bo);
            for (int64_t q = lane; q < r.rtotal; q += LANES) {
                acc += static_cast<double>(S::get(gy + bg + i * sg)) *
                       static_cast<double>(S::get(other + bo + i * so));
                i += LANES;
                if (i >= inner_r) {
                    oq += i / inner_r;
                    i %= inner_r;
                    outer(oq, bg, bo);
                }
            }
        }
        part[threadIdx.x] = acc;
        __syncthreads();
#pragma unroll
        for (int w = LANES / 2; w > 0; w /= 2) {
            if (lane < w) part[threadIdx.x] += part[threadIdx.x + w];
            __syncthreads();
        }
        if (lane == 0 && j < n_out) {
            const double old = accumulate ? static_cast<double>(d[j]) : 0.0;
            d[j] = static_cast<float>(old + part[threadIdx.x]);
        }
        __syncthreads();
    }
}

// The same product with 16-byte accesses, when the innermost axis is
// contiguous (stride 1) or broadcast (stride 0) in both operands, its extent a
// multiple of the slot width and every base 16-byte aligned.  A run's base
// offsets are computed once per workgroup and a broadcast operand's value once
// per run; the lanes walk the run's slots.  Same roundings as the element-wise
// kernel, so the results are the same bits.
template <class S>
__global__ __launch_bounds__(kBcastBlock) void bcast_mul_vec_kernel(
    const typename S::T* __restrict__ a, const typename S::T* __restrict__ b,
    typename S::T* __restrict__ y, const BcastGeom g, int64_t runs, int accumulate) {
    using T = typename S::T;
    constexpr int W = S::kVec;
    const int last = g.nd - 1;
    const int64_t inner = g.size[last];
    const int64_t nvec = inner / W;
    const bool a_vec = g.sa[last] != 0;
    const bool b_vec = g.sb[last] != 0;
    for (int64_t run = blockIdx.y; run < runs; run += gridDim.y) {
        int64_t oa = 0, ob = 0, rem = run;
        for (int d = last - 1; d >= 0; --d) {
            const int64_t c = rem % g.size[d];
            rem /= g.size[d];
            oa += c * g.sa[d];
            ob += c * g.sb[d];
        }
        const T* ar = a + oa;
        const T* br = b + ob;
        T* yr = y + run * inner;
        const float as = a_vec ? 0.0f : S::get(ar);
        const float bs = b_vec ? 0.0f : S::get(br);
        for (int64_t v = static_cast<int64_t>(blockIdx.x) * kBcastBlock + threadIdx.x; v < nvec;
             v += static_cast<int64_t>(gridDim.x) * kBcastBlock) {
            float fa[W], fb[W], p[W];
            if (a_vec) {
                S::unpack(load16<S>(ar + v * W), fa);
            } else {
#pragma unroll
                for (int e = 0; e < W; ++e) fa[e] = as;
            }
            if (b_vec) {
                S::unpack(load16<S>(br + v * W), fb);
            } else {
#pragma unroll
                for (int e = 0; e < W; ++e) fb[e] = bs;
            }
#pragma unroll
            for (int e = 0; e < W; ++e) p[e] = fa[e] * fb[e];
            if (accumulate) {
                float old[W];
                S::unpack(load16<S>(yr + v * W), old);
#pragma unroll
                for (int e = 0; e < W; ++e) p[e] = acc_add(old[e], S::stored(p[e]));
            }
            store16_stream<S>(yr + v * W, S::pack(p));
        }
    }
}

// A reduction whose output keeps the innermost axis (e.g. [B, T, D] summed to
// [B, 1, D]): each workgroup takes 64 consecutive outputs, one per lane, so a
// wave's loads are contiguous in gy.  The reduced index space is cut into four
// contiguous quarters, one per wave; a wave walks its quarter along the
// innermost reduced axis (divisions only when it moves to the next outer
// reduced position), accumulating exact products in fp64.  The quarters'
// partials are added in quarter order: a fixed order for the shapes.
template <class S>
__global__ __launch_bounds__(kBcastBlock) void bcast_reduce_cols_kernel(
    const typename S::T* __restrict__ gy, const typename S::T* __restrict__ other,
    float* __restrict__ d, const BcastRed r, int64_t n_out, int accumulate) {
    __shared__ double part[4][64];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int inner_ax = r.nr - 1;
    const int64_t inner_r = r.rsize[inner_ax];
    const int64_t sg = r.rgy[inner_ax], so = r.ro[inner_ax];
    const int64_t q0 = r.rtotal * w / 4, q1 = r.rtotal * (w + 1) / 4;
    for (int64_t base = static_cast<int64_t>(blockIdx.x) * 64; base < n_out;
         base += static_cast<int64_t>(gridDim.x) * 64) {
        const int64_t j = base + lane;
        double acc = 0.0;
        if (j < n_out) {
            int64_t og = 0, oo = 0, rem = j;
            for (int k = r.nk - 1; k >= 0; --k) {
                const int64_t c = rem % r.ksize[k];
                rem /= r.ksize[k];
                og += c * r.kgy[k];
                oo += c * r.ko[k];
            }
            for (int64_t q = q0; q < q1;) {
                const int64_t oq = q / inner_r;
                const int64_t i0 = q - oq * inner_r;
                int64_t pg = og, po = oo, qr = oq;
                for (int k = inner_ax - 1; k >= 0; --k) {
                    const int64_t c = qr % r.rsize[k];
                    qr /= r.rsize[k];
                    pg += c * r.rgy[k];
                    po += c * r.ro[k];
                }
                const int64_t i1 = inner_r - i0 < q1 - q ? inner_r : i0 + (q1 - q);
#pragma unroll 4
                for (int64_t i = i0; i < i1; ++i)
                    acc += static_cast<double>(S::get(gy + pg + i * sg)) *
                           static_cast<double>(S::get(other + po + i * so));
                q += i1 - i0;
            }
        }
        part[w][lane] = acc;
        __syncthreads();
        if (w == 0 && j < n_out) {
            const double s = ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane];
            const double old = accumulate ? static_cast<double>(d[j]) : 0.0;
            d[j] = static_cast<float>(old + s);
        }
        __syncthreads();
    }
}

// ---- rows x cols views -----------------------------------------------------------
// The full operand as rows of cols contiguous elements; the other is a vector of
// cols elements per group of `group` consecutive rows (row r uses vector
// r / group), or with SCALAR one element per row.  cols holds at least one slot.

// First column of slot `slot`: the last slot is moved back to end with the row.
template <int W>
__device__ __forceinline__ int64_t view_col(int64_t slot, int64_t cols) {
    const int64_t c = slot * W;
    return c + W > cols ? cols - W : c;
}

// A slot of the full operand or of gy.  STREAM: past the caches.
template <class S, bool STREAM>
__device__ __forceinline__ u32x4 view_load(const typename S::T* p) {
    if constexpr (STREAM) return load16_any_stream<S>(p);
    else return load16_any<S>(p);
}

// y (+)= r for one slot, leaving out the first `dup` elements when adding.
template <class S>
__device__ __forceinline__ void view_store(typename S::T* y, float (&r)[S::kVec], int dup,
                                           int accumulate) {
    constexpr int W = S::kVec;
    if (accumulate) {
        if (dup > 0) {
#pragma unroll
            for (int e = 0; e < W; ++e)
                if (e >= dup) S::put(y + e, acc_add(S::get(y + e), S::stored(r[e])));
            return;
        }
        float old[W];
        S::unpack(load16_any_stream<S>(y), old);
#pragma unroll
        for (int e = 0; e < W; ++e) r[e] = acc_add(old[e], S::stored(r[e]));
    }
    store16_any_stream<S>(y, S::pack(r));
}

// y (+)= full * other.  TPR lanes per row and chunk of 4 TPR slots, so that a
// workgroup streams 16 KiB: HBM-bound (reads full, writes y; `other` comes from
// the caches).
// Measured on MI355X (us, before / now, the element-wise and run-per-workgroup
// kernels before): bf16 32 x 2048 x 4096 by 32 x 1 x 4096 209 / 174 (6.2 TB/s), by 65536 x
// 1 184 / 167; bf16 2 x 2048 x 4001 by 2 x 1 x 4001 78 / 16; f32 355 / 352.  With the
// backward kernels below, both gradients: bf16 411 / 257, 587 / 274, 129 / 64; f32
// 742 / 545, 794 / 573, 130 / 71.
//
// Workgroup `id` takes one row block and chunk (view_block).  Rows of 8 chunks and
// more: chunk c runs on XCD c % 8 (workgroup L runs on XCD L % 8), for one row block
// after the other, so that c's part of `other` is read into one XCD's L2 once.
constexpr int kViewSlots = 4;
constexpr uint32_t kViewXcds = 8;

struct ViewBlocks {
    uint32_t nrow, nchunk;  // row blocks, chunks of a row
    __host__ __device__ bool wide() const { return nchunk >= kViewXcds; }
    __host__ __device__ uint32_t total() const {  // with the padding
        return nrow * (wide() ? (nchunk + kViewXcds - 1) / kViewXcds * kViewXcds : nchunk);
    }
};

__device__ __forceinline__ void view_block(const ViewBlocks& b, uint32_t id, uint32_t& row,
                                           uint32_t& chunk) {
    const uint32_t q = b.wide() ? id / kViewXcds : id;
    row = q % b.nrow;
    chunk = q / b.nrow;
    if (b.wide()) chunk = chunk * kViewXcds + id % kViewXcds;
}

template <class S, int TPR, bool SCALAR, bool STREAM>
__global__ __launch_bounds__(kBcastBlock) void bcast_rows_mul_kernel(
    const typename S::T* __restrict__ full, const typename S::T* __restrict__ other,
    typename S::T* __restrict__ y, int64_t rows, int64_t cols, int64_t group, int accumulate,
    ViewBlocks blocks) {
    constexpr int W = S::kVec, NV = kViewSlots, RPB = kBcastBlock / TPR;
    const int t = threadIdx.x % TPR;
    const int64_t nslot = (cols + W - 1) / W;
    const uint32_t total = blocks.total();
    for (uint32_t id = blockIdx.x; id < total; id += gridDim.x) {
        uint32_t rb, chunk;
        view_block(blocks, id, rb, chunk);
        const int64_t row = static_cast<int64_t>(rb) * RPB + threadIdx.x / TPR;
        const int64_t s0 = static_cast<int64_t>(chunk) * (TPR * NV) + t;
        if (row < rows && s0 < nslot) {
            const typename S::T* fr = full + row * cols;
            typename S::T* yr = y + row * cols;
            const typename S::T* orow = SCALAR ? other + row : other + row / group * cols;
            const float os = SCALAR ? S::get(orow) : 0.0f;
            u32x4 fv[NV], ov[SCALAR ? 1 : NV];
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const int64_t s = s0 + k * TPR < nslot ? s0 + k * TPR : nslot - 1;
                fv[k] = view_load<S, STREAM>(fr + view_col<W>(s, cols));
                if constexpr (!SCALAR) ov[k] = load16_any<S>(orow + view_col<W>(s, cols));
            }
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                if (s0 + k * TPR >= nslot) break;
                const int64_t col = view_col<W>(s0 + k * TPR, cols);
                float f[W], o[W];
                S::unpack(fv[k], f);
                if constexpr (SCALAR) {
#pragma unroll
                    for (int e = 0; e < W; ++e) o[e] = os;
                } else {
                    S::unpack(ov[k], o);
                }
#pragma unroll
                for (int e = 0; e < W; ++e) f[e] = f[e] * o[e];
                view_store<S>(yr + col, f, static_cast<int>((s0 + k * TPR) * W - col), accumulate);
            }
        }
    }
}

// Both gradients of full * (a vector per group of rows) in one pass over gy and
// full: dfull (+)= gy * other (nullptr: not wanted), dother[group][col] (+)= the
// group's sum of gy * full, exact products in fp64.  A workgroup takes TW slots of
// columns of one group; its LANES / TW row lanes take the group's rows in turn,
// BATCH of them in flight (loads past the group's end repeat its last row), and
// their sums are added in lane order: an order fixed by the sizes.  HBM-bound at gy
// + full + dfull; narrow tiles of 1024 lanes where wide ones would leave CUs idle.
template <class S, int TW, int LANES, int BATCH, bool STREAM>
__global__ __launch_bounds__(LANES) void bcast_group_grad_kernel(
    const typename S::T* __restrict__ gy, const typename S::T* __restrict__ full,
    const typename S::T* __restrict__ other, typename S::T* __restrict__ dfull,
    float* __restrict__ dother, int64_t groups, int64_t group, int64_t cols, int acc_full,
    int acc_other) {
    constexpr int W = S::kVec, RG = LANES / TW;
    __shared__ double part[RG > 1 ? RG : 1][RG > 1 ? TW * W : 1];
    const int t = threadIdx.x % TW;
    const int g = threadIdx.x / TW;
    const int64_t nslot = (cols + W - 1) / W;
    const int64_t slot0 = static_cast<int64_t>(blockIdx.x) * TW;
    const bool active = slot0 + t < nslot;
    const int64_t slot = active ? slot0 + t : nslot - 1;
    const int64_t col = view_col<W>(slot, cols);
    const int dup = static_cast<int>(slot * W - col);
    for (int64_t o = blockIdx.y; o < groups; o += gridDim.y) {
        const int64_t base = o * group * cols + col;
        float ov[W];
#pragma unroll
        for (int e = 0; e < W; ++e) ov[e] = 0.0f;
        if (dfull) S::unpack(load16_any<S>(other + o * cols + col), ov);
        double acc[W];
#pragma unroll
        for (int e = 0; e < W; ++e) acc[e] = 0.0;
        u32x4 gv[BATCH], fv[BATCH];
        auto load = [&](int u, int64_t r) {
            gv[u] = view_load<S, STREAM>(gy + base + r * cols);
            fv[u] = view_load<S, STREAM>(full + base + r * cols);
        };
        auto use = [&](int u, int64_t r) {
            float a[W], b[W];
            S::unpack(gv[u], a);
            S::unpack(fv[u], b);
#pragma unroll
            for (int e = 0; e < W; ++e)
                acc[e] += static_cast<double>(a[e]) * static_cast<double>(b[e]);
            if (dfull && active) {
#pragma unroll
                for (int e = 0; e < W; ++e) a[e] = a[e] * ov[e];
                view_store<S>(dfull + base + r * cols, a, dup, acc_full);
            }
        };
        int64_t r = g;
        if constexpr (LANES <= 256) {  // whole batches (1024 lanes have no registers for both)
            for (; r + (BATCH - 1) * RG < group; r += BATCH * RG) {
#pragma unroll
                for (int u = 0; u < BATCH; ++u) load(u, r + u * RG);
#pragma unroll
                for (int u = 0; u < BATCH; ++u) use(u, r + u * RG);
            }
        }
        for (; r < group; r += BATCH * RG) {  // partial batches: loads stay in the group
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                load(u, r + u * RG < group ? r + u * RG : group - 1);
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                if (r + u * RG < group) use(u, r + u * RG);
        }
        auto put = [&](int64_t at, double sum) {  // column `at` of this group
            float* d = dother + o * cols + at;
            *d = static_cast<float>((acc_other ? static_cast<double>(*d) : 0.0) + sum);
        };
        if constexpr (RG == 1) {
#pragma unroll
            for (int e = 0; e < W; ++e)
                if (active && e >= dup) put(col + e, acc[e]);
        } else {
#pragma unroll
            for (int e = 0; e < W; ++e) part[g][t * W + e] = acc[e];
            __syncthreads();
            for (int c = threadIdx.x; c < TW * W; c += LANES) {
                const int64_t sl = slot0 + c / W;
                if (sl >= nslot) break;
                const int64_t c0 = view_col<W>(sl, cols);
                double sum = part[0][c];
#pragma unroll 8
                for (int q = 1; q < RG; ++q) sum += part[q][c];
                if (c % W >= sl * W - c0) put(c0 + c % W, sum);
            }
            __syncthreads();
        }
    }
}

// Both gradients of full * (a scalar per row): dfull (+)= gy * other[row]
// (nullptr: not wanted), dother[row] (+)= the row's sum of gy * full, exact products
// in fp64.  TPR lanes (one wave at most) per row; lane sums meet in a fixed
// butterfly.  HBM-bound at gy + full + dfull.
template <class S, int TPR>
__global__ __launch_bounds__(kBcastBlock) void bcast_row_grad_kernel(
    const typename S::T* __restrict__ gy, const typename S::T* __restrict__ full,
    const typename S::T* __restrict__ other, typename S::T* __restrict__ dfull,
    float* __restrict__ dother, int64_t rows, int64_t cols, int acc_full, int acc_other) {
    constexpr int W = S::kVec, NV = kViewSlots, RPB = kBcastBlock / TPR;
    const int t = threadIdx.x % TPR;
    const int64_t nslot = (cols + W - 1) / W;
    for (int64_t r0 = static_cast<int64_t>(blockIdx.x) * RPB; r0 < rows;
         r0 += static_cast<int64_t>(gridDim.x) * RPB) {
        const bool active = r0 + threadIdx.x / TPR < rows;
        const int64_t row = active ? r0 + threadIdx.x / TPR : rows - 1;
        const float ov = dfull ? S::get(other + row) : 0.0f;
        double acc[W];
#pragma unroll
        for (int e = 0; e < W; ++e) acc[e] = 0.0;
        for (int64_t s0 = t; s0 < nslot; s0 += TPR * NV) {
            u32x4 gv[NV], fv[NV];
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const int64_t s = s0 + k * TPR < nslot ? s0 + k * TPR : nslot - 1;
                gv[k] = load16_any_stream<S>(gy + row * cols + view_col<W>(s, cols));
                fv[k] = load16_any_stream<S>(full + row * cols + view_col<W>(s, cols));
            }
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                if (s0 + k * TPR >= nslot) break;
                const int64_t col = view_col<W>(s0 + k * TPR, cols);
                const int dup = static_cast<int>((s0 + k * TPR) * W - col);
                float a[W], b[W];
                S::unpack(gv[k], a);
                S::unpack(fv[k], b);
#pragma unroll
                for (int e = 0; e < W; ++e) {
                    const double p = static_cast<double>(a[e]) * static_cast<double>(b[e]);
                    acc[e] = e < dup ? acc[e] : acc[e] + p;
                }
                if (dfull && active) {
#pragma unroll
                    for (int e = 0; e < W; ++e) a[e] = a[e] * ov;
                    view_store<S>(dfull + row * cols + col, a, dup, acc_full);
                }
            }
        }
        double s = acc[0];
#pragma unroll
        for (int e = 1; e < W; ++e) s += acc[e];
#pragma unroll
        for (int m = TPR / 2; m > 0; m /= 2) s += __shfl_xor(s, m, 64);
        if (active && t == 0)
            dother[row] =
                static_cast<float>((acc_other ? static_cast<double>(dother[row]) : 0.0) + s);
    }
}

// Zeros n 16-bit words (a kernel rather than a memset node, so that the call
// can be captured into a graph).
__global__ __launch_bounds__(kBcastBlock) void bcast_zero_kernel(uint16_t* __restrict__ p,
                                                                int64_t n) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBcastBlock + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kBcastBlock)
        p[i] = 0;
}

// ---- host side -------------------------------------------------------------------

// Row-major contiguous strides of an operand aligned to nd output axes (its
// missing leading axes and its extent-1 axes get stride 0).
struct Aligned {
    int64_t size[kBcastMaxDims];
    int64_t stride[kBcastMaxDims];
};

inline bool align_operand(const int64_t* shape, int ndim, int nd, Aligned& out) {
    int64_t s = 1;
    for (int i = nd - 1; i >= 0; --i) {
        const int src = i - (nd - ndim);
        const int64_t e = src >= 0 ? shape[src] : 1;
        if (e < 0) return false;
        out.size[i] = e;
        out.stride[i] = e == 1 ? 0 : s;
        if (e > 0 && s > INT64_MAX / e) return false;
        s *= e;
    }
    return true;
}

// The broadcast output shape of a and b; false when incompatible or too many axes.
inline bool broadcast_shape(const int64_t* as, int an, const int64_t* bs, int bn, int& nd,
                            Aligned& a, Aligned& b, int64_t (&osize)[kBcastMaxDims],
                            int64_t& numel) {
    if (an < 0 || bn < 0 || an > kBcastMaxDims || bn > kBcastMaxDims) return false;
    if ((an && !as) || (bn && !bs)) return false;
    nd = an > bn ? an : bn;
    if (!align_operand(as, an, nd, a) || !align_operand(bs, bn, nd, b)) return false;
    numel = 1;
    for (int i = 0; i < nd; ++i) {
        const int64_t x = a.size[i], y = b.size[i];
        if (x != y && x != 1 && y != 1) return false;
        osize[i] = x == 1 ? y : x;
        if (osize[i] > 0 && numel > INT64_MAX / osize[i]) return false;
        numel *= osize[i];
    }
    return true;
}

// Merges adjacent output axes that both operands walk contiguously and drops
// extent-1 axes; at least one axis remains.
inline BcastGeom make_geom(int nd, const int64_t* osize, const Aligned& a, const Aligned& b) {
    BcastGeom g{};
    g.nd = 0;
    for (int i = 0; i < nd; ++i) {
        if (osize[i] == 1) continue;
        const int64_t sa = a.size[i] == 1 ? 0 : a.stride[i];
        const int64_t sb = b.size[i] == 1 ? 0 : b.stride[i];
        if (g.nd > 0) {
            const int p = g.nd - 1;
            if (g.sa[p] == sa * osize[i] && g.sb[p] == sb * osize[i]) {
                g.size[p] *= osize[i];
                g.sa[p] = sa;
                g.sb[p] = sb;
                continue;
            }
        }
        g.size[g.nd] = osize[i];
        g.sa[g.nd] = sa;
        g.sb[g.nd] = sb;
        ++g.nd;
    }
    if (g.nd == 0) {
        g.nd = 1;
        g.size[0] = 1;
        g.sa[0] = g.sb[0] = 0;
    }
    return g;
}

// The rows x cols view of a product of a full operand and a broadcast one; kind
// 0: none applies.
struct RowsView {
    enum Kind { kNone = 0, kGroup = 1, kScalar = 2 };
    int kind = kNone;
    int64_t rows = 0, cols = 0, group = 1;
};

// g: make_geom's axes with the full operand first (its strides are the output's).
inline RowsView rows_view(const BcastGeom& g, int w) {
    RowsView v;
    const int last = g.nd - 1;
    if (g.nd == 2 && g.sb[0] == 0 && g.sb[1] == 1)
        v = {RowsView::kGroup, g.size[0], g.size[1], g.size[0]};
    else if (g.nd == 3 && g.sb[0] == g.size[2] && g.sb[1] == 0 && g.sb[2] == 1)
        v = {RowsView::kGroup, g.size[0] * g.size[1], g.size[2], g.size[1]};
    else if (g.nd == 2 && g.sb[0] == 1 && g.sb[1] == 0)
        v = {RowsView::kScalar, g.size[0], g.size[1], 1};
    else if (g.nd == 1 && g.sb[0] == 0)
        v = {RowsView::kScalar, 1, g.size[0], 1};
    if (v.cols < w || g.sa[last] != 1) v.kind = RowsView::kNone;
    return v;
}

inline int64_t view_elems(const RowsView& v) { return v.rows * v.cols; }
inline int64_t view_other_elems(const RowsView& v) {
    return v.kind == RowsView::kScalar ? v.rows : v.rows / v.group * v.cols;
}

// Whether the one-pass gradient kernels take the view: long single rows spread
// better over bcast_reduce_kernel's workgroups.
inline bool grad_view_fits(const RowsView& v) {
    if (v.kind == RowsView::kScalar) return v.cols <= 16384 || v.rows >= 1024;
    return v.kind == RowsView::kGroup;
}

// Full operands of this many bytes and more are loaded past the caches: with y they
// exceed the 256 MiB Infinity Cache, where smaller ones may still lie from the
// kernel that wrote them, and stay for the one that reads them next.  Measured on
// MI355X by a scalar per row, ordinary / streaming loads (us, operands in the cache
// where they fit; from HBM): 20 MB 5.7 / 8.8; 8.3 / 10.2, 100 MB 33 / 39; 32 / 40,
// 200 MB 64 / 76; 64 / 77, 400 MB 134 / 126; 135 / 126.
constexpr int64_t kStreamBytes = 256LL << 20;

template <class S>
int launch_rows_mul(const void* full, const void* other, void* y, const RowsView& v,
                    int accumulate, hipStream_t st) {
    using T = typename S::T;
    const int64_t nslot = row_slots(v.cols, S::kVec);
    const int64_t need = (nslot + kViewSlots - 1) / kViewSlots;
    const int tpr = need <= 16 ? 16 : need <= 64 ? 64 : need <= 128 ? 128 : 256;
    // (a workgroup moves at least 256 bytes: the counts fit 32 bits)
    ViewBlocks blocks;
    blocks.nrow = static_cast<uint32_t>((v.rows + kBcastBlock / tpr - 1) / (kBcastBlock / tpr));
    blocks.nchunk = static_cast<uint32_t>((nslot + tpr * kViewSlots - 1) / (tpr * kViewSlots));
    const dim3 grid(capped_blocks(blocks.total(), kBcastBlock));
    const bool stream = view_elems(v) * static_cast<int64_t>(sizeof(T)) >= kStreamBytes;
#define AGK_ROWS_MUL(TPR, SCALAR, STREAM)                                                         \
    hipLaunchKernelGGL((bcast_rows_mul_kernel<S, TPR, SCALAR, STREAM>), grid, dim3(kBcastBlock),  \
                       0, st, static_cast<const T*>(full), static_cast<const T*>(other),          \
                       static_cast<T*>(y), v.rows, v.cols, v.group, accumulate, blocks)
#define AGK_ROWS_MUL_TPR(TPR)                                                                     \
    do {                                                                                          \
        if (v.kind == RowsView::kScalar) {                                                        \
            if (stream) AGK_ROWS_MUL(TPR, true, true);                                            \
            else AGK_ROWS_MUL(TPR, true, false);                                                  \
        } else {                                                                                  \
            if (stream) AGK_ROWS_MUL(TPR, false, true);                                           \
            else AGK_ROWS_MUL(TPR, false, false);                                                 \
        }                                                                                         \
    } while (0)
    if (tpr == 16) AGK_ROWS_MUL_TPR(16);
    else if (tpr == 64) AGK_ROWS_MUL_TPR(64);
    else if (tpr == 128) AGK_ROWS_MUL_TPR(128);
    else AGK_ROWS_MUL_TPR(256);
#undef AGK_ROWS_MUL_TPR
#undef AGK_ROWS_MUL
    return check_launch();
}

// The gradient of the broadcast operand, with dfull (nullptr: not wanted) in the
// same pass.
template <class S>
int launch_rows_grad(const void* gy, const void* full, const void* other, void* dfull,
                     float* dother, const RowsView& v, int acc_full, int acc_other,
                     hipStream_t st) {
    using T = typename S::T;
    const T *g = static_cast<const T*>(gy), *f = static_cast<const T*>(full),
            *o = static_cast<const T*>(other);
    T* df = static_cast<T*>(dfull);
    const int64_t nslot = row_slots(v.cols, S::kVec);
    if (v.kind == RowsView::kScalar) {
        const int tpr = nslot <= 32 ? 16 : 64;
        const int64_t bx = (v.rows + kBcastBlock / tpr - 1) / (kBcastBlock / tpr);
        const dim3 grid(capped_blocks(bx, kBcastBlock));
#define AGK_ROW_GRAD(TPR)                                                                       \
    hipLaunchKernelGGL((bcast_row_grad_kernel<S, TPR>), grid, dim3(kBcastBlock), 0, st, \
                       g, f, o, df, dother, v.rows, v.cols, acc_full, acc_other)
        if (tpr == 16) AGK_ROW_GRAD(16);
        else AGK_ROW_GRAD(64);
#undef AGK_ROW_GRAD
        return check_launch();
    }
    const int64_t groups = v.rows / v.group;
    // One row lane for short groups; else whole kilobytes per row (four row
    // lanes), or narrower tiles of 16 to 256 row lanes where those would leave CUs
    // without a workgroup.  Measured on MI355X, both gradients (us, 4- / 16- / 64-slot
    // tiles): f32 8 x 2048 x 1024 86 / 50 / -, bf16 42 / 51 / -; f32 2 x 2048 x 4001 126 /
    // 71 / -; bf16 20 groups' rows of 117520 - / 32 / 16; f32 2 x 2048 x 64 15 / 28 / -
    // (the two passes this replaces: 76, 73, 130, 15, 32); bf16 sums alone 40 x 73 x 513
    // to 40 x 513 - / 4.7 (256 lanes) / 7.7.
    auto tiles = [&](int64_t tw) { return (nslot + tw - 1) / tw; };
    int tw = v.group <= 8 ? 256 : 64;
    if (v.group > 8 && tiles(64) * groups < 256)
        tw = v.group >= 512 && tiles(16) * groups < 100 ? 4 : 16;
    if (tiles(tw) > 0x7fffffffLL) return AGK_EINVAL;
    const dim3 grid(static_cast<unsigned>(tiles(tw)),
                    static_cast<unsigned>(groups < 65535 ? groups : 65535));
    // Loads stream past the caches unless tiles share 128-byte lines, which then stay
    // for the neighbour.  Measured on MI355X, both gradients, ordinary / streaming loads
    // (us, operands from HBM): f32 2 x 97465 x 513 by 2 x 513 (odd widths, all sizes of 400
    // MB) 724 / 906, 2 x 64-column rows of 200 MB 339 / 370, but 8 x 24366 x 513 by 24366 x
    // 513 241 / 221.
    const uintptr_t at = reinterpret_cast<uintptr_t>(gy) | reinterpret_cast<uintptr_t>(full) |
                         static_cast<uintptr_t>(v.cols * static_cast<int64_t>(sizeof(T)));
    const bool stream = tw == 256 || (tw >= 16 && at % 128 == 0);
#define AGK_GROUP_GRAD(TW, LANES, BATCH, STREAM)                                              \
    hipLaunchKernelGGL((bcast_group_grad_kernel<S, TW, LANES, BATCH, STREAM>), grid,          \
                       dim3(LANES), 0, st, g, f, o, df, dother, groups, v.group, v.cols,      \
                       acc_full, acc_other)
#define AGK_GROUP_GRAD_TW(TW, LANES, BATCH)                                                   \
    do {                                                                                      \
        if (stream) AGK_GROUP_GRAD(TW, LANES, BATCH, true);                                   \
        else AGK_GROUP_GRAD(TW, LANES, BATCH, false);                                         \
    } while (0)
    if (tw == 256) AGK_GROUP_GRAD_TW(256, 256, 8);
    else if (tw == 64) AGK_GROUP_GRAD_TW(64, 256, 8);
    else if (tw == 16 && v.group < 128) AGK_GROUP_GRAD_TW(16, 256, 8);
    else if (tw == 16) AGK_GROUP_GRAD_TW(16, 1024, 4);
    else AGK_GROUP_GRAD_TW(4, 1024, 4);
#undef AGK_GROUP_GRAD_TW
#undef AGK_GROUP_GRAD
    return check_launch();
}

template <class S>
int launch_bcast_mul(const void* a, const void* b, void* y, const BcastGeom& g, int accumulate,
                     hipStream_t st) {
    const int64_t inner = g.size[g.nd - 1];
    int64_t runs = 1;
    for (int d = 0; d + 1 < g.nd; ++d) runs *= g.size[d];
    const int last = g.nd - 1;
    const bool vec = inner % S::kVec == 0 && (g.sa[last] == 0 || g.sa[last] == 1) &&
                     (g.sb[last] == 0 || g.sb[last] == 1) && aligned16(a) && aligned16(b) &&
                     aligned16(y);
    const int64_t per_run = vec ? inner / S::kVec : inner;
    const int64_t bx = (per_run + kBcastBlock - 1) / kBcastBlock;
    const dim3 grid(static_cast<unsigned>(bx < 1024 ? bx : 1024),
                    static_cast<unsigned>(runs < 65535 ? runs : 65535));
    const auto* ap = static_cast<const typename S::T*>(a);
    const auto* bp = static_cast<const typename S::T*>(b);
    auto* yp = static_cast<typename S::T*>(y);
    if (vec)
        hipLaunchKernelGGL(bcast_mul_vec_kernel<S>, grid, dim3(kBcastBlock), 0, st, ap, bp, yp, g,
                           runs, accumulate);
    else
        hipLaunchKernelGGL(bcast_mul_kernel<S>, grid, dim3(kBcastBlock), 0, st, ap, bp, yp, g, runs,
                           accumulate);
    return check_launch();
}

// The reduction that produces the gradient of operand `t` (aligned to the
// output) from gy and the other operand `o`.
inline BcastRed make_red(int nd, const int64_t* osize, const Aligned& t, const Aligned& o,
                         int64_t& n_out) {
    BcastRed r{};
    int64_t sgy[kBcastMaxDims];
    int64_t s = 1;
    for (int i = nd - 1; i >= 0; --i) {
        sgy[i] = s;
        s *= osize[i];
    }
    n_out = 1;
    r.rtotal = 1;
    for (int i = 0; i < nd; ++i) {
        if (osize[i] == 1) continue;
        const int64_t so = o.size[i] == 1 ? 0 : o.stride[i];
        if (t.size[i] == osize[i]) {
            r.ksize[r.nk] = osize[i];
            r.kgy[r.nk] = sgy[i];
            r.ko[r.nk] = so;
            ++r.nk;
            n_out *= osize[i];
        } else {
            r.rsize[r.nr] = osize[i];
            r.rgy[r.nr] = sgy[i];
            r.ro[r.nr] = so;
            ++r.nr;
            r.rtotal *= osize[i];
        }
    }
    return r;
}

template <class S>
int launch_bcast_reduce(const void* gy, const void* other, float* d, const BcastRed& r,
                        int64_t n_out, int accumulate, hipStream_t st) {
    const auto* g = static_cast<const typename S::T*>(gy);
    const auto* o = static_cast<const typename S::T*>(other);
    if (r.nk >= 1 && r.kgy[r.nk - 1] == 1) {  // the output keeps the innermost axis
        const int64_t blocks = (n_out + 63) / 64;
        hipLaunchKernelGGL(bcast_reduce_cols_kernel<S>,
                           dim3(static_cast<unsigned>(blocks < 65536 ? blocks : 65536)),
                           dim3(kBcastBlock), 0, st, g, o, d, r, n_out, accumulate);
        return check_launch();
    }
    const bool wide = r.rtotal >= 4096;
    const int per = wide ? 1 : kBcastBlock / 64;
    const int64_t blocks = (n_out + per - 1) / per;
    const dim3 grid(static_cast<unsigned>(blocks < 65536 ? blocks : 65536));
    if (wide)
        hipLaunchKernelGGL((bcast_reduce_kernel<S, kBcastBlock>), grid, dim3(kBcastBlock), 0, st,
                           g, o, d, r, n_out, accumulate);
    else
        hipLaunchKernelGGL((bcast_reduce_kernel<S, 64>), grid, dim3(kBcastBlock), 0, st, g, o,
                           d, r, n_out, accumulate);
    return check_launch();
}

// Whether an aligned operand covers the whole output (its gradient is then
// the element-wise product, in the storage dtype).
inline bool is_full(int nd, const int64_t* osize, const Aligned& t) {
    for (int i = 0; i < nd; ++i)
        if (t.size[i] != osize[i]) return false;
    return true;
}

// The rows x cols view of a * b written to y (or of a gradient gy * other): which
// operand is full and which broadcast; none when y overlaps one of them (a slot
// moved back to the row's end may be stored before its neighbour is loaded).
inline RowsView product_view(int nd, const int64_t* osize, const Aligned& al, const Aligned& bl,
                             const void* a, const void* b, const void* y, int dtype,
                             const void** full, const void** other) {
    const bool af = is_full(nd, osize, al), bf = is_full(nd, osize, bl);
    if (af == bf) return RowsView{};
    const int w = dtype == AGK_F32 ? F32::kVec : BF16::kVec;
    const RowsView v = rows_view(af ? make_geom(nd, osize, al, bl) : make_geom(nd, osize, bl, al), w);
    *full = af ? a : b;
    *other = af ? b : a;
    const int64_t es = 16 / w, bytes = view_elems(v) * es;
    if (v.kind != RowsView::kNone && (!disjoint(y, *full, bytes) ||
                                      !disjoint(y, bytes, *other, view_other_elems(v) * es)))
        return RowsView{};
    return v;
}

// Whether the rows x cols kernel takes a product: not tiny ones off the 16-byte grid,
// where the element-wise kernel's shorter start counts, nor, on it, rows of many chunks
// in tiny tensors, or by one vector in many rows of large ones.  Measured on MI355X
// (us, general / rows x cols): bf16 8 x 6 x 513 by 6 x 513 2.4 / 2.9, f32 8 x 3 x 4096 by
// 3 x 4096 2.2 / 2.7 (2 x 610 x 4096 by 610 x 4096 6.7 / 4.7), f32 40 x 305 x 4096 by 305 x
// 4096 55 / 59, bf16 40 x 1220 x 4096 by 1220 x 4096 135 / 149 (8 rows: 167 / 164).
template <class S>
inline bool rows_mul_fits(const RowsView& v, const void* full, const void* other, const void* y) {
    constexpr int64_t kTiny = 1 << 16, kTinyWide = 1 << 18, kLarge = 128LL << 20;
    const int64_t n = view_elems(v);
    if (v.cols % S::kVec != 0 || !aligned16(full) || !aligned16(other) || !aligned16(y))
        return n >= kTiny;
    if (v.kind != RowsView::kGroup || v.cols < kViewXcds * kBcastBlock * kViewSlots * S::kVec)
        return true;
    return n >= kTinyWide && (v.group != v.rows || v.rows < 16 ||
                              n * static_cast<int64_t>(sizeof(typename S::T)) < kLarge);
}

template <class S>
int bcast_bwd_one(const void* gy, const void* other, const Aligned& t, const Aligned& o,
                  const Aligned& gyal, int nd, const int64_t* osize, void* d, int accumulate,
                  hipStream_t st) {
    if (is_full(nd, osize, t)) {
        // d (+)= gy * other: the forward kernels with gy as the full operand
        const void *full = nullptr, *bc = nullptr;
        const int dtype = S::kVec == 4 ? AGK_F32 : AGK_BF16;
        const RowsView v = product_view(nd, osize, gyal, o, gy, other, d, dtype, &full, &bc);
        if (v.kind != RowsView::kNone && rows_mul_fits<S>(v, full, bc, d))
            return launch_rows_mul<S>(full, bc, d, v, accumulate, st);
        const BcastGeom g = make_geom(nd, osize, gyal, o);
        return launch_bcast_mul<S>(gy, other, d, g, accumulate, st);
    }
    int64_t n_out = 0;
    const BcastRed r = make_red(nd, osize, t, o, n_out);
    return launch_bcast_reduce<S>(gy, other, static_cast<float*>(d), r, n_out, accumulate, st);
}

}  // namespace agk

namespace agk {

// dst[i] = value for i < n (a grid-stride loop of 256-lane workgroups).
template <class S>
__global__ __launch_bounds__(256) void fill_kernel(typename S::T* __restrict__ dst, int64_t n,
                                                   float value) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride)
        S::put(dst + i, value);
}

}  // namespace agk

extern "C" int agk_fill(void* dst, int64_t n, float value, int dtype, agk_stream_t stream) {
    using namespace agk;
    if (n < 0) return AGK_EINVAL;
    if (dtype != AGK_F32 && dtype != AGK_BF16) return AGK_EDTYPE;
    if (n == 0) return AGK_OK;
    if (!dst) return AGK_EINVAL;
    clear_pending_error();
    const int64_t blocks64 = (n + 255) / 256;
    const unsigned blocks = static_cast<unsigned>(blocks64 < 4096 ? blocks64 : 4096);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (dtype == AGK_F32)
        hipLaunchKernelGGL(fill_kernel<F32>, dim3(blocks), dim3(256), 0, st,
                           static_cast<float*>(dst), n, value);
    else
        hipLaunchKernelGGL(fill_kernel<BF16>, dim3(blocks), dim3(256), 0, st,
                           static_cast<uint16_t*>(dst), n, value);
    return check_launch();
}

extern "C" int agk_mul_bcast_shape(const int64_t* a_shape, int a_ndim, const int64_t* b_shape,
                                   int b_ndim, int64_t* out_shape, int* out_ndim) {
    using namespace agk;
    int nd = 0;
    Aligned a, b;
    int64_t osize[kBcastMaxDims];
    int64_t numel = 0;
    if (!out_ndim) return AGK_EINVAL;
    if (!broadcast_shape(a_shape, a_ndim, b_shape, b_ndim, nd, a, b, osize, numel))
        return AGK_EINVAL;
    *out_ndim = nd;
    if (out_shape)
        for (int i = 0; i < nd; ++i) out_shape[i] = osize[i];
    return AGK_OK;
}

extern "C" int agk_mul_bcast_fwd(const void* a, const int64_t* a_shape, int a_ndim,
                                 const void* b, const int64_t* b_shape, int b_ndim, void* y,
                                 int dtype, int accumulate, agk_stream_t stream) {
    using namespace agk;
    if (!valid_dtype(dtype)) return AGK_EDTYPE;
    int nd = 0;
    Aligned al, bl;
    int64_t osize[kBcastMaxDims];
    int64_t numel = 0;
    if (!broadcast_shape(a_shape, a_ndim, b_shape, b_ndim, nd, al, bl, osize, numel))
        return AGK_EINVAL;
    if (numel == 0) return AGK_OK;
    if (!a || !b || !y) return AGK_EINVAL;
    clear_pending_error();
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int acc = accumulate != 0;
    const void *full = nullptr, *other = nullptr;
    const RowsView v = product_view(nd, osize, al, bl, a, b, y, dtype, &full, &other);
    if (v.kind != RowsView::kNone &&
        (dtype == AGK_F32 ? rows_mul_fits<F32>(v, full, other, y)
                          : rows_mul_fits<BF16>(v, full, other, y)))
        return dtype == AGK_F32 ? launch_rows_mul<F32>(full, other, y, v, acc, st)
                                : launch_rows_mul<BF16>(full, other, y, v, acc, st);
    const BcastGeom g = make_geom(nd, osize, al, bl);
    return dtype == AGK_F32 ? launch_bcast_mul<F32>(a, b, y, g, acc, st)
                            : launch_bcast_mul<BF16>(a, b, y, g, acc, st);
}

extern "C" int agk_mul_bcast_bwd(const void* gy, const void* a, const int64_t* a_shape,
                                 int a_ndim, const void* b, const int64_t* b_shape, int b_ndim,
                                 void* da, void* db, int dtype, int accumulate,
                                 agk_stream_t stream) {
    using namespace agk;
    if (!valid_dtype(dtype)) return AGK_EDTYPE;
    if (accumulate & ~AGK_ACCUM_ALL) return AGK_EINVAL;
    int nd = 0;
    Aligned al, bl;
    int64_t osize[kBcastMaxDims];
    int64_t numel = 0;
    if (!broadcast_shape(a_shape, a_ndim, b_shape, b_ndim, nd, al, bl, osize, numel))
        return AGK_EINVAL;
    if (!da && !db) return AGK_OK;
    // an empty output: the gradients are empty sums (zeros), or unchanged
    // when accumulating; an empty operand has an empty gradient
    if (numel == 0) {
        if (accumulate == AGK_ACCUM_ALL) return AGK_OK;
        clear_pending_error();
        hipStream_t st = reinterpret_cast<hipStream_t>(stream);
        for (int w = 0; w < 2; ++w) {
            void* d = w ? db : da;
            const Aligned& t = w ? bl : al;
            if (!d || (accumulate & (w ? AGK_ACCUM_DGAMMA : AGK_ACCUM_DX))) continue;
            int64_t n = 1;
            for (int i = 0; i < nd; ++i) n *= t.size[i];
            if (n == 0) continue;
            const int64_t words = n * (is_full(nd, osize, t) && dtype == AGK_BF16 ? 1 : 2);
            const int64_t blocks = (words + kBcastBlock - 1) / kBcastBlock;
            hipLaunchKernelGGL(bcast_zero_kernel, dim3(static_cast<unsigned>(blocks < 4096 ? blocks : 4096)),
                               dim3(kBcastBlock), 0, st, static_cast<uint16_t*>(d), words);
            const int rc = check_launch();
            if (rc != AGK_OK) return rc;
        }
        return AGK_OK;
    }
    if (!gy || (da && !b) || (db && !a)) return AGK_EINVAL;
    clear_pending_error();
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    Aligned gyal;  // gy in the output layout
    if (!align_operand(osize, nd, nd, gyal)) return AGK_EINVAL;
    int rc = AGK_OK;
    // One operand full and the other a vector per group of rows or a scalar per
    // row: the broadcast operand's gradient and the full one's in one pass.  Not
    // where either gradient overlaps what the pass reads (or the other gradient): a
    // workgroup may read an element that its neighbour has already overwritten.
    // In two passes the first one has read everything before the second writes.
    {
        const bool a_full = is_full(nd, osize, al);
        void* dfull = a_full ? da : db;
        void* dother = a_full ? db : da;
        const int acc_full = (accumulate & (a_full ? AGK_ACCUM_DX : AGK_ACCUM_DGAMMA)) != 0;
        const int acc_other = (accumulate & (a_full ? AGK_ACCUM_DGAMMA : AGK_ACCUM_DX)) != 0;
        const void *full = nullptr, *other = nullptr;
        const RowsView v = product_view(nd, osize, al, bl, a, b, dfull, dtype, &full, &other);
        const int64_t bytes = view_elems(v) * (dtype == AGK_F32 ? 4 : 2);
        const int64_t obytes = view_other_elems(v) * (dtype == AGK_F32 ? 4 : 2);
        const int64_t dbytes = view_other_elems(v) * 4;  // a sum: fp32
        if (dother && grad_view_fits(v) && disjoint(dfull, gy, bytes) &&
            disjoint(dother, dbytes, gy, bytes) && disjoint(dother, dbytes, full, bytes) &&
            disjoint(dother, dbytes, other, obytes) && disjoint(dother, dbytes, dfull, bytes))
            return dtype == AGK_F32
                       ? launch_rows_grad<F32>(gy, full, other, dfull, static_cast<float*>(dother),
                                               v, acc_full, acc_other, st)
                       : launch_rows_grad<BF16>(gy, full, other, dfull,
                                                static_cast<float*>(dother), v, acc_full,
                                                acc_other, st);
    }
    if (da) {
        const int acc = (accumulate & AGK_ACCUM_DX) != 0;
        rc = dtype == AGK_F32 ? bcast_bwd_one<F32>(gy, b, al, bl, gyal, nd, osize, da, acc, st)
                              : bcast_bwd_one<BF16>(gy, b, al, bl, gyal, nd, osize, da, acc, st);
        if (rc != AGK_OK) return rc;
    }
    if (db) {
        const int acc = (accumulate & AGK_ACCUM_DGAMMA) != 0;
        rc = dtype == AGK_F32 ? bcast_bwd_one<F32>(gy, a, bl, al, gyal, nd, osize, db, acc, st)
                              : bcast_bwd_one<BF16>(gy, a, bl, al, gyal, nd, osize, db, acc, st);
    }
    return rc;
}
