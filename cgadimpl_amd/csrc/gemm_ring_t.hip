// gemm_ring_t.hip -- the ring kernels of gemm_ring.hpp for A k-strided ([K][M])
// (one translation unit per layout of A, to compile side by side).
#define AGK_RING_KERNELS
#include "gemm_ring.hpp"

namespace agk_gemm {

template int launch_ring<true, false>(int shape, bool f32, const GemmCall& c);
template int launch_ring<true, true>(int shape, bool f32, const GemmCall& c);

}  // namespace agk_gemm
