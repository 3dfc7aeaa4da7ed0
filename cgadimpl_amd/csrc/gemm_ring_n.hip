// gemm_ring_n.hip -- the ring kernels of gemm_ring.hpp for A k-contiguous ([M][K])
// (one translation unit per layout of A, to compile side by side).
#define AGK_RING_KERNELS
#include "gemm_ring.hpp"

namespace agk_gemm {

template int launch_ring<false, false>(int shape, bool f32, const GemmCall& c);
template int launch_ring<false, true>(int shape, bool f32, const GemmCall& c);

}  // namespace agk_gemm
