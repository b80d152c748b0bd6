// The block kernel on NVFP4 weights.
#include "gemm_block.h"

namespace dro {
int launch_block_nvfp4(const GemmArgs& a, const block::Plan& p, hipStream_t stream) { return block::launch_format<LX_W_NVFP4, LX_MATH_BF16>(a, p, stream); }
}  // namespace dro
