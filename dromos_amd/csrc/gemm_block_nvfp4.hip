// The block kernel on NVFP4 weights.
#include "gemm_block.h"

namespace dro {
bool launch_block_nvfp4(const GemmArgs& a, int* status, hipStream_t stream) { return block::launch_format<LX_W_NVFP4, LX_MATH_BF16>(a, status, stream); }
}  // namespace dro
