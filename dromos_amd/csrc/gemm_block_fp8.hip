// The block kernel on FP8 weights.
#include "gemm_block.h"

namespace dro {
int launch_block_fp8(const GemmArgs& a, const block::Plan& p, hipStream_t stream) { return block::launch_format<LX_W_FP8, LX_MATH_BF16>(a, p, stream); }
}  // namespace dro
