// The block kernel under the FP8 math.
#include "gemm_block.h"

namespace dro {
int launch_block_fp8_math(const GemmArgs& a, const block::Plan& p, hipStream_t stream) { return block::launch_format<LX_W_FP8, LX_MATH_FP8>(a, p, stream); }
}  // namespace dro
