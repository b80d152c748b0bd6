// The block kernel on BF16 weights.
#include "gemm_block.h"

namespace dro {
int launch_block_bf16(const GemmArgs& a, const block::Plan& p, hipStream_t stream) { return block::launch_format<LX_W_BF16, LX_MATH_BF16>(a, p, stream); }
}  // namespace dro
