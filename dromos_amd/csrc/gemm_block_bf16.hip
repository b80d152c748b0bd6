// The block kernel on BF16 weights.
#include "gemm_block.h"

namespace dro {
bool launch_block_bf16(const GemmArgs& a, int* status, hipStream_t stream) { return block::launch_format<LX_W_BF16, LX_MATH_BF16>(a, status, stream); }
}  // namespace dro
