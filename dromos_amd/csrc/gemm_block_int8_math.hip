// The block kernel under the INT8 math.
#include "gemm_block.h"

namespace dro {
int launch_block_int8_math(const GemmArgs& a, const block::Plan& p, hipStream_t stream) { return block::launch_format<LX_W_INT8, LX_MATH_INT8>(a, p, stream); }
}  // namespace dro
