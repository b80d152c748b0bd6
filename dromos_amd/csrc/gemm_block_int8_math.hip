// The block kernel under the INT8 math.
#include "gemm_block.h"

namespace dro {
bool launch_block_int8_math(const GemmArgs& a, int* status, hipStream_t stream) { return block::launch_format<LX_W_INT8, LX_MATH_INT8>(a, status, stream); }
}  // namespace dro
