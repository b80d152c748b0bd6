// The block kernel on INT8 weights.
#include "gemm_block.h"

namespace dro {
bool launch_block_int8(const GemmArgs& a, int* status, hipStream_t stream) { return block::launch_format<LX_W_INT8, LX_MATH_BF16>(a, status, stream); }
}  // namespace dro
