// The experts' block kernels on FP8 weights.
#include "moe_block_kernels.h"

namespace dro {
int launch_expert_block_fp8(const ExpertBlock& a, int max_tiles, hipStream_t stream) { return block::launch_experts<LX_W_FP8>(a, max_tiles, stream); }
}  // namespace dro
