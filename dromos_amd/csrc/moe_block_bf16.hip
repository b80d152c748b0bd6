// The experts' block kernels on BF16 weights.
#include "moe_block_kernels.h"

namespace dro {
int launch_expert_block_bf16(const ExpertBlock& a, int max_tiles, hipStream_t stream) { return block::launch_experts<LX_W_BF16>(a, max_tiles, stream); }
}  // namespace dro
