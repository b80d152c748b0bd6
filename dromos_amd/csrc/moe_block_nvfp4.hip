// The experts' block kernels on NVFP4 weights.
#include "moe_block_kernels.h"

namespace dro {
int launch_expert_block_nvfp4(const ExpertBlock& a, int max_tiles, hipStream_t stream) { return block::launch_experts<LX_W_NVFP4>(a, max_tiles, stream); }
}  // namespace dro
