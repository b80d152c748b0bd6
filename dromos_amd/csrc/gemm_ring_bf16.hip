// The ring kernel on BF16 weights.
#include "gemm_ring.h"

namespace dro {
bool launch_ring_bf16(const GemmArgs& a, int cols, int* status, hipStream_t stream) { return ring::launch_ring<LX_W_BF16>(a, cols, status, stream); }
}  // namespace dro
