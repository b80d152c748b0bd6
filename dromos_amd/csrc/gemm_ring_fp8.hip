// The ring kernel on FP8 weights.
#include "gemm_ring.h"

namespace dro {
bool launch_ring_fp8(const GemmArgs& a, int cols, int* status, hipStream_t stream) { return ring::launch_ring<LX_W_FP8>(a, cols, status, stream); }
}  // namespace dro
