// The ring kernel on NVFP4 weights.
#include "gemm_ring.h"

namespace dro {
bool launch_ring_nvfp4(const GemmArgs& a, int cols, int* status, hipStream_t stream) { return ring::launch_ring<LX_W_NVFP4>(a, cols, status, stream); }
int launch_fed_nvfp4(const GemmArgs& a, hipStream_t stream) { return ring::launch_fed(a, stream); }
}  // namespace dro
