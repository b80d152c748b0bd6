// The ring kernel on INT8 weights.
#include "gemm_ring.h"

namespace dro {
bool launch_ring_int8(const GemmArgs& a, int cols, int* status, hipStream_t stream) { return ring::launch_ring<LX_W_INT8>(a, cols, status, stream); }
}  // namespace dro
