// Instantiates the persistent kernels for few rows per slice (moe_matmul_ring.h).
#include "moe_matmul_ring.h"

namespace tamd {
int ring_mm_f16(const tamd_matmul_args &a, int rows, hipStream_t st) { return dispatch_ring<TAMD_F16>(a, rows, st); }
}  // namespace tamd
