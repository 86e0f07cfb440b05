// Instantiates the persistent kernels for few rows per slice (moe_matmul_ring.h).
#include "moe_matmul_ring.h"

namespace tamd {
int ring_mm_fp4(const tamd_matmul_args &a, int rows, hipStream_t st) { return dispatch_ring<TAMD_MXFP4>(a, rows, st); }
}  // namespace tamd
