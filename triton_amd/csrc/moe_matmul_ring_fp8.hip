// Instantiates the persistent kernels for few rows per slice (moe_matmul_ring.h).
#include "moe_matmul_ring.h"

namespace tamd {
int ring_mm_fp8e4m3(const tamd_matmul_args &a, int rows, hipStream_t st) { return dispatch_ring<TAMD_FP8_E4M3>(a, rows, st); }
}  // namespace tamd
