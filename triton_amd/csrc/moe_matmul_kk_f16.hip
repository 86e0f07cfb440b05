// Instantiates the matmul of two K-contiguous operands (moe_matmul_kk.h) for f16.
#include "moe_matmul_kk.h"

namespace tamd {
int dispatch_mm_kk_f16(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  return dispatch_kk<TAMD_F16>(a, block_m, grid_m, st);
}
}  // namespace tamd
