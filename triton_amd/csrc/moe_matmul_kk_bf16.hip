// Instantiates the matmul of two K-contiguous operands (moe_matmul_kk.h) for bf16.
#include "moe_matmul_kk.h"

namespace tamd {
int dispatch_mm_kk_bf16(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  return dispatch_kk<TAMD_BF16>(a, block_m, grid_m, st);
}
}  // namespace tamd
