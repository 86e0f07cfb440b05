// Instantiates the matmul of two K-contiguous operands (moe_matmul_kk.h) for float8_e4m3fn and float8_e5m2.
#include "moe_matmul_kk.h"

namespace tamd {
int dispatch_mm_kk_fp8e4m3(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  return dispatch_kk<TAMD_FP8_E4M3>(a, block_m, grid_m, st);
}
int dispatch_mm_kk_fp8e5m2(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  return dispatch_kk<TAMD_FP8_E5M2>(a, block_m, grid_m, st);
}
}  // namespace tamd
