// Instantiates the tiled MXFP4 grouped matmul kernels (moe_matmul_impl.h) with the fused SwiGLU epilogue.
#include "moe_matmul_mx.h"

namespace tamd {
int tiled_mm_swiglu_bf16(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  return dispatch_x16_act<TAMD_BF16, TAMD_ACT_SWIGLU>(a, block_m, grid_m, st);
}
}  // namespace tamd
