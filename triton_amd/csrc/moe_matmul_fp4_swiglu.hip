// Instantiates the kernels for microscaled e2m1 activations x MXFP4 weights (moe_matmul_mx.h) with the fused SwiGLU epilogue.
#include "moe_matmul_mx.h"

namespace tamd {
int tiled_mm_swiglu_fp4(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  return dispatch_mx_act<TAMD_MXFP4, TAMD_ACT_SWIGLU>(a, block_m, grid_m, st);
}
}  // namespace tamd
