// Instantiates the kernels for microscaled e2m1 activations x MXFP4 weights (moe_matmul_mx.h) with the plain epilogue (the SwiGLU
// ones are compiled in moe_matmul_fp4_swiglu.hip).
#include "moe_matmul_mx.h"

namespace tamd {
int dispatch_mm_fp4(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  if (a.activation == TAMD_ACT_SWIGLU) return tiled_mm_swiglu_fp4(a, block_m, grid_m, st);
  return dispatch_mx_act<TAMD_MXFP4, TAMD_ACT_NONE>(a, block_m, grid_m, st);
}
}  // namespace tamd
