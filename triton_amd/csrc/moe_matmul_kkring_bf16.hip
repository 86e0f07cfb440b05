// Instantiates the persistent kernels for unquantised bf16 weights (moe_matmul_kkring.h).
#include "moe_matmul_kkring.h"

namespace tamd {
int kk_ring_mm_bf16(const tamd_matmul_args &a, int rows, hipStream_t st) { return dispatch_kk_ring<TAMD_BF16>(a, rows, st); }
}  // namespace tamd
