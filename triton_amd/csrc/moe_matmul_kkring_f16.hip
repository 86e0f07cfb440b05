// Instantiates the persistent kernels for unquantised f16 weights (moe_matmul_kkring.h).
#include "moe_matmul_kkring.h"

namespace tamd {
int kk_ring_mm_f16(const tamd_matmul_args &a, int rows, hipStream_t st) { return dispatch_kk_ring<TAMD_F16>(a, rows, st); }
}  // namespace tamd
