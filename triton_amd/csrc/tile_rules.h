// Which kernel and which row block a product takes: rules on the arguments alone, shared by the kernels' launchers and the host path
// (no HIP here).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include "../../include/triton_amd.h"

namespace tamd {

inline bool aligned(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

// The pitch of one matrix is never used: it takes part in no check.
inline void drop_unused_pitches(tamd_matmul_args &a) {
  if (a.n_experts == 1) a.w_stride_e = a.w_mx_stride_e = a.bias_stride_e = 0;
}

// Whether the streaming kernel covers the problem: rows without block scales (bf16 does not hold value times scale over the range that
// the scaled MFMA takes: scales of 2^119 and above overflow, values below 2^-133 vanish), K contiguous and dense per column for codes and
// scales, 16-byte aligned column groups, N a multiple of 16, K <= 4096, whole tensors addressable
// with 32-bit offsets.
inline bool stream16_applicable(const tamd_matmul_args &a) {
  const int64_t lim = 0x7FFFFF00;
  const int64_t G = a.K / 32;
  if (a.K > 4096 || a.K % 32 != 0) return false;
  if (a.x_mx_scale) return false;
  const bool cdna4 = a.w_mx_layout == TAMD_SCALE_CDNA4;
  const bool wnat = a.w_layout == TAMD_W_CDNA4_BLOCKS;
  if (!wnat && (a.w_stride_k != 1 || a.w_stride_n != a.K / 2)) return false;
  if (!cdna4 && (a.w_mx_stride_k != 1 || a.w_mx_stride_n != G)) return false;
  if (!aligned(a.w, 16) || a.w_stride_e % 16 != 0 || !aligned(a.w_mx_scale, 16) || a.w_mx_stride_e % 16 != 0) return false;
  if ((int64_t)a.n_experts * a.w_stride_e + (wnat ? (int64_t)0 : (int64_t)a.N * a.w_stride_n) >= lim) return false;
  if ((int64_t)a.n_experts * a.w_mx_stride_e + (int64_t)(a.N + 32) * (G + 8) >= lim) return false;
  if (a.bias && ((int64_t)a.n_experts * a.bias_stride_e + a.N) * 4 >= lim) return false;
  if (a.bias && !aligned(a.bias, a.bias_dtype == TAMD_F32 ? 4 : 2)) return false;
  if (a.N % 16 != 0) return false;  // whole 16-column groups only (their scale run is then a multiple of 16 bytes)
  if (a.block_schedule && !a.block_offs) return false;
  if (a.y_mx_scale) return false;  // a unit is 16 columns, an output scale group 32
  return true;
}

// The same for the arguments as a caller has them: whether the row blocks of 16 of a product with MXFP4 weights would stream.
inline bool blocks_of_16_stream(tamd_matmul_args a) {
  drop_unused_pitches(a);
  return a.w_dtype == TAMD_MXFP4 && stream16_applicable(a);
}

// Row block size of a dense / batched problem: the block whose tiles take the fewest rounds over the CUs, weighted with what a
// tile of it takes.  MXFP4 weights: one and a half tiles per CU (fp8 and packed rows one and a quarter) run at the speed of one, a tile of 64 or 32
// rows takes 0.45 or 0.35 of one of 128.  Kernels for operands of one type hold one tile per CU: 0.6 and 0.45 where the weights are
// contiguous along K, 0.8 and 0.76 where they are contiguous along N (the LDS reads of the weights do not follow the rows).
// (Fitted to products timed with every block.  800 of 1 to 4096 rows, against the largest block that gave every CU a tile: one type along K 9 %
// faster in the mean -- 2000 rows of K 2000 and N 1600 two rounds of 64 rows instead of one of 128 on half the CUs, up to 1.7 times --,
// MXFP4 2.5 %, none slower by more than 5 %.  150 of 16 to 16384 rows along N: 0.7 % slower than the best block of each
// in the mean, 12 % with the MXFP4 figures; 3943 x 6144 x 7464 815 us in blocks of 64, 471 in blocks of 128, 5749 x 2432 x 512 68 in
// blocks of 32, 39 in blocks of 64.)
inline int dense_block_m(const tamd_matmul_args &a, int cus) {
  const bool x16 = a.x_dtype == TAMD_BF16 || a.x_dtype == TAMD_F16, mxfp4 = a.w_dtype == TAMD_MXFP4;
  const bool along_n = !mxfp4 && a.w_stride_k != 1;
  const int64_t cols = (int64_t)((a.N + 255) / 256) * a.n_experts, slots = !mxfp4 ? cus : (x16 ? cus * 3 / 2 : cus * 5 / 4);
  const int extra = x16 && !along_n ? 32 : 0;   // remainder that a block of 128 absorbs
  const int bm[3] = {128, 64, 32}, weight[3] = {100, mxfp4 ? 45 : (along_n ? 80 : 60), mxfp4 ? 35 : (along_n ? 76 : 45)};
  int best = 0;
  int64_t least = 0;
  for (int i = 0; i < 3; ++i) {
    const int64_t m = i == 0 && a.M > 128 ? a.M - extra : a.M;
    const int64_t cost = ((m + bm[i] - 1) / bm[i] * cols + slots - 1) / slots * weight[i];
    if (best == 0 || cost < least) best = bm[i], least = cost;
  }
  return best;
}

}  // namespace tamd
