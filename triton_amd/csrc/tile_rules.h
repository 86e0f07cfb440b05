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

}  // namespace tamd
