// Which kernel and which row block a product or a routing takes: rules on the arguments alone, shared by the kernels' launchers and the host path
// (no HIP here).
#pragma once
#include <math.h>
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

// Slices of a ragged problem that have rows, if they are spread at random; all of a batch.
inline double live_slices(const tamd_matmul_args &a) {
  return a.block_schedule ? -expm1(a.M * log1p(-1.0 / a.n_experts)) * a.n_experts : a.n_experts;
}

// The most of them that its rows can fall on.
inline int most_live_slices(const tamd_matmul_args &a) { return a.M < a.n_experts ? a.M : a.n_experts; }

// The row blocks that a ragged schedule may have.
inline bool known_block(int block_m) { return block_m == 16 || block_m == 32 || block_m == 64 || block_m == 128; }

inline int64_t output_size(int dtype) { return dtype == TAMD_F32 ? 4 : (dtype == TAMD_FP8_E4M3 || dtype == TAMD_FP8_E5M2 ? 1 : 2); }

// Products of 8- and 4-bit rows x MXFP4 weights, row blocks of up to 32, that K groups share (moe_matmul_mx.h): up to half as many tiles of
// 256 columns as CUs, four stages of 256 K and more.  1500 products, dense: K 769 to 1024 0.95 of the tiled kernel's time, 1025 to 1280
// (two stages for some groups) 1.0, to 2048 0.83, to 4096 0.74, to 8192 0.58; three stages 1.05.
inline bool mx_groups(const tamd_matmul_args &a, int cus, int block_m) {
  if (a.K <= 768 || block_m > 32) return false;
  const double blocks = a.block_schedule ? live_slices(a) * ceil((double)a.M / a.n_experts / block_m) : (double)a.n_experts * ((a.M + block_m - 1) / block_m);
  return 2.0 * blocks * ((a.N + 255) / 256) <= cus;
}

// What the persistent kernel of few rows per slice (moe_matmul_ring.h) covers: ragged problems with weights in 4 KB blocks and pre-shuffled
// scales or both strided along K, outputs of the usual type in pairs of columns that 32-bit offsets reach.
inline bool ring_applicable(const tamd_matmul_args &a) {
  if (!a.block_schedule || a.force_variant) return false;
  if ((a.w_layout == TAMD_W_CDNA4_BLOCKS) != (a.w_mx_layout == TAMD_SCALE_CDNA4)) return false;
  if (a.n_experts > 256 || (a.N + 63) / 64 > 0x8000 || ((int64_t)a.M + a.n_experts) * ((a.N + 63) / 64) > 0x7FFFFFF0) return false;
  const bool x16 = a.x_dtype == TAMD_BF16 || a.x_dtype == TAMD_F16, sw = a.activation == TAMD_ACT_SWIGLU;
  if (!x16 && a.x_dtype != TAMD_FP8_E4M3 && a.x_dtype != TAMD_MXFP4) return false;
  const int64_t lim = 0x7FFFFF00, size = output_size(a.y_dtype);
  if (a.y_rows <= 0 || a.y_stride_m < 0 || a.y_rows * a.y_stride_m * size >= lim) return false;
  if (a.y_mx_scale && a.y_rows * a.y_mx_stride_m >= lim) return false;
  if (!sw && (((a.N | (int)a.y_stride_m) & 1) != 0 || !aligned(a.y, 2 * (size_t)size))) return false;
  const bool flex = a.y_expected_scale || a.y_actual_scale;
  if (x16) return !a.y_mx_scale && !flex && a.y_dtype == a.x_dtype;
  // (fp8 rows whose row blocks stream stay there: widened to bf16 their sums are 5e-9 off 64-bit ones, 4e-6 with the MFMA that takes them
  // as they are)
  if (a.x_dtype == TAMD_FP8_E4M3 && a.block_m == 16 && stream16_applicable(a)) return false;
  return a.y_dtype == TAMD_FP8_E4M3 || (a.y_dtype == TAMD_BF16 && !flex);
}

// Strided weights come in pieces of 64 bytes, at 3 to 4.7 TB/s in either kernel, and the copies no longer run ahead of anything over
// several rounds (1.0 to 1.05 there): it is the faster where most CUs have no tile or one and narrower tiles share them out, and for the
// larger blocks of 16-bit rows.  4000 products, time over the tiled kernel's, where it is taken: packed rows 0.83, MXFP8 0.89, fp8 0.89,
// 16-bit rows 0.93; one in ten above 1.04.
// (16-bit rows in blocks of 64 with 0.85 to 1.0 tiles per CU, slices spread as a router's: K 800 to 1200 1.00, to 1800 0.94, to 2880 0.89;
// with 1.0 to 1.15 1.06, 1.00, 0.94.)
inline int ring_rows_strided(const tamd_matmul_args &a, double cover, double tiles) {
  if (a.x_dtype == TAMD_BF16 || a.x_dtype == TAMD_F16) {
    if (cover <= 16.0 || cover > 64.0) return 0;
    if (cover <= 32.0) return tiles > 0.3 && tiles <= 1.0 ? 32 : 0;
    return (tiles > 0.5 && tiles <= 1.0) || (tiles > 2.0 && a.K > 128) ? 64 : 0;   // (K 32 to 96 1.05 of the tiled kernel's time, to 256 0.92)
  }
  const bool packed = a.x_dtype == TAMD_MXFP4;
  if (cover > (packed ? 64.0 : 32.0) || tiles > 0.75 || tiles <= (packed ? 0.0 : a.x_mx_scale ? 0.15 : 0.3)) return 0;
  return cover <= 32.0 ? 32 : 64;
}

// A tile alone on its CU wins by copies that run ahead, which takes stages: with fewer, the start of a workgroup of twelve waves and its table
// cost more than they give, against tiles (not against streaming, the blocks of 16, which is slower still there).  Rows of 8 and 4 bits
// win again where one stage or two are all of K.  4700 products of K 32 to 1500, time over the tiled kernel's:
//   16-bit rows         strided K to 512 1.08, to 640 1.04, to 768 1.00, to 1500 0.96; in 4 KB blocks 1.15, 1.07, 1.05, 0.98
//   MXFP8               strided K to 256 0.87, to 768 1.08; 4 KB blocks to 256 0.95, to 768 1.04
//   fp8 and packed rows strided K to 256 0.89, to 512 1.04 (64 rows 1.09), to 768 1.01; 4 KB blocks to 512 0.99 (64 rows 1.06)
inline bool ring_stages_too_few(const tamd_matmul_args &a, double cover) {
  if (a.block_m <= 16) return false;
  if (a.x_dtype == TAMD_BF16 || a.x_dtype == TAMD_F16) return a.K <= 768;
  const bool scaled = a.x_dtype == TAMD_FP8_E4M3 && a.x_mx_scale;
  return a.K > 256 && a.K <= (scaled ? 768 : 512) && (scaled || a.w_layout != TAMD_W_CDNA4_BLOCKS || cover > 32.0);
}

// SwiGLU products of 8- and 4-bit rows with more than 64 rows per slice: the persistent kernel's blocks of 96 against tiles of 128, by what each
// is estimated to take (us): a start, and rounds over the CUs (two tiles of 128 to a CU) whose last is paid for in part.  The epilogue of
// such a tile is a third of its time, which the persistent kernel hides behind the next tile's products; without SwiGLU, and from
// about a thousand rows per slice on, tiles are the faster.  Fitted to 2300 products (8 to 128 slices of 24 to 2000 rows, K 512 to 5760, slices as
// uneven as a router's).  900 others, a third each with even slices, 0.2 and 0.45 in the logarithm: 0.857 of the tiles' time in the mean, 38
// above 1.05, 1.23 at worst.  25 of those have even slices: with 97 to 126 and 200 to 226 rows one tile takes what two blocks of 96 share,
// or two what three, 1.02 in the mean and up to 1.23 (0.86 to 0.93 if slices are uneven).  Where that one round of tiles is nearly full
// as well, 18 products took 0.75 to 1.29, 0.98 in the mean: left to the tiles.
inline bool ring_96_before_tiles(const tamd_matmul_args &a, int cus, double mean, double cover) {
  if (a.activation != TAMD_ACT_SWIGLU || a.K < 800 || mean < 60.0 || mean > 1024.0) return false;
  const bool packed = a.x_dtype == TAMD_MXFP4, scaled = !packed && a.x_mx_scale;
  const double cols = live_slices(a) * ((a.N + 255) / 256) / cus, k = a.K / 1000.0;
  const double r = cols * fmax(1.0, mean / 96.0 + 0.5), m = cols * 0.5 * fmax(1.0, mean / 128.0 + 0.5);
  if (m < 0.75) return false;
  if (cover <= 128.0 && cols > 1.4 && cols <= 2.0) return false;   // one round of tiles of 128, nearly full
  const double ring = 5.0 + (packed ? 3.2 + 3.5 * k : scaled ? 4.2 + 4.8 * k : 3.2 + 4.4 * k) * (r + 0.6 * (ceil(r) - r) + 0.1);
  const double tiles = 5.0 + (packed ? 5.9 + 11.1 * k : scaled ? 9.7 + 13.9 * k : 7.9 + 11.6 * k) * (m + 0.05 * (ceil(m) - m) + 0.07);
  return ring < (scaled ? 1.0 : 0.97) * tiles;
}

// Rows of the persistent kernel's blocks, 0 where another kernel is the faster (or the only one).  The block is the smallest that covers a
// slice's mean size and two standard deviations, up to 96; the lines between the kernels are in tiles per CU, one row block for every slice
// that has rows (on the average of random choices).  Up to one, a tile is alone on its CU and wins by its depth; just above, the second
// round is nearly empty, where smaller tiles, three and four to a CU, lose less; from two on the rounds fill.  Below K 1024 the loop over K
// is too short to hide the tile before, unless there is none.
// 16-bit rows of up to 16 per slice are the streaming kernel's, except where its parts of K (multiples of 1024) fit badly; their larger
// blocks are bound by the conversion of the codes, as in the other kernels.
// From 38 000 products (layers of 1 to 16384 tokens, 8 to 128 slices, K and N 512 to 5760, random choices), time with this rule where it
// chooses this kernel over the time without: 16-bit rows 0.905, fp8 0.907, MXFP8 0.95, packed 0.914; more than 10 % slower in 1 to 2 % of
// them.
inline int ring_rows(const tamd_matmul_args &a, int cus) {
  if (!ring_applicable(a)) return 0;
  const bool x16 = a.x_dtype == TAMD_BF16 || a.x_dtype == TAMD_F16;
  // (16-bit rows: no line lies below 0.3 tiles per CU; a few rows have fewer whichever slices they fall on)
  if (x16 && 10.0 * most_live_slices(a) * ((a.N + 255) / 256) <= 3.0 * cus) return 0;
  const double mean = (double)a.M / a.n_experts, cover = mean + 2.0 * sqrt(mean);
  const double tiles = live_slices(a) * ((a.N + 255) / 256) / cus;
  // (K groups, mx_groups, against this kernel: MXFP8 0.65 to 0.9, fp8 0.6 to 0.95, packed rows 0.75 to 1.0; with more tiles 1.0 to 1.5)
  const bool x8 = a.x_dtype == TAMD_FP8_E4M3;
  if ((x8 || a.x_dtype == TAMD_MXFP4) && a.block_m <= 32 && a.K > 1280 && cover <= 32.0 && tiles <= (x8 && a.K > 2048 ? 0.375 : 0.25)) return 0;
  if (tiles <= 1.0 && ring_stages_too_few(a, cover)) return 0;
  if (a.w_layout != TAMD_W_CDNA4_BLOCKS) return ring_rows_strided(a, cover, tiles);
  const bool packed = a.x_dtype == TAMD_MXFP4, scaled = !packed && a.x_mx_scale;
  // (of blocks of 96 rows what the products of a layer write is built)
  const bool rows_96 = !x16 && cover > 64.0 && (a.y_dtype != TAMD_FP8_E4M3 || (a.activation == TAMD_ACT_SWIGLU && !(packed && a.y_mx_scale)));
  if (rows_96 && ring_96_before_tiles(a, cus, mean, cover)) return 96;
  if (mean > 96.0 || (a.K < 1024 && tiles > 1.0)) return 0;
  const bool alone = tiles <= 1.0;
  if (x16) {
    if (cover <= 16.0 && a.K <= 4096) {
      const bool padded = a.K > 1024 && (a.K + 1023) / 1024 * 1024 >= 1.3 * a.K;
      return (alone && tiles > (mean < 3.0 ? 0.75 : 0.5)) || (padded && tiles > 2.0) ? 32 : 0;
    }
    if (cover <= 32.0) return (alone && tiles > 0.3) || tiles > (cover <= 16.0 ? 2.2 : 8.0) ? 32 : 0;
    if (mean < 50.0) return alone && tiles > 0.75 ? 64 : 0;
    return mean <= 80.0 && tiles > 1.1 && tiles < 8.0 ? 64 : 0;
  }
  if (cover <= 32.0) {
    if (scaled) return alone || tiles > 2.0 ? 32 : 0;
    if (packed) return alone || tiles > 1.4 ? 32 : 0;
    // (A slice in two blocks of 32 costs more than a block of 64, and a router picks some experts more often than others.  476 products with
    // slices spread as a router's, 0.45 in the logarithm, time over that with blocks of 32: above 6 tiles per CU mean 12 to 16 0.989, to 23 0.964,
    // below 12 0.999; up to 6 tiles 0.99 to 1.00 for any mean.  With even slices 1.00 to 1.01 throughout.)
    if (tiles > 6.0 && mean >= 12.0) return 64;
    return (alone && tiles > (mean < 10.0 ? 0.27 : 0.1)) || tiles > 2.0 ? 32 : 0;
  }
  if (cover <= 64.0) return tiles > 2.0 || (alone && !scaled && tiles > (packed ? 0.0 : 0.6)) ? 64 : 0;
  return rows_96 && tiles > (packed ? 1.4 : 2.0) ? 96 : 0;
}

// What the persistent kernel for unquantised 16-bit weights (moe_matmul_kkring.h) covers, of the products that the tiled kernel of two
// operands along K takes: ragged problems of four stages of K and more, outputs of the rows' type in pairs of columns that 32-bit offsets
// reach.
inline bool kk_ring_applicable(const tamd_matmul_args &a) {
  if (!a.block_schedule || a.force_variant || a.K < 256 || a.n_experts > 256) return false;
  if ((a.x_dtype != TAMD_BF16 && a.x_dtype != TAMD_F16) || a.w_dtype != a.x_dtype || a.y_dtype != a.x_dtype) return false;
  if (a.y_mx_scale || a.y_expected_scale || a.y_actual_scale) return false;
  if ((a.N + 63) / 64 > 0x8000 || ((int64_t)a.M + a.n_experts) * ((a.N + 63) / 64) > 0x7FFFFFF0) return false;
  if (a.y_rows <= 0 || a.y_stride_m < 0 || a.y_rows * a.y_stride_m * 2 >= (int64_t)0x7FFFFF00) return false;
  return a.activation == TAMD_ACT_SWIGLU || (((a.N | (int)a.y_stride_m) & 1) == 0 && aligned(a.y, 4));
}

// Rows of its blocks, 0 where the tiled kernels are the faster.  The lines are in thirds of a tile of 256 columns per CU, row blocks of 160 counted:
// where there are few, one workgroup's stages are all latency (four rows for 8 slices, 1760 x 3904: 13.4 us, 16 with this one).
// From one third on, 486 products of 1 to 16384 tokens, 8 to 128 slices, K and N 512 to 5760: 0.876 of the time in the mean (0.866 with the
// best choice for each), none above 1.05.  Blocks of 64 up to 56 rows per slice lose up to 1.21, where slices come in two.
// Below it tiles of one to three strips of 64 columns and blocks of 64 rows reach every CU, where the tiled kernel leaves most of them without
// a tile: the more rows per slice, the earlier.  675 products below the line (8 to 60 slices, bf16 and f16, even slices, 0.2 and 0.45 in the
// logarithm): 0.84 of the time in the mean; up to K 640 0.87 to 1.05, beyond 0.75 to 0.99.  Above 1.05 are 24, 1.10 at worst but for one
// of five rows per slice (1.25), 21 of them of K up to 832; of 48 to 64 rows and K up to 400 were 16 of 40, 1.03 in the mean: not taken.  Layer
// of 102 rows for each of 8 slices, f16, 5376 -> 992, 112 -> 93 us.  Under four rows per slice up to 1.9; half a line further down 0.93 to
// 1.25, 2.1 at worst.  Just above the line blocks of 64 for up to 128 rows per slice take 0.88 of what those of 160 do in the mean of 125
// products, 1.054 at worst, with K above 4096 up to 1.3; from 1.3 thirds on up to 1.5.
inline double kk_ring_thirds(const tamd_matmul_args &a, int cus) {
  const double mean = (double)a.M / a.n_experts, tiles = live_slices(a) * ((a.N + 255) / 256) / cus;
  return 3.0 * tiles * (mean > 160.0 ? mean / 160.0 : 1.0);
}
inline int kk_ring_rows(const tamd_matmul_args &a, int cus) {
  if (!kk_ring_applicable(a)) return 0;
  // (the line below, whichever slices the rows fall on)
  if (a.M <= a.n_experts && 3 * (int64_t)most_live_slices(a) * ((a.N + 255) / 256) < cus) return 0;
  const double mean = (double)a.M / a.n_experts, thirds = kk_ring_thirds(a, cus);
  if (thirds < 1.0) {
    if (a.K <= 400 && mean >= 48.0 && mean < 64.0) return 0;
    return mean >= 4.0 && thirds >= (mean < 32.0 ? 0.9 : mean < 48.0 ? 0.6 : mean < 128.0 ? 0.5 : 0.4) ? 64 : 0;
  }
  return mean <= 48.0 || (mean < 128.0 && thirds < 1.15 && a.K <= 4096) ? 64 : 160;
}

// Float32 sums that a result of a block of 64 rows is made of: below the line no fewer than in the tiled kernels, which products take there otherwise.
// Two, of the halves of every stage, are those of their wide tiles to the bit; four, of the quarters of K, those of the narrow tiles, which only
// products of more than ten stages take.  Above the line one, as in blocks of 160.
inline int kk_ring_sums(const tamd_matmul_args &a, int cus) { return kk_ring_thirds(a, cus) >= 1.0 ? 1 : a.K <= 640 ? 2 : 4; }

// Row block size of a dense / batched problem: the block whose tiles take the fewest rounds over the CUs, weighted with what a
// tile of it takes, of one of 128 rows: `weight` (in percent) for 64 and 32 rows, `slots` tiles at the speed of one round.
// Fitted to products timed with every block (mean and worst time against the best block of each):
//   16-bit rows x MXFP4, 130 of 64 to 16384 rows: one and a half tiles per CU, 0.45 and 0.35; from K 3072 down, where a block of 128 has
//     its scales in LDS, one per CU, 0.58 and 0.4 for strided weights and from four rounds on.  1.009, 1.14; with the first figures for all 1.019,
//     1.23 (14716 x 2080 x 8144 481 us in blocks of 64, 413 of 128; block layout, 16384 x 2880 x 2880 232 and 217, 3337 x 608 x 4768 24 and
//     31), with the largest block that gives every CU a tile 1.041, 1.47;
//   fp8 x MXFP4, the same: one and three quarters, 0.68 and 0.4.  1.009, 1.18 (the figures of 16-bit rows 1.039, 1.24: 8192 x 2880 x
//     5760 131 us in blocks of 64, 118 of 128; the largest block 1.011, 1.19);
//   packed rows, the same: one, 0.58 and 0.4.  1.014, 1.15 (1.037, 1.27: 4122 x 7808 x 3152 119 us, 90; 1.028, 1.24);
//   one type along K, 800 of 1 to 4096 rows: one, 0.6 and 0.45, 9 % faster in the mean than the largest block (2000 rows of K 2000 and N 1600
//     two rounds of 64 rows instead of one of 128 on half the CUs, up to 1.7 times);
//   one type along N, 150 of 16 to 16384 rows: one, 0.8 and 0.76 (the LDS reads of the weights do not follow the rows).  1.007; 3943 x 6144 x 7464
//     815 us in blocks of 64, 471 of 128, 5749 x 2432 x 512 68 of 32, 39 of 64.
inline int dense_block_m(const tamd_matmul_args &a, int cus) {
  const bool x16 = a.x_dtype == TAMD_BF16 || a.x_dtype == TAMD_F16, mxfp4 = a.w_dtype == TAMD_MXFP4;
  const bool along_n = !mxfp4 && a.w_stride_k != 1;
  const int64_t cols = (int64_t)((a.N + 255) / 256) * a.n_experts;
  int slots = cus, w64 = 58, w32 = 40;
  if (!mxfp4) {
    w64 = along_n ? 80 : 60, w32 = along_n ? 76 : 45;
  } else if (x16 && (a.K > 3072 || (a.w_layout == TAMD_W_CDNA4_BLOCKS && (a.M + 127) / 128 * cols < 4 * (int64_t)cus))) {
    slots = cus * 3 / 2, w64 = 45, w32 = 35;
  } else if (!x16 && a.x_dtype != TAMD_MXFP4) {
    slots = cus * 7 / 4, w64 = 68, w32 = 40;
  }
  const int extra = x16 && !along_n ? 32 : 0;   // remainder that a block of 128 absorbs
  const int bm[3] = {128, 64, 32}, weight[3] = {100, w64, w32};
  int best = 0;
  int64_t least = 0;
  for (int i = 0; i < 3; ++i) {
    const int64_t m = i == 0 && a.M > 128 ? a.M - extra : a.M;
    const int64_t cost = ((m + bm[i] - 1) / bm[i] * cols + slots - 1) / slots * weight[i];
    if (best == 0 || cost < least) best = bm[i], least = cost;
  }
  return best;
}

// ---------------------------------------------------------------------------
// routing
// ---------------------------------------------------------------------------
// Lanes that share a row of up to 512 logits, eight of them or fewer each, a lane for every pick.
inline int lanes_per_row(int n_cols, int k) {
  const int need = (n_cols + 7) / 8 > k ? (n_cols + 7) / 8 : k;
  return need <= 8 ? 8 : (need <= 16 ? 16 : (need <= 32 ? 32 : 64));
}

// How the two launches of the routing (routing.hip) cut n_rows rows: blocks of RB rows, TH threads each.
struct RowPlan {
  int TH, RB, pitch, lg_cols, nb, sub, nbo, W;
  size_t lds;
};
constexpr int kMaxRowsPerBlock = 128;   // (a byte would count 255; RB is a power of two)

// Fills the plan, or returns false where the table or the counts do not fit or the older launches are the faster: more than 65535 rows (the sums of
// the table's bytes have 16 bits), more than 512 experts, and the two lines below.  The workgroups of the first launch are the smallest whose
// table is read with four loads per thread (16 KB); a longer input makes the blocks larger, so that a workgroup passes over its rows several times.
// There the chip idles: above 256 experts, 16 rows to a pass, from four passes on (79 workgroups for 10000 rows; k 1 1.32 to 1.41 of the other
// launches' time, k 8 1.57 to 1.68, 24000 rows 1.02 to 1.06 and 0.90 to 0.93, two passes 0.44 to 1.06); below, where the workgroups no longer are one
// round over 256 CUs (from 32769 rows) and a row gives fewer than four entries to place (200 experts, 33000 rows, k 1 1.35, k 2
// 1.38, k 4 1.07, k 8 1.02; 65000 1.27, 1.25, 0.91, 0.82; 128 experts 1.14, 1.15, 0.82, 0.76 and 1.09, 1.13, 0.72, 0.63).
inline bool make_row_plan(int64_t n_rows, int E, int k, int L, int64_t workspace_ints, RowPlan &p) {
  if (n_rows < 1 || n_rows > 65535 || E > 512) return false;
  p.pitch = 16;
  while (p.pitch < E) p.pitch *= 2;
  p.lg_cols = __builtin_ctz(p.pitch / 4);
  p.TH = 256;
  while (p.TH < 1024 && (n_rows + p.TH / L - 1) / (p.TH / L) * p.pitch > 16384) p.TH *= 2;
  p.RB = p.TH / L;
  while (2 * p.RB <= kMaxRowsPerBlock && (n_rows + p.RB - 1) / p.RB * p.pitch > 65536) p.RB *= 2;
  p.nb = (int)((n_rows + p.RB - 1) / p.RB);
  const int passes = p.RB / (p.TH / L);
  if (E > 256 ? passes >= 4 : passes > 1 && p.nb > 256 && k < 4) return false;
  if ((int64_t)p.nb * (p.pitch / 4) > workspace_ints) return false;
  p.sub = 1;
  while (p.RB * p.sub * 2 * k <= 1024 && p.RB * p.sub * 2 <= 128 && p.sub < p.nb) p.sub *= 2;
  p.nbo = (p.nb + p.sub - 1) / p.sub;
  p.W = (p.RB * p.sub + 31) / 32;
  if ((int64_t)p.RB * p.sub * k * k >= 1 << 19) return false;  // over_k
  const int64_t waves = p.RB * p.sub * k >= 1024 ? 16 : (p.RB * p.sub * k + 64 - 1) / 64;
  const int64_t copies = waves * E > 6 * (E + 1) ? waves * E : 6 * (E + 1);
  p.lds = (size_t)(p.pitch + (int64_t)E * p.W + copies) * 4;
  return p.lds <= 150 * 1024;
}

}  // namespace tamd
