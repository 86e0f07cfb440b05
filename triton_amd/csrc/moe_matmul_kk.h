// Grouped / dense matmul of two operands of the same element type that are both contiguous along K: unquantised 16-bit
// weights (bf16 x bf16, f16 x f16) and fp8 x fp8 with per-tensor scales.
//
// A tile is up to 128 rows (160 with 16-bit operands: a remainder of up to 32 rows is absorbed, as in moe_matmul_impl.h)
// x 256 columns; a workgroup of eight waves owns a CU.  Both operands travel HBM -> LDS by 16-byte DMA in stages of 128
// bytes per row and column (64 K of 16-bit values, 128 K of fp8), through a ring of three or four stages that is two or
// three ahead of the matrix cores; rows and columns are 128-byte lines, requested whole.
//
// What bounds it.  With few rows per expert: HBM (the ring holds 64 KB or more of weights in flight per CU).  With full tiles
// the stages themselves: a stage's copies (one holds its wave for about a hundred cycles), its barrier and its LDS reads
// follow one another.  In the layer of 1021 tokens over 32 experts (K 2880) the matrix cores are busy 25 % of the cycles, the
// address units 63 %, LDS 11 %; at 1024 x 8192 x 8192 of fp8 53, 27 and 11 %.  Hence the two K groups: waves 0-3 and 4-7 share
// the tile's four 64-column strips, each group multiplying one half of every stage, so that a SIMD holds two waves for the
// operand reads of one (waves of 64 x 64 would read a third more), and group 0 requests the next stage's copies before its
// products and group 1 after them: with both groups issuing at the same time the matrix cores idled meanwhile.  The groups'
// partial sums meet in LDS after the loop, each group finishing one half of the row fragments.
//
// fp8 operands stay fp8 up to the registers and are widened there, so that the products are those of the widened operands:
// exact, with float32 sums.  The MFMAs that take fp8 directly (32x32x16 and the scaled 32x32x64 alike) align the products of a
// step at the largest one and drop what falls below: measured against 64-bit sums over K 512 .. 8192, they are off by 0.9 to
// 1.5e-5 of the result (normal operands) and 6e-5 (operands over twelve binades) at every K, the bf16 MFMA by 0.2 to 3e-7.
// 1024 x 8192 x 8192: 110 us, 1.25 PFLOP/s (large bf16 products of the library reach 1.14 on this part; matrix cores busy 53 % of
// the cycles, a stage holds 2048 cycles of MFMA then); 348 widened in a pass of its own, 67 with the fp8 MFMA.
#pragma once
#include "moe_matmul_impl.h"

namespace tamd {

template <int XDT>
struct KK {
  static constexpr bool FP8 = is_fp8(XDT);
  static constexpr int ESZ = FP8 ? 1 : 2;
  static constexpr int KS = 128 / ESZ;                 // K per stage
  typedef Mma<FP8 ? TAMD_BF16 : XDT> M;                // (every fp8 number is a bf16 number)
  typedef typename M::frag_t frag_t;
  // MFMA steps that a 16-byte chunk of a row or column feeds, and the operand of step s
  static constexpr int STEPS = FP8 ? 2 : 1;
  static TAMD_DEVICE frag_t operand(const uint4 &v, int s) {
    if constexpr (!FP8) {
      return __builtin_bit_cast(frag_t, v);
    } else {
      const uint32_t w[2] = {s ? v.z : v.x, s ? v.w : v.y};
      bf16x2_t p[4];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (XDT == TAMD_FP8_E5M2) {
          p[2 * i] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w[i], 1.0f, false);
          p[2 * i + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w[i], 1.0f, true);
        } else {
          p[2 * i] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[i], 1.0f, false);
          p[2 * i + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[i], 1.0f, true);
        }
      }
      return frag_t{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
    }
  }
};
template <int XDT, int BM>
struct KKShape {
  typedef TileShape<XDT, BM> T;
  static constexpr int STAGE = (T::LDS_ROWS + BLOCK_N) * 128;
  static constexpr int RING = T::LDS_ROWS <= 32 ? 4 : 3;
  static constexpr int EXCHANGE = T::MF * 4 * kWave * NF * 16 * 4;   // partial sums of MF row fragments
  static constexpr int LDS = RING * STAGE > EXCHANGE ? RING * STAGE : EXCHANGE;
  static_assert(LDS <= 160 * 1024, "one workgroup per CU");
};

template <int XDT, int NFR, int BM, int ACT, bool ONCE>
TAMD_DEVICE void run_tile_kk(const tamd_matmul_args &a, const Tile &t, uint8_t *lds) {
  typedef KK<XDT> O;
  typedef typename O::frag_t frag_t;
  typedef KKShape<XDT, BM> S;
  constexpr bool FP8 = KK<XDT>::FP8;
  constexpr int ESZ = KK<XDT>::ESZ, KS = KK<XDT>::KS, EPC = 16 / ESZ;
  constexpr int LDS_ROWS = S::T::LDS_ROWS, STAGE = S::STAGE, RING = S::RING;
  constexpr uint32_t kOob = 0x7FFFFFFFu;
  const int wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int grp = wave8 >> 2, wave = wave8 & 3;        // K group, column strip
  const int c32 = lane % 32, h = lane / 32;
  const int K = a.K, N = a.N;
  const v4i_t rx = make_rsrc((const uint8_t *)a.x + (int64_t)t.z * a.x_stride_z * ESZ, kOob);
  const v4i_t rw = make_rsrc((const uint8_t *)a.w + (int64_t)t.expert * a.w_stride_e * ESZ, kOob);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;

  // ---- copies: instruction q of an operand moves its LDS rows 8q .. 8q + 7, lane -> (row 8q + lane / 8, slot lane % 8),
  // slot s of row r holding chunk s ^ ((r >> 1) & 7); wave w takes the instructions w, w + 8, ... of both operands
  const int rin = lane / 8;
  const int chunk = (lane % 8) ^ ((wave8 & 1) * 4 + (rin >> 1));
  constexpr int NA0 = (NFR + 1) / 2, NA1 = NFR / 2, NB = 4;   // copies per wave and stage: group 0, group 1; columns
  uint32_t a_off[NA0], b_off[NB];
#pragma unroll
  for (int u = 0; u < NA0; ++u) {
    const int r = (wave8 + 8 * u) * 8 + rin;
    const int rr = t.off_m + (r < t.rows ? r : t.rows - 1);
    const uint32_t src = a.gather_indx ? (uint32_t)a.gather_indx[t.start_m + rr] : (uint32_t)(t.start_m + rr);
    a_off[u] = r < t.rows ? src * (uint32_t)(a.x_stride_m * ESZ) + chunk * 16 : kOob;
  }
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int p = (wave8 + 8 * u) * 8 + rin;                  // position 64 strip + 32 f + c holds column 64 strip + 2 c + f
    const int col = t.n0 + (p & ~63) + 2 * (p % 32) + (p % 64) / 32;
    b_off[u] = col < N ? (uint32_t)col * (uint32_t)(a.w_stride_n * ESZ) + chunk * 16 : kOob;
  }
  auto issue = [&](int it, int slot) {   // (chunks past K are not read: zeros)
    const int kb = it * KS;
    const uint32_t kill = kb + chunk * EPC < K ? 0u : kOob;
    const uint32_t sa = lds_base + slot * STAGE + wave8 * 1024;
#pragma unroll
    for (int u = 0; u < NA0; ++u)
      if (u < NA1 || grp == 0) dma16(rx, sa + u * 8192, a_off[u] | kill, kb * ESZ);
    const uint32_t sb = sa + LDS_ROWS * 128;
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if constexpr (ONCE) dma16_nt(rw, sb + u * 8192, b_off[u] | kill, kb * ESZ);
      else dma16(rw, sb + u * 8192, b_off[u] | kill, kb * ESZ);
    }
  };

  f32x16_t acc[NFR][NF];
#pragma unroll
  for (int i = 0; i < NFR; ++i)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[i][f][j] = 0.f;

  const bool live = t.n0 + wave * 64 < N;
  const int swz = (c32 >> 1) & 7;
  // the group's two 16-byte chunks of a row or column
  const int slot0 = (h * 4 + 2 * grp) ^ swz, slot1 = (h * 4 + 2 * grp + 1) ^ swz;
  const int a_lane = c32 * 128, b_lane = LDS_ROWS * 128 + (wave * 64 + c32) * 128;
  const int n_k = (K + KS - 1) / KS;
#pragma unroll
  for (int s = 0; s < RING - 1; ++s) issue(s, s);
  int rd = 0, wr = RING - 1;
  for (int it = 0; it < n_k; ++it) {
    // copies complete in the order of their requests: all but those of the newest RING - 2 stages have landed
    if (grp == 0) wait_vmcnt<(RING - 2) * (NA0 + NB)>(); else wait_vmcnt<(RING - 2) * (NA1 + NB)>();
    sync_threads();   // stage `it` is visible; every wave is done with the slot that is refilled now
    const uint8_t *buf = lds + rd * STAGE;
    uint4 av[NFR][2], bv[NF][2];
    if (live) {
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        bv[f][0] = *(const uint4 *)(buf + b_lane + f * 4096 + slot0 * 16);
        bv[f][1] = *(const uint4 *)(buf + b_lane + f * 4096 + slot1 * 16);
      }
#pragma unroll
      for (int i = 0; i < NFR; ++i) {
        av[i][0] = *(const uint4 *)(buf + a_lane + i * 4096 + slot0 * 16);
        av[i][1] = *(const uint4 *)(buf + a_lane + i * 4096 + slot1 * 16);
      }
    }
    if (grp == 0) issue(it + RING - 1, wr);
    if (live) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int s = 0; s < O::STEPS; ++s) {
          frag_t b[NF];
#pragma unroll
          for (int f = 0; f < NF; ++f) b[f] = O::operand(bv[f][c], s);
#pragma unroll
          for (int i = 0; i < NFR; ++i) {
            const frag_t ai = O::operand(av[i][c], s);
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[i][f] = O::M::mma(ai, b[f], acc[i][f]);
          }
        }
    }
    if (grp == 1) issue(it + RING - 1, wr);
    rd = rd + 1 == RING ? 0 : rd + 1;
    wr = wr + 1 == RING ? 0 : wr + 1;
  }
  wait_dma();
  sync_threads();

  // ---- the groups' partial sums: group 0 finishes the row fragments [0, N0), group 1 the rest.  Plane (fragment,
  // strip) of the exchange is [NF x 4][64 lanes] of four accumulators; a wave reads only what its partner left for it.
  constexpr int N0 = (NFR + 1) / 2, N1 = NFR / 2;
  f32x4_t *ex = (f32x4_t *)lds;
  constexpr int PLANE = NF * 4 * kWave;
  auto put = [&](int i) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        ex[(i * 4 + wave) * PLANE + (f * 4 + j) * kWave + lane] =
            f32x4_t{acc[i][f][4 * j], acc[i][f][4 * j + 1], acc[i][f][4 * j + 2], acc[i][f][4 * j + 3]};
  };
  auto take = [&](int i, f32x16_t (&to)[NF]) {   // (group 0's part first, whichever group adds)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4_t v = ex[(i * 4 + wave) * PLANE + (f * 4 + j) * kWave + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) to[f][4 * j + e] += v[e];
      }
  };
  constexpr int FAST = FP8 ? TAMD_BF16 : XDT;
  if (grp == 0) {
#pragma unroll
    for (int i = N0; i < NFR; ++i) put(i);
  } else {
#pragma unroll
    for (int i = 0; i < N0; ++i) put(i);
  }
  sync_threads();
  if (grp == 0) {
    f32x16_t mine[N0][NF];
#pragma unroll
    for (int i = 0; i < N0; ++i) {
#pragma unroll
      for (int f = 0; f < NF; ++f) mine[i][f] = acc[i][f];
      take(i, mine[i]);
    }
    Tile t0 = t;
    t0.rows = t.rows < 32 * N0 ? t.rows : 32 * N0;
    tile_epilogue<N0, ACT, FAST, FP8>(kernel_args_late(), t0, mine, lds + wave * PLANE * 16);   // (its plane has been read)
  } else {
    if constexpr (N1 > 0) {
      f32x16_t mine[N1][NF];
#pragma unroll
      for (int i = 0; i < N1; ++i) {
#pragma unroll
        for (int f = 0; f < NF; ++f) mine[i][f] = acc[N0 + i][f];
        take(N0 + i, mine[i]);
      }
      Tile t1 = t;
      t1.off_m = t.off_m + 32 * N0;
      t1.rows = t.rows - 32 * N0;
      tile_epilogue<N1, ACT, FAST, FP8>(kernel_args_late(), t1, mine, lds + (N0 * 4 + wave) * PLANE * 16);
    }
  }
}

// ONCE: weights are copied non-temporally (a slice of more than one row block reads them again).
template <int XDT, int BM, int ACT, bool ONCE>
__global__ __launch_bounds__(512, 1) void mm_kk_kernel(tamd_matmul_args a, int grid_n, int64_t grid_total, int group_m) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  typedef TileShape<XDT, BM> S;
  Tile t;
  if (S::EXTRA > 0 && group_m < 0) {
    if (!locate_tile_live<BM, S::EXTRA>(a, grid_n, -group_m, t)) return;
  } else if (!locate_tile<BM, S::EXTRA>(a, grid_n, grid_total, group_m, t)) return;
  const int nfr = (t.rows + 31) / 32;
#define TAMD_CASE(n)                                                         \
  case n:                                                                    \
    if constexpr (n <= S::MF) run_tile_kk<XDT, n, BM, ACT, ONCE>(a, t, lds); \
    break;
  switch (nfr) { TAMD_CASE(1) TAMD_CASE(2) TAMD_CASE(3) TAMD_CASE(4) TAMD_CASE(5) }
#undef TAMD_CASE
}

// ---- Few tiles: 32 rows x 64 columns, K split over the workgroup's four waves.
// A problem of few rows has ceil(N / 256) tiles per row block; with fewer tiles than CUs the chip idles while each tile's
// K loop streams 256 columns through one CU (10 x 6496 x 3096: 13 tiles of 3.3 MB each, 54 us; now 19).  Here a tile is one 64-column
// strip, and a wave has a quarter of K to itself: its copies go through a ring of its own (three stages of up to 12 KB), so
// the loop has no barrier; the partial sums meet in LDS, added in the order of the waves.  Bound by the copies a wave can
// issue (27 x 6912 x 8192: twelve copies of 8 lines per stage, 157 cycles of a wave's life for each; the address units of the CUs
// at work are busy 57 % of the time, their matrix cores 9 %): NA, the row copies of a stage, follows the tile's rows.
template <int NA>
struct NarrowShape {
  static constexpr int A_LINES = 8 * NA, STAGE = (A_LINES + 64) * 128, RING = 3;
};
constexpr int kNarrowLds = 4 * NarrowShape<4>::RING * NarrowShape<4>::STAGE;
static_assert(kNarrowLds <= 160 * 1024, "one workgroup per CU");

template <int XDT, int NA, int ACT>
TAMD_DEVICE void run_tile_narrow(const tamd_matmul_args &a, const Tile &t, uint8_t *lds) {
  typedef KK<XDT> O;
  typedef typename O::frag_t frag_t;
  typedef NarrowShape<NA> S;
  constexpr bool FP8 = KK<XDT>::FP8;
  constexpr int ESZ = KK<XDT>::ESZ, KS = KK<XDT>::KS, EPC = 16 / ESZ;
  constexpr int RING = S::RING, STAGE = S::STAGE, NB = 8;
  constexpr uint32_t kOob = 0x7FFFFFFFu;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int c32 = lane % 32, h = lane / 32;
  const int K = a.K, N = a.N;
  const v4i_t rx = make_rsrc((const uint8_t *)a.x + (int64_t)t.z * a.x_stride_z * ESZ, kOob);
  const v4i_t rw = make_rsrc((const uint8_t *)a.w + (int64_t)t.expert * a.w_stride_e * ESZ, kOob);
  uint8_t *ring = lds + wave * (RING * STAGE);
  const uint32_t ring_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)ring;
  // the wave's stages: [first, first + n_w) of the problem's n_k, the same number for every wave
  const int n_k = (K + KS - 1) / KS, n_w = (n_k + 3) / 4, first = wave * n_w;
  // copy u of an operand moves its lines 8u .. 8u + 7, lane -> (line 8u + lane / 8, slot lane % 8); slot s of line r holds
  // chunk s ^ ((r >> 1) & 7)
  const int rin = lane / 8;
  const int chunk[2] = {(lane % 8) ^ (rin >> 1), (lane % 8) ^ (4 + (rin >> 1))};   // even, odd copies
  uint32_t a_off[NA], b_off[NB];
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    const int r = u * 8 + rin;
    const int rr = t.off_m + (r < t.rows ? r : t.rows - 1);
    const uint32_t src = a.gather_indx ? (uint32_t)a.gather_indx[t.start_m + rr] : (uint32_t)(t.start_m + rr);
    a_off[u] = r < t.rows ? src * (uint32_t)(a.x_stride_m * ESZ) + chunk[u & 1] * 16 : kOob;
  }
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int p = u * 8 + rin;                          // position 32 f + c holds column 2 c + f
    const int col = t.n0 + 2 * (p % 32) + p / 32;
    b_off[u] = col < N ? (uint32_t)col * (uint32_t)(a.w_stride_n * ESZ) + chunk[u & 1] * 16 : kOob;
  }
  auto issue = [&](int it, int slot) {   // (chunks past K, and stages past the wave's own, are not read: zeros)
    const int kb = (first + it) * KS;
    const uint32_t kill[2] = {it < n_w && kb + chunk[0] * EPC < K ? 0u : kOob, it < n_w && kb + chunk[1] * EPC < K ? 0u : kOob};
    const uint32_t sa = ring_base + slot * STAGE, sb = sa + S::A_LINES * 128;
#pragma unroll
    for (int u = 0; u < NA; ++u) dma16(rx, sa + u * 1024, a_off[u] | kill[u & 1], kb * ESZ);
#pragma unroll
    for (int u = 0; u < NB; ++u) dma16(rw, sb + u * 1024, b_off[u] | kill[u & 1], kb * ESZ);
  };
  f32x16_t acc[1][NF];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[0][f][j] = 0.f;
  // (rows past the tile's lines repeat earlier ones: their results are not stored)
  const int a_line = c32 & (S::A_LINES - 1), a_swz = (a_line >> 1) & 7, b_swz = (c32 >> 1) & 7;
  const int a_lane = a_line * 128, b_lane = (S::A_LINES + c32) * 128;
#pragma unroll
  for (int s = 0; s < RING - 1; ++s) issue(s, s);
  int rd = 0, wr = RING - 1;
#pragma unroll 1
  for (int it = 0; it < n_w; ++it) {
    wait_vmcnt<(RING - 2) * (NA + NB)>();   // copies complete in the order of their requests: stage `it` has landed
    const uint8_t *buf = ring + rd * STAGE;
    uint4 av[4], bv[NF][4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int ch = 4 * h + c;   // (lanes 0-31 take chunks 0 .. 3, the others 4 .. 7)
      av[c] = *(const uint4 *)(buf + a_lane + (ch ^ a_swz) * 16);
#pragma unroll
      for (int f = 0; f < NF; ++f) bv[f][c] = *(const uint4 *)(buf + b_lane + f * 4096 + (ch ^ b_swz) * 16);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // everything read so far is in registers: the slot of stage it - 1 is free
    issue(it + RING - 1, wr);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int s = 0; s < O::STEPS; ++s) {
        const frag_t ai = O::operand(av[c], s);
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[0][f] = O::M::mma(ai, O::operand(bv[f][c], s), acc[0][f]);
      }
    rd = rd + 1 == RING ? 0 : rd + 1;
    wr = wr + 1 == RING ? 0 : wr + 1;
  }
  wait_dma();
  sync_threads();   // every ring is dead
  f32x4_t *ex = (f32x4_t *)lds;
  constexpr int PLANE = NF * 4 * kWave;
  if (wave > 0) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        ex[wave * PLANE + (f * 4 + j) * kWave + lane] =
            f32x4_t{acc[0][f][4 * j], acc[0][f][4 * j + 1], acc[0][f][4 * j + 2], acc[0][f][4 * j + 3]};
  }
  sync_threads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 1; w < 4; ++w)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4_t v = ex[w * PLANE + (f * 4 + j) * kWave + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[0][f][4 * j + e] += v[e];
      }
  constexpr int FAST = FP8 ? TAMD_BF16 : XDT;
  tile_epilogue<1, ACT, FAST, FP8>(kernel_args_late(), t, acc, lds);   // (plane 0 was not used)
}

template <int XDT, int BM, int ACT>
__global__ __launch_bounds__(256, 1) void mm_kk_narrow_kernel(tamd_matmul_args a, int grid_n, int64_t grid_total, int group_m) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  Tile t;
  if (!locate_tile<BM, 0>(a, grid_n, grid_total, group_m, t)) return;
  t.n0 /= 4;   // 64-column tiles
  if (t.rows <= 8) run_tile_narrow<XDT, 1, ACT>(a, t, lds);
  else if (t.rows <= 16) run_tile_narrow<XDT, 2, ACT>(a, t, lds);
  else run_tile_narrow<XDT, 4, ACT>(a, t, lds);
}

template <int XDT, int BM, int ACT>
int launch_kk(const tamd_matmul_args &a, int grid_m, hipStream_t st) {
  const int grid_n = (a.N + BLOCK_N - 1) / BLOCK_N;
  const int64_t total = (int64_t)grid_m * grid_n;
  if (total <= 0) return 0;
  const int64_t launch = ((total + 7) / 8) * 8;
  if (launch > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
  // row blocks walked together (see launch_x16_act)
  const int64_t rows_per_slice = a.block_schedule ? a.M / a.n_experts : a.M;
  int64_t group_m = (rows_per_slice + BM - 1) / BM;
  group_m = group_m < 1 ? 1 : (group_m > 8 ? 8 : group_m);
  if constexpr (BM <= 32) {
    // Narrow tiles where their rounds of a quarter of K, and about eight stages of start and finish each, are less than the
    // K loop of a wide tile.  (5472 x 5760 and 2880 x 5472, one row for each of 3 experts: layer 132 us wide, 78 narrow; K of
    // 576, four rows x 7752 columns: 8.3 us wide, 10.2 narrow.)
    int cus = 0;
    if (int rc = cu_count(cus)) return rc;
    const int grid64 = (a.N + 63) / 64;
    const int64_t n_k = (a.K + KK<XDT>::KS - 1) / KK<XDT>::KS;
    const int64_t rounds = ((int64_t)grid_m * grid64 + cus - 1) / cus;
    if (total < cus && rounds * (n_k + 32) < 4 * n_k) {
      auto narrow = mm_kk_narrow_kernel<XDT, BM, ACT>;
      if (int rc = raise_lds_limit_once((const void *)narrow)) return rc;
      const int64_t tiles = (int64_t)grid_m * grid64;
      narrow<<<dim3((unsigned)((tiles + 7) / 8 * 8)), 256, kNarrowLds, st>>>(a, grid64, tiles, 1);
      return launch_status();
    }
  }
  // 16-bit weights of slices that hardly ever need two row blocks are copied non-temporally where their columns are whole lines and a call
  // reads more of them (320 MB) than the 256 MB behind the L2s keep for the next one.  Of what the persistent kernel leaves here, us, ordinary
  // copies -> these: float32 outputs, K 2880, 1200 rows of 32 slices, N 5760 203 -> 192, N 2880 118 -> 108, 64 rows, N 5760 180 -> 161 (6.6 TB/s);
  // 300 slices, K and N 1024, 300 rows 76 -> 66, 3000 rows 119 -> 108; dense, 8192 x 28672, 16 rows 115 -> 110, 64 rows 131 -> 130 (8192 x 24576
  // 110 -> 111).  Below 320 MB 1.0 to 1.5 of the time, with lines that two stages share 1.08 (0.95 to 1.3).
  auto kern = mm_kk_kernel<XDT, BM, ACT, false>;
  if constexpr (!KK<XDT>::FP8) {
    const bool lines = aligned(a.w, 128) && (a.w_stride_n * 2) % 128 == 0 && (a.w_stride_e * 2) % 128 == 0;
    if (lines && 4 * rows_per_slice <= 3 * BM && live_slices(a) * a.N * ((double)a.K * 2) >= 320.0 * (1 << 20))
      kern = mm_kk_kernel<XDT, BM, ACT, true>;
  }
  if (int rc = raise_lds_limit_once((const void *)kern)) return rc;
  // (one workgroup per CU: an XCD holds 32 tiles, and an expert's blocks share a column tile only side by side; 32 experts
  // of 250 bf16 rows, 2880 x 2880: 181 us in fours, 199 one after the other, 217 in schedule order)
  if (TileShape<XDT, BM>::EXTRA > 0 && counts_live_blocks(a) && group_m <= 2) group_m = -4;
  kern<<<dim3((unsigned)launch), 512, KKShape<XDT, BM>::LDS, st>>>(a, grid_n, total, (int)group_m);
  return launch_status();
}

int kk_ring_mm_bf16(const tamd_matmul_args &a, int rows, hipStream_t st);
int kk_ring_mm_f16(const tamd_matmul_args &a, int rows, hipStream_t st);

// Both operands contiguous along K, 16-byte aligned rows and columns, whole 16-byte chunks along K, and offsets inside
// an operand below 2 GB: anything else is refused (TAMD_E_UNSUPPORTED / _ALIGNMENT).
template <int XDT>
int dispatch_kk(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  constexpr int ESZ = KK<XDT>::ESZ;
  dense_grid(a, block_m, grid_m);
  if (a.w_stride_k != 1 || a.K % (16 / ESZ) != 0) return TAMD_E_UNSUPPORTED;
  if (!aligned(a.w, 16) || (a.w_stride_n * ESZ) % 16 != 0 || (a.w_stride_e * ESZ) % 16 != 0) return TAMD_E_ALIGNMENT;
  if (!aligned(a.x, 16) || (a.x_stride_m * ESZ) % 16 != 0 || (a.x_stride_z * ESZ) % 16 != 0) return TAMD_E_ALIGNMENT;
  const int64_t x_rows = a.x_rows > 0 ? a.x_rows : a.M, lim = 0x7FFFFF00;
  if (x_rows * a.x_stride_m * ESZ >= lim || (int64_t)a.N * a.w_stride_n * ESZ >= lim) return TAMD_E_UNSUPPORTED;
  if constexpr (!KK<XDT>::FP8) {
    if (known_block(block_m) && kk_ring_applicable(a)) {
      int cus = 0;
      if (int rc = cu_count(cus)) return rc;
      if (const int rows = kk_ring_rows(a, cus)) return XDT == TAMD_BF16 ? kk_ring_mm_bf16(a, rows, st) : kk_ring_mm_f16(a, rows, st);
    }
  }
  const bool sw = a.activation == TAMD_ACT_SWIGLU;
  switch (block_m) {
    case 16: return sw ? launch_kk<XDT, 16, TAMD_ACT_SWIGLU>(a, grid_m, st) : launch_kk<XDT, 16, TAMD_ACT_NONE>(a, grid_m, st);
    case 32: return sw ? launch_kk<XDT, 32, TAMD_ACT_SWIGLU>(a, grid_m, st) : launch_kk<XDT, 32, TAMD_ACT_NONE>(a, grid_m, st);
    case 64: return sw ? launch_kk<XDT, 64, TAMD_ACT_SWIGLU>(a, grid_m, st) : launch_kk<XDT, 64, TAMD_ACT_NONE>(a, grid_m, st);
    case 128: return sw ? launch_kk<XDT, 128, TAMD_ACT_SWIGLU>(a, grid_m, st) : launch_kk<XDT, 128, TAMD_ACT_NONE>(a, grid_m, st);
    default: return TAMD_E_UNSUPPORTED;
  }
}

}  // namespace tamd
