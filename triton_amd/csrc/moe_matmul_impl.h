// Grouped (ragged-M) / dense matmul for gfx950: 16-bit activations x MXFP4 weights, and what every tiled kernel shares.
//
//   y[dst(r), :] = act(((x[src(r), :] . deq(w[e])) * sx * sw + bias[e, :] * beta[r]) * alpha) * gamma[r]
//
// (matmul_details/_matmul.py:43-669 of the reference; epilogue order :540-559.)
//
// Work decomposition
//   workgroup (4 waves) = one BLOCK_M x 256 output tile of one expert, taken from the ragged
//     block schedule ((block << 16) | expert, -1 = padding);
//   wave w owns the 64 columns [64w, 64w+64) of the tile and ALL its rows;
//   both operands travel HBM -> LDS by 16-byte DMA (buffer_load ... lds): activation rows (gathered)
//     in 128-byte stages, double buffered, chunks XOR-swizzled by row; the weights of a wave's own
//     columns into a wave-private region, 128 K per stage.
//   bf16 / f16 activations: the fp4 codes are expanded in registers with v_cvt_scalef32_pk_*_fp4
//     (scale applied by the instruction) and feed v_mfma_f32_32x32x16, which sustains twice the rate
//     of 16x16x32 on this part (measured 2.45 vs 1.25 PFLOP/s for bf16).
//   (fp8 and packed activations: moe_matmul_mx.h.)
//
// K order inside a 128-K weight stage: lane half h = lane/32 holds K [64q + 32h, 64q + 32h + 32) of
// its column for q = 0, 1 (two 128-bit LDS reads); MFMA step s = 4q + u consumes elements [8u, 8u+8) of load q in
// both halves, for A and B alike.
#pragma once
#include <type_traits>

#include "common.h"

namespace tamd {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr bool is_fp8(int dt) { return dt == TAMD_FP8_E4M3 || dt == TAMD_FP8_E5M2; }

constexpr int KB = 128;  // K per weight (super-)stage
constexpr int NF = 2;              // 32-column fragments per wave
constexpr int BLOCK_N = 4 * 32 * NF;

template <int XDT>
struct Mma;
template <>
struct Mma<TAMD_BF16> {
  typedef bf16x8_t frag_t;
  static TAMD_DEVICE frag_t expand(uint32_t codes, float scale) {
    bf16x2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, scale, 0);
    bf16x2_t p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, scale, 1);
    bf16x2_t p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, scale, 2);
    bf16x2_t p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, scale, 3);
    return frag_t{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
  }
  static TAMD_DEVICE f32x16_t mma(frag_t a, frag_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mma<TAMD_F16> {
  typedef f16x8_t frag_t;
  static TAMD_DEVICE frag_t expand(uint32_t codes, float scale) {
    f16x2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(codes, scale, 0);
    f16x2_t p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(codes, scale, 1);
    f16x2_t p2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(codes, scale, 2);
    f16x2_t p3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(codes, scale, 3);
    return frag_t{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
  }
  static TAMD_DEVICE f32x16_t mma(frag_t a, frag_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

TAMD_DEVICE float load_any_f32(const void *p, int dt, int64_t i) {
  if (dt == TAMD_F32) return ((const float *)p)[i];
  if (dt == TAMD_BF16) return bf16_bits_to_f32(((const uint16_t *)p)[i]);
  return f16_bits_to_f32(((const uint16_t *)p)[i]);
}

TAMD_DEVICE void store_any(void *p, int dt, int64_t i, float v) {
  if (dt == TAMD_F32) ((float *)p)[i] = v;
  else if (dt == TAMD_BF16) ((uint16_t *)p)[i] = (uint16_t)f32_to_bf16_bits(v);
  else ((uint16_t *)p)[i] = (uint16_t)f32_to_f16_bits(v);
}

// Gate for the fused epilogue (swiglu_details/_swiglu.py:55-65): exp and reciprocal on the
// hardware transcendental unit (relative error ~1e-6, far inside the 16-bit output rounding).
TAMD_DEVICE float swiglu_fast(float g, float l, float alpha, float limit, bool has_limit) {
  if (has_limit) {
    g = __builtin_fminf(g, limit);
    l = __builtin_fminf(__builtin_fmaxf(l, -limit), limit);
  }
  float e = __builtin_amdgcn_exp2f(-alpha * 1.4426950408889634f * g);
  float s = g * __builtin_amdgcn_rcpf(1.0f + e);
  return __builtin_fmaf(s, l, s);
}

// Tile coordinates of a workgroup.
struct Tile {
  int expert;   // weight slice
  int z;        // batch index (dense batched) else 0
  int start_m;  // first expert-sorted row of the slice
  int off_m;    // first row of the tile inside the slice
  int rows;     // valid rows in the tile (1..BLOCK_M)
  int n0;       // first column of the tile
};

template <int BLOCK_M, int EXTRA>
TAMD_DEVICE bool locate_tile(const tamd_matmul_args &a, int grid_n, int64_t grid_total, int group_m, Tile &t) {
  // XCD-aware remap: hardware deals workgroups round-robin to the 8 XCDs; give each XCD a
  // contiguous range of tiles so neighbours (same expert, adjacent columns) share one L2.
  // A ragged launch is sized for the worst split of the rows over the experts (grid_total), about twice what a
  // balanced routing needs; the schedule's real entries come first and their number is block_offs[n_experts].  The
  // XCD ranges are cut from that number, read here, so that all eight XCDs share the real tiles; the rest exit.
  // (the launchers keep a grid below 2^31 tiles: 32-bit unsigned arithmetic, whose divisions cost a third of the 64-bit ones)
  uint32_t total = (uint32_t)grid_total;
  const uint32_t gn = (uint32_t)grid_n;
  if (a.block_schedule && a.block_offs) {
    const uint64_t real_total = (uint64_t)(uint32_t)a.block_offs[a.n_experts] * gn;
    total = real_total < total ? (uint32_t)real_total : total;
  }
  const uint32_t per_xcd = (total + 7) / 8;
  const uint32_t bx = blockIdx.x;
  if (bx / 8 >= per_xcd) return false;
  const uint32_t pid = (bx % 8) * per_xcd + bx / 8;
  if (pid >= total) return false;
  // Tiles are walked in groups of `group_m` row blocks: row block fastest inside a group, then the
  // column tile.  With many row blocks per expert the workgroups running together then share one
  // column tile of weights while the group's activation rows stay in L2; group_m = 1 is the plain
  // row-block-major order (right when an expert has only a block or two).
  int pid_m, pid_n;
  if (group_m > 1) {
    const uint32_t gm = (uint32_t)group_m;
    const uint32_t grid_m = total / gn;
    const uint32_t in_group = gm * gn;
    const uint32_t gi = pid / in_group;
    const uint32_t first_m = gi * gm;
    const uint32_t size_m = grid_m - first_m < gm ? grid_m - first_m : gm;
    const uint32_t r = pid - gi * in_group;
    const uint32_t q = r / size_m;
    pid_m = (int)(first_m + (r - q * size_m));
    pid_n = (int)q;
  } else {
    const uint32_t q = pid / gn;
    pid_m = (int)q;
    pid_n = (int)(pid - q * gn);
  }
  t.n0 = pid_n * BLOCK_N;
  t.z = 0;
  int slice_rows;
  if (a.block_schedule) {
    int sched = a.block_schedule[pid_m];
    if (sched == -1) return false;
    t.expert = sched & 0xFFFF;
    int blk = sched >> 16;
    slice_rows = a.slice_sizes[t.expert];
    t.start_m = a.slice_offs[t.expert];
    t.off_m = blk * BLOCK_M;
  } else {
    int bm = (a.M + BLOCK_M - 1) / BLOCK_M;
    int z = pid_m / bm;
    t.expert = z;
    t.z = z;
    slice_rows = a.M;
    t.start_m = 0;
    t.off_m = (pid_m - z * bm) * BLOCK_M;
  }
  // A 128-row block also takes a remainder of up to 32 rows that follows it (one more 32-row
  // fragment), and that remainder's own block does nothing: with about 128 rows per expert this
  // avoids a second, nearly empty pass over the expert's weights.
  const int left = slice_rows - t.off_m;
  if (EXTRA > 0 && t.off_m > 0 && left <= EXTRA) return false;
  t.rows = left > BLOCK_M + EXTRA ? BLOCK_M : left;
  return t.rows > 0;
}

// Tile of a workgroup of a ragged problem, from the slices' sizes alone: one round trip to memory where the schedule takes three
// (its length, the entry, the slice), each about 0.8 us of a tile that may last 10 (with the row indices requested before the
// first weights, see run_tile: 333 tokens over 32 experts, 2016 -> 2112, f16, layer 83.4 us -> 81.3).
// Blocks that absorb remainders (EXTRA > 0) leave the absorbed ones out: at 128 rows per expert they are a third of the schedule,
// and XCD ranges of equal numbers of its entries leave the XCDs with unequal work (32 experts, 2880 x 2880, 128 bf16 rows
// each: 98 us, 76 so).  The ranges are in expert order; up to `group` blocks of an expert run next to each other on
// a column tile.  (XCD ranges of equal estimated time with the longest tiles first take 2 us to find and read an expert's
// weights once per block: 128 experts, 200 rows each, 2880 x 2880: 462 us against 414, fp8 rows 387 against 293 in plain order.
// Where a launch is one to three rounds of tiles they win up to 7 % (32 experts of 160 bf16 rows, 2880 x 5760: 179 against 190),
// but over 16 to 128 experts of 40 to 250 rows they lose 6 %.)
//
// Every wave finds the tile by itself, without LDS or barriers and with one round trip to memory: lane l holds the experts
// [l n, (l + 1) n), n = ceil(experts / 64) up to kLivePerLane, and a scan over the lanes counts the blocks before them.
constexpr int kLivePerLane = 8;
template <int BLOCK_M, int EXTRA>
TAMD_DEVICE bool locate_tile_live(const tamd_matmul_args &a, int grid_n, int group, Tile &t) {
  const int lane = threadIdx.x % kWave, E = a.n_experts, n_lane = (E + kWave - 1) / kWave;
  const uint32_t gn = (uint32_t)grid_n;
  int rows[kLivePerLane], offs[kLivePerLane];
#pragma unroll
  for (int u = 0; u < kLivePerLane; ++u) {
    rows[u] = offs[u] = 0;
    if (u == 0 || u < n_lane) {   // (wave uniform)
      const int e = lane * n_lane + u;
      if (e < E) rows[u] = a.slice_sizes[e], offs[u] = a.slice_offs[e];
    }
  }
  // (a block that starts past the first needs more than EXTRA rows)
  auto blocks = [](int n) { return n > BLOCK_M ? (n - EXTRA + BLOCK_M - 1) / BLOCK_M : (n > 0 ? 1 : 0); };
  int own = blocks(rows[0]);
#pragma unroll
  for (int u = 1; u < kLivePerLane; ++u)
    if (u < n_lane) own += blocks(rows[u]);
  const int incl = wave_incl_scan(own);
  const uint32_t total = (uint32_t)__builtin_amdgcn_readlane(incl, kWave - 1) * gn;
  const uint32_t per_xcd = (total + 7) / 8, bx = blockIdx.x;
  const uint32_t idx = (bx % 8) * per_xcd + bx / 8;
  if (bx / 8 >= per_xcd || idx >= total) return false;
  const int m = (int)(idx / gn);                     // the m-th block that has rows
  int first = incl - own, e = 0, n = 0, off = 0, before = 0;
  bool here = false;
#pragma unroll
  for (int u = 0; u < kLivePerLane; ++u) {
    if (u > 0 && u >= n_lane) continue;
    const int c = blocks(rows[u]);
    if (m >= first && m < first + c) here = true, e = lane * n_lane + u, n = rows[u], off = offs[u], before = first;
    first += c;
  }
  const int src = __builtin_ctzll(__ballot(here));   // (exactly one lane)
  t.expert = __builtin_amdgcn_readlane(e, src);
  t.start_m = __builtin_amdgcn_readlane(off, src);
  const int slice_rows = __builtin_amdgcn_readlane(n, src);
  const uint32_t local = idx - (uint32_t)__builtin_amdgcn_readlane(before, src) * gn;   // tile of the expert
  const uint32_t b = (uint32_t)blocks(slice_rows);
  uint32_t g = b < (uint32_t)group ? b : (uint32_t)group, blk, col;
  if (g > 1) {
    g = (b + (b + g - 1) / g - 1) / ((b + g - 1) / g);   // (groups of about one size)
    const uint32_t gi = local / (g * gn), r = local - gi * g * gn;
    const uint32_t size = b - gi * g < g ? b - gi * g : g;
    col = r / size;
    blk = gi * g + (r - col * size);
  } else {
    blk = local / gn;
    col = local - blk * gn;
  }
  t.n0 = (int)col * BLOCK_N;
  t.z = 0;
  t.off_m = (int)blk * BLOCK_M;
  const int left = slice_rows - t.off_m;
  t.rows = left > BLOCK_M + EXTRA ? BLOCK_M : left;
  return true;
}

// What a row of x is below: the rows that a gathered index can name.  An index outside of them (-1) names none: the row is read as
// zeros, by the buffer descriptors where the address leaves their 2 GB, and by this limit where loads have no descriptor.
template <typename Args>
TAMD_DEVICE uint32_t gather_limit(const Args &a) {
  const int64_t rows = a.x_rows > 0 ? a.x_rows : (int64_t)a.M;
  return a.gather_indx && rows < 0x80000000ll ? (uint32_t)rows : 0x80000000u;
}

// 128-bit global -> LDS copy that bypasses registers (buffer_load ... lds).  The LDS destination of
// lane L is lds_addr + 16*L; out-of-range offsets (>= num_records of the descriptor) deliver zeros.
// Issued through inline asm so that the compiler does not serialise later LDS reads behind it; the
// kernel waits for these copies itself (wait_dma) before the barrier that publishes a stage.  The
// five wait states cover an SGPR operand written by a v_readfirstlane just before the block (the
// compiler's hazard recognizer does not look inside inline asm) and the write of M0.
typedef int v4i_t __attribute__((ext_vector_type(4)));
TAMD_DEVICE void dma16(v4i_t rsrc, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(rsrc),
                 "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory", "m0");
}
// The same for data that is read once (non-temporal).
TAMD_DEVICE void dma16_nt(v4i_t rsrc, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(rsrc),
                 "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory", "m0");
}
// 2- and 4-byte global -> LDS copies: lane L's value lands (zero-extended) in the dword at
// lds_addr + 4*L; out-of-range offsets deliver zero.  The five wait states before the load cover an
// SGPR operand that a v_readfirstlane wrote just before the asm block (the compiler's hazard
// recognizer does not look inside inline asm) as well as the write of M0.
TAMD_DEVICE void dma2(v4i_t rsrc, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_ushort %1, %2, %3 offen lds"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(rsrc),
                 "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory", "m0");
}
TAMD_DEVICE void dma4(v4i_t rsrc, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dword %1, %2, %3 offen lds"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(rsrc),
                 "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory", "m0");
}
// Four consecutive 1 KB pieces of a linear image with ONE M0 value: the instruction's immediate offset is added to the
// global offset and to the LDS address alike.
TAMD_DEVICE void dma16_x4(v4i_t rsrc, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
  asm volatile(
      "s_mov_b32 m0, %0\n\ts_nop 4\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen lds\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen offset:1024 lds\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen offset:2048 lds\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen offset:3072 lds"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(soff))
      : "memory", "m0");
}
// The same for data that is read once (non-temporal).
TAMD_DEVICE void dma16_x4_nt(v4i_t rsrc, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
  asm volatile(
      "s_mov_b32 m0, %0\n\ts_nop 4\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen nt lds\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen offset:1024 nt lds\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen offset:2048 nt lds\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen offset:3072 nt lds"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voff), "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(soff))
      : "memory", "m0");
}
TAMD_DEVICE void wait_dma() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding).
template <int N>
TAMD_DEVICE void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
  asm volatile("" ::: "memory");
}

TAMD_DEVICE v4i_t make_rsrc(const void *base, uint32_t num_records) {
  uint64_t p = (uint64_t)base;
  return v4i_t{__builtin_amdgcn_readfirstlane((int)(uint32_t)p),
               __builtin_amdgcn_readfirstlane((int)((uint32_t)(p >> 32) & 0xFFFFu)), (int)num_records, 0x00020000};
}

constexpr int A_ROW_BYTES = 128;       // LDS bytes per activation row per stage (64 K of 16-bit values)
constexpr int B_BYTES = 4 * 64 * 64;   // 4 waves x 64 columns x 64 bytes (128 K of fp4)
// LDS of the K pipeline.  Row blocks of 128: two activation stages, one weight stage (4 KB per wave), the e8m0 scales
// of the whole tile staged once.  Row blocks of at most 32 (KS = 1): the counted waits and stages of one of two K groups.
// K groups (KS = 2 on tiles of four strips, 8 on tiles of two; row blocks of at most 32 rows): KS groups of a wave per strip share a tile,
// each taking a contiguous part of K through a pipeline of its own with counted waits, four activation stages and two weight stages (two
// and one); their partial sums meet in LDS.  A problem with fewer tiles than the part has CUs is bound by what one wave per SIMD can issue
// (a copy instruction holds its wave for about a hundred cycles); more waves per SIMD fill those gaps.
struct PipeShape {
  int da, db;        // activation / weight stages
  int bytes;
};
constexpr PipeShape pipe_shape(int lds_rows, int ks = 1, int strips = 4) {
  PipeShape p{};
  const bool deep = ks == 2 || (ks == 1 && lds_rows <= 32);
  p.da = deep ? 4 : 2;
  p.db = deep ? 2 : 1;
  p.bytes = p.da * lds_rows * 128 + p.db * strips * (B_BYTES / 4);
  return p;
}

// Copies that a stage of the counted-wait loop (K groups) may leave in flight.  The requests are made in this order:
// stage j -- the stages before 0 are the loop's prologue -- asks for the activations of stage j + DA - 1 (NA copies)
// and, if j is even, after them for the weights of pair j/2 + DB (NB copies).  A stage needs its own activations and,
// if it is even, its pair's weights; copies complete in the order of their requests, so everything requested after
// the last of those may still be outstanding when the stage begins.
constexpr int ring_outstanding(int DA, int DB, int NA, int NB, bool odd) {
  const int s = 64 + (odd ? 1 : 0);   // any stage in the steady state
  int pos = 0, need_end = 0;
  for (int j = 0; j < s; ++j) {
    pos += NA;
    if (j + DA - 1 == s) need_end = pos;
    if (j % 2 == 0) {
      pos += NB;
      if (!odd && j / 2 + DB == s / 2 && pos > need_end) need_end = pos;
    }
  }
  return pos - need_end;
}
static_assert(ring_outstanding(4, 2, 1, 4, false) == 6 && ring_outstanding(4, 2, 1, 4, true) == 10, "ring bookkeeping");
static_assert(ring_outstanding(3, 2, 2, 4, false) == 6 && ring_outstanding(3, 2, 2, 4, true) == 6, "ring bookkeeping");
static_assert(ring_outstanding(2, 1, 2, 4, false) == 0 && ring_outstanding(2, 1, 2, 4, true) == 4, "ring bookkeeping");

// Flexpoint actual scale: the wave's max|result| by one atomic; positive floats order like their bit patterns.
TAMD_DEVICE void store_actual_scale(float *actual, uint32_t amax, float out_max, int lane) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t other = (uint32_t)__shfl_xor((int)amax, o);
    amax = other > amax ? other : amax;
  }
  if (lane == 0) {
    amax = amax < 0x7F800000u ? amax : 0x7F800000u;  // NaN counts as +inf
    atomicMax((unsigned int *)actual, f32_to_bits(__builtin_fmaf(bits_to_f32(amax), 1.0f / out_max, 1.0e-30f)));
  }
}

// Epilogue of one output tile (shared by every tiled kernel).  The accumulators hold, for fragment
// (i, f), element j: row 32i + 8(j/4) + 4h + j%4, column t.n0 + wave*64 + c32*NF + f.
//
// A wave finishes its 64 columns by itself: the destination of each of the tile's rows (a byte offset into y; out of
// range for a row that is not stored) and the rows' factors go into a table of the wave's own in LDS, from which four
// consecutive rows are read at a time by a broadcast; every element is then computed and stored from registers, a row's
// 32 lanes writing 32 consecutive outputs (one half or whole line of a 16-bit type).  Nothing is masked by control flow:
// a store whose offset is out of range is dropped by the buffer descriptor.  There is no barrier either, so waves
// leave the tile one by one.  (Staging the tile through LDS for 16-byte stores, as before, took a fifth to a
// quarter of a tile's time: two barriers, a pass of narrow LDS writes and a copy-out between them.)
//
// YDT: output type, or a width whose type is read at run time (kAny8, kAny16; float32 is one of its own); ROWSC: per-row
// betas / gammas may be present; FLEX: flexpoint output (expected / actual scale) may be present; MXO: MXFP8 output
// (a.y_mx_scale).  The element loops must unroll completely (the accumulators are indexed by them and would otherwise live in
// scratch memory).
// pairs: a lane's two outputs lie whole on one aligned word, which is stored at once (only read by the forms of one width;
// the others are entered with such outputs).
// ready: the operands whose table is written already, or null.  pace: called after every four rows of a lane.
// Args: tamd_matmul_args, or the same structure read in place from the kernel-argument segment (see kernel_args_late).
// tab: LDS that belongs to the wave alone, epilogue_table_bytes(NFR).
struct NoPace {
  TAMD_DEVICE void operator()() const {}
};
// Two float32 in range (or NaN) -> e4m3fn bytes in the low or high half of `into`.
template <bool HIGH>
TAMD_DEVICE uint32_t e4m3_pair_bits(float lo, float hi, uint32_t into) {
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(lo, hi, (int)into, HIGH);
}
constexpr int epilogue_table_bytes(int nfr) { return nfr * 32 * 16; }
// Maximum over a lane's aligned group of 32 / NO lanes, by moves in the register file (mirrored lanes serve once the blocks of four and
// eight hold one value; for 32 the rows of 16 lanes change places).
template <int NO>
TAMD_DEVICE uint32_t group_max_lanes(uint32_t m) {
  auto with = [&](uint32_t other) { m = other > m ? other : m; };
  with((uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
  with((uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xF, 0xF, true));    // quad_perm [2,3,0,1]
  with((uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xF, 0xF, true));   // row_half_mirror
  with((uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x140, 0xF, 0xF, true));   // row_mirror
  if constexpr (NO == 1) {
    const auto r = __builtin_amdgcn_permlane16_swap(m, m, false, false);
    m = r[0] > r[1] ? r[0] : r[1];
  }
  return m;
}

// What the epilogue of a tile reads from memory, as it lies there: a lane's rows of the table (64 u + lane), its columns' bias, the
// per-tensor scales.  Nothing is computed from the values where they are loaded, so that they may be requested long before.
template <int NFR>
struct EpilogueOperands {
  static constexpr int PER_LANE = (NFR + 1) / 2;
  int dst[PER_LANE];
  float beta[PER_LANE], gamma[PER_LANE];
  uint32_t bias[NF];
  float x_scale, w_scale;
};
TAMD_DEVICE uint32_t load_any_bits(const void *p, int dt, int64_t i) {
  return dt == TAMD_F32 ? ((const uint32_t *)p)[i] : (uint32_t)((const uint16_t *)p)[i];
}
TAMD_DEVICE float bits_of_type(uint32_t v, int dt) {
  return dt == TAMD_F32 ? bits_to_f32(v) : (dt == TAMD_BF16 ? bf16_bits_to_f32(v) : f16_bits_to_f32(v));
}
template <int NFR, bool ROWSC, typename Args>
TAMD_DEVICE void epilogue_operands(const Args &a, const Tile &t, EpilogueOperands<NFR> &o) {
  const int wave = (threadIdx.x / kWave) & 3, lane = threadIdx.x % kWave;
#pragma unroll
  for (int u = 0; u < EpilogueOperands<NFR>::PER_LANE; ++u) {
    const int r = u * kWave + lane;
    const int erow = t.start_m + t.off_m + (r < t.rows ? r : t.rows - 1);  // expert-sorted row
    o.dst[u] = a.scatter_indx ? a.scatter_indx[erow] : erow;
    o.beta[u] = o.gamma[u] = 1.0f;
    if constexpr (ROWSC) {
      if (a.betas) o.beta[u] = a.betas[erow];
      if (a.gammas) o.gamma[u] = a.gammas[erow];
    }
  }
  const int col0 = t.n0 + wave * 64 + lane % 32 * NF, last = a.N - 1;
#pragma unroll
  for (int f = 0; f < NF; ++f)
    o.bias[f] = a.bias ? load_any_bits(a.bias, a.bias_dtype, (int64_t)t.expert * a.bias_stride_e + (col0 + f < last ? col0 + f : last)) : 0u;
  o.x_scale = a.x_scale ? *a.x_scale : 1.0f;
  o.w_scale = a.w_scale ? *a.w_scale : 1.0f;
}

// The wave's row table: [rows] destinations (byte offsets into y, out of range for a row that is not stored), [rows] betas, [rows] gammas,
// [rows] destinations of the scales (MXO).
template <int NFR, int OSZ, bool ROWSC, bool MXO, typename Args>
TAMD_DEVICE void epilogue_table(const Args &a, const Tile &t, const int *dsts, const float *betas, const float *gammas, uint8_t *tab) {
  constexpr uint32_t kDrop = 0x80000000u;
  const int lane = threadIdx.x % kWave;
  uint32_t *tab_dst = (uint32_t *)tab;
  float *tab_beta = (float *)tab + NFR * 32, *tab_gamma = (float *)tab + NFR * 64;
#pragma unroll
  for (int u = 0; u < (NFR + 1) / 2; ++u) {
    const int r = u * kWave + lane, dst = dsts[u];
    if (NFR % 2 == 0 || r < NFR * 32) {
      const bool keep = r < t.rows && dst >= 0;
      tab_dst[r] = keep ? (uint32_t)dst * (uint32_t)(a.y_stride_m * OSZ) : kDrop;
      if constexpr (MXO) tab_dst[NFR * 96 + r] = keep ? (uint32_t)dst * (uint32_t)a.y_mx_stride_m : kDrop;
      if constexpr (ROWSC) {
        tab_beta[r] = betas[u];
        tab_gamma[r] = gammas[u];
      }
    }
  }
}

// Four rows of a quad of lanes change places with its columns: lane q ends with what the four lanes hold of row q, in the order of the
// lanes.  A register holds a byte of each row (one column per lane), or 16 bits of two rows each (two columns).
TAMD_DEVICE uint32_t quad_xor1(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true); }
TAMD_DEVICE uint32_t quad_xor2(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true); }
// (The selectors by arithmetic on a constant that the compiler does not see through: as selections between two constants it keeps both
// in vector registers over the tiles of a persistent kernel.)
TAMD_DEVICE uint32_t flip_where(uint32_t base, int bit_mask, uint32_t diff) {
  asm volatile("" : "+s"(diff));
  return base ^ ((uint32_t)bit_mask & diff);
}
TAMD_DEVICE uint32_t quad_rows(uint32_t rows0123, int lane) {
  const uint32_t x = __builtin_amdgcn_perm(quad_xor1(rows0123), rows0123, flip_where(0x06020400u, __builtin_amdgcn_sbfe(lane, 0, 1), 0x05050505u));
  return __builtin_amdgcn_perm(quad_xor2(x), x, flip_where(0x05040100u, __builtin_amdgcn_sbfe(lane, 1, 1), 0x06060606u));
}
TAMD_DEVICE u32x2_t quad_rows(uint32_t rows01, uint32_t rows23, int lane) {
  const uint32_t sel = flip_where(0x05040100u, __builtin_amdgcn_sbfe(lane, 0, 1), 0x06060606u);
  const uint32_t a = __builtin_amdgcn_perm(quad_xor1(rows01), rows01, sel), b = __builtin_amdgcn_perm(quad_xor1(rows23), rows23, sel);
  const bool up = (lane & 2) != 0;
  const uint32_t r = quad_xor2(up ? a : b);
  return up ? u32x2_t{r, b} : u32x2_t{a, r};
}

// Whole quads of lanes, of NO columns each, inside the output, and whole words.
template <int NO, typename Args>
TAMD_DEVICE bool epilogue_stores_quads(const Args &a, int n_out) {
  return n_out % (4 * NO) == 0 && (((uint32_t)(uintptr_t)a.y | (uint32_t)a.y_stride_m | (uint32_t)a.y_stride_z) & 3u) == 0;
}

constexpr int kAny16 = 0x100, kAny8 = 0x101;
// float8_e4m3fn: bounded by flexpoint, without factors, in whole quads (`quads` below), which a layer's rows are: four rows at once without a
// branch; everything else row by row.  Deciding by branches in one form for all took 1.02 to 1.07 of the time of row by row where a CU has one
// tile (700 products of 5 to 12 us; the 4-row form was 1.025 with SwiGLU, as it is now 0.98): blocks of four rows whose latencies no
// other wave hides.  16384 fp8 tokens x 4 of 32, layer 1551 -> 1531 us.
constexpr int kQuads8 = 0x102, kRows8 = 0x103;
template <int NFR, int ACT, int YDT, bool ROWSC, bool FLEX, bool MXO, typename Args, typename Pace>
TAMD_DEVICE void tile_epilogue_t(const Args &a, const Tile &t, f32x16_t (&acc)[NFR][NF], uint8_t *tab, const EpilogueOperands<NFR> *ready,
                                 Pace &pace, bool pairs = true) {
  constexpr bool BYTES = is_fp8(YDT) || YDT == kQuads8;
  const int wave = (threadIdx.x / kWave) & 3;
  int lane = threadIdx.x % kWave;
  float log2e = 1.4426950408889634f, inf = __builtin_inff();
  uint32_t kDrop = 0x80000000u;                             // an offset that no descriptor here covers
  // (nothing made of these is kept in registers over the tiles of a persistent kernel)
  if constexpr (BYTES) asm volatile("" : "+v"(lane), "+s"(log2e), "+s"(inf), "+s"(kDrop));
  const int c32 = lane % 32, h = lane / 32;
  const int N = a.N;
  const int col0 = t.n0 + wave * 64 + c32 * NF;
  constexpr bool ANY = YDT == kAny16 || YDT == kAny8 || YDT == TAMD_F32;   // one width
  const int ydt = ANY ? a.y_dtype : (YDT == kQuads8 || YDT == kRows8 ? TAMD_FP8_E4M3 : YDT);
  constexpr int NO = ACT == TAMD_ACT_SWIGLU ? NF / 2 : NF;  // outputs per lane per row
  const int n_out = ACT == TAMD_ACT_SWIGLU ? N / 2 : N;
  const int out_col0 = ACT == TAMD_ACT_SWIGLU ? col0 / 2 : col0;
  constexpr int osz = YDT == TAMD_F32 ? 4 : (BYTES || YDT == kRows8 || YDT == kAny8 ? 1 : 2);   // bytes per output
  if (t.n0 + wave * 64 >= N) return;
  uint32_t *tab_dst = (uint32_t *)tab;
  float *tab_beta = (float *)tab + NFR * 32, *tab_gamma = (float *)tab + NFR * 64;
  EpilogueOperands<NFR> ops;
  if (ready) {
    ops = *ready;
  } else {
    epilogue_operands<NFR, ROWSC, Args>(a, t, ops);
    epilogue_table<NFR, osz, ROWSC, MXO, Args>(a, t, ops.dst, ops.beta, ops.gamma, tab);
  }
  const float flex = ops.x_scale * ops.w_scale * a.out_alpha;
  // without per-row factors bias * beta * out_alpha is one value per column
  float bias_a[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) bias_a[f] = (a.bias && col0 + f < N ? bits_of_type(ops.bias[f], a.bias_dtype) : 0.f) * a.out_alpha;
  const bool has_limit = a.act_has_limit != 0;
  // flexpoint output: scale by 1 / expected, optionally clamp, and track max|result| for the actual scale
  const float inv_expected = (FLEX && a.y_expected_scale) ? 1.0f / *a.y_expected_scale : 1.0f;
  const bool clamp_out = YDT == kQuads8 || (FLEX && a.y_expected_scale != nullptr && a.y_saturate_inf != 0);
  const float out_max = max_finite_of(ydt);
  const bool track_max = FLEX && a.y_actual_scale != nullptr;
  const uint32_t track_mask = track_max ? 0x7FFFFFFFu : 0u;
  uint32_t amax = 0;
  auto narrow = [&](float v) -> uint32_t {  // one output value as 8 / 16 bits
    return ydt == TAMD_BF16 ? f32_to_bf16_bits(v) : (ydt == TAMD_F16 ? f32_to_f16_bits(v) : f32_to_fp8_bits(v, ydt));
  };
  auto narrow2 = [&](float lo, float hi) -> uint32_t {  // two 16-bit outputs in one word (one packed conversion)
    if (ydt == TAMD_BF16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, f16x2_t));
  };
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((uint8_t *)a.y + (int64_t)t.z * a.y_stride_z * osz, 0,
                                                                     0x7FFFFFFF, 0x00020000);
  const uint32_t col_off = (uint32_t)out_col0 * (uint32_t)osz, col_kill = out_col0 < n_out ? 0u : kDrop;
  const uint32_t col_kill1 = out_col0 + 1 < n_out ? 0u : kDrop;   // (the second output of a pair that N cuts)
  // Bytes: whole quads of lanes inside the output, whole words: one store of four or eight bytes per lane and four rows.  (Of 16 bits the
  // stores are not what a tile waits for: 8 and 16 bytes per lane took 1 to 3 % longer for the exchange between the lanes.)
  const bool quads = YDT == kQuads8 || (BYTES && epilogue_stores_quads<NO>(a, n_out));
  const bool factors = ROWSC && (a.betas || a.gammas);
  const float act_scale = ACT == TAMD_ACT_SWIGLU ? -a.act_alpha * log2e : 0.f, limit = ACT == TAMD_ACT_SWIGLU ? a.act_limit : 0.f;
  const float limit_lo = __builtin_fminf(-limit, limit);
  const __amdgpu_buffer_rsrc_t rsc = __builtin_amdgcn_make_buffer_rsrc(
      MXO ? a.y_mx_scale + (int64_t)t.z * a.y_mx_stride_z : nullptr, 0, MXO ? 0x7FFFFFFF : 0, 0x00020000);
  // the scales of four rows go out together: in a group's lanes, lane jj takes row jj's
  const uint32_t sc_off = ((c32 & (32 / NO - 1)) < 4 && (out_col0 & ~31) < n_out) ? (uint32_t)(out_col0 / 32) : kDrop;
  // four rows of the table at a time, read one step ahead; the scheduling barrier keeps the compiler from reading the
  // whole table up front (registers)
  // (of bytes a lane stores one row in four: only that row's destination is read)
  constexpr bool DST_AHEAD = !BYTES;
  uint4 next_dst = DST_AHEAD ? *(const uint4 *)(tab_dst + h * 4) : uint4{0u, 0u, 0u, 0u};
  // (the factors of a SwiGLU tile, which a layer has none of, are read where they are used: registers)
  constexpr bool FACTORS_AHEAD = ROWSC && (!BYTES || ACT != TAMD_ACT_SWIGLU);
  f32x4_t next_beta = f32x4_t{1.f, 1.f, 1.f, 1.f}, next_gamma = next_beta;
  if constexpr (FACTORS_AHEAD) {
    next_beta = *(const f32x4_t *)(tab_beta + h * 4);
    next_gamma = *(const f32x4_t *)(tab_gamma + h * 4);
  }
#pragma unroll
  for (int i = 0; i < NFR; ++i) {
#pragma unroll (ANY ? 1 : 4)
    for (int jq = 0; jq < 4; ++jq) {
      const uint32_t dst4[4] = {next_dst.x, next_dst.y, next_dst.z, next_dst.w};
      const f32x4_t beta4 = next_beta, gamma4 = next_gamma;
      if (ANY || i * 4 + jq + 1 < NFR * 4) {   // (one row past the last: still the table)
        const int r1 = (i * 4 + jq + 1) * 8 + h * 4;
        if constexpr (DST_AHEAD) next_dst = *(const uint4 *)(tab_dst + r1);
        if constexpr (FACTORS_AHEAD) {
          next_beta = *(const f32x4_t *)(tab_beta + r1);
          next_gamma = *(const f32x4_t *)(tab_gamma + r1);
        }
      }
      auto result = [&](int jj, float (&o)[NO]) {
        const int j = ANY ? jj : jq * 4 + jj;
        float v[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) v[f] = __builtin_fmaf(acc[i][f][j], flex, ROWSC ? bias_a[f] * beta4[jj] : bias_a[f]);
        if constexpr (ACT == TAMD_ACT_SWIGLU) {
          o[0] = swiglu_fast(v[0], v[1], a.act_alpha, a.act_limit, has_limit);
        } else {
#pragma unroll
          for (int p = 0; p < NO; ++p) o[p] = v[p];
        }
        if constexpr (ROWSC) {
#pragma unroll
          for (int p = 0; p < NO; ++p) o[p] *= gamma4[jj];
        }
      };
      const int r0 = (i * 4 + jq) * 8 + h * 4;
      const uint32_t own = DST_AHEAD ? 0u : tab_dst[r0 + (lane & 3)];
      float out4[4][NO];
      if constexpr (!BYTES) {
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          float (&o)[NO] = out4[jj];
          result(jj, o);
          if constexpr (YDT == kRows8) {
            // (selections, no branches: a branch per element breaks the fragment into hundreds of blocks)
#pragma unroll
            for (int p = 0; p < NO; ++p) {
              const uint32_t b = f32_to_bits(o[p]) & ((dst4[jj] | col_kill) & kDrop ? 0u : track_mask);
              amax = b > amax ? b : amax;
              o[p] *= inv_expected;
              const float oc = __builtin_fminf(__builtin_fmaxf(o[p], -out_max), out_max);
              o[p] = clamp_out ? oc : o[p];
            }
            const int off = (int)((dst4[jj] + col_off) | col_kill);
            if constexpr (NO == 2) __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(narrow(o[0]) | (narrow(o[NO - 1]) << 8)), ry, off, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b8((uint8_t)narrow(o[0]), ry, off, 0, 0);
          } else if constexpr (!ANY) {
            const int off = (int)((dst4[jj] + col_off) | col_kill);
            if constexpr (NO == 2) __builtin_amdgcn_raw_buffer_store_b32(narrow2(o[0], o[NO - 1]), ry, off, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b16((uint16_t)narrow(o[0]), ry, off, 0, 0);
          }
        }
      } else {
        // Four rows at once, and what is the same for the launch decided by a branch for all of them (the empty asm keeps it one): the
        // epilogue of a tile of 128 x 256 with SwiGLU is a third of a short tile's time, bound by its instructions -- 270 per four rows
        // with MXFP8 output when everything was selected per value, each row's scale made by every lane and every byte stored by
        // itself, 130 now.  1028 MXFP8 tokens x 6 of 32 slices, 1248 -> 2688: 60.2 -> 51.4 us (the epilogue 12.4 -> 8.4 of a tile's 30);
        // 5670 x 4 of 64, 2144 -> 1472, strided, 135 -> 123; fp8, 16384 x 4 of 32, 2880 -> 5760: 961 -> 942.
        float v[4][NF];
        if (ROWSC && factors) {
          const f32x4_t beta = FACTORS_AHEAD ? beta4 : *(const f32x4_t *)(tab_beta + r0);
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int f = 0; f < NF; ++f) v[jj][f] = __builtin_fmaf(acc[i][f][jq * 4 + jj], flex, bias_a[f] * beta[jj]);
        } else {
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int f = 0; f < NF; ++f) v[jj][f] = __builtin_fmaf(acc[i][f][jq * 4 + jj], flex, bias_a[f]);
        }
        if constexpr (ACT == TAMD_ACT_SWIGLU) {   // swiglu_fast, a step for four rows at a time
          if (has_limit) {
            asm volatile("");
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
              v[jj][0] = __builtin_fminf(v[jj][0], limit);
              v[jj][1] = __builtin_amdgcn_fmed3f(v[jj][1], limit_lo, limit);   // (a NaN gives the lower bound, as the maximum does)
            }
          }
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            const float e = __builtin_amdgcn_exp2f(act_scale * v[jj][0]);
            const float g = v[jj][0] * __builtin_amdgcn_rcpf(1.0f + e);
            out4[jj][0] = __builtin_fmaf(g, v[jj][1], g);
          }
        } else {
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int p = 0; p < NO; ++p) out4[jj][p] = v[jj][p];
        }
        if (ROWSC && factors) {
          asm volatile("");
          const f32x4_t gamma = FACTORS_AHEAD ? gamma4 : *(const f32x4_t *)(tab_gamma + r0);
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int p = 0; p < NO; ++p) out4[jj][p] *= gamma[jj];
        }
      }
      if constexpr (MXO) {
        // MXFP8 output: a group is 32 consecutive output columns of a row = the outputs of one half wave (of
        // half of it when a lane holds two columns).  max |o| over the group, scale = 2^ceil(log2(max / 448)), o / scale
        // (within +-448 by the choice of the scale); the cast below rounds to nearest even (as tamd_downcast_mxfp does).  The maxima
        // of non-negative numbers are those of their bits (a NaN counts as 0); lane jj of every quad makes row jj's scale and
        // hands it to the others.
        const float cap = out_col0 < n_out ? inf : 0.f, cap1 = out_col0 + 1 < n_out ? inf : 0.f;
        uint32_t m4[4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          m4[jj] = f32_to_bits(__builtin_amdgcn_fmed3f(__builtin_fabsf(out4[jj][0]), 0.f, cap));
          if constexpr (NO == 2) {
            const uint32_t m1 = f32_to_bits(__builtin_amdgcn_fmed3f(__builtin_fabsf(out4[jj][NO - 1]), 0.f, cap1));
            m4[jj] = m1 > m4[jj] ? m1 : m4[jj];
          }
        }
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) m4[jj] = group_max_lanes<NO>(m4[jj]);
        const uint32_t mine = (c32 & 2) ? ((c32 & 1) ? m4[3] : m4[2]) : ((c32 & 1) ? m4[1] : m4[0]);
        const uint32_t se = ceil_scale_byte<TAMD_FP8_E4M3>(bits_to_f32(mine));
        const uint32_t qs = se == 0u || se == 255u ? 0u : (254u - se) << 23;   // 1 / 2^(se - 127)
        const float qs4[4] = {bits_to_f32((uint32_t)__builtin_amdgcn_update_dpp(0, (int)qs, 0x00, 0xF, 0xF, true)),
                              bits_to_f32((uint32_t)__builtin_amdgcn_update_dpp(0, (int)qs, 0x55, 0xF, 0xF, true)),
                              bits_to_f32((uint32_t)__builtin_amdgcn_update_dpp(0, (int)qs, 0xAA, 0xF, 0xF, true)),
                              bits_to_f32((uint32_t)__builtin_amdgcn_update_dpp(0, (int)qs, 0xFF, 0xF, 0xF, true))};
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
          for (int p = 0; p < NO; ++p) out4[jj][p] *= qs4[jj];
        const uint32_t sdst = tab_dst[NFR * 96 + (i * 4 + jq) * 8 + h * 4 + (c32 & 3)];
        __builtin_amdgcn_raw_buffer_store_b8((uint8_t)se, rsc, (int)(((sdst | sc_off) & kDrop) | (sdst + sc_off)), 0, 0);
      }
      if constexpr (FLEX && YDT != kRows8) {
        if (ANY || track_max) {
          const uint4 d = DST_AHEAD ? uint4{dst4[0], dst4[1], dst4[2], dst4[3]} : *(const uint4 *)(tab_dst + r0);
          const uint32_t rows[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int p = 0; p < NO; ++p) {
              const uint32_t amask = (rows[jj] | (ANY && p == 1 ? col_kill1 : col_kill)) & kDrop ? 0u : track_mask;
              const uint32_t b = f32_to_bits(out4[jj][p]) & amask;
              amax = b > amax ? b : amax;
            }
        }
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
          for (int p = 0; p < NO; ++p) out4[jj][p] *= inv_expected;
        if (clamp_out) {
          if constexpr (YDT != kQuads8) asm volatile("");
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int p = 0; p < NO; ++p) out4[jj][p] = __builtin_amdgcn_fmed3f(out4[jj][p], -out_max, out_max);
        }
      }
      if constexpr (BYTES) {
        // the bytes of a column's four rows (of two columns' rows two by two)
        uint32_t w[NO];
        bool in_range = clamp_out;   // then the conversion alone
        if constexpr (MXO) {         // unless one is a NaN, whose sign it would lose
          bool nan = false;
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) nan |= __builtin_isunordered(out4[jj][0], out4[jj][NO - 1]);
          in_range = __ballot(nan) == 0;
        }
        if (in_range) {
          if constexpr (NO == 1) w[0] = e4m3_pair_bits<true>(out4[2][0], out4[3][0], e4m3_pair_bits<false>(out4[0][0], out4[1][0], 0u));
          else {
            w[0] = e4m3_pair_bits<true>(out4[1][0], out4[1][NO - 1], e4m3_pair_bits<false>(out4[0][0], out4[0][NO - 1], 0u));
            w[NO - 1] = e4m3_pair_bits<true>(out4[3][0], out4[3][NO - 1], e4m3_pair_bits<false>(out4[2][0], out4[2][NO - 1], 0u));
          }
        } else {
          asm volatile("");
          if constexpr (NO == 1) w[0] = narrow(out4[0][0]) | narrow(out4[1][0]) << 8 | narrow(out4[2][0]) << 16 | narrow(out4[3][0]) << 24;
          else {
            w[0] = narrow(out4[0][0]) | narrow(out4[0][NO - 1]) << 8 | narrow(out4[1][0]) << 16 | narrow(out4[1][NO - 1]) << 24;
            w[NO - 1] = narrow(out4[2][0]) | narrow(out4[2][NO - 1]) << 8 | narrow(out4[3][0]) << 16 | narrow(out4[3][NO - 1]) << 24;
          }
        }
        if (quads) {
          const int off = (int)((own + col_off - (uint32_t)((lane & 3) * NO)) | col_kill);
          if constexpr (NO == 1) __builtin_amdgcn_raw_buffer_store_b32(quad_rows(w[0], lane), ry, off, 0, 0);
          else __builtin_amdgcn_raw_buffer_store_b64(quad_rows(w[0], w[NO - 1], lane), ry, off, 0, 0);
        } else {
          asm volatile("");
          const uint4 d = *(const uint4 *)(tab_dst + r0);
          const uint32_t rows[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            const int off = (int)((rows[jj] + col_off) | col_kill);
            if constexpr (NO == 1) __builtin_amdgcn_raw_buffer_store_b8((uint8_t)(w[0] >> 8 * jj), ry, off, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(w[(jj >> 1) * (NO - 1)] >> 16 * (jj & 1)), ry, off, 0, 0);
          }
        }
      }
      if constexpr (ANY) {
        // the type and the way to store are the same for the whole launch: one branch each for four rows
        uint32_t w[4][NO];
        auto all = [&](auto f) {
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int p = 0; p < NO; ++p) w[jj][p] = f(out4[jj][p]);
        };
        if constexpr (osz == 4) {
          all([](float v) { return f32_to_bits(v); });
        } else if constexpr (osz == 2) {
          if (ydt == TAMD_BF16) all([](float v) { return f32_to_bf16_bits(v); });
          else all([](float v) { return f32_to_f16_bits(v); });
        } else {
          if (ydt == TAMD_FP8_E5M2) all([](float v) { return f32_to_e5m2_bits(v, false); });
          else all([](float v) { return f32_to_e4m3_bits(v, false); });
        }
        auto store1 = [&](uint32_t v, int off) {
          if constexpr (osz == 4) __builtin_amdgcn_raw_buffer_store_b32(v, ry, off, 0, 0);
          else if constexpr (osz == 2) __builtin_amdgcn_raw_buffer_store_b16((uint16_t)v, ry, off, 0, 0);
          else __builtin_amdgcn_raw_buffer_store_b8((uint8_t)v, ry, off, 0, 0);
        };
        if (NO == 1 || !pairs) {
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            store1(w[jj][0], (int)((dst4[jj] + col_off) | col_kill));
            if constexpr (NO == 2) store1(w[jj][NO - 1], (int)((dst4[jj] + col_off + osz) | col_kill1));
          }
        } else {
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            const int off = (int)((dst4[jj] + col_off) | col_kill);
            if constexpr (osz == 4) __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{w[jj][0], w[jj][NO - 1]}, ry, off, 0, 0);
            else if constexpr (osz == 2) __builtin_amdgcn_raw_buffer_store_b32(w[jj][0] | (w[jj][NO - 1] << 16), ry, off, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(w[jj][0] | (w[jj][NO - 1] << 8)), ry, off, 0, 0);
          }
        }
      }
      // (the running maximum is taken here and not after the last row, with every result kept until then)
      if constexpr (FLEX) asm volatile("" : "+v"(amax));
      if constexpr (ANY) {   // a rolled loop: the next four rows move to where it looks for them
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int e = 0; e < 12; ++e) acc[i][f][e] = acc[i][f][e + 4];
      }
      __builtin_amdgcn_sched_barrier(0);
      pace();
    }
  }
  if constexpr (FLEX) {
    if (track_max) store_actual_scale(a.y_actual_scale, amax, out_max, lane);
  }
}

// The general epilogue: any output type, alignment and size, every feature read at run time, stores through 64-bit
// addresses.  A row fragment's accumulators are taken four at a time in a rolled loop and move up by four after each
// step, so that the loop indexes registers with constants.
template <int NFR, int ACT, typename Args, typename Pace>
TAMD_DEVICE void tile_epilogue_general(const Args &a, const Tile &t, f32x16_t (&acc)[NFR][NF], uint8_t *tab, Pace &pace) {
  const int wave = (threadIdx.x / kWave) & 3, lane = threadIdx.x % kWave;
  const int c32 = lane % 32, h = lane / 32;
  const int N = a.N;
  const int col0 = t.n0 + wave * 64 + c32 * NF;
  constexpr int NO = ACT == TAMD_ACT_SWIGLU ? NF / 2 : NF;
  const int n_out = ACT == TAMD_ACT_SWIGLU ? N / 2 : N;
  const int out_col0 = ACT == TAMD_ACT_SWIGLU ? col0 / 2 : col0;
  if (t.n0 + wave * 64 >= N) return;
  int32_t *tab_dst = (int32_t *)tab;
  float *tab_beta = (float *)tab + NFR * 32, *tab_gamma = (float *)tab + NFR * 64;
  for (int r = lane; r < NFR * 32; r += kWave) {
    const int erow = t.start_m + t.off_m + (r < t.rows ? r : t.rows - 1);
    const int dst = a.scatter_indx ? a.scatter_indx[erow] : erow;
    tab_dst[r] = r < t.rows ? dst : -1;
    tab_beta[r] = a.betas ? a.betas[erow] : 1.0f;
    tab_gamma[r] = a.gammas ? a.gammas[erow] : 1.0f;
  }
  float flex = 1.0f;
  if (a.x_scale) flex *= *a.x_scale;
  if (a.w_scale) flex *= *a.w_scale;
  flex *= a.out_alpha;
  float bias_a[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f)
    bias_a[f] = ((a.bias && col0 + f < N) ? load_any_f32(a.bias, a.bias_dtype, (int64_t)t.expert * a.bias_stride_e + col0 + f)
                                          : 0.f) * a.out_alpha;
  const bool has_limit = a.act_has_limit != 0;
  const int ydt = a.y_dtype;
  const float inv_expected = a.y_expected_scale ? 1.0f / *a.y_expected_scale : 1.0f;
  const bool clamp_out = a.y_expected_scale != nullptr && a.y_saturate_inf != 0;
  const float out_max = max_finite_of(ydt);
  uint32_t amax = 0;
#pragma unroll
  for (int i = 0; i < NFR; ++i)
#pragma unroll 1
  for (int q = 0; q < 4; ++q) {
    const int r0 = i * 32 + q * 8 + h * 4;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int dst = tab_dst[r0 + jj];
      const float beta = tab_beta[r0 + jj], gamma = tab_gamma[r0 + jj];
      float v[NF], o[NO];
#pragma unroll
      for (int f = 0; f < NF; ++f) v[f] = __builtin_fmaf(acc[i][f][jj], flex, bias_a[f] * beta);
      if constexpr (ACT == TAMD_ACT_SWIGLU) {
        o[0] = swiglu_fast(v[0], v[1], a.act_alpha, a.act_limit, has_limit);
      } else {
#pragma unroll
        for (int p = 0; p < NO; ++p) o[p] = v[p];
      }
#pragma unroll
      for (int p = 0; p < NO; ++p) o[p] *= gamma;
      if (a.y_mx_scale) {  // MXFP8 output, as in tile_epilogue_t
        float m = 0.f;
#pragma unroll
        for (int p = 0; p < NO; ++p) m = __builtin_fmaxf(m, out_col0 + p < n_out ? __builtin_fabsf(o[p]) : 0.f);
        for (int sh = 16 / NO; sh > 0; sh >>= 1) m = __builtin_fmaxf(m, __shfl_xor(m, sh));
        const uint32_t sb = (f32_to_bits(m / 448.0f) + 0x007FFFFFu) & 0x7F800000u;
        const float ds = bits_to_f32(sb);
        const float qs = ds == 0.f ? 0.f : 1.0f / ds;
#pragma unroll
        for (int p = 0; p < NO; ++p) {
          const float w = o[p] * qs;
          o[p] = w != w ? w : __builtin_fminf(__builtin_fmaxf(w, -448.0f), 448.0f);
        }
        if (dst >= 0 && (c32 & (32 / NO - 1)) == 0 && out_col0 < n_out)
          a.y_mx_scale[(int64_t)t.z * a.y_mx_stride_z + (int64_t)dst * a.y_mx_stride_m + out_col0 / 32] = (uint8_t)(sb >> 23);
      }
      if (dst >= 0) {
        const int64_t at = (int64_t)t.z * a.y_stride_z + (int64_t)dst * a.y_stride_m + out_col0;
#pragma unroll
        for (int p = 0; p < NO; ++p) {
          if (out_col0 + p < n_out) {
            if (a.y_actual_scale) amax = absmax_bits(amax, o[p]);
            float w = o[p] * inv_expected;
            if (clamp_out) w = __builtin_fminf(__builtin_fmaxf(w, -out_max), out_max);
            if (ydt == TAMD_F32) ((float *)a.y)[at + p] = w;
            else if (ydt == TAMD_BF16) ((uint16_t *)a.y)[at + p] = (uint16_t)f32_to_bf16_bits(w);
            else if (ydt == TAMD_F16) ((uint16_t *)a.y)[at + p] = (uint16_t)f32_to_f16_bits(w);
            else ((uint8_t *)a.y)[at + p] = (uint8_t)f32_to_fp8_bits(w, ydt);
          }
        }
      }
    }
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 12; ++j) acc[i][f][j] = acc[i][f][j + 4];
    pace();
  }
  if (a.y_actual_scale) store_actual_scale(a.y_actual_scale, amax, out_max, lane);
}

// Whether 32-bit offsets reach every output of a batch entry, and whether a lane's two outputs lie whole on one aligned word
// (float32 pairs are stored as two words, which need no more than their own alignment).
template <typename Args>
TAMD_DEVICE bool epilogue_spans_32_bits(const Args &a) {
  const int osz = a.y_dtype == TAMD_F32 ? 4 : (is_fp8(a.y_dtype) ? 1 : 2);
  const int64_t lim = 0x7FFFFF00;
  if (a.y_rows <= 0 || a.y_stride_m < 0 || a.y_rows * a.y_stride_m * osz >= lim) return false;
  return !a.y_mx_scale || a.y_rows * a.y_mx_stride_m < lim;
}
template <int ACT, typename Args>
TAMD_DEVICE bool epilogue_stores_pairs(const Args &a) {
  if (ACT == TAMD_ACT_SWIGLU) return true;   // one output per lane
  if (a.y_dtype == TAMD_F32) return (a.N & 1) == 0;
  const int osz = is_fp8(a.y_dtype) ? 1 : 2;
  return ((a.N | (int)a.y_stride_m | (int)a.y_stride_z) & 1) == 0 && ((uintptr_t)a.y & (2 * osz - 1)) == 0;
}
template <int ACT, typename Args>
TAMD_DEVICE bool epilogue_is_regular(const Args &a) {
  return epilogue_spans_32_bits(a) && epilogue_stores_pairs<ACT>(a);
}
// FAST_YDT: the 16-bit output type that gets epilogues of its own (the activations' type; bf16 for fp8 activations); FP8_ROWS:
// the kernel's activations are fp8, then float8_e4m3fn output (the rows the next matmul of an MoE layer consumes, usually with
// a flexpoint scale) has one as well.  Everything else -- another type, flexpoint scales, odd sizes or strides -- takes the form of
// its width, and only an output of 2 GB or more (or of unknown rows) and MXFP8 output in odd rows the general epilogue.  The
// general one, a branch and a 64-bit address per element, is slower by (4096 x 2880, MXFP4 weights): fp8 rows, 5759 columns of
// bf16 116 us against 88; bf16 rows, 5760 columns of float32 145 against 128, of e4m3 with a flexpoint scale 161 against 126.
template <int NFR, int ACT, int FAST_YDT, bool FP8_ROWS, typename Args>
TAMD_DEVICE void tile_epilogue(const Args &a, const Tile &t, f32x16_t (&acc)[NFR][NF], uint8_t *tab) {
  const NoPace pace;
  const bool flexo = a.y_expected_scale != nullptr || a.y_actual_scale != nullptr;
  const bool spans = epilogue_spans_32_bits(a), pairs = epilogue_stores_pairs<ACT>(a);
  if (spans && pairs && a.y_mx_scale) {  // always e4m3 values and no flexpoint output (checked by the entry point)
    tile_epilogue_t<NFR, ACT, TAMD_FP8_E4M3, true, false, true, Args>(a, t, acc, tab, nullptr, pace);
  } else if (!spans || a.y_mx_scale) {
    tile_epilogue_general<NFR, ACT, Args>(a, t, acc, tab, pace);
  } else if (FP8_ROWS && pairs && a.y_dtype == TAMD_FP8_E4M3) {
    if constexpr (FP8_ROWS) {
      constexpr int NO = ACT == TAMD_ACT_SWIGLU ? NF / 2 : NF;
      if (a.y_expected_scale && a.y_saturate_inf && !a.betas && !a.gammas && epilogue_stores_quads<NO>(a, ACT == TAMD_ACT_SWIGLU ? a.N / 2 : a.N))
        tile_epilogue_t<NFR, ACT, kQuads8, false, true, false, Args>(a, t, acc, tab, nullptr, pace);
      else tile_epilogue_t<NFR, ACT, kRows8, true, true, false, Args>(a, t, acc, tab, nullptr, pace);
    }
  } else if (pairs && a.y_dtype == FAST_YDT && !flexo) {
    if (a.betas || a.gammas) tile_epilogue_t<NFR, ACT, FAST_YDT, true, false, false, Args>(a, t, acc, tab, nullptr, pace);
    else tile_epilogue_t<NFR, ACT, FAST_YDT, false, false, false, Args>(a, t, acc, tab, nullptr, pace);
  } else if (a.y_dtype == TAMD_F32) {
    tile_epilogue_t<NFR, ACT, TAMD_F32, true, true, false, Args>(a, t, acc, tab, nullptr, pace, pairs);
  } else if (is_fp8(a.y_dtype)) {
    tile_epilogue_t<NFR, ACT, kAny8, true, true, false, Args>(a, t, acc, tab, nullptr, pace, pairs);
  } else {
    tile_epilogue_t<NFR, ACT, kAny16, true, true, false, Args>(a, t, acc, tab, nullptr, pace, pairs);
  }
}

// The kernel's tamd_matmul_args (its first parameter) read in place from the kernel-argument segment, through a
// pointer the compiler cannot see through.  The compiler loads every field of a by-value kernel argument that is
// used anywhere into scalar registers at the top of the kernel; the few dozen that only the epilogue needs then
// stay live through the K loop, the scalar registers overflow into vector registers, and a kernel that sits at 256
// of those starts spilling accumulators.  Read this way, the epilogue's fields are fetched when it begins.
typedef const __attribute__((address_space(4))) tamd_matmul_args late_args_t;
TAMD_DEVICE late_args_t &kernel_args_late() {
  late_args_t *p = (late_args_t *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}

// The K groups' partial sums of one row fragment meet in LDS: group g > 0 leaves its accumulators in plane g - 1 and ends (false); group 0
// adds the planes in the order of the groups and finishes the tile alone (a barrier waits only for the waves that are still alive).
// (16 bytes per lane and access: a plane is [NS waves][NF x 4 quads][64 lanes] of four accumulators)
template <int KS, int NS>
TAMD_DEVICE bool k_groups_add(f32x16_t (&acc)[NF], uint8_t *lds, int grp, int wave) {
  const int lane = threadIdx.x % kWave;
  f32x4_t *red = (f32x4_t *)lds;
  constexpr int PLANE = NS * NF * 4 * kWave;
  if (grp > 0) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        red[(grp - 1) * PLANE + ((wave * NF + f) * 4 + j) * kWave + lane] = f32x4_t{acc[f][4 * j], acc[f][4 * j + 1], acc[f][4 * j + 2], acc[f][4 * j + 3]};
  }
  sync_threads();
  if (grp > 0) return false;
#pragma unroll
  for (int g = 1; g < KS; ++g)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4_t v = red[(g - 1) * PLANE + ((wave * NF + f) * 4 + j) * kWave + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[f][4 * j + e] += v[e];
      }
  // (added here: left for the epilogue, which has several forms, the planes would not fit the registers until then)
#pragma unroll
  for (int f = 0; f < NF; ++f) asm volatile("" : "+v"(acc[f]));
  sync_threads();   // the epilogue's tables take the same memory
  return true;
}

// One output tile with NFR (compile time) active 32-row fragments.
// LDS: [A stages (2 to 4) | B: 4 wave-private regions, one or two stages | the e8m0 scales of the whole tile]; with K groups (KS > 1) one
// such pipeline per group, the tile's scales behind them.
//
// Both operands reach LDS by DMA.  Activations: 64 K per stage; wave w copies rows
// 8w..8w+7 of every 32-row fragment (8 lanes x 16 B per row); chunk c of row r sits at slot
// c ^ ((r>>1)&7), which makes the 32-row MFMA operand reads bank-conflict free.  Weights: every
// second stage each wave copies 128 K of its own 64 columns into its private region: position
// p' = f*32 + c holds global column 2c + f of the wave's strip (so a lane ends up with a gate/linear column pair), the
// four 16-byte parts rotated by ((p'>>2)&3) ^ 2f.  From column-strided weights that is 64 contiguous bytes of each
// column; weights in the block layout (TAMD_W_CDNA4_BLOCKS) hold exactly this image, 4 KB per strip and 128 K, and
// are copied as they lie.  The wave reads the region into registers at the start of the stage and immediately
// requests the next 128 K into it, so weights need no barrier.
// Loops: two stages and full waits; counted waits over a deeper ring (K groups), see pipe_shape.
template <int XDT, int NFR, int LDS_ROWS, int ACT, bool SC_LDS, int KS = 1, int NS = 4>
TAMD_DEVICE void run_tile(const tamd_matmul_args &a, const Tile &t, uint8_t *lds_wg) {
  typedef Mma<XDT> M;
  typedef typename M::frag_t frag_t;
  constexpr int ESZ = 2;                      // bytes per activation element
  constexpr int KA = A_ROW_BYTES / ESZ;       // K per activation stage
  constexpr int A_STAGE = LDS_ROWS * A_ROW_BYTES;
  constexpr bool DEEP = KS > 1 || LDS_ROWS <= 32;   // counted waits
  static_assert(!DEEP || (SC_LDS && NFR == 1 && (KS == 1 || KS == 2 || KS == 8)), "counted waits: scales in LDS, one row fragment");
  static_assert(NS == 4 || (NS == 2 && KS > 1), "a tile is four strips of 64 columns, with K groups two or four");
  constexpr PipeShape PS = pipe_shape(LDS_ROWS, KS, NS);
  constexpr int DA = PS.da, DB = PS.db;
  constexpr int COLS = 64 * NS, WB_STAGE = NS * 4096;
  auto a_slot = [](int it) { return DA == 2 ? (it & 1) : it % DA; };
  constexpr uint32_t kOob = 0x7FFFFFFFu;
  const int tid = threadIdx.x;
  // K group of the wave (0 unless KS > 1) and its place among the group's NS waves, one per strip
  const int grp = KS > 1 ? __builtin_amdgcn_readfirstlane(tid / (kWave * NS)) : 0;
  const int wave = KS > 1 ? __builtin_amdgcn_readfirstlane((tid / kWave) & (NS - 1)) : tid / kWave, lane = tid % kWave;
  const int c32 = lane % 32, h = lane / 32;
  const int K = a.K, N = a.N, G = K / 32;
  // a wave whose 64 columns lie beyond N (last column tile) copies its share of the activations and keeps the
  // barriers, but neither fetches weights nor runs MFMAs
  const bool wave_live = t.n0 + wave * 64 < N;
  // the pipeline buffers of the wave's K group; the tile's scale image behind the last group's is shared
  constexpr int PIPE_G = PS.bytes;
  uint8_t *lds = lds_wg + grp * PIPE_G;
  // the group's part of K: whole 128-K pairs [sup0, sup0 + n_sup), the same number for every group (a group whose
  // part reaches past K copies zeros there: out-of-range offsets)
  const int n_kb_all = (K + KB - 1) / KB;
  const int n_sup = (n_kb_all + KS - 1) / KS;
  const int sup0 = grp * n_sup;
  const int k0 = sup0 * KB;
  const int k_hi = KS > 1 ? (k0 + n_sup * KB < K ? k0 + n_sup * KB : K) : K;

  const v4i_t rx = make_rsrc((const uint8_t *)a.x + (int64_t)t.z * a.x_stride_z * ESZ, kOob);
  const v4i_t rw = make_rsrc((const uint8_t *)a.w + (int64_t)t.expert * a.w_stride_e, kOob);
  const uint8_t *s_base = a.w_mx_scale + (int64_t)t.expert * a.w_mx_stride_e;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
  const uint32_t lds_b = lds_base + DA * A_STAGE + wave * 4096;
  const uint8_t *bbuf = lds + DA * A_STAGE + wave * 4096;
  uint8_t *lds_sc = KS > 1 ? lds_wg + KS * PIPE_G : lds + DA * A_STAGE + DB * WB_STAGE;

  // ---- scales of the whole tile, once.  Strided: 256 columns x G bytes, contiguous in memory.  CDNA4
  // pre-shuffle: the tile's 8 blocks of 32 columns are contiguous too (KSP*32 bytes each); byte
  // 256*(k/8) + 64*(k%4) + 4*(n%16) + 2*((k%8)/4) + (n%32)/16 of a block is the scale of (group k, column n).
  const bool cdna4 = a.w_mx_layout == TAMD_SCALE_CDNA4;
  const int KSP = (G + 7) / 8 * 8;
  const int tile_cols = N - t.n0 < COLS ? N - t.n0 : COLS;
  const int64_t sc_tile_off = cdna4 ? (int64_t)(t.n0 / 32) * KSP * 32 : (int64_t)t.n0 * G;
  auto stage_scales = [&]() {
  if constexpr (SC_LDS) {
    const uint8_t *sc_src = s_base + sc_tile_off;
    const int sc_tile_bytes = COLS * (cdna4 ? KSP : G);
    const int sc_avail = cdna4 ? ((N + 31) / 32 * 32 - t.n0) * KSP : (N - t.n0) * G;  // bytes up to the expert's end
    if (cdna4 || ((((uintptr_t)sc_src) & 15) == 0 && (N * G) % 16 == 0)) {
      // by DMA, 1 KB per instruction: in flight together with the first activation / weight stages and
      // awaited with them at the first barrier of the K loop
      const v4i_t rs = make_rsrc(sc_src, (uint32_t)sc_avail);
      const uint32_t lds_sc_addr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds_sc;
      for (int i = wave + NS * grp; i * 1024 < sc_tile_bytes; i += NS * KS)
        dma16(rs, lds_sc_addr + i * 1024, i * 1024 + lane * 16, 0);
    } else {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)sc_src, 0, (uint32_t)(tile_cols * G),
                                                                        0x00020000);
      const int n_dw = (COLS * G + 3) / 4;
      const int avail = tile_cols * G;
      for (int i = tid; i < n_dw; i += kWave * NS * KS) {
        uint32_t v;
        if (i * 4 + 4 <= avail || i * 4 >= avail) {
          v = __builtin_amdgcn_raw_buffer_load_b32(rs, i * 4, 0, 0);  // whole, or wholly outside (zeros)
        } else {
          // the dword that straddles the end of the scales: a dword load that is partly out of range returns
          // zeros for all four bytes, so the bytes inside are fetched one by one
          v = 0;
          for (int b = 0; i * 4 + b < avail; ++b)
            v |= (uint32_t)(uint8_t)__builtin_amdgcn_raw_buffer_load_b8(rs, i * 4 + b, 0, 0) << (8 * b);
        }
        ((uint32_t *)lds_sc)[i] = v;
      }
    }
  }
  };
  // offset of a column's scales inside the tile's image (LDS) or, without staging, from the expert's first scale
  int sc_col_off[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int tc = wave * 64 + c32 * NF + f;  // tile column
    if constexpr (SC_LDS) {
      sc_col_off[f] = cdna4 ? (tc / 32) * KSP * 32 + (tc % 16) * 4 + (tc % 32) / 16 : tc * G;
    } else {
      const int col = t.n0 + tc < N ? t.n0 + tc : N - 1;
      sc_col_off[f] = cdna4 ? (col / 32) * KSP * 32 + (col % 16) * 4 + (col % 32) / 16 : 0;  // strided: 64-bit below
    }
  }

  const int sc_lane_off[2] = {h * (cdna4 ? 64 : 1), (2 + h) * (cdna4 ? 64 : 1)};  // the (2q + h) part of a group's offset
  const int sc_clamp = cdna4 ? 0x7FFFFFFF : G - 1;

  // Copies per request, as the counted waits of the ring loops below see them (a wave's copies complete in the order
  // of their requests): the loops of the issue_* functions run to these numbers and the waits are written in them.
  constexpr int PIECES = 4 / NS;   // (of eight rows of a fragment, NS pieces apart)
  constexpr int CP_A = NFR * PIECES;   // issue_a: one copy per row fragment and piece
  constexpr int CP_B = 4;          // issue_b: four 1 KB pieces
  // ---- activation DMA: one instruction per 32-row fragment, lane -> (row 8w + lane/8, slot lane%8)
  const int a_rin = wave * 8 + lane / 8;
  const int a_chunk = (lane % 8) ^ ((a_rin >> 1) & 7);
  // Rows past the end of the slice are never stored: they are copied as zeros (out-of-range offset), which keeps the matrix
  // cores' inputs quiet for the padding of a ragged tile.
  uint32_t a_off[CP_A];
  const int row0 = t.start_m + t.off_m;
  auto piece = [](int i) { return i / PIECES * 32 + i % PIECES * (8 * NS); };   // first row of copy i, of wave 0
  auto row_off = [&](int r, uint32_t src) { return r < t.rows ? src * (uint32_t)(a.x_stride_m * ESZ) + a_chunk * 16 : kOob; };
  // The rows' indices are the first thing requested, and the first weights, which do not depend on them, while they come.  They
  // travel by LDS, each in front of the row pieces that the wave will copy there (an ordinary load would be waited for with a count
  // that takes in the copies requested after it, which the compiler does not see).
  const v4i_t rg = make_rsrc(a.gather_indx + row0, (uint32_t)__builtin_amdgcn_readfirstlane(t.rows) * 4u);
  const int idx_at = wave * 8 * A_ROW_BYTES;
  if (a.gather_indx) {
#pragma unroll
    for (int i = 0; i < CP_A; ++i) dma4(rg, lds_base + idx_at + piece(i) * A_ROW_BYTES, (uint32_t)(piece(i) + a_rin) * 4u, 0);
  }
  auto rows_known = [&](auto newer) {   // (after `newer` further requests of the wave)
    if (a.gather_indx) wait_vmcnt<decltype(newer)::value>();
#pragma unroll
    for (int i = 0; i < CP_A; ++i) {
      const int at = idx_at + piece(i) * A_ROW_BYTES + lane * 4;
      a_off[i] = row_off(piece(i) + a_rin, a.gather_indx ? *(const uint32_t *)(lds + at) : (uint32_t)(row0 + piece(i) + a_rin));
    }
    if (a.gather_indx) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // read before the rows are copied over them
  };
  // ---- weight DMA: instruction j copies LDS positions j*16 + lane/4, part slot lane%4
  // Codes in the block layout (TAMD_W_CDNA4_BLOCKS): a stage of this wave's strip is one 4 KB block that already has
  // the LDS image's order, so the four copies are linear (whole, aligned lines) and the K stage enters through the
  // scalar offset; K and N are padded with zero codes, nothing is masked.
  const bool wnat = a.w_layout == TAMD_W_CDNA4_BLOCKS;
  const int w_stage_shift = wnat ? 12 : 6;   // bytes from one K stage to the next: a 4 KB block, or 64 bytes of a column
  // (the lane's 16-byte part of a column is the same for copies 0, 1 and, two further on, for copies 2, 3:
  // (pos >> 2) & 3 = (lane / 16) & 3 for every j, (pos >> 5) << 1 = 2 (j / 2))
  uint32_t w_off[4];
  const int w_part0 = (lane % 4) ^ ((lane / 16) & 3);
  const int w_kpart0 = wnat ? 0 : w_part0 * 32;   // K offset (codes) of the lane's bytes inside a stage; block layout: padded, 0
  auto w_kpart = [&](int j) { return wnat ? 0 : (w_kpart0 ^ ((j >> 1) << 6)); };
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int pos = j * 16 + lane / 4;  // f*32 + c
    const int col = t.n0 + wave * 64 + 2 * (pos % 32) + pos / 32;
    const int part = w_part0 ^ ((j >> 1) << 1);
    w_off[j] = wnat ? (uint32_t)(((t.n0 >> 6) + wave) * ((K + KB - 1) / KB)) * 4096u + (uint32_t)(j * 1024 + lane * 16)
                    : (uint32_t)(col < N ? col : N - 1) * (uint32_t)a.w_stride_n + part * 16;
  }
  // ---- this lane's MFMA columns
  const int col0 = t.n0 + wave * 64 + c32 * NF;

  f32x16_t acc[NFR][NF];
#pragma unroll
  for (int i = 0; i < NFR; ++i)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[i][f][j] = 0.f;

  const int n_ka = (K + KA - 1) / KA;      // activation stages
  const int n_kb = (K + KB - 1) / KB;      // weight super-stages (two activation stages each)
  auto issue_a = [&](int it) {             // clamped: past the end the last stage is copied again
    if constexpr (!DEEP) it = it < n_ka ? it : n_ka - 1;   // (K groups: chunks past K are not read at all)
    const int kb = k0 + it * KA;
    const uint32_t akill = kb + a_chunk * (16 / ESZ) < k_hi ? 0u : kOob;
    const uint32_t sb = lds_base + a_slot(it) * A_STAGE + wave * 8 * A_ROW_BYTES;
#pragma unroll
    for (int i = 0; i < CP_A; ++i) dma16(rx, sb + piece(i) * A_ROW_BYTES, a_off[i] | akill, kb * ESZ);
  };
  auto issue_b = [&](int sup) {
    const uint32_t region = DB == 2 ? (uint32_t)(sup & 1) * WB_STAGE : 0u;
    if constexpr (!DEEP) sup = sup < n_kb ? sup : n_kb - 1;
    const int kb = k0 + sup * KB;
    static_assert(CP_B == 4, "dma16_x4 makes four copies");
    if (wnat) {   // one 4 KB block, copied as it lies
      dma16_x4(rw, lds_b + region, w_off[0] | ((wave_live && kb < k_hi) ? 0u : kOob), (uint32_t)(sup0 + sup) << 12);
      return;
    }
#pragma unroll
    for (int j = 0; j < CP_B; ++j) {
      const uint32_t bkill = (wave_live && kb + w_kpart(j) < k_hi) ? 0u : kOob;
      dma16(rw, lds_b + region + j * 1024, w_off[j] | bkill, (uint32_t)(sup0 + sup) << w_stage_shift);
    }
  };
  uint4 raw[NF][2];
  float scf[NF][2];      // 2^(e-127) as a float
  // registers <- this wave's weights and scales of super-stage `sup`
  auto load_b = [&](int sup) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int pos = f * 32 + c32;
        const int rot = ((pos >> 2) & 3) ^ (f << 1);   // slot of part p of position pos: p ^ rot
        raw[f][q] = *(const uint4 *)(bbuf + (DB == 2 ? (sup & 1) * WB_STAGE : 0) + pos * 64 + (((2 * q + h) ^ rot) * 16));
        // group kg = 4*sup + 2q + h of this lane's column.  Strided: byte kg, kept inside the column's G bytes
        // (groups past the end of K meet zero codes and zero activations; their scale only has to be some finite
        // value of this column).  Pre-shuffled: byte 256*(kg/8) + 64*(kg%4) + 2*((kg%8)/4); the padding up to a
        // multiple of 8 groups is stored (zeros), so nothing is clamped.
        // (K groups: a group's pairs past the end of K hold zero codes and meet the last pair's scales)
        const int sg = KS > 1 ? (sup0 + sup < n_kb_all ? sup0 + sup : n_kb_all - 1) : sup;
        const int sup_off = cdna4 ? (sg >> 1) * 256 + (sg & 1) * 2 : sg * 4;  // wave uniform
        int kg_off = sup_off + sc_lane_off[q];
        kg_off = kg_off < sc_clamp ? kg_off : sc_clamp;
        uint32_t sbyte;
        if constexpr (SC_LDS) sbyte = lds_sc[sc_col_off[f] + kg_off];
        else if (cdna4) sbyte = s_base[sc_col_off[f] + kg_off];
        else sbyte = s_base[(int64_t)(col0 + f < N ? col0 + f : N - 1) * a.w_mx_stride_n + kg_off];
        scf[f][q] = bits_to_f32(sbyte << 23);
      }
  };

  auto compute = [&](int it, auto qc) {
    constexpr int q = decltype(qc)::value;
    if (!wave_live) return;
    const uint8_t *buf = lds + a_slot(it) * A_STAGE;
    auto read_frags = [&](int s, frag_t *af) {
      const int slot = (h * 4 + s) ^ ((c32 >> 1) & 7);
#pragma unroll
      for (int i = 0; i < NFR; ++i) af[i] = *(const frag_t *)(buf + (i * 32 + c32) * A_ROW_BYTES + slot * 16);
    };
    frag_t af[2][NFR];
    read_frags(0, af[0]);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (s < 3) read_frags(s + 1, af[(s + 1) & 1]);
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const uint4 r = raw[f][q];
        const uint32_t codes = s == 0 ? r.x : (s == 1 ? r.y : (s == 2 ? r.z : r.w));
        const frag_t bf = M::expand(codes, scf[f][q]);
#pragma unroll
        for (int i = 0; i < NFR; ++i) acc[i][f] = M::mma(af[s & 1][i], bf, acc[i][f]);
      }
    }
  };

  typedef std::integral_constant<int, 0> Even;
  typedef std::integral_constant<int, 1> Odd;
  // (the scales of the whole tile are first read in stage 0: requested behind that stage's own copies, before any later one)
  issue_b(0);
  rows_known(std::integral_constant<int, CP_B>{});
  issue_a(0);
  if constexpr (SC_LDS) stage_scales();
  if constexpr (DEEP) {
    // Stage s requests the activations of stage s + DA - 1, an even stage after them the weights of pair s/2 + DB
    // (a weight region is free once its pair's weights are in registers).  Copies complete in the order of their
    // requests: a stage waits until only the requests made after the ones it needs are outstanding
    // (ring_outstanding).  The requests before the loop are those of the stages before 0, in the same order, so the
    // counts hold from the first stage on.
    // (The first stage's own copies, and the tile's scales, have been requested above.)
    constexpr int PRE = DA - 1 > 2 * DB ? DA - 1 : 2 * DB;
#pragma unroll
    for (int j = -PRE; j < 0; ++j) {
      if (j + DA - 1 > 0) issue_a(j + DA - 1);
      if (j % 2 == 0 && j / 2 + DB > 0) issue_b(j / 2 + DB);
    }
    const int n_stage = 2 * n_sup;   // (the same trip count, and barriers, for every group)
    for (int it = 0; it < n_stage; it += 2) {
      wait_vmcnt<ring_outstanding(DA, DB, CP_A, CP_B, false)>();
      sync_threads();
      load_b(it >> 1);
      issue_a(it + DA - 1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // weights are in registers: the region may be refilled
      issue_b((it >> 1) + DB);
      compute(it, Even{});
      if (it + 1 < n_stage) {
        wait_vmcnt<ring_outstanding(DA, DB, CP_A, CP_B, true)>();
        sync_threads();
        issue_a(it + DA);
        compute(it + 1, Odd{});
      }
    }
  } else {
    for (int it = 0; it < n_ka; it += 2) {
      wait_dma();
      sync_threads();
      load_b(it >> 1);
      issue_a(it + 1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // weights are in registers: the region may be refilled
      issue_b((it >> 1) + 1);
      compute(it, Even{});
      if (it + 1 < n_ka) {
        // the weight copies just issued (4, after the activation stage it + 1) are not needed before the next
        // even stage and take the longest (weights stream from HBM, activations mostly hit L2): leave them in flight
        wait_vmcnt<CP_B>();
        sync_threads();
        issue_a(it + 2);
        compute(it + 1, Odd{});
      }
    }
  }
  wait_dma();

  if constexpr (KS > 1) {
    sync_threads();   // (the pipelines are dead: every copy has landed and every operand has been read)
    if (!k_groups_add<KS, NS>(acc[0], lds_wg, grp, wave)) return;
  }
  // (the wave's own weight region is free by now: its table goes there)
  uint8_t *tab = KS > 1 ? lds_wg + wave * 4096 : lds + DA * A_STAGE + wave * 4096;
  static_assert(epilogue_table_bytes(NFR) <= 4096, "a wave's table fits its weight region");
  tile_epilogue<NFR, ACT, XDT, false>(kernel_args_late(), t, acc, tab);
}

// Row fragments a workgroup can hold: a 128-row block of 16-bit activations also takes a remainder of
// up to 32 rows (fifth fragment); the fp8 path keeps four (its A operands are twice as wide).
template <int XDT, int BM>
struct TileShape {
  static constexpr int EXTRA = (BM == 128 && !is_fp8(XDT)) ? 32 : 0;
  static constexpr int MF = BM <= 32 ? 1 : (BM + EXTRA) / 32;
  static constexpr int LDS_ROWS = 32 * MF;
};

// BM: block size of the ragged schedule the kernel consumes (16..128).
template <int XDT, int BM, int ACT, bool SC_LDS, int KS = 1, int NS = 4>
TAMD_DEVICE void tile_entry(const tamd_matmul_args &a, int grid_n, int64_t grid_total, int group_m, uint8_t *lds) {
  typedef TileShape<XDT, BM> S;
  Tile t;
  if (group_m < 0) {  // from the slices' sizes; up to -group_m blocks of an expert together
    if (!locate_tile_live<BM, S::EXTRA>(a, grid_n, -group_m, t)) return;
  } else if (!locate_tile<BM, S::EXTRA>(a, grid_n, grid_total, group_m, t)) return;
  t.n0 = t.n0 / BLOCK_N * (64 * NS);
  const int nfr = (t.rows + 31) / 32;  // active row fragments (workgroup uniform)
#define TAMD_CASE(n)                                                                     \
  case n:                                                                                \
    if constexpr (n <= S::MF) run_tile<XDT, n, S::LDS_ROWS, ACT, SC_LDS, KS, NS>(a, t, lds); \
    break;
  switch (nfr) { TAMD_CASE(1) TAMD_CASE(2) TAMD_CASE(3) TAMD_CASE(4) TAMD_CASE(5) }
#undef TAMD_CASE
}

template <int XDT, int BM, int ACT, bool SC_LDS>
__global__ __launch_bounds__(256, 2) void mm_x16_mxfp4_kernel(tamd_matmul_args a, int grid_n, int64_t grid_total,
                                                                  int group_m) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  tile_entry<XDT, BM, ACT, SC_LDS>(a, grid_n, grid_total, group_m, lds);
}

// K groups: KS x NS waves per tile of at most 32 rows and NS strips, scales of the tile in LDS (see pipe_shape).
template <int XDT, int BM, int ACT, int KS, int NS>
__global__ __launch_bounds__(kWave * NS * KS, 1) void mm_x16_mxfp4_kgroups_kernel(tamd_matmul_args a, int grid_n, int64_t grid_total,
                                                                            int group_m) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  tile_entry<XDT, BM, ACT, true, KS, NS>(a, grid_n, grid_total, group_m, lds);
}

// Whether a problem takes locate_tile_live: it is ragged and the experts fit the lanes.
inline bool counts_live_blocks(const tamd_matmul_args &a) { return a.block_schedule && a.n_experts <= kWave * kLivePerLane; }

// Blocks of up to 64 rows: moe_matmul_mx.h.
template <int XDT, int BM, int ACT>
int launch_mx(const tamd_matmul_args &a, int grid_m, hipStream_t st);

template <int XDT, int BM, int ACT>
int launch_x16_act(const tamd_matmul_args &a, int grid_m, hipStream_t st) {
  constexpr int LDS_ROWS = TileShape<XDT, BM>::LDS_ROWS;
  int grid_n = (a.N + BLOCK_N - 1) / BLOCK_N;
  int64_t total = (int64_t)grid_m * grid_n;
  if (total <= 0) return 0;
  int64_t launch = ((total + 7) / 8) * 8;
  if (launch > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
  const int64_t G = a.K / 32;
  const bool cdna4 = a.w_mx_layout == TAMD_SCALE_CDNA4;
  const int64_t sc_bytes = (BLOCK_N * (cdna4 ? (G + 7) / 8 * 8 : G) + 1023) / 1024 * 1024;  // whole 1 KB copies
  const bool dense_sc = cdna4 || (a.w_mx_stride_k == 1 && a.w_mx_stride_n == G && a.w_mx_stride_e % 4 == 0 &&
                                  aligned(a.w_mx_scale, 4) && (BLOCK_N * G) % 4 == 0);
  // row blocks walked together: as many as one expert (or batch entry) has, while their activation
  // rows (BM x K each) fit comfortably in one XCD's 4 MB L2
  const int64_t rows_per_slice = a.block_schedule ? a.M / a.n_experts : a.M;
  int64_t group_m = rows_per_slice / BM;
  const int64_t fit = (int64_t)(2.5 * 1024 * 1024) / ((int64_t)BM * a.K * 2);
  group_m = group_m > fit ? fit : group_m;
  group_m = group_m < 1 ? 1 : (group_m > 16 ? 16 : group_m);
  if (counts_live_blocks(a)) group_m = -group_m;
  if constexpr (BM <= 32) {
    // Fewer tiles than CUs: K groups, so that every SIMD of the CUs that do get a tile holds two to four waves (the groups' pipelines and
    // the tile's scales have to fit one CU's LDS).
    // Up to half as many tiles as CUs: tiles of 128 columns on twice as many CUs, eight groups, K of 928 to 7168.  A wave then has half the
    // stages to wait for; against four groups on 256 columns 300 products take 0.57 to 0.95 of the time (256 x 2048 x 4096, block layout,
    // 13.4 -> 11.5 us; 208 x 2656 x 2848 19.9 -> 14.3; 46 rows of 3 slices, 6496 x 352, 32.5 -> 19.0).  Shorter K pays for the exchange of
    // the partial sums more than it gains (K 800 1.0 to 1.1 of launch_mx's time, 500 1.25).
    // Four groups and two such tiles per CU for up to 256 tiles: 0.95 to 1.1, not taken.
    // Else two groups on 256 columns from K 1312 on (over 700 layers with up to 256 tiles of 32 rows: without groups 0.96 of the time at K
    // 1200, 1.06 at 2100, 1.2 at 3600, 1.35 at 5000).
    int cus = 0;
    if (int rc = cu_count(cus)) return rc;
    const int64_t pairs = (a.K + KB - 1) / KB;
    constexpr size_t PIPE8 = 8 * (size_t)pipe_shape(LDS_ROWS, 8, 2).bytes, PIPE2 = 2 * (size_t)pipe_shape(LDS_ROWS, 2).bytes;
    const int64_t sc_half = (sc_bytes / 2 + 1023) / 1024 * 1024;
    if (dense_sc && pairs >= 8 && total * 2 <= cus && PIPE8 + sc_half <= 156 * 1024) {
      auto kk = mm_x16_mxfp4_kgroups_kernel<XDT, BM, ACT, 8, 2>;
      if (int rc = raise_lds_limit_once((const void *)kk)) return rc;
      const int grid128 = (a.N + 127) / 128;
      const int64_t tiles = (int64_t)grid_m * grid128;
      kk<<<dim3((unsigned)((tiles + 7) / 8 * 8)), 1024, PIPE8 + sc_half, st>>>(a, grid128, tiles, (int)group_m);
      return launch_status();
    }
    if (dense_sc && pairs >= 11 && total <= cus && PIPE2 + sc_bytes <= 156 * 1024) {
      auto kk = mm_x16_mxfp4_kgroups_kernel<XDT, BM, ACT, 2, 4>;
      if (int rc = raise_lds_limit_once((const void *)kk)) return rc;
      kk<<<dim3((unsigned)launch), 512, PIPE2 + sc_bytes, st>>>(a, grid_n, total, (int)group_m);
      return launch_status();
    }
  }
  if constexpr (BM <= 32) {
    // Weights of slices of one row block whose columns do not start on 64 bytes: pieces of 64 bytes of a column, two and more stages ahead,
    // instead of launch_mx's pieces of 128.  The other way round where columns are aligned, where slices share their weights' lines between
    // row blocks, with pre-shuffled scales, and for short K (953 rows of 64 slices, 2496 x 3552: 77 us against 104; 539 x 2 of 60, 1024 x
    // 5488, aligned: 48 against 38; 161 x 4 of 60, 3776 x 5488: 182 against 242; 1159 of 60, 5024 x 1616: 78 against 91; 157 x 2 of 16, 992
    // x 1392 11.5 against 10.7).
    constexpr int PIPE_BYTES = pipe_shape(LDS_ROWS).bytes;
    if (a.block_schedule && rows_per_slice <= LDS_ROWS && a.w_layout != TAMD_W_CDNA4_BLOCKS && a.w_stride_n % 64 != 0 && a.K > 1024 &&
        !cdna4 && dense_sc && PIPE_BYTES + sc_bytes <= 156 * 1024) {
      auto kern = mm_x16_mxfp4_kernel<XDT, BM, ACT, true>;
      if (int rc = raise_lds_limit_once((const void *)kern)) return rc;
      kern<<<dim3((unsigned)launch), 256, PIPE_BYTES + sc_bytes, st>>>(a, grid_n, total, (int)group_m);
      return launch_status();
    }
  }
  if constexpr (BM <= 64) {
    return launch_mx<XDT, BM, ACT>(a, grid_m, st);
  } else {
    // scales of a tile are staged in LDS when they are dense ([N][K/32]) or pre-shuffled and two workgroups still fit a CU
    constexpr int PIPE_BYTES = pipe_shape(LDS_ROWS).bytes;
    const bool sc_in_lds = dense_sc && PIPE_BYTES + sc_bytes <= 80 * 1024;
    auto kern = sc_in_lds ? mm_x16_mxfp4_kernel<XDT, BM, ACT, true> : mm_x16_mxfp4_kernel<XDT, BM, ACT, false>;
    if (int rc = raise_lds_limit_once((const void *)kern)) return rc;
    kern<<<dim3((unsigned)launch), 256, PIPE_BYTES + (sc_in_lds ? sc_bytes : 0), st>>>(a, grid_n, total, (int)group_m);
    return launch_status();
  }
}

// Whether a dense / batched problem has enough 32-row tiles for the tiled kernels: more than `tiles`.  Fewer run as 16-row blocks through
// the streaming kernel, whose units of 16 columns reach every CU.  (900 products, time in tiles that K groups share over the streaming
// kernel's: 16-bit rows, K up to 2048, 33 to 48 tiles 1.1 to 1.25, 65 to 72 0.94 to 1.04, 73 to 80 0.75 to 0.95; longer K, 17 to 32 1.06 to
// 1.28, 49 to 64 0.93 to 1.06, 65 to 80 0.7 to 0.9.  fp8 rows would be faster in tiles from 24 on, 0.7 to 0.95, but their products are
// exact in the streaming kernel: 5e-9 off 64-bit sums, 4e-6 in tiles.)
inline bool dense_prefers_tiles(const tamd_matmul_args &a, int tiles) {
  return (int64_t)((a.M + 31) / 32) * a.n_experts * ((a.N + BLOCK_N - 1) / BLOCK_N) > tiles;
}
// Row blocks of a dense / batched problem (block_m == 0 on entry of a dispatcher).
inline void dense_grid(const tamd_matmul_args &a, int &block_m, int &grid_m) {
  if (block_m != 0) return;
  int cus = 0;
  if (cu_count(cus) != 0) cus = 256;
  block_m = dense_block_m(a, cus);
  grid_m = ((a.M + block_m - 1) / block_m) * a.n_experts;
}

// The tiled kernels of one activation type and one epilogue activation.  The two activations are compiled in
// translation units of their own (moe_matmul_<type>.hip: none, moe_matmul_<type>_swiglu.hip: SwiGLU), which
// is all that separates them: each unit holds 16 kernels of up to five tile sizes with all the forms of their epilogue.
template <int XDT, int ACT>
int dispatch_x16_act(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  dense_grid(a, block_m, grid_m);
  switch (block_m) {
    case 16: return launch_x16_act<XDT, 16, ACT>(a, grid_m, st);
    case 32: return launch_x16_act<XDT, 32, ACT>(a, grid_m, st);
    case 64: return launch_x16_act<XDT, 64, ACT>(a, grid_m, st);
    case 128: return launch_x16_act<XDT, 128, ACT>(a, grid_m, st);
    default: return TAMD_E_UNSUPPORTED;
  }
}
int tiled_mm_swiglu_bf16(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st);
int tiled_mm_swiglu_f16(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st);

}  // namespace tamd
