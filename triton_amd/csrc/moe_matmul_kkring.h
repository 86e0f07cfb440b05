// Grouped (ragged) matmul of 16-bit activations x unquantised weights of their type, both contiguous along K: a persistent kernel whose
// copies never stop at the end of a tile.
//
// Bound by HBM up to some 150 rows per slice, then by the matrix units.  One tile per workgroup (moe_matmul_kk.h) starts with an empty
// pipeline, exchanges partial sums and ends with an epilogue beside which it copies nothing, and its waves wait for their own copies
// between the products (one holds its wave for a hundred cycles): 4.3 TB/s of the 6.4 to 7 that copies alone read, matrix cores busy 29 %
// of the cycles.  Here a workgroup owns a CU and walks over tiles:
//   * four waves copy and do nothing else, through a ring of three stages (64 K of a tile's rows and columns, 128-byte lines of both) that
//     runs on into the next tile; they find the tiles and leave them for the others in LDS;
//   * eight waves multiply, two halves of the row fragments times four strips of 64 columns, and finish the tile from registers; the two
//     stages ahead cover the copies for most of that time;
//   * weights of slices with one row block are copied non-temporally where their columns are whole lines and the call reads more than the
//     caches keep (300 tokens x 4 of 32 slices, 2880 -> 2 x 2880: 188 -> 170 us; of columns off the lines 137 -> 150 and 28 -> 34, so not there);
//   * tiles of fewer strips where that fills the rounds over the workgroups (1021 tokens x 4 of 32: 228 -> 216); blocks of one slice are of one
//     size.
// Sums.  In blocks of 160 rows one float32 accumulator for all of K, where the tiled kernel has two (of either half of every stage): a wave has
// the registers for one.  Results of K 2880 against 64-bit sums (2-norm): bf16 1.662372e-3 from both, which is what rounding the exact sums gives;
// f16 2.077690e-4, 2.077689e-4 from the tiled kernel, 2.077687e-4 from rounding alone; of K 5376 bf16 1.6563609e-3 all three, f16 2.0717160e-4,
// 2.0717133e-4 and 2.0717109e-4.  Blocks of 64 have the registers for two sets: products below the line of kk_ring_rows are summed as the tiled
// kernels do, up to ten stages in the same two sums to the bit, beyond in four, one for each quarter of K, which are those of the narrow
// tiles to the bit.  Results that are not the 64-bit sum rounded, f16, tiled kernels / one sum / now: 8 slices of 55 rows, 576 -> 2152, of
// 951184 743 / 761 / 743; 8 of 12, 3784 -> 2560, of 238080 347 / 446 / 347 (narrow tiles); 8 of 60, 2544 -> 1856, of 885312 1406 / 1451 / 1195.  Of 100 products
// of 3 to 200 rows per slice, K 256 to 5600, 16 of the 19 below the line had more than the tiled kernels with one sum, none now.  The second set costs up to 3 %
// of a short tile.
// Blocks of 160 rows, the most that three stages have LDS for (128: 1021 tokens 225, 2000 tokens 357 where 160 take 311; 96: 266 and 393);
// of 64 where slices are smaller, whose copies of rows that are not there cost 2 to 4 % (300 tokens: 170 -> 165; blocks of 32 with a ring
// of four: 208).
//
// Layers of 32 slices, 2880 -> 2880, bf16, tokens x 4, tiled kernel -> now, us: 300 tokens 355 -> 279, 600 349 -> 316, 1021 392 -> 372,
// 2000 612 -> 536; 4000 tokens x 4 of 16 slices 1056 -> 797.  What is left of the 1021 tokens' time without one part of the work: without
// the products 0.98, without the copies of the rows 0.91, without the stores 0.92.  Matrix cores are busy 28 % of the cycles (25 before),
// the address units 80 % (63): 1.12 GB are fetched for 1.06 of weights.
#pragma once
#include <algorithm>
#include <type_traits>

#include "moe_matmul_kk.h"

namespace tamd {

constexpr int kKKRingCopiers = 4, kKKRingPerLane = 4;   // copying waves; slices that a lane of them holds

template <int XDT, int MF_>
struct KKRingShape {
  typedef typename KK<XDT>::M M;
  typedef typename KK<XDT>::frag_t frag_t;
  static constexpr int MF = MF_, ROWS = 32 * MF, KS = KK<XDT>::KS;
  static constexpr int N0 = (MF + 1) / 2;                                    // row fragments of a wave, at most
  static constexpr bool TWO = N0 == 1;                                       // registers for two sums
  static constexpr int STAGE = (ROWS + BLOCK_N) * 128, RING = 3;
  static constexpr int COPIES = 8 + MF;                                      // of a copying wave and stage
  static constexpr int CONSUMERS = 8, THREADS = (CONSUMERS + kKKRingCopiers) * kWave;
  static constexpr int TABLE = N0 * 32 * 12;                                 // destinations, betas, gammas of half of the rows
  static constexpr int TABLE_AT = RING * STAGE, INDEX_AT = TABLE_AT + 2 * TABLE, TILE_AT = INDEX_AT + kKKRingCopiers * 256;
  static constexpr int LDS = TILE_AT + 4 * 32 + 16;
  static_assert(LDS <= 160 * 1024 && (RING - 1) * COPIES < 64, "one workgroup per CU, copies that vmcnt can count");
  static_assert(RING * KS <= 256, "a tile has RING stages and more (kk_ring_applicable): its row indices are requested a tile ahead");
};

// A tile: up to four strips of 64 columns from t.n0 on.
struct KKRingTile {
  Tile t;
  int strips;
  bool once;   // no other row block reads its weights
};

// The tiles of a workgroup, as a copying wave knows them: lane l holds the slices [l n, (l + 1) n).
template <int ROWS>
struct KKRingWork {
  int rows[kKKRingPerLane], offs[kKKRingPerLane], before;   // (blocks before the lane's)
  int n_lane, group, n_tiles;
  uint32_t strips, gn, first, step;
  static TAMD_DEVICE int blocks(int n) { return (n + ROWS - 1) / ROWS; }

  template <typename Args>
  TAMD_DEVICE void init(const Args &a, int group_) {
    const int lane = threadIdx.x % kWave, E = a.n_experts;
    n_lane = (E + kWave - 1) / kWave, group = group_;
    int own = 0;
#pragma unroll
    for (int u = 0; u < kKKRingPerLane; ++u) {
      rows[u] = offs[u] = 0;
      const int e = lane * n_lane + u;
      if (u < n_lane && e < E) rows[u] = a.slice_sizes[e], offs[u] = a.slice_offs[e];
    }
#pragma unroll
    for (int u = 0; u < kKKRingPerLane; ++u) own += blocks(rows[u]);
    const int incl = wave_incl_scan(own);
    before = incl - own;
    const uint32_t n_blocks = (uint32_t)__builtin_amdgcn_readlane(incl, kWave - 1), wgs = gridDim.x;
    strips = (uint32_t)(a.N + 63) / 64;
    gn = (strips + 3) / 4;
    if (n_blocks > 0) {   // narrower tiles where they fill the rounds over the workgroups
      const uint32_t rounds = (n_blocks * gn + wgs - 1) / wgs, fill = rounds * wgs / n_blocks;
      gn = fill < strips ? fill : strips;
    }
    const uint32_t total = n_blocks * gn, per_xcd = (total + 7) / 8, xcd = blockIdx.x % 8;
    const uint32_t begin = xcd * per_xcd < total ? xcd * per_xcd : total, end = begin + per_xcd < total ? begin + per_xcd : total;
    step = gridDim.x / 8;
    first = begin + blockIdx.x / 8;
    n_tiles = first < end ? (int)((end - first + step - 1) / step) : 0;
  }

  TAMD_DEVICE void tile(int i, KKRingTile &k) const {
    const int lane = threadIdx.x % kWave;
    const uint32_t idx = first + (uint32_t)i * step;
    const int m = (int)(idx / gn);
    int at = before, e = 0, n = 0, off = 0, lead = 0;
    bool here = false;
#pragma unroll
    for (int u = 0; u < kKKRingPerLane; ++u) {
      const int c = blocks(rows[u]);
      if (m >= at && m < at + c) here = true, e = lane * n_lane + u, n = rows[u], off = offs[u], lead = at;
      at += c;
    }
    const int src = __builtin_ctzll(__ballot(here));   // (exactly one lane)
    k.t.expert = __builtin_amdgcn_readlane(e, src);
    k.t.z = 0;
    k.t.start_m = __builtin_amdgcn_readlane(off, src);
    const int slice = __builtin_amdgcn_readlane(n, src);
    const uint32_t local = idx - (uint32_t)__builtin_amdgcn_readlane(lead, src) * gn;
    const uint32_t b = (uint32_t)blocks(slice);
    k.once = b == 1;
    uint32_t g = b < (uint32_t)group ? b : (uint32_t)group, blk, col;
    if (g > 1) {   // (as in locate_tile_live)
      g = (b + (b + g - 1) / g - 1) / ((b + g - 1) / g);
      const uint32_t gi = local / (g * gn), r = local - gi * g * gn;
      const uint32_t size = b - gi * g < g ? b - gi * g : g;
      col = r / size;
      blk = gi * g + (r - col * size);
    } else {
      blk = local / gn;
      col = local - blk * gn;
    }
    const uint32_t strip0 = col * strips / gn;
    k.strips = (int)((col + 1) * strips / gn - strip0);
    k.t.n0 = (int)strip0 * 64;
    // a slice's blocks are of about one size, whole fragments
    const int per = (int)(((uint32_t)slice + b - 1) / b + 31) & ~31;
    k.t.off_m = (int)blk * per;
    const int left = slice - k.t.off_m;
    k.t.rows = left > per ? per : left;
  }
};

// Copying waves: strip w's columns, rows 8 w .. of every row fragment.  Stage s goes to slot s % RING and is requested RING - 1 stages
// ahead; copies complete in the order of their requests, so a stage has landed once only those of the stages after it are outstanding (the
// indices of the next tile's rows, requested behind a tile's first stage, only make that wait a little longer).
template <int XDT, int MF, typename Args>
TAMD_DEVICE void kk_ring_copy(const Args &a, int group, bool nt, uint8_t *lds) {
  typedef KKRingShape<XDT, MF> S;
  constexpr uint32_t kOob = 0x7FFFFFFFu;
  constexpr int RING = S::RING, NB = 8;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) - S::CONSUMERS, lane = threadIdx.x % kWave;
  const int K = a.K, N = a.N, n_k = (K + S::KS - 1) / S::KS;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
  KKRingWork<S::ROWS> work;
  work.init(a, group);
  if (w == 0 && lane == 0) *(int *)(lds + S::TILE_AT + 4 * 32) = work.n_tiles;
  KKRingTile k, next;
  // (what the multiplying waves have to know of it, some stages before they come to it)
  auto publish = [&](int i, const KKRingTile &v) {
    if (w == 0 && lane == 0) {
      int4 *to = (int4 *)(lds + S::TILE_AT + (i & 3) * 32);
      to[0] = int4{v.t.expert, v.t.start_m, v.t.off_m, v.t.rows};
      to[1] = int4{v.t.n0, v.strips, 0, 0};
    }
  };
  if (work.n_tiles > 0) {
    work.tile(0, next);
    publish(0, next);
  }
  sync_threads();
  if (work.n_tiles == 0) return;
  // chunks of row or column r lie at slot chunk ^ ((r >> 1) & 7)
  const int rin = lane / 8, a_rin = w * 8 + rin;
  const int a_chunk = (lane % 8) ^ ((a_rin >> 1) & 7), b_chunk[2] = {(lane % 8) ^ (rin >> 1), (lane % 8) ^ (4 + (rin >> 1))};
  const uint32_t x_rows = gather_limit(a);
  const int idx_at = S::INDEX_AT + w * 256;
  // lane 8 i + r asks for the index of the wave's row r in fragment i
  auto request_rows = [&](const Tile &t) {
    if (!a.gather_indx) return;
    const v4i_t rg = make_rsrc(a.gather_indx + t.start_m + t.off_m, (uint32_t)__builtin_amdgcn_readfirstlane(t.rows) * 4u);
    dma4(rg, lds_base + idx_at, lane < 8 * MF ? (uint32_t)((lane / 8) * 32 + w * 8 + lane % 8) * 4u : kOob, 0);
  };
  request_rows(next.t);
  const v4i_t rx = make_rsrc(a.x, kOob);
  const uint8_t *w_base = nullptr;
  uint32_t a_off[MF], b_off[NB];
  bool once = false;
  int i_tile = 0, p = 0;
  auto issue = [&](int slot) {
    const bool fresh = p == 0;
    if (fresh) {
      k = next;
      w_base = (const uint8_t *)a.w + (int64_t)k.t.expert * a.w_stride_e * 2;
      once = nt && k.once;
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int q = u * 8 + rin, col = k.t.n0 + w * 64 + 2 * (q % 32) + q / 32;   // position 32 f + c holds column 2 c + f
        b_off[u] = w < k.strips && col < N ? (uint32_t)col * (uint32_t)(a.w_stride_n * 2) + b_chunk[u & 1] * 16 : kOob;
      }
    }
    const v4i_t rw = make_rsrc(w_base, kOob);
    const uint32_t sb = lds_base + slot * S::STAGE;
    const int kb = p * S::KS;
    const uint32_t kill[2] = {kb + b_chunk[0] * 8 < K ? 0u : kOob, kb + b_chunk[1] * 8 < K ? 0u : kOob};
    const uint32_t to_b = sb + S::ROWS * 128 + w * 64 * 128;
    if (once) {
#pragma unroll
      for (int u = 0; u < NB; ++u) dma16_nt(rw, to_b + u * 1024, b_off[u] | kill[u & 1], kb * 2);
    } else {
#pragma unroll
      for (int u = 0; u < NB; ++u) dma16(rw, to_b + u * 1024, b_off[u] | kill[u & 1], kb * 2);
    }
    if (fresh) {
      if (a.gather_indx && i_tile == 0) wait_vmcnt<NB>();
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        const int r = i * 32 + a_rin;
        const uint32_t src = a.gather_indx ? *(const uint32_t *)(lds + idx_at + (i * 8 + rin) * 4) : (uint32_t)(k.t.start_m + k.t.off_m + r);
        a_off[i] = r < k.t.rows && src < x_rows ? src * (uint32_t)(a.x_stride_m * 2) + a_chunk * 16 : kOob;
      }
    }
    const uint32_t kill_a = kb + a_chunk * 8 < K ? 0u : kOob;
#pragma unroll
    for (int i = 0; i < MF; ++i) dma16(rx, sb + i * 4096 + w * 1024, a_off[i] | kill_a, kb * 2);
    if (fresh && i_tile + 1 < work.n_tiles) {
      work.tile(i_tile + 1, next);
      publish(i_tile + 1, next);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (this tile's indices have been read)
      request_rows(next.t);
    }
    if (++p == n_k) p = 0, ++i_tile;
  };
  const int stages = work.n_tiles * n_k;
  int slot = 0, s = 0;
  auto advance = [&]() { slot = slot + 1 == RING ? 0 : slot + 1; };
#pragma unroll 1
  for (int q = 0; q < RING - 1; ++q) {   // (a tile has at least RING stages)
    issue(slot);
    advance();
  }
#pragma unroll 1
  for (; s + RING - 1 < stages; ++s) {
    wait_vmcnt<(RING - 2) * S::COPIES>();
    sync_threads();
    issue(slot);
    advance();
  }
  // the last RING - 1 stages, with nothing left to request
  static_assert(RING == 3, "stages written out below");
  wait_vmcnt<S::COPIES>();
  sync_threads();
  wait_vmcnt<0>();
  sync_threads();
}

// A multiplying wave's part of a tile, NFR row fragments of one strip: the K loop, into `sums` float32 sums (kk_ring_sums), and the epilogue.
template <int XDT, int MF, int NFR, int ACT, typename Args>
TAMD_DEVICE void kk_ring_products(const Args &a, const Tile &t, int half, int first_row, int sums, uint8_t *lds, int &slot) {
  typedef KKRingShape<XDT, MF> S;
  const int strip = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) & 3, lane = threadIdx.x % kWave;
  const int c32 = lane % 32, h = lane / 32, n_k = (a.K + S::KS - 1) / S::KS;
  EpilogueOperands<NFR> ops;
  epilogue_operands<NFR, true>(kernel_args_late(), t, ops);
  const uint32_t at = (uint32_t)(c32 * 128 + ((4 * h) ^ ((c32 >> 1) & 7)) * 16);
  const uint32_t a_lane = at + (uint32_t)first_row * 128, b_lane = at + (uint32_t)(S::ROWS + strip * 64) * 128;
  static_assert(S::STAGE % 128 == 0, "chunks are picked by the low seven address bits");
  f32x16_t acc[NFR][NF];
#pragma unroll
  for (int i = 0; i < NFR; ++i)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[i][f][j] = 0.f;
  f32x16_t other[S::TWO ? NFR : 1][NF];   // of the upper halves of the stages, or of the parts that are through
  if constexpr (S::TWO) {
#pragma unroll
    for (int i = 0; i < NFR; ++i)
#pragma unroll
      for (int f = 0; f < NF; ++f) other[i][f] = acc[i][f];
  }
  auto add = [&](f32x16_t (&to)[NFR][NF], const f32x16_t (&from)[NFR][NF]) {
#pragma unroll
    for (int i = 0; i < NFR; ++i)
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int j = 0; j < 16; ++j) to[i][f][j] += from[i][f][j];
  };
  auto stage = [&](auto halves) {
    sync_threads();
    const uint32_t buf = (uint32_t)slot * S::STAGE;
    slot = slot + 1 == S::RING ? 0 : slot + 1;
    typename S::frag_t af[2][NFR], bf[2][NF];
    auto read = [&](int v) {   // the operands of 16 K: chunk v of either half of the 64
#pragma unroll
      for (int f = 0; f < NF; ++f)
        bf[v & 1][f] = __builtin_bit_cast(typename S::frag_t, *(const uint4 *)(lds + ((buf + b_lane) ^ (uint32_t)(v * 16)) + f * 4096));
#pragma unroll
      for (int i = 0; i < NFR; ++i)
        af[v & 1][i] = __builtin_bit_cast(typename S::frag_t, *(const uint4 *)(lds + ((buf + a_lane) ^ (uint32_t)(v * 16)) + i * 4096));
    };
    read(0);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (v < 3) read(v + 1);
#pragma unroll
      for (int i = 0; i < NFR; ++i)
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          f32x16_t &to = halves.value && v >= 2 ? other[S::TWO ? i : 0][f] : acc[i][f];
          to = S::M::mma(af[v & 1][i], bf[v & 1][f], to);
        }
    }
  };
  if (S::TWO && sums == 2) {
    if constexpr (S::TWO) {
#pragma unroll 1
      for (int p = 0; p < n_k; ++p) stage(std::true_type{});
      add(acc, other);
    }
  } else {
    const int n_part = (n_k + sums - 1) / sums;
    int left = n_part;
#pragma unroll 1
    for (int p = 0; p < n_k; ++p) {
      stage(std::false_type{});
      if constexpr (S::TWO) {
        if (--left == 0 && p + 1 < n_k) {
          left = n_part;
          add(other, acc);
#pragma unroll
          for (int i = 0; i < NFR; ++i)
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[i][f] = f32x16_t{};
        }
      }
    }
    if constexpr (S::TWO) {
      if (sums > 1) add(acc, other);
    }
  }
  // The waves of a half write the same table; all of them have passed a barrier since the last tile's was read.
  uint8_t *tab = lds + S::TABLE_AT + half * S::TABLE;
  NoPace pace;
  const Args &late = kernel_args_late();
  epilogue_table<NFR, 2, true, false>(late, t, ops.dst, ops.beta, ops.gamma, tab);
  if (late.betas || late.gammas) tile_epilogue_t<NFR, ACT, XDT, true, false, false, Args>(late, t, acc, tab, &ops, pace);
  else tile_epilogue_t<NFR, ACT, XDT, false, false, false, Args>(late, t, acc, tab, &ops, pace);
}

// Multiplying waves: two halves of the tile's row fragments, four strips.
template <int XDT, int MF, int ACT, typename Args>
TAMD_DEVICE void kk_ring_compute(const Args &a, int sums, uint8_t *lds) {
  typedef KKRingShape<XDT, MF> S;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), strip = wave & 3, half = wave >> 2;
  const int n_k = (a.K + S::KS - 1) / S::KS;
  sync_threads();
  const int n_tiles = __builtin_amdgcn_readfirstlane(*(const int *)(lds + S::TILE_AT + 4 * 32));
  int slot = 0;
#pragma unroll 1
  for (int i = 0; i < n_tiles; ++i) {
    const int4 *from = (const int4 *)(lds + S::TILE_AT + (i & 3) * 32);
    const int4 lo = from[0], hi = from[1];
    Tile t;
    t.expert = __builtin_amdgcn_readfirstlane(lo.x), t.z = 0;
    t.start_m = __builtin_amdgcn_readfirstlane(lo.y), t.off_m = __builtin_amdgcn_readfirstlane(lo.z);
    t.rows = __builtin_amdgcn_readfirstlane(lo.w), t.n0 = __builtin_amdgcn_readfirstlane(hi.x);
    const int strips = __builtin_amdgcn_readfirstlane(hi.y);
    const int nfr = (t.rows + 31) / 32, n0 = (nfr + 1) / 2, first_row = half ? 32 * n0 : 0, mine = strip < strips ? (half ? nfr - n0 : n0) : 0;
    t.off_m += first_row;
    t.rows = half ? t.rows - first_row : (t.rows < 32 * n0 ? t.rows : 32 * n0);
    if (mine == 0) {
#pragma unroll 1
      for (int p = 0; p < n_k; ++p) sync_threads();
      slot = (slot + n_k) % S::RING;
    } else if (S::N0 == 1 || mine == 1) {
      kk_ring_products<XDT, MF, 1, ACT>(a, t, half, first_row, sums, lds, slot);
    } else if (S::N0 == 2 || mine == 2) {
      kk_ring_products<XDT, MF, (S::N0 < 2 ? S::N0 : 2), ACT>(a, t, half, first_row, sums, lds, slot);
    } else {
      kk_ring_products<XDT, MF, S::N0, ACT>(a, t, half, first_row, sums, lds, slot);
    }
  }
}

template <int XDT, int MF, int ACT>
__global__ __launch_bounds__((KKRingShape<XDT, MF>::THREADS), 1) void mm_kk_ring_kernel(tamd_matmul_args, int group, int nt, int sums) {
  extern __shared__ __attribute__((aligned(128))) uint8_t lds_ring[];
  // (the arguments are read where they are used, see kernel_args_late)
  if (threadIdx.x >= KKRingShape<XDT, MF>::CONSUMERS * kWave) kk_ring_copy<XDT, MF>(kernel_args_late(), group, nt != 0, lds_ring);
  else kk_ring_compute<XDT, MF, ACT>(kernel_args_late(), sums, lds_ring);
}

template <int XDT, int MF, int ACT>
int launch_kk_ring(const tamd_matmul_args &a, hipStream_t st) {
  typedef KKRingShape<XDT, MF> S;
  int cus = 0;
  if (int rc = cu_count(cus)) return rc;
  const int64_t blocks = a.M / S::ROWS + (a.M < a.n_experts ? a.M : a.n_experts), strips = (a.N + 63) / 64;
  const int64_t wgs = (std::min<int64_t>(blocks * strips, cus) + 7) / 8 * 8;
  int64_t group = (a.M / a.n_experts + S::ROWS - 1) / S::ROWS + 1;
  group = group < 2 ? 2 : (group > 8 ? 8 : group);
  auto kern = mm_kk_ring_kernel<XDT, MF, ACT>;
  if (int rc = raise_lds_limit_once((const void *)kern)) return rc;
  const bool lines = aligned(a.w, 128) && (a.w_stride_n * 2) % 128 == 0 && (a.w_stride_e * 2) % 128 == 0;
  const bool nt = lines && live_slices(a) * a.N * ((double)a.K * 2) >= 320.0 * (1 << 20);
  kern<<<dim3((unsigned)wgs), S::THREADS, S::LDS, st>>>(a, (int)group, (int)nt, S::TWO ? kk_ring_sums(a, cus) : 1);
  return launch_status();
}

template <int XDT>
int dispatch_kk_ring(const tamd_matmul_args &a, int rows, hipStream_t st) {
  const bool sw = a.activation == TAMD_ACT_SWIGLU;
  switch (rows) {
    case 64: return sw ? launch_kk_ring<XDT, 2, TAMD_ACT_SWIGLU>(a, st) : launch_kk_ring<XDT, 2, TAMD_ACT_NONE>(a, st);
    case 160: return sw ? launch_kk_ring<XDT, 5, TAMD_ACT_SWIGLU>(a, st) : launch_kk_ring<XDT, 5, TAMD_ACT_NONE>(a, st);
    default: return TAMD_E_UNSUPPORTED;
  }
}

}  // namespace tamd
