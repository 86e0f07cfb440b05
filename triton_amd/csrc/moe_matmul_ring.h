// Grouped (ragged) matmul of up to about 96 rows per slice x MXFP4 weights in 4 KB blocks with pre-shuffled scales, or both strided: a
// persistent kernel whose copies never stop at the end of a tile.
//
// With few rows per slice HBM is the bound, and one tile per workgroup (moe_matmul_mx.h) reaches 5.3 TB/s of the 7 that copies alone read:
// a tile starts with an empty pipeline and ends with an epilogue beside which it copies nothing, 8 of its 46 us, and three such workgroups
// per CU fill only part of one another's gaps.  Here one workgroup owns a CU and walks over its tiles:
//   * four waves copy and do nothing else, through a ring of three to six stages that runs on into the next tile; a stage is its tile's rows,
//     weights and the block scales of both, so that no other wave waits for memory inside the K loop (an ordinary load there is served
//     behind the CU's outstanding copies: row scales loaded by the multiplying waves took 3 000 cycles, with one piece of 256 K in advance
//     every stage waited);
//   * two sets of four waves (one per strip of 64 columns, all rows of the tile) take the tiles in turn: while one multiplies, the other
//     finishes the tile before, one barrier of the stages for every four rows, and requests what its next tile's epilogue needs.  (Eight
//     waves on every tile, epilogue at its end: 3 and 8 % slower on the 509 fp8 and the 2048 packed tokens below.)
//   * the weights of a slice with one row block are read once: non-temporal copies (0.89 of the time on the first of the layers below);
//   * tiles of fewer than four strips where that fills the one or two rounds over the workgroups.
// Barriers of the whole workgroup, one per stage, publish a stage and free the one before.
//
// Strided weights (blocks of up to 64 rows): pieces of 64 bytes per column and 128 K, sixteen bytes of scales per column and 256 K.  They
// read 3 to 4.7 TB/s, by whether a piece crosses a line, as in moe_matmul_mx.h; what is won is the narrower tiles of small calls and, for
// 16-bit rows, multiplying waves that do not copy.  (Scales a dword at a time asked for twice as many lines as the weights, 5 to 15 %
// slower.)  Layers, tiled kernel -> now, us: 100 packed tokens x 4 of 16 slices, 2880 -> 1440, 52.8 -> 48.1; 60 fp8 x 4 of 16, 1760 ->
// 1440, 38.1 -> 34.6; 80 bf16 x 4 of 16, 2048 -> 1024, 44.1 -> 37.4; 512 bf16 x 4 of 60, 2880 -> 2880, 284 -> 271.
//
// Time of a layer (routing, both products, sum), tiled kernels -> now, us: 509 fp8 tokens x 4 of 128 slices, 5760 -> 2880, 643 -> 583;
// 2880 -> 2880, 128 slices: 512 tokens fp8 353 -> 325, MXFP8 363 -> 346, packed 372 -> 343, 1024 fp8 388 -> 374, packed 409 -> 381, 2048
// packed 471 -> 437, fp8 453 -> 434.  (ring_rows in tile_rules.h says which problems.)
//
// What is left of the 509, the 2048 packed and the 2048 fp8 tokens' time without one part of the work: without the products 1.00, 0.99,
// 0.99; without the copies of the rows 0.98, 0.95, 0.89; without the stores 0.92, 0.87, 0.88.  The copies are the bound, and what the
// stores take from them: scattered lines between the reads.  Weights are read once (2.27 GB fetched for 2.26 of weights, 1.26 for 1.13),
// matrix cores are busy 16 to 12 % of the cycles.
#pragma once
#include <algorithm>

#include "moe_matmul_mx.h"

namespace tamd {

constexpr int kRingSlices = 256;   // slices that the table of the work holds
constexpr int kRingProducers = 4;

// Weights of up to four strips, columns' scales: eight blocks of 32 columns x 256 bytes (256 K, also where a stage is 128 K).  A deeper
// ring changes nothing: copies alone reach their rate with two stages in flight, and 5 stages were 1 % faster than 7.

template <int XDT, int MF_, bool XMX = false>
struct RingShape {
  typedef MxShape<XDT, 32> M;
  static constexpr bool FP4 = M::FP4, X16 = M::X16;
  static constexpr int ESZ = M::ESZ, PLANE_K = M::PLANE_K;
  static constexpr int MF = MF_, ROWS = 32 * MF, BM = ROWS;
  static constexpr int KA = FP4 ? 256 : 128;                 // K per stage
  static constexpr int PLANES = KA / PLANE_K, BLOCKS = KA / KB;
  static constexpr int AHEAD = X16 ? 1 : 0;                  // stages past its own whose operands a wave reads
  static constexpr int A_STAGE = PLANES * ROWS * A_ROW_BYTES, B_STAGE = 4 * BLOCKS * 4096;
  // Strided column scales: sixteen bytes of every column from the dword on that holds the first of 256 K (a stage of 128 K: every other one).
  static constexpr bool STRIDED = MF <= 2;                   // (blocks of 96 rows have neither the LDS nor the registers)
  static constexpr int SC_STAGE = STRIDED ? 4096 : 2048;
  // Block scales of the rows (XMX): the dwords that cover a row's bytes of the stage, whatever their alignment, for whole waves of rows.
  static constexpr int XS_WORDS = XMX ? KA / 128 + 1 : 0, XS_WAVES = (MF + 1) / 2, XS_STAGE = XS_WORDS * XS_WAVES * kWave * 4;
  static constexpr int STAGE = A_STAGE + B_STAGE + SC_STAGE + XS_STAGE;
  static constexpr int CONSUMERS = 8, THREADS = (CONSUMERS + kRingProducers) * kWave;   // two sets of four, a wave per strip
  static constexpr int TABLE = epilogue_table_bytes(MF) + BLOCK_N * 4, WORK = 3 * kRingSlices * 4 + 16, INDEX = (kRingProducers + 2) * 2 * 256;
  static constexpr int FIXED = 4 * TABLE + WORK + INDEX;   // (two tables of a set's rows, in turn)
  static constexpr int FIT = (160 * 1024 - FIXED) / STAGE;
  static constexpr int RING = FIT > 5 + AHEAD ? 5 + AHEAD : FIT;
  static constexpr int LDS = RING * STAGE + FIXED;
  static constexpr int COPIES = 4 * BLOCKS + PLANES * MF;   // of a copying wave and stage, without scales
  static_assert(RING >= 2 + AHEAD && (RING - 2) * (COPIES + 1 + XS_WORDS) < 64, "ring does not fit the vmcnt counter");
};

// The tiles of a workgroup: every step-th of its XCD's range, so that the workgroups of an XCD are at about the same slices.
struct RingWork {
  const int32_t *tab;    // LDS: first block, rows, first row of every slice; number of blocks
  int E, group, n_tiles;
  uint32_t strips, gn, first, step;   // strips of 64 columns, column tiles of up to four of them
};

template <int BM>
TAMD_DEVICE int ring_blocks(int rows) { return (rows + BM - 1) / BM; }

// The first wave makes the table (one round trip to memory, see locate_tile_live); every wave then goes by it.
template <int BM, typename Args>
TAMD_DEVICE void ring_work(const Args &a, int group, int32_t *tab, RingWork &w) {
  const int E = a.n_experts;
  if (threadIdx.x < kWave) {
    const int lane = threadIdx.x, n_lane = (E + kWave - 1) / kWave;
    constexpr int PER = kRingSlices / kWave;
    int rows[PER], offs[PER], own = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      rows[u] = offs[u] = 0;
      const int e = lane * n_lane + u;
      if (u < n_lane && e < E) rows[u] = a.slice_sizes[e], offs[u] = a.slice_offs[e];
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) own += ring_blocks<BM>(rows[u]);
    const int incl = wave_incl_scan(own);
    int first = incl - own;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = lane * n_lane + u;
      if (u < n_lane && e < E) {
        tab[e] = first, tab[kRingSlices + e] = rows[u], tab[2 * kRingSlices + e] = offs[u];
        first += ring_blocks<BM>(rows[u]);
      }
    }
    if (lane == kWave - 1) tab[3 * kRingSlices] = incl;
  }
  sync_threads();
  w.tab = tab, w.E = E, w.group = group;
  const uint32_t blocks = (uint32_t)__builtin_amdgcn_readfirstlane(tab[3 * kRingSlices]), wgs = gridDim.x;
  w.strips = (uint32_t)(a.N + 63) / 64;
  w.gn = (w.strips + 3) / 4;
  if (blocks > 0) {   // narrower tiles where they fill one or two rounds (later on they only repeat the rows' copies: 1 % slower)
    const uint32_t rounds = (blocks * w.gn + wgs - 1) / wgs, fill = rounds * wgs / blocks;
    if (rounds <= 2) w.gn = fill < w.strips ? fill : w.strips;
  }
  const uint32_t total = blocks * w.gn, per_xcd = (total + 7) / 8, xcd = blockIdx.x % 8;
  const uint32_t begin = xcd * per_xcd < total ? xcd * per_xcd : total, end = begin + per_xcd < total ? begin + per_xcd : total;
  w.step = gridDim.x / 8;
  w.first = begin + blockIdx.x / 8;
  w.n_tiles = w.first < end ? (int)((end - w.first + w.step - 1) / w.step) : 0;
}

// The i-th tile: up to `strips` strips from t.n0 on; once: no other row block reads its weights.
template <int BM>
TAMD_DEVICE void ring_tile(const RingWork &w, int i, Tile &t, int &strips, bool &once) {
  const int lane = threadIdx.x % kWave;
  const uint32_t idx = w.first + (uint32_t)i * w.step, m = idx / w.gn;
  int e = -1;   // the last slice whose first block is not past the m-th
  for (int u = 0; u * kWave < w.E; ++u) {
    const int s = u * kWave + lane;
    const int first = w.tab[s < w.E ? s : 0];
    e += __builtin_popcountll(__ballot(s < w.E && first <= (int)m));
  }
  t.expert = e;
  t.z = 0;
  const int rows = __builtin_amdgcn_readfirstlane(w.tab[kRingSlices + e]);
  t.start_m = __builtin_amdgcn_readfirstlane(w.tab[2 * kRingSlices + e]);
  const uint32_t local = idx - (uint32_t)__builtin_amdgcn_readfirstlane(w.tab[e]) * w.gn;
  const uint32_t b = (uint32_t)ring_blocks<BM>(rows);
  once = b == 1;
  uint32_t g = b < (uint32_t)w.group ? b : (uint32_t)w.group, blk, col;
  if (g > 1) {   // (as in locate_tile_live)
    g = (b + (b + g - 1) / g - 1) / ((b + g - 1) / g);
    const uint32_t gi = local / (g * w.gn), r = local - gi * g * w.gn;
    const uint32_t size = b - gi * g < g ? b - gi * g : g;
    col = r / size;
    blk = gi * g + (r - col * size);
  } else {
    blk = local / w.gn;
    col = local - blk * w.gn;
  }
  const uint32_t strip0 = col * w.strips / w.gn;
  strips = (int)((col + 1) * w.strips / w.gn - strip0);
  t.n0 = (int)strip0 * 64;
  t.off_m = (int)blk * BM;
  const int left = rows - t.off_m;
  t.rows = left > BM ? BM : left;
}

// Copying waves: strip w's weights, rows 8 w .. of every row fragment, the column scales (waves 0 and 1, four blocks of 32 columns each) or
// the row scales (waves 2 and, past 64 rows, 3).  Stage s goes to slot s % RING and is requested RING - 1 stages ahead; copies complete in
// the order of their requests, so a stage has landed once only those of the stages after it are outstanding (the indices of the next tile's
// rows, requested in front of a tile's first stage, only make that wait a little longer).
template <int XDT, int MF, bool XMX, typename Args>
TAMD_DEVICE void ring_copy(const Args &a, const RingWork &work, uint8_t *lds) {
  typedef RingShape<XDT, MF, XMX> S;
  constexpr uint32_t kOob = 0x7FFFFFFFu;
  constexpr int KA = S::KA, RING = S::RING;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) - S::CONSUMERS, lane = threadIdx.x % kWave;
  const int K = a.K, N = a.N, n_k = (K + KA - 1) / KA, n_kb = (K + KB - 1) / KB, KSP = (K / 32 + 7) / 8 * 8;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
  const int idx_at = RING * S::STAGE + 4 * S::TABLE + S::WORK + w * 512;
  const int a_rin = w * 8 + lane / 8, a_chunk = (lane % 8) ^ ((a_rin >> 1) & 7);
  const uint32_t x_rows = gather_limit(a);
  const bool row_scales = XMX && w >= 2 && w - 2 < S::XS_WAVES;
  // lane 8 i + r asks for the index of the wave's row r in fragment i
  auto request_rows = [&](int i, const Tile &t) {
    if (!a.gather_indx) return;
    const v4i_t rg = make_rsrc(a.gather_indx + t.start_m + t.off_m, (uint32_t)__builtin_amdgcn_readfirstlane(t.rows) * 4u);
    dma4(rg, lds_base + idx_at + (i & 1) * 256, lane < 8 * MF ? (uint32_t)((lane / 8) * 32 + w * 8 + lane % 8) * 4u : kOob, 0);
    if (row_scales) dma4(rg, lds_base + idx_at + 1024 + (i & 1) * 256, (uint32_t)((w - 2) * kWave + lane) * 4u, 0);
  };
  Tile t, next;
  int strips, next_strips;
  bool once, next_once;
  ring_tile<S::BM>(work, 0, next, next_strips, next_once);
  request_rows(0, next);
  int i_tile = 0, p = 0;
  const v4i_t rx = make_rsrc(a.x, kOob);
  const uint8_t *w_base = nullptr, *s_base = nullptr;
  uint32_t a_off[MF], w_off = kOob, s_off = kOob, xs_off = kOob;
  // Strided weights: instruction j copies positions 16 j + lane / 4 of a strip, 16-byte part `part` (j > 1: part ^ 2) of 64 bytes, so that
  // they lie in LDS as blocks do; position 32 f + c holds column 2 c + f.
  const bool strided = S::STRIDED && a.w_layout != TAMD_W_CDNA4_BLOCKS;
  const int part = (lane % 4) ^ ((lane / 16) & 3);
  uint32_t c_off[4], s_end = kOob;
  // the row scales as aligned dwords, up to the one that holds the last row's last byte
  const uint32_t xs_mis = XMX ? (uint32_t)(uintptr_t)a.x_mx_scale & 3u : 0u;
  const v4i_t rxs = make_rsrc(a.x_mx_scale - xs_mis,
                              (uint32_t)__builtin_amdgcn_readfirstlane(
                                  (int)((xs_mis + (uint32_t)(((a.x_rows > 0 ? a.x_rows : (int64_t)a.M) - 1) * a.x_mx_stride_m + K / 32) + 3u) & ~3u)));
  auto issue = [&](int slot) {
    const bool fresh = p == 0;
    if (fresh) {
      t = next, strips = next_strips, once = next_once;
      if (i_tile + 1 < work.n_tiles) {
        ring_tile<S::BM>(work, i_tile + 1, next, next_strips, next_once);
        request_rows(i_tile + 1, next);
      }
      w_base = (const uint8_t *)a.w + (int64_t)t.expert * a.w_stride_e;
      s_base = a.w_mx_scale + (int64_t)t.expert * a.w_mx_stride_e;
      if (strided) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int col = t.n0 + w * 64 + 2 * (lane / 4 + 16 * j % 32) + 16 * j / 32;
          c_off[j] = w < strips ? (uint32_t)(col < N ? col : N - 1) * (uint32_t)a.w_stride_n + (uint32_t)(part ^ (j >> 1) << 1) * 16u : kOob;
        }
        // (scales as aligned dwords, up to the one that holds the last column's last byte)
        const uint32_t mis = (uint32_t)(uintptr_t)s_base & 3u, col = (uint32_t)(t.n0 + w * 64 + lane);
        s_base -= mis;
        s_end = (mis + (uint32_t)((N - 1) * a.w_mx_stride_n + K / 32) + 3u) & ~3u;
        s_off = w < strips && (int)col < N ? (mis + col * (uint32_t)a.w_mx_stride_n) & ~3u : kOob;
      } else {
        w_off = w < strips ? (uint32_t)(((t.n0 >> 6) + w) * n_kb) * 4096u + (uint32_t)lane * 16u : kOob;
        const int blk = (t.n0 >> 5) + 4 * w + lane / 16;
        s_off = blk * 32 < N && (4 * w + lane / 16) / 2 < strips ? (uint32_t)(blk * KSP * 32 + (lane % 16) * 16) : kOob;
      }
    }
    const v4i_t rw = make_rsrc(w_base, kOob), rs = make_rsrc(s_base, strided ? (uint32_t)__builtin_amdgcn_readfirstlane((int)s_end) : kOob);
    const uint32_t sb = lds_base + slot * S::STAGE;
#pragma unroll
    for (int u = 0; u < S::BLOCKS; ++u) {
      const uint32_t to = sb + S::A_STAGE + (w * S::BLOCKS + u) * 4096;
      if (strided) {
        const int kb = p * KA + u * KB;
#pragma unroll
        for (int j = 0; j < 4; ++j) dma16(rw, to + j * 1024, c_off[j] | (kb + (part ^ (j >> 1) << 1) * 32 < K ? 0u : kOob), kb >> 1);
        continue;
      }
      const uint32_t from = w_off | (p * KA + u * KB < K ? 0u : kOob);
      const uint32_t so = (uint32_t)(S::BLOCKS * p + u) * 4096u;
      if (once) dma16_x4_nt(rw, to, from, so);
      else dma16_x4(rw, to, from, so);
    }
    if (strided) {
      if (KA == 256 || (p & 1) == 0) dma16(rs, sb + S::A_STAGE + S::B_STAGE + w * 1024, s_off + (uint32_t)(p * (KA / 32)), 0);
    } else if (w < 2) dma16(rs, sb + S::A_STAGE + S::B_STAGE + w * 1024, s_off, (uint32_t)(p * KA / 256) * 256u);
    if (fresh) {
      if (a.gather_indx && (i_tile == 0 || n_k < RING)) wait_vmcnt<4 * S::BLOCKS>();
      auto index = [&](int at) { return *(const uint32_t *)(lds + idx_at + (i_tile & 1) * 256 + at * 4); };
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        const int r = i * 32 + a_rin;
        const uint32_t src = a.gather_indx ? index(i * 8 + lane / 8) : (uint32_t)(t.start_m + t.off_m + r);
        a_off[i] = r < t.rows && src < x_rows ? src * (uint32_t)(a.x_stride_m * S::ESZ) + a_chunk * 16 : kOob;
      }
      if (row_scales) {
        const int r = (w - 2) * kWave + lane;
        const uint32_t src = a.gather_indx ? index(256 + lane) : (uint32_t)(t.start_m + t.off_m + r);
        xs_off = r < t.rows && src < x_rows ? (src * (uint32_t)a.x_mx_stride_m + xs_mis) & ~3u : kOob;
      }
    }
#pragma unroll
    for (int u = 0; u < S::PLANES; ++u) {
      constexpr int CHUNK_K = S::PLANE_K / 8;
      const int kb = p * KA + u * S::PLANE_K;
      const uint32_t kill = kb + a_chunk * CHUNK_K < K ? 0u : kOob;
      const uint32_t to = sb + u * S::ROWS * A_ROW_BYTES + w * 8 * A_ROW_BYTES;
#pragma unroll
      for (int i = 0; i < MF; ++i) dma16(rx, to + i * 32 * A_ROW_BYTES, a_off[i] | kill, S::FP4 ? kb >> 1 : kb * S::ESZ);
    }
    if (row_scales) {
#pragma unroll
      for (int j = 0; j < S::XS_WORDS; ++j)
        dma4(rxs, sb + S::A_STAGE + S::B_STAGE + S::SC_STAGE + (j * S::XS_WAVES + w - 2) * (kWave * 4), xs_off + (uint32_t)(p * (KA / 32) + 4 * j), 0);
    }
    if (++p == n_k) p = 0, ++i_tile;
  };
  auto wait = [&](auto newer) {
    constexpr int n = decltype(newer)::value;
    // (strided and 128 K: with the column scales of every other stage one or two more may be outstanding than are waited for)
    constexpr int SC = KA == 256 ? 1 : 0;
    if (strided && row_scales) wait_vmcnt<n * (S::COPIES + SC + S::XS_WORDS)>();
    else if (strided) wait_vmcnt<n * (S::COPIES + SC)>();
    else if (w < 2) wait_vmcnt<n * (S::COPIES + 1)>();
    else if (row_scales) wait_vmcnt<n * (S::COPIES + S::XS_WORDS)>();
    else wait_vmcnt<n * S::COPIES>();
  };
  const int stages = work.n_tiles * n_k;
  int slot = 0, s = 0;
  auto advance = [&]() { slot = slot + 1 == RING ? 0 : slot + 1; };
#pragma unroll 1
  for (int q = 0; q < RING - 1 && q < stages; ++q) {
    issue(slot);
    advance();
  }
  if constexpr (S::AHEAD > 0) {   // the first stage is read before the first stage's barrier
    if (stages >= RING - 1) wait(std::integral_constant<int, RING - 2>{});
    else wait(std::integral_constant<int, 0>{});
    sync_threads();
  }
#pragma unroll 1
  for (; s + RING - 1 < stages; ++s) {
    wait(std::integral_constant<int, RING - 2 - S::AHEAD>{});
    sync_threads();
    issue(slot);
    advance();
  }
  // the last RING - 1 stages, with nothing left to request
  auto drain = [&](auto newer) {
    constexpr int n = decltype(newer)::value;
    if (n >= stages) return;
    wait(std::integral_constant<int, (n > S::AHEAD ? n - S::AHEAD : 0)>{});
    sync_threads();
  };
  static_assert(RING <= 6, "stages written out below");
#define TAMD_DRAIN(n) if constexpr (RING - 2 >= n) drain(std::integral_constant<int, (RING - 2 >= n ? n : 0)>{});
  TAMD_DRAIN(4) TAMD_DRAIN(3) TAMD_DRAIN(2) TAMD_DRAIN(1) TAMD_DRAIN(0)
#undef TAMD_DRAIN
}

// Barriers that a set owes while the other one multiplies: one after every four rows of its epilogue, the rest behind it.
struct RingPace {
  int left;
  TAMD_DEVICE void operator()() {
    if (left > 0) {
      sync_threads();
      --left;
    }
  }
};

// What a kernel writes: the 16-bit type of 16-bit rows (bf16 for others), float8_e4m3fn with or without flexpoint scales, MXFP8.
enum { kRing16, kRingFp8, kRingMx };

// A tile of a set: NFR row fragments, the K loop and the epilogue.  xs_sel: where a row's scales start in the dwords that hold them.
// 16-bit rows: bound by the conversions and what they wait for (a stage of 128 K is 512 cycles of MFMA per fragment and took 1 060), so a
// stage's operands are read while the one before is multiplied.
template <int XDT, int MF, int NFR, int ACT, int OUT, bool XMX, typename Args>
TAMD_DEVICE void ring_products(const Args &a, const Tile &t, uint8_t *lds, uint8_t *tab, int slot, const EpilogueOperands<MF> &ops,
                               const uint32_t (&xs_sel)[MF], float flex, RingPace &pace) {
  typedef RingShape<XDT, MF, XMX> S;
  constexpr bool FP4 = S::FP4, X16 = S::X16;
  constexpr int KA = S::KA, STEPS = KA / 64;
  constexpr int FMT = FP4 ? 4 : 0;
  const int strip = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) & 3;
  int lane = threadIdx.x % kWave;
  if constexpr (NFR >= 3 && !XMX) asm volatile("" : "+v"(lane));   // (nothing made of it is kept over the tiles: registers)
  const int c32 = lane % 32, h = lane / 32;
  const int K = a.K, G = K / 32, n_k = (K + KA - 1) / KA;
  const bool strided = S::STRIDED && a.w_layout != TAMD_W_CDNA4_BLOCKS;
  // Column scales of 256 K: bytes h, 2 + h, ... of eight (strided: of the sixteen that start with their dword).
  uint32_t sc_sel[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    if (strided) {
      const uint32_t at = (uint32_t)(uintptr_t)(a.w_mx_scale + (int64_t)t.expert * a.w_mx_stride_e) +
                          (uint32_t)(t.n0 + strip * 64 + 2 * c32 + f) * (uint32_t)a.w_mx_stride_n;
      sc_sel[f] = 0x0C0C0200u + ((at & 3u) + h) * 0x0101u;
    } else {
      sc_sel[f] = 0x06020400u + (uint32_t)((c32 >> 3) & 1) * 0x01010101u;
    }
  }
  // Offsets into a stage: a lane's first chunk of a row and of a column, the others an exclusive or away (a stage starts on 128 bytes),
  // so that one address register serves all of them.
  static_assert(S::STAGE % 128 == 0 && S::A_STAGE % 128 == 0, "chunks are picked by the low seven address bits");
  const uint32_t a_lane = (uint32_t)(c32 * A_ROW_BYTES + (((X16 ? 4 * h : h) ^ ((c32 >> 1) & 7)) * 16));
  const uint32_t b_lane = (uint32_t)(S::A_STAGE + strip * S::BLOCKS * 4096 + c32 * 64 + ((h ^ ((c32 >> 2) & 3)) * 16));
  const uint32_t sc_lane = S::A_STAGE + S::B_STAGE + (uint32_t)(strided ? strip * 1024 + 32 * c32 : (2 * strip + c32 / 16) * 256 + 64 * h + 8 * (c32 % 8));
  const uint32_t sc_lane1 = sc_lane + (strided ? 16 : 128);
  epilogue_table<NFR, OUT == kRing16 ? 2 : 1, true, OUT == kRingMx>(kernel_args_late(), t, ops.dst, ops.beta, ops.gamma, tab);
  u32x2_t *tab_bias = (u32x2_t *)(tab + epilogue_table_bytes(MF)) + strip * 32 + c32;
  *tab_bias = u32x2_t{ops.bias[0], ops.bias[1]};
  f32x16_t acc[NFR][NF];
#pragma unroll
  for (int i = 0; i < NFR; ++i)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[i][f][j] = 0.f;
  auto next_slot = [&](int s) { return s + 1 == S::RING ? 0 : s + 1; };
  // codes of step q, column fragment f, of a stage
  auto read_b = [&](uint32_t buf, int q, int f) {
    return *(const uint4 *)(lds + ((buf + b_lane) ^ (uint32_t)(((q & 1) ^ f) * 32)) + f * 2048 + (q >> 1) * 4096);
  };
  // groups past K, whose place the next row's or column's scales take: zero bytes
  auto within = [&](int left, int n) {   // (of n groups, `left` of them before K ends)
    if (left >= n) return 0xFFFFFFFFu;
    const int steps = (left + 1 - h) / 2;
    return steps > 0 ? 0xFFFFFFFFu >> (32 - 8 * steps) : 0u;
  };
  // the column scales of a stage's steps, a byte each
  auto take_w = [&](const uint2 &s0, const uint2 &s1, int p, uint32_t buf, uint32_t (&sw)[NF]) {
    if (S::STRIDED && KA == 128 && (p & 1) != 0) {   // the second half of the 256 K
      sw[0] >>= 16, sw[1] >>= 16;
    } else if (strided) {   // s0, s1: the first eight bytes of either column
      const uint32_t third[NF] = {*(const uint32_t *)(lds + buf + sc_lane + 8), *(const uint32_t *)(lds + buf + sc_lane1 + 8)};
      const uint2 of[NF] = {s0, s1};
      const uint32_t keep = within(G - p * (KA / 32), 8);
#pragma unroll
      for (int f = 0; f < NF; ++f)
        sw[f] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(third[f], of[f].y, sc_sel[f]), __builtin_amdgcn_perm(of[f].y, of[f].x, sc_sel[f]), 0x05040100u) & keep;
    } else {
      sw[0] = __builtin_amdgcn_perm(s1.x, s0.x, sc_sel[0]);
      sw[1] = __builtin_amdgcn_perm(s1.y, s0.y, sc_sel[1]);
      if (!S::STRIDED && KA == 128 && (p & 1) != 0) sw[0] >>= 16, sw[1] >>= 16;   // (read again: registers)
    }
  };
  // operand of step q (of 64 K), fragment i; of 16-bit rows of the u-th 16 K in it
  auto read_a = [&](uint32_t buf, int q, int i, int u = 0) {
    auto chunk = [&](int c) {
      return *(const uint4 *)(lds + ((buf + a_lane) ^ (uint32_t)(c * 16)) + q * 64 / S::PLANE_K * S::ROWS * A_ROW_BYTES + i * 32 * A_ROW_BYTES);
    };
    if constexpr (X16) {
      return __builtin_bit_cast(typename RowMma<XDT>::frag_t, chunk(u));
    } else if constexpr (FP4) {
      const uint4 v = chunk(2 * q);
      return i32x8_t{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0};
    } else {
      const uint4 lo = chunk(4 * (q & 1)), hi = chunk(4 * (q & 1) + 2);
      return i32x8_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    }
  };
  uint32_t sw[NF];
  if constexpr (X16) {
    uint4 raw[STEPS][NF];
    // The operands of the next stage are read while this one's are multiplied; after the last one whatever its slot holds, for nothing.
    typedef Mma<XDT> M;
    typename M::frag_t af[2][NFR];
    uint32_t buf = (uint32_t)slot * S::STAGE;
#pragma unroll
    for (int q = 0; q < STEPS; ++q)
#pragma unroll
      for (int f = 0; f < NF; ++f) raw[q][f] = read_b(buf, q, f);
    take_w(*(const uint2 *)(lds + buf + sc_lane), *(const uint2 *)(lds + buf + sc_lane1), 0, buf, sw);
#pragma unroll
    for (int i = 0; i < NFR; ++i) af[0][i] = read_a(buf, 0, i);
#pragma unroll 1
    for (int p = 0; p < n_k; ++p) {
      sync_threads();
      slot = next_slot(slot);
      const uint32_t ahead = (uint32_t)slot * S::STAGE;
      uint4 raw_next[STEPS][NF];
      uint2 s0, s1;
#pragma unroll
      for (int v = 0; v < 4 * STEPS; ++v) {
        const int q = v / 4, u = v % 4;
#pragma unroll
        for (int i = 0; i < NFR; ++i)
          af[(v + 1) & 1][i] = v + 1 < 4 * STEPS ? read_a(buf, (v + 1) / 4, i, (v + 1) % 4) : read_a(ahead, 0, i);
        if (u == 1) {
#pragma unroll
          for (int f = 0; f < NF; ++f) raw_next[q][f] = read_b(ahead, q, f);
        }
        if (v == 2) s0 = *(const uint2 *)(lds + ahead + sc_lane), s1 = *(const uint2 *)(lds + ahead + sc_lane1);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const uint32_t codes = u == 0 ? raw[q][f].x : (u == 1 ? raw[q][f].y : (u == 2 ? raw[q][f].z : raw[q][f].w));
          const auto bf = M::expand(codes, bits_to_f32((sw[f] >> (8 * q) & 0xFFu) << 23));
#pragma unroll
          for (int i = 0; i < NFR; ++i) acc[i][f] = M::mma(af[v & 1][i], bf, acc[i][f]);
        }
      }
#pragma unroll
      for (int q = 0; q < STEPS; ++q)
#pragma unroll
        for (int f = 0; f < NF; ++f) raw[q][f] = raw_next[q][f];
      take_w(s0, s1, p + 1, ahead, sw);
      buf = ahead;
    }
  } else {
    uint32_t sa[NFR];
#pragma unroll
    for (int i = 0; i < NFR; ++i) sa[i] = 0x7F7F7F7Fu;
    auto row_scales = [&](int p, uint32_t buf) {
      if constexpr (XMX) {
        // bytes h, 2 + h, ... of the stage's groups
        const uint32_t keep = within(G - p * (KA / 32), KA / 32);
        const uint32_t *words = (const uint32_t *)(lds + buf + S::A_STAGE + S::B_STAGE + S::SC_STAGE) + c32;
#pragma unroll
        for (int i = 0; i < NFR; ++i) {
          auto word = [&](int j) { return words[j * S::XS_WAVES * kWave + i * 32]; };
          sa[i] = __builtin_amdgcn_perm(word(1), word(0), xs_sel[i]);
          if constexpr (KA == 256) sa[i] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(word(2), word(1), xs_sel[i]), sa[i], 0x05040100u);
          sa[i] &= keep;
        }
      }
    };
#pragma unroll 1
    for (int p = 0; p < n_k; ++p) {
      sync_threads();
      uint32_t buf = (uint32_t)slot * S::STAGE;
      slot = next_slot(slot);
      if constexpr (FP4 && NFR >= 3) {   // (scales before the operands, for their registers)
        row_scales(p, buf);
        __builtin_amdgcn_sched_barrier(0);
      }
      constexpr int NB = NFR < 3 ? 2 : 1;   // steps whose codes are in registers (as many as there are registers for)
      uint4 raw[NB][NF];
#pragma unroll
      for (int f = 0; f < NF; ++f) raw[0][f] = read_b(buf, 0, f);
      typename RowMma<XDT>::frag_t af[NFR];
#pragma unroll
      for (int i = 0; i < NFR; ++i) af[i] = read_a(buf, 0, i);
      const uint2 s0 = *(const uint2 *)(lds + buf + sc_lane), s1 = *(const uint2 *)(lds + buf + sc_lane1);
      if constexpr (NB > 1) {
#pragma unroll
        for (int f = 0; f < NF; ++f) raw[NB - 1][f] = read_b(buf, 1, f);
      }
      take_w(s0, s1, p, buf, sw);
      if constexpr (XMX && !(FP4 && NFR >= 3)) row_scales(p, buf);
      // (the operands of the next step are requested one by one behind the last MFMA that uses those of this one)
#define TAMD_STEP(q)                                                                                                        \
  if constexpr (q < STEPS) {                                                                                                \
    constexpr int r = q % NB;                                                                                               \
    i32x8_t bf[NF];                                                                                                         \
    _Pragma("unroll") for (int f = 0; f < NF; ++f) bf[f] =                                                                  \
        i32x8_t{(int)raw[r][f].x, (int)raw[r][f].y, (int)raw[r][f].z, (int)raw[r][f].w, 0, 0, 0, 0};                        \
    _Pragma("unroll") for (int i = 0; i < NFR; ++i) {                                                                       \
      _Pragma("unroll") for (int f = 0; f < NF; ++f) acc[i][f] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(           \
          af[i], bf[f], acc[i][f], FMT, 4, q, (int)sa[i], q, (int)sw[f]);                                                   \
      if constexpr (q + 1 < STEPS) af[i] = read_a(buf, q + 1, i);                                                           \
    }                                                                                                                       \
    if constexpr (q + NB < STEPS) _Pragma("unroll") for (int f = 0; f < NF; ++f) raw[r][f] = read_b(buf, q + NB, f);        \
  }
      TAMD_STEP(0) TAMD_STEP(1) TAMD_STEP(2) TAMD_STEP(3)
#undef TAMD_STEP
    }
  }
  const Args &late = kernel_args_late();
  EpilogueOperands<NFR> operands;   // (the rows' are in the table)
  const u32x2_t bias = *tab_bias;
  operands.bias[0] = bias[0], operands.bias[1] = bias[1];
  operands.x_scale = flex, operands.w_scale = 1.0f;
  if constexpr (OUT == kRingMx) {
    tile_epilogue_t<NFR, ACT, TAMD_FP8_E4M3, true, false, true, Args>(late, t, acc, tab, &operands, pace);
  } else if constexpr (OUT == kRingFp8) {
    tile_epilogue_t<NFR, ACT, TAMD_FP8_E4M3, true, true, false, Args>(late, t, acc, tab, &operands, pace);
  } else if (late.betas || late.gammas) {
    tile_epilogue_t<NFR, ACT, X16 ? XDT : TAMD_BF16, true, false, false, Args>(late, t, acc, tab, &operands, pace);
  } else {
    tile_epilogue_t<NFR, ACT, X16 ? XDT : TAMD_BF16, false, false, false, Args>(late, t, acc, tab, &operands, pace);
  }
}

// A multiplying wave.  Both sets pass every stage's barrier: their own tiles' in the K loop, the other's in the epilogue and behind it.
template <int XDT, int MF, int ACT, int OUT, bool XMX, typename Args>
TAMD_DEVICE void ring_compute(const Args &a, const RingWork &work, uint8_t *lds) {
  typedef RingShape<XDT, MF, XMX> S;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), strip = wave & 3, set = wave >> 2, lane = threadIdx.x % kWave;
  const int n_k = (a.K + S::KA - 1) / S::KA;
  Tile t, next;
  int strips, next_strips;
  bool once;
  EpilogueOperands<MF> ops;   // of the set's next tile
  uint32_t src[MF];           // its rows' indices (XMX)
  auto request = [&](int i) {
    if (i >= work.n_tiles) return;
    ring_tile<S::BM>(work, i, next, next_strips, once);
    epilogue_operands<MF, true>(kernel_args_late(), next, ops);
    if constexpr (XMX) {
#pragma unroll
      for (int u = 0; u < MF; ++u) {
        int r = u * 32 + lane % 32;
        r = next.start_m + next.off_m + (r < next.rows ? r : next.rows - 1);
        src[u] = (uint32_t)(a.gather_indx ? a.gather_indx[r] : r);
      }
    }
  };
  // (one scale for every tile, in a scalar register)
  const float flex = bits_to_f32(__builtin_amdgcn_readfirstlane((int)f32_to_bits((a.x_scale ? *a.x_scale : 1.0f) * (a.w_scale ? *a.w_scale : 1.0f))));
  request(set);
  if constexpr (S::AHEAD > 0) sync_threads();
  if (set == 1) {
#pragma unroll 1
    for (int p = 0; p < n_k; ++p) sync_threads();
  }
#pragma unroll 1
  for (int i = set; i < work.n_tiles; i += 2) {
    t = next, strips = next_strips;
    RingPace pace{i + 1 < work.n_tiles ? n_k : 0};
    if (strip >= strips) {
#pragma unroll 1
      for (int p = 0; p < n_k; ++p) sync_threads();
    } else {
      uint32_t sel[MF];   // where a row's scales start in the dwords that hold them (none: zero bytes)
      if constexpr (XMX) {
        const uint32_t mis = (uint32_t)(uintptr_t)a.x_mx_scale & 3u, x_rows = gather_limit(a);
#pragma unroll
        for (int u = 0; u < MF; ++u)
          sel[u] = src[u] < x_rows ? 0x0C0C0200u + ((src[u] * (uint32_t)a.x_mx_stride_m + mis & 3u) + lane / 32) * 0x0101u : 0x0C0C0C0Cu;
      }
      // The waves of a set write the same table.  One may start a tile while another still finishes the last one, never the one before.
      uint8_t *tab = lds + S::RING * S::STAGE + (2 * set + (i >> 1 & 1)) * S::TABLE;
      const int slot = (int)((uint32_t)(i * n_k) % (uint32_t)S::RING);
      if (MF == 1 || t.rows <= 32) ring_products<XDT, MF, 1, ACT, OUT, XMX>(a, t, lds, tab, slot, ops, sel, flex, pace);
      else if (MF == 2 || t.rows <= 64) ring_products<XDT, MF, (MF < 2 ? MF : 2), ACT, OUT, XMX>(a, t, lds, tab, slot, ops, sel, flex, pace);
      else ring_products<XDT, MF, MF, ACT, OUT, XMX>(a, t, lds, tab, slot, ops, sel, flex, pace);
    }
    request(i + 2);
#pragma unroll 1
    for (; pace.left > 0; --pace.left) sync_threads();
  }
}

template <int XDT, int MF, int ACT, int OUT, bool XMX>
__global__ __launch_bounds__((RingShape<XDT, MF, XMX>::THREADS), 1) void mm_ring_kernel(tamd_matmul_args, int group) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  typedef RingShape<XDT, MF, XMX> S;
  // (the arguments are read where they are used, see kernel_args_late)
  RingWork work;
  ring_work<S::BM>(kernel_args_late(), group, (int32_t *)(lds + S::RING * S::STAGE + 4 * S::TABLE), work);
  if (work.n_tiles == 0) return;
  if (threadIdx.x >= S::CONSUMERS * kWave) ring_copy<XDT, MF, XMX>(kernel_args_late(), work, lds);
  else ring_compute<XDT, MF, ACT, OUT, XMX>(kernel_args_late(), work, lds);
}

template <int XDT, int MF, int ACT, int OUT, bool XMX>
int launch_ring(const tamd_matmul_args &a, hipStream_t st) {
  typedef RingShape<XDT, MF, XMX> S;
  int cus = 0;
  if (int rc = cu_count(cus)) return rc;
  // (a workgroup for every strip of every block, if that is not one per CU: ring_applicable keeps their number below 2^31)
  const int64_t blocks = a.M / S::BM + (a.M < a.n_experts ? a.M : a.n_experts), strips = (a.N + 63) / 64;
  const int64_t wgs = (std::min<int64_t>(blocks * strips, cus) + 7) / 8 * 8;
  int64_t group = a.M / a.n_experts / S::BM;
  group = group < 1 ? 1 : (group > 16 ? 16 : group);
  auto kern = mm_ring_kernel<XDT, MF, ACT, OUT, XMX>;
  if (int rc = raise_lds_limit_once((const void *)kern)) return rc;
  kern<<<dim3((unsigned)wgs), S::THREADS, S::LDS, st>>>(a, (int)group);
  return launch_status();
}

// What is built: for blocks of 96 rows the outputs that the products of a layer write, fp8 and MXFP8 with SwiGLU, 16 bits (MXFP8 not from
// packed rows: registers).
template <int XDT, int MF, int ACT, int OUT>
constexpr bool kRingBuilt = MF < 3 || OUT == kRing16 || (ACT == TAMD_ACT_SWIGLU && !(XDT == TAMD_MXFP4 && OUT == kRingMx));

template <int XDT, int MF, int ACT, int OUT>
int launch_ring_scales(const tamd_matmul_args &a, hipStream_t st) {
  if constexpr (!kRingBuilt<XDT, MF, ACT, OUT>) {
    return TAMD_E_UNSUPPORTED;
  } else if constexpr (XDT == TAMD_BF16 || XDT == TAMD_F16) {
    return launch_ring<XDT, MF, ACT, OUT, false>(a, st);
  } else {
    if constexpr (XDT != TAMD_MXFP4) {
      if (!a.x_mx_scale) return launch_ring<XDT, MF, ACT, OUT, false>(a, st);
    }
    return launch_ring<XDT, MF, ACT, OUT, true>(a, st);
  }
}
template <int XDT, int MF, int ACT>
int launch_ring_out(const tamd_matmul_args &a, hipStream_t st) {
  if constexpr (XDT != TAMD_BF16 && XDT != TAMD_F16) {
    if (a.y_mx_scale) return launch_ring_scales<XDT, MF, ACT, kRingMx>(a, st);
    if (a.y_dtype == TAMD_FP8_E4M3) return launch_ring_scales<XDT, MF, ACT, kRingFp8>(a, st);
  }
  return launch_ring_scales<XDT, MF, ACT, kRing16>(a, st);
}

template <int XDT>
int dispatch_ring(const tamd_matmul_args &a, int rows, hipStream_t st) {
  const bool sw = a.activation == TAMD_ACT_SWIGLU;
  switch (rows) {
    case 32: return sw ? launch_ring_out<XDT, 1, TAMD_ACT_SWIGLU>(a, st) : launch_ring_out<XDT, 1, TAMD_ACT_NONE>(a, st);
    case 64: return sw ? launch_ring_out<XDT, 2, TAMD_ACT_SWIGLU>(a, st) : launch_ring_out<XDT, 2, TAMD_ACT_NONE>(a, st);
    case 96:
      if constexpr (XDT != TAMD_BF16 && XDT != TAMD_F16) return sw ? launch_ring_out<XDT, 3, TAMD_ACT_SWIGLU>(a, st) : launch_ring_out<XDT, 3, TAMD_ACT_NONE>(a, st);
      [[fallthrough]];
    default: return TAMD_E_UNSUPPORTED;
  }
}

}  // namespace tamd
