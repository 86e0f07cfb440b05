// Grouped / dense matmul of fp8, packed e2m1 or (blocks of up to 64 rows) 16-bit activations x MXFP4 weights.  fp8 and packed rows:
// v_mfma_scale_f32_32x32x64_f8f6f4 on the bytes or codes of both operands and their e8m0 bytes, without any conversion.  16-bit
// rows: codes expanded in registers, as in moe_matmul_impl.h.
//
// Tile, epilogue, tile location and LDS images are those of moe_matmul_impl.h.  A stage is 256 K (128 K for 16-bit rows and for fp8
// rows in blocks of 128): one or two planes of 128 bytes per row against one or two 4 KB weight blocks per wave, four MFMA steps of 64 K (two).
// Step q takes, for lane half h, the 32 codes K 64 q + 32 h .. of a column (part 2 (q % 2) + h of weight block q / 2) and of a
// packed row (chunk 2 q + h); of an fp8 row it takes the 16 values K 64 q + 16 h .. followed by the 16 at K 64 q + 32 + 16 h ..
// (the operand layout of the instruction, established by one-hot probing).  The scale operand of lane half h is group 2 q + h's.
//
// What bounds it: few rows per expert HBM (in the K loop 5 TB/s of 6.1) and the start and end of a tile, 8 us of the 46 that a tile
// of 23 stages of 128 K lasts; full blocks the matrix rate (16384 tokens over 32 experts 2.1 PFLOP/s of the library's 2.6).  The block
// scales of both operands come straight to registers, eight bytes (256 K) per row or column and lane: through LDS, staged with the
// tile or travelling with the weights, they took copies of one to four bytes per row, eight byte-sized LDS reads per 128 K
// and, with strided scales that did not fit, four copies of 64 lines per 128 K.  Everything a stage needs is requested
// one stage ahead, so small blocks have stages of 256 K (with 128 K and five workgroups per CU 16 fp8 rows per expert run 4 %
// slower), and a CU holds as many workgroups as its registers do (a third 128-K weight slot, half a stage further ahead,
// changed nothing).  Packed rows, against being widened to fp8 in front of the kernel: half the MFMA cycles, row copies and LDS reads,
// no pass over the rows.
// Before -> now, layers: packed rows, widening included, 2048 tokens, 128 experts (top-4) 531 -> 471 us, 2331 over 16 (top-8) 212 -> 177;
// fp8 16384 over 32 1587 -> 1550, 13 over 64 (top-2) 34.3 -> 32.2, 509 over 128 the same; dense fp8, 3425 x 5600 x 2312
// (strided scales) 104 -> 73, 2 x 3680 x 1336 19.4 -> 14.5, 158 x 640 x 1080 7.3 -> 6.6.
// 16-bit rows in blocks of up to 64: a barrier per 128 K instead of 64, no scales in LDS, three workgroups per CU (blocks of 32: four; with
// strided weights, which take twice the LDS, two and three) where the kernel with deeper rings beside the tile's scales held one or two:
// 816 x 4960 x 2776 f16 62.3 -> 35.8 us, 2351 x 1664 x 6992 62 -> 55; 256 tokens over 16 experts, 3776 -> 1280, layer 74.9 -> 66.8.
#pragma once
#include "moe_matmul_impl.h"

namespace tamd {

// Eight bytes at base + voff, any alignment; of a row or column with fewer groups (n < 8) its own, zeros behind them.  Ordinary
// loads, which the compiler waits for by itself: the loop below uses them behind a wait for everything.
TAMD_DEVICE uint64_t load_scales(const uint8_t *base, uint32_t voff, int n) {
  uint64_t v = 0;
  if (n >= 8) {
    __builtin_memcpy(&v, base + voff, 8);
  } else {
    for (int b = 0; b < n; ++b) v |= (uint64_t)base[voff + b] << (8 * b);
  }
  return v;
}

template <int XDT, int BM>
struct MxShape {
  static constexpr bool FP4 = XDT == TAMD_MXFP4, X16 = XDT == TAMD_BF16 || XDT == TAMD_F16;
  static constexpr int ESZ = X16 ? 2 : 1;                    // bytes per unit of the rows' strides
  static constexpr int MF = BM <= 32 ? 1 : BM / 32;
  static constexpr int ROWS = 32 * MF;
  static constexpr int KA = FP4 || (!X16 && BM <= 64) ? 256 : 128;     // K per stage
  static constexpr int PLANE_K = FP4 ? 256 : (X16 ? 64 : 128);         // K of 128 bytes of a row
  static constexpr int PLANES = KA / PLANE_K;                // 128-byte pieces of a row per stage
  static constexpr int BLOCKS = KA / KB;                     // weight blocks per wave and stage
  static constexpr int A_STAGE = PLANES * ROWS * A_ROW_BYTES;
  static constexpr bool PAIRS = BLOCKS == 1;                 // strided weights: 256 K at a time, every other stage
  static constexpr int b_wave(bool blocks) { return (PAIRS && !blocks ? 2 : BLOCKS) * 4096; }   // weight bytes of a wave
  static constexpr int lds(bool blocks) { return 2 * A_STAGE + 4 * b_wave(blocks); }
  static constexpr int WGS = BM >= 128 ? 2 : (FP4 || X16 ? (BM == 64 ? 3 : 4) : (BM == 64 ? 2 : 3));   // workgroups per CU (block layout)
  static_assert(!X16 || BM <= 64, "larger blocks of 16-bit rows: run_tile");
};

template <int XDT>
struct RowMma {   // scaled MFMA: raw dwords
  typedef i32x8_t frag_t;
};
template <>
struct RowMma<TAMD_BF16> : Mma<TAMD_BF16> {};
template <>
struct RowMma<TAMD_F16> : Mma<TAMD_F16> {};

// KS > 1: K groups of NS waves share a tile of NS strips (blocks of up to 32 rows), as in moe_matmul_impl.h.
template <int XDT, int NFR, int BM, int ACT, int KS = 1, int NS = 4>
TAMD_DEVICE void run_tile_mx(const tamd_matmul_args &a, const Tile &t, uint8_t *lds_wg) {
  typedef MxShape<XDT, BM> S;
  constexpr bool FP4 = S::FP4, X16 = S::X16;
  constexpr int KA = S::KA, PLANES = S::PLANES, BLOCKS = S::BLOCKS, STEPS = KA / 64, A_STAGE = S::A_STAGE;
  constexpr int FMT = XDT == TAMD_MXFP4 ? 4 : (XDT == TAMD_FP8_E5M2 ? 1 : 0);
  constexpr uint32_t kOob = 0x7FFFFFFFu;
  const int wave_wg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), wave = KS > 1 ? wave_wg % NS : wave_wg, grp = KS > 1 ? wave_wg / NS : 0;
  static_assert(KS == 1 ? NS == 4 : NFR == 1 && !X16 && !S::PAIRS, "K groups: one row fragment, stages of 256 K");
  const int lane = threadIdx.x % kWave;
  const int c32 = lane % 32, h = lane / 32;
  const int K = a.K, N = a.N, G = K / 32;
  uint8_t *lds = lds_wg + grp * (2 * A_STAGE + NS * S::b_wave(true));
  const bool wave_live = t.n0 + wave * 64 < N;
  const v4i_t rx = make_rsrc((const uint8_t *)a.x + (int64_t)t.z * a.x_stride_z * S::ESZ, kOob);
  const v4i_t rw = make_rsrc((const uint8_t *)a.w + (int64_t)t.expert * a.w_stride_e, kOob);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
  const bool wnat = a.w_layout == TAMD_W_CDNA4_BLOCKS;
  const int b_at = 2 * A_STAGE + wave * S::b_wave(wnat);   // the wave's weights
  const uint32_t lds_b = lds_base + b_at;
  const uint8_t *bbuf = lds + b_at;
  const int n_k = (K + KA - 1) / KA;
  const int n_p = (n_k + KS - 1) / KS, p0 = grp * n_p;   // the group's stages (past K: nothing is copied or multiplied)
  const bool x_mx = FP4 || (!X16 && a.x_mx_scale != nullptr);

  // ---- row indices: of the rows whose values the lane copies, and of the rows whose scales its MFMAs use; by LDS, each in front of
  // the row pieces that the wave will copy there (see run_tile)
  const int a_rin = wave * 8 + lane / 8;
  const int a_chunk = (lane % 8) ^ ((a_rin >> 1) & 7);
  const int idx_at = wave * 8 * A_ROW_BYTES;
  constexpr int PIECES = 4 / NS, CP_A = NFR * PIECES;   // copies of rows: eight of a fragment each, a wave's NS pieces apart
  auto piece = [](int i) { return i / PIECES * 32 + i % PIECES * (8 * NS); };   // first row of copy i, of wave 0
  if (a.gather_indx) {
    const v4i_t rg = make_rsrc(a.gather_indx + t.start_m + t.off_m, (uint32_t)__builtin_amdgcn_readfirstlane(t.rows) * 4u);
#pragma unroll
    for (int i = 0; i < CP_A; ++i) dma4(rg, lds_base + idx_at + piece(i) * A_ROW_BYTES, (uint32_t)(piece(i) + a_rin) * 4u, 0);
    if constexpr (!X16) {
#pragma unroll
      for (int i = 0; i < NFR; ++i) {
        const int rs = i * 32 + c32;
        dma4(rg, lds_base + idx_at + i * 32 * A_ROW_BYTES + 4 * kWave, (uint32_t)(rs < t.rows ? rs : t.rows - 1) * 4u, 0);
      }
    }
  }

  // ---- weights: the stage's 4 KB blocks as they lie, or 64 contiguous bytes of every column per 128 K (128 of a pair of blocks:
  // eight lanes per column, whole lines where the column's piece lies inside one).  Where a stage is 128 K such a pair is copied
  // every other stage: half lines passed the caches twice (3168 fp8 tokens x 8 over 16 experts, 3008 -> 1568, layer 433 us
  // -> 423, with the halves' shared scale loads below 446 -> 433; 333 f16 tokens x 4 over 32, 2016 -> 1056, 79.2 -> 75.2; 16-bit
  // stages of 256 K, which hold whole lines too, run blocks of 16 and 32 rows at 0.97 to 1.05 of the speed).
  const uint32_t w_nat = (uint32_t)(((t.n0 >> 6) + wave) * ((K + KB - 1) / KB)) * 4096u + (uint32_t)lane * 16;
  constexpr int WIDE = S::PAIRS ? 2 : BLOCKS;         // blocks of K that strided weights are copied by
  constexpr int W_LANES = 4 * WIDE;                   // lanes per column
  const int w_col = t.n0 + wave * 64 + 2 * (lane / W_LANES);
  auto issue_b = [&](int p) {
    const int kb = p * KA;
    if (wnat) {
#pragma unroll
      for (int u = 0; u < BLOCKS; ++u)
        dma16_x4(rw, lds_b + u * 4096, w_nat | ((wave_live && kb + u * KB < K) ? 0u : kOob), (uint32_t)(BLOCKS * p + u) * 4096u);
      return;
    }
    if (S::PAIRS && (p & 1) != 0) return;   // (came with the stage before)
#pragma unroll
    for (int j = 0; j < 4 * WIDE; ++j) {
      // instruction j copies positions (64 / W_LANES) j + lane / W_LANES; position 32 f + c holds column 2 c + f
      constexpr int PER = 64 / W_LANES;
      const int part = WIDE == 2 ? (lane % 8) ^ ((4 * j + lane / 16) & 7) : (lane % 4) ^ ((lane / 16) & 3) ^ ((j >> 1) << 1);
      const int pos0 = PER * j, col = w_col + 2 * (pos0 % 32) + pos0 / 32;
      const uint32_t kill = (wave_live && kb + part * 32 < K) ? 0u : kOob;
      dma16(rw, lds_b + j * 1024, ((uint32_t)(col < N ? col : N - 1) * (uint32_t)a.w_stride_n + part * 16) | kill, kb >> 1);
    }
  };

  // ---- block scales, eight groups (256 K) at a time.  The last eight bytes end with the row or column (nothing past it
  // is read) and are shifted down, zeros behind them; the pre-shuffled layout pads K to whole eights and is read as it is.
  const bool cdna4 = a.w_mx_layout == TAMD_SCALE_CDNA4;
  const uint8_t *xs_base = a.x_mx_scale + (int64_t)t.z * a.x_mx_stride_z;
  const uint8_t *ws_base = a.w_mx_scale + (int64_t)t.expert * a.w_mx_stride_e;
  constexpr uint32_t kSel = 0x06040200u;             // byte selectors: every second scale, from the lane half's first on
  uint32_t as_off[NFR], as_sel[NFR], ws_off[NF];
  const int col0 = t.n0 + wave * 64 + c32 * NF, half = (c32 >> 3) & 1;
  if (cdna4) {   // ws_off[0]: groups h and 2 + h of both columns lie 128 bytes apart
    const int KSP = (G + 7) / 8 * 8, last = (N - 1) / 32, blk = col0 / 32;
    ws_off[0] = (uint32_t)((blk < last ? blk : last) * KSP * 32 + 64 * h + 4 * (col0 % 16));
    ws_off[1] = ws_off[0] + 128;
  } else {
    // a load touches a line per lane, so each half of the wave loads one of its lanes' two columns and the halves exchange them
    ws_off[0] = ws_off[1] = (uint32_t)(col0 + h < N ? col0 + h : N - 1) * (uint32_t)a.w_mx_stride_n;
  }
  const int g_last = G > 8 ? G - 8 : 0;               // where the last eight bytes start
  uint64_t as_raw[NFR], ws_raw[NF];
#pragma unroll
  for (int i = 0; i < NFR; ++i) as_raw[i] = 0x7F7F7F7F7F7F7F7Full;
  auto load_sc = [&](int e) {   // of the e-th 256 K
    const int last = (G - 1) / 8;
    e = e < last ? e : last;
    const int at = 8 * e < g_last ? 8 * e : g_last;
    if (x_mx) {
#pragma unroll
      for (int i = 0; i < NFR; ++i) as_raw[i] = load_scales(xs_base + at, as_off[i], G);
    }
    const uint8_t *w = ws_base + (cdna4 ? 256 * e : at);
    ws_raw[0] = load_scales(w, ws_off[0], cdna4 ? 8 : G);
    if (cdna4) ws_raw[1] = load_scales(w, ws_off[1], 8);
  };
  uint32_t sa[NFR], sw[NF];   // byte q: the scale of step q
  auto take_sc = [&](int e) {
    const int shift = 8 * (8 * e > g_last ? 8 * e - g_last : 0);
    auto pick = [&](uint64_t v, uint32_t sel) {
      const uint64_t x = v >> shift;
      return __builtin_amdgcn_perm((uint32_t)(x >> 32), (uint32_t)x, sel);
    };
#pragma unroll
    for (int i = 0; i < NFR; ++i) sa[i] = x_mx ? pick(as_raw[i], as_sel[i]) : 0x7F7F7F7Fu;
    if (cdna4) {
      const uint32_t s2 = 0x06020400u + (uint32_t)half * 0x01010101u;
#pragma unroll
      for (int f = 0; f < NF; ++f) sw[f] = __builtin_amdgcn_perm((uint32_t)(ws_raw[1] >> (32 * f)), (uint32_t)(ws_raw[0] >> (32 * f)), s2);
    } else {
      // (the lane's own column's: column 2 c32 + h)
      const uint64_t x = ws_raw[0] >> shift;
      const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)x, false, false);
      const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)(x >> 32), (uint32_t)(x >> 32), false, false);
#pragma unroll
      for (int f = 0; f < NF; ++f) sw[f] = __builtin_amdgcn_perm(hi[f], lo[f], kSel + (uint32_t)h * 0x01010101u);
    }
    // (made before the next ones are requested, which then come to the same registers)
#pragma unroll
    for (int i = 0; i < NFR; ++i) asm volatile("" : "+v"(sa[i]));
#pragma unroll
    for (int f = 0; f < NF; ++f) asm volatile("" : "+v"(sw[f]));
  };

  f32x16_t acc[NFR][NF];
#pragma unroll
  for (int i = 0; i < NFR; ++i)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[i][f][j] = 0.f;

  uint32_t a_off[CP_A];
  auto issue_a = [&](int p) {   // (chunks past K are not read: zeros)
    constexpr int PLANE_K = S::PLANE_K, CHUNK_K = PLANE_K / 8;
#pragma unroll
    for (int u = 0; u < PLANES; ++u) {
      const int kb = p * KA + u * PLANE_K;
      const uint32_t kill = kb + a_chunk * CHUNK_K < K ? 0u : kOob;
      const uint32_t to = lds_base + ((p - p0) & 1) * A_STAGE + u * S::ROWS * A_ROW_BYTES + wave * 8 * A_ROW_BYTES;
#pragma unroll
      for (int i = 0; i < CP_A; ++i) dma16(rx, to + piece(i) * A_ROW_BYTES, a_off[i] | kill, FP4 ? kb >> 1 : kb * S::ESZ);
    }
  };

  const uint32_t x_rows = gather_limit(a);
  issue_b(p0);
  if (a.gather_indx) wait_vmcnt<4 * BLOCKS>();   // (the copies of the weights may be outstanding)
  const int row0 = t.start_m + t.off_m;
#pragma unroll
  for (int i = 0; i < CP_A; ++i) {
    const int r = piece(i) + a_rin;
    const uint32_t src = a.gather_indx ? ((const uint32_t *)(lds + idx_at + piece(i) * A_ROW_BYTES))[lane] : (uint32_t)(row0 + r);
    a_off[i] = r < t.rows && src < x_rows ? src * (uint32_t)(a.x_stride_m * S::ESZ) + a_chunk * 16 : kOob;
  }
#pragma unroll
  for (int i = 0; i < NFR; ++i) {
    const int rs = i * 32 + c32;
    const uint32_t *idx = (const uint32_t *)(lds + idx_at + i * 32 * A_ROW_BYTES) + lane;
    const uint32_t srs = a.gather_indx ? idx[X16 ? 0 : kWave] : (uint32_t)(row0 + (rs < t.rows ? rs : t.rows - 1));
    // rows past the end of the slice are never stored: they are copied as zeros, which keeps the matrix cores' inputs quiet; so
    // is the row of an index that names none (-1), for which the first row's scales are read (ordinary loads have no descriptor that
    // would end with them) and zero bytes taken (selector 12)
    as_off[i] = srs < x_rows ? srs * (uint32_t)a.x_mx_stride_m : 0u;
    as_sel[i] = srs < x_rows ? kSel + (uint32_t)h * 0x01010101u : 0x0C0C0C0Cu;
  }
  if (a.gather_indx) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // read before the rows are copied over them
  issue_a(p0);
  load_sc(KA == 256 ? p0 : 0);
  const int swz = (c32 >> 1) & 7;
  for (int p = p0; p < p0 + n_p; ++p) {
    wait_vmcnt<0>();   // (everything requested so far belongs to this stage)
    sync_threads();   // stage p is visible; every wave is done with the buffer that stage p + 1 goes to
    const uint8_t *buf = lds + ((p - p0) & 1) * A_STAGE;
    uint4 raw[STEPS][NF];
#pragma unroll
    for (int q = 0; q < STEPS; ++q)
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const int pos = f * 32 + c32, rot = ((pos >> 2) & 3) ^ (f << 1);
        const int qp = S::PAIRS ? q + (p & 1) * STEPS : q;   // the step in its piece of a strided column
        raw[q][f] = wnat || WIDE == 1 ? *(const uint4 *)(bbuf + (q >> 1) * 4096 + pos * 64 + (((2 * (q & 1) + h) ^ rot) * 16))
                                      : *(const uint4 *)(bbuf + pos * 128 + (((2 * qp + h) ^ ((pos >> 1) & 7)) * 16));
      }
    // operand of step q (of 64 K), fragment i; of 16-bit rows of the u-th 16 K in it
    auto read_a = [&](int q, int i, int u = 0) {
      const uint8_t *row = buf + q * 64 / S::PLANE_K * S::ROWS * A_ROW_BYTES + (i * 32 + c32) * A_ROW_BYTES;
      auto chunk = [&](int c) { return *(const uint4 *)(row + ((c ^ swz) * 16)); };
      if constexpr (X16) {
        return __builtin_bit_cast(typename RowMma<XDT>::frag_t, chunk(4 * h + u));
      } else if constexpr (FP4) {
        const uint4 v = chunk(2 * q + h);
        return i32x8_t{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0};
      } else {
        const uint4 lo = chunk(4 * (q & 1) + h), hi = chunk(4 * (q & 1) + 2 + h);
        return i32x8_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
      }
    };
    typename RowMma<XDT>::frag_t af[X16 ? 2 : 1][NFR];
#pragma unroll
    for (int i = 0; i < NFR; ++i) af[0][i] = read_a(0, i);
    const int e = KA == 256 ? p : p >> 1;
    if (KA == 256 || (p & 1) == 0) {
      take_sc(e);
    } else {   // the second half of the 256 K
#pragma unroll
      for (int i = 0; i < NFR; ++i) sa[i] >>= 16;
#pragma unroll
      for (int f = 0; f < NF; ++f) sw[f] >>= 16;
    }
    // (the stage after a group's last is the next group's: copied for nothing, and waited for behind the loop, dense fp8 256 x 2048 x 4096 took
    // 8.6 us instead of 8.1; without groups it lies past K, where nothing is read)
    const bool more = KS == 1 || p + 1 < p0 + n_p;
    if (more) {
      issue_a(p + 1);
      if (KA == 256 || (p & 1) == 1) load_sc(e + 1);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the weights are in registers: their buffer may be refilled
    if (more) issue_b(p + 1);
    if (!wave_live || (KS > 1 && p >= n_k)) continue;
    if constexpr (X16) {
      // codes expanded in registers, the scale applied by the instruction
      typedef Mma<XDT> M;
#pragma unroll
      for (int v = 0; v < 4 * STEPS; ++v) {
        const int q = v / 4, u = v % 4;
        if (v + 1 < 4 * STEPS) {
#pragma unroll
          for (int i = 0; i < NFR; ++i) af[(v + 1) & 1][i] = read_a((v + 1) / 4, i, (v + 1) % 4);
        }
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const uint32_t codes = u == 0 ? raw[q][f].x : (u == 1 ? raw[q][f].y : (u == 2 ? raw[q][f].z : raw[q][f].w));
          const auto bf = M::expand(codes, bits_to_f32((sw[f] >> (8 * q) & 0xFFu) << 23));
#pragma unroll
          for (int i = 0; i < NFR; ++i) acc[i][f] = M::mma(af[v & 1][i], bf, acc[i][f]);
        }
      }
    } else {
      // (the fragments of the next step are requested one by one behind the last MFMA that uses those of this one)
#define TAMD_STEP(q)                                                                                                        \
  if constexpr (q < STEPS) {                                                                                                \
    constexpr int r = q < STEPS ? q : 0;                                                                                    \
    i32x8_t bf[NF];                                                                                                         \
    _Pragma("unroll") for (int f = 0; f < NF; ++f) bf[f] =                                                                  \
        i32x8_t{(int)raw[r][f].x, (int)raw[r][f].y, (int)raw[r][f].z, (int)raw[r][f].w, 0, 0, 0, 0};                        \
    _Pragma("unroll") for (int i = 0; i < NFR; ++i) {                                                                       \
      _Pragma("unroll") for (int f = 0; f < NF; ++f) acc[i][f] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(           \
          af[0][i], bf[f], acc[i][f], FMT, 4, q, (int)sa[i], q, (int)sw[f]);                                                \
      if constexpr (q + 1 < STEPS) af[0][i] = read_a(q + 1, i);                                                             \
    }                                                                                                                       \
  }
      TAMD_STEP(0) TAMD_STEP(1) TAMD_STEP(2) TAMD_STEP(3)
#undef TAMD_STEP
    }
  }
  wait_vmcnt<0>();
  if constexpr (KS > 1) {
    sync_threads();   // (every copy has landed, every operand has been read)
    if (!k_groups_add<KS, NS>(acc[0], lds_wg, grp, wave)) return;
  }
  // (the wave's own weight region is free by now: its table goes there)
  tile_epilogue<NFR, ACT, X16 ? XDT : TAMD_BF16, !X16>(kernel_args_late(), t, acc, lds + b_at);
}

template <int XDT, int BM, int ACT>
__global__ __launch_bounds__(256, (MxShape<XDT, BM>::WGS)) void mm_mx_kernel(tamd_matmul_args a, int grid_n, int64_t grid_total,
                                                                           int group_m) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  typedef MxShape<XDT, BM> S;
  static_assert(S::WGS * S::lds(true) <= 160 * 1024, "the workgroups that the registers are limited for fit a CU's LDS");
  Tile t;
  if (group_m < 0) {
    if (!locate_tile_live<BM, 0>(a, grid_n, -group_m, t)) return;
  } else if (!locate_tile<BM, 0>(a, grid_n, grid_total, group_m, t)) return;
  const int nfr = (t.rows + 31) / 32;
#define TAMD_CASE(n)                                                   \
  case n:                                                              \
    if constexpr (n <= S::MF) run_tile_mx<XDT, n, BM, ACT>(a, t, lds); \
    break;
  switch (nfr) { TAMD_CASE(1) TAMD_CASE(2) TAMD_CASE(3) TAMD_CASE(4) }
#undef TAMD_CASE
}

// Few tiles: four K groups of two waves on tiles of 128 columns.  A tile's stages wait for a trip to memory each, which only the tile's own
// waves could fill, and half of the CUs and more have none: four times as many waves on twice as many CUs, a quarter of the stages each.
// Tiled kernel -> this one, us: dense fp8, 256 x 2048 x 4096 10.1 -> 8.1, 208 x 2656 x 2848, strided, 17.4 -> 10.9, 60 x 6144 x 3000
// 24.9 -> 13.8; layers: one packed token x 4 of 128 slices, 2880 -> 2880, 45.4 -> 38.6, one MXFP8 token x 4 of 32 44.8 -> 35.7, 100 fp8 tokens x 2
// of 8, 5760 -> 768, 45.9 -> 36.5.
// (mx_groups in tile_rules.h says which problems.)
constexpr int kMxGroups = 4, kMxStrips = 2;
template <int XDT, int BM>
constexpr int kMxGroupsLds = kMxGroups * (2 * MxShape<XDT, BM>::A_STAGE + kMxStrips * MxShape<XDT, BM>::b_wave(true));
template <int XDT, int BM, int ACT>
__global__ __launch_bounds__(kWave * kMxGroups * kMxStrips, 1) void mm_mx_kgroups_kernel(tamd_matmul_args a, int grid_n, int64_t grid_total, int group_m) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  Tile t;
  if (group_m < 0) {
    if (!locate_tile_live<BM, 0>(a, grid_n, -group_m, t)) return;
  } else if (!locate_tile<BM, 0>(a, grid_n, grid_total, group_m, t)) return;
  t.n0 = t.n0 / BLOCK_N * (64 * kMxStrips);
  run_tile_mx<XDT, 1, BM, ACT, kMxGroups, kMxStrips>(a, t, lds);
}

template <int XDT, int BM, int ACT>
int launch_mx(const tamd_matmul_args &a, int grid_m, hipStream_t st) {
  const int grid_n = (a.N + BLOCK_N - 1) / BLOCK_N;
  const int64_t total = (int64_t)grid_m * grid_n;
  if (total <= 0) return 0;
  const int64_t launch = ((total + 7) / 8) * 8;
  if (launch > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
  // row blocks walked together (see launch_x16_act)
  const int64_t rows_per_slice = a.block_schedule ? a.M / a.n_experts : a.M;
  const int64_t fit = (int64_t)(2.5 * 1024 * 1024) / ((int64_t)BM * a.K * MxShape<XDT, BM>::ESZ / (XDT == TAMD_MXFP4 ? 2 : 1));
  int64_t group_m = rows_per_slice / BM;
  group_m = group_m > fit ? fit : group_m;
  group_m = group_m < 1 ? 1 : (group_m > 16 ? 16 : group_m);
  if constexpr (BM <= 32 && !MxShape<XDT, BM>::X16) {
    int cus = 0;
    if (int rc = cu_count(cus)) return rc;
    if (mx_groups(a, cus, BM)) {
      auto kk = mm_mx_kgroups_kernel<XDT, BM, ACT>;
      if (int rc = raise_lds_limit_once((const void *)kk)) return rc;
      const int grid128 = (a.N + 127) / 128;
      const int64_t tiles = (int64_t)grid_m * grid128;
      kk<<<dim3((unsigned)((tiles + 7) / 8 * 8)), kWave * kMxGroups * kMxStrips, kMxGroupsLds<XDT, BM>, st>>>(a, grid128, tiles, (int)(counts_live_blocks(a) ? -group_m : group_m));
      return launch_status();
    }
  }
  auto kern = mm_mx_kernel<XDT, BM, ACT>;
  if (int rc = raise_lds_limit_once((const void *)kern)) return rc;
  const bool blocks = a.w_layout == TAMD_W_CDNA4_BLOCKS;
  size_t lds_bytes = MxShape<XDT, BM>::lds(blocks);
  // Columns that do not start on 64 bytes: a line that two pieces of a column share is read for each, a stage or two apart, and with
  // three workgroups per CU an XCD's L2 has lost it by then (3 x 32 CUs x 256 columns, requested and requested next).  Two per CU from K
  // 1920 on, ragged: 120 x 4 packed rows of 60 slices, 2368 x 3584 80 -> 71 us, 512 x 2 of 128, 3744 x 2176 193 -> 168, fp8 184 -> 172;
  // 320 of 64, 1760 x 2352 40.5 -> 42.2, 64 x 4 of 128, 704 x 1536 18.8 -> 20.
  if (BM <= 32 && a.block_schedule && !blocks && a.w_stride_n % 64 != 0 && a.K >= 1920 && lds_bytes < 56 * 1024) lds_bytes = 56 * 1024;
  kern<<<dim3((unsigned)launch), 256, lds_bytes, st>>>(a, grid_n, total, (int)(counts_live_blocks(a) ? -group_m : group_m));
  return launch_status();
}

// The two activations are compiled in translation units of their own (moe_matmul_<type>.hip, moe_matmul_<type>_swiglu.hip).
template <int XDT, int ACT>
int dispatch_mx_act(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  dense_grid(a, block_m, grid_m);
  switch (block_m) {
    case 16: return launch_mx<XDT, 16, ACT>(a, grid_m, st);
    case 32: return launch_mx<XDT, 32, ACT>(a, grid_m, st);
    case 64: return launch_mx<XDT, 64, ACT>(a, grid_m, st);
    case 128:
      if constexpr (XDT != TAMD_BF16 && XDT != TAMD_F16) return launch_mx<XDT, 128, ACT>(a, grid_m, st);
      [[fallthrough]];
    default: return TAMD_E_UNSUPPORTED;
  }
}
int tiled_mm_swiglu_fp4(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st);
int tiled_mm_swiglu_fp8e4m3(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st);
int tiled_mm_swiglu_fp8e5m2(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st);

}  // namespace tamd
