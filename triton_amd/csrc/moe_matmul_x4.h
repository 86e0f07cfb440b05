// Grouped / dense matmul of microscaled e2m1 activations x MXFP4 weights: v_mfma_scale_f32_32x32x64_f8f6f4 on the codes of both
// operands and their e8m0 bytes.
//
// Tile, epilogue, tile location and LDS images are those of moe_matmul_impl.h; a stage is 256 K here: 128 bytes of a row (four
// MFMA steps) against two 4 KB weight blocks per wave.  Step q takes, for lane half h, the 32 codes K 64 q + 32 h .. of both
// operands: chunk 2 q + h of the row, part 2 (q % 2) + h of the column in weight block q / 2.
//
// What bounds it: with 64 to 128 rows per expert HBM (in the K loop 5 TB/s of 6.1) and the start and end of a tile, 8 of its 46 us.
// Rows widened to fp8 in front of the kernel (as the fp8 path takes them, and as they went before) need an MFMA of twice the
// cycles, twice the row copies and LDS reads, a barrier per 128 K and a pass over the rows.  The block scales of both
// operands come straight to registers, eight bytes (a stage) per row or column and lane: through LDS they took copies of two bytes per
// row and eight byte-sized LDS reads per 128 K.  Everything a stage needs is requested one stage ahead (a third
// 128-K weight slot, half a stage further ahead, changed nothing: 276 us); a CU holds two workgroups of 128-row blocks, three of 64, four of 32.
// Widening included, before -> now: 2048 tokens over 128 experts (top-4), 2880 -> 5760 304 -> 278 us, 2880 -> 2880 187 -> 157, layer
// 531 -> 471; 2331 over 16 (top-8), 2240 -> 1792 109 -> 85, 896 -> 2240 63 -> 49; 39 over 16 (top-6), 2272 -> 1152 25.6 -> 17.8.
#pragma once
#include "moe_matmul_impl.h"

namespace tamd {

// Eight bytes at base + voff, any alignment.  An ordinary load, which the compiler waits for by itself: the loop below uses it
// behind a wait for everything.
TAMD_DEVICE uint64_t load_scales(const uint8_t *base, uint32_t voff) {
  uint64_t v;
  __builtin_memcpy(&v, base + voff, 8);
  return v;
}

template <int BM>
struct X4Shape {
  static constexpr int MF = BM <= 32 ? 1 : BM / 32;
  static constexpr int ROWS = 32 * MF;
  static constexpr int A_STAGE = ROWS * A_ROW_BYTES;
  static constexpr int LDS = 2 * A_STAGE + 2 * B_BYTES;
  static constexpr int WGS = BM >= 128 ? 2 : (BM == 64 ? 3 : 4);   // workgroups per CU
};

template <int NFR, int BM, int ACT>
TAMD_DEVICE void run_tile_x4(const tamd_matmul_args &a, const Tile &t, uint8_t *lds) {
  typedef X4Shape<BM> S;
  constexpr int KA = 256, A_STAGE = S::A_STAGE;
  constexpr uint32_t kOob = 0x7FFFFFFFu;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int c32 = lane % 32, h = lane / 32;
  const int K = a.K, N = a.N, G = K / 32;
  const bool wave_live = t.n0 + wave * 64 < N;
  const v4i_t rx = make_rsrc((const uint8_t *)a.x + (int64_t)t.z * a.x_stride_z, kOob);
  const v4i_t rw = make_rsrc((const uint8_t *)a.w + (int64_t)t.expert * a.w_stride_e, kOob);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
  const uint32_t lds_b = lds_base + 2 * A_STAGE + wave * 8192;
  const uint8_t *bbuf = lds + 2 * A_STAGE + wave * 8192;
  const int n_k = (K + KA - 1) / KA;

  // ---- row indices: of the rows whose codes the lane copies, and of the rows whose scales its MFMAs use
  const int a_rin = wave * 8 + lane / 8;
  const int a_chunk = (lane % 8) ^ ((a_rin >> 1) & 7);
  const v4i_t rg = make_rsrc(a.gather_indx ? a.gather_indx + t.start_m + t.off_m : nullptr,
                             a.gather_indx ? (uint32_t)__builtin_amdgcn_readfirstlane(t.rows) * 4u : 0u);
  uint32_t row_idx[2 * NFR];
#pragma unroll
  for (int i = 0; i < NFR; ++i) {
    const int rs = i * 32 + c32;
    row_idx[i] = request_dword(rg, (uint32_t)(i * 32 + a_rin) * 4u);
    row_idx[NFR + i] = request_dword(rg, (uint32_t)(rs < t.rows ? rs : t.rows - 1) * 4u);
  }

  // ---- weights: two 4 KB blocks as they lie, or 128 contiguous bytes of every column (issue_b_pair of run_tile)
  const bool wnat = a.w_layout == TAMD_W_CDNA4_BLOCKS;
  const uint32_t w_nat = (uint32_t)(((t.n0 >> 6) + wave) * ((K + KB - 1) / KB)) * 4096u + (uint32_t)lane * 16;
  const int w_col = t.n0 + wave * 64 + 2 * (lane / 8);
  auto issue_b = [&](int p) {
    const int kb = p * KA;
    if (wnat) {
      dma16_x4(rw, lds_b, w_nat | ((wave_live && kb < K) ? 0u : kOob), (uint32_t)(2 * p) * 4096u);
      dma16_x4(rw, lds_b + 4096, w_nat | ((wave_live && kb + KB < K) ? 0u : kOob), (uint32_t)(2 * p + 1) * 4096u);
      return;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int part = (lane % 8) ^ ((4 * j + lane / 16) & 7);
      const int col = w_col + 16 * (j % 4) + j / 4;
      const uint32_t kill = (wave_live && kb + part * 32 < K) ? 0u : kOob;
      dma16(rw, lds_b + j * 1024, ((uint32_t)(col < N ? col : N - 1) * (uint32_t)a.w_stride_n + part * 16) | kill, kb >> 1);
    }
  };

  // ---- block scales: eight groups per stage.  The last stage's eight bytes end with the row or column (so nothing past it
  // is read) and are shifted down, zeros behind them; the layouts that pad K to whole stages are read as they are.
  const bool cdna4 = a.w_mx_layout == TAMD_SCALE_CDNA4;
  const uint8_t *xs_base = a.x_mx_scale + (int64_t)t.z * a.x_mx_stride_z;
  const uint8_t *ws_base = a.w_mx_scale + (int64_t)t.expert * a.w_mx_stride_e;
  uint32_t as_off[NFR], ws_off[NF];
  const int col0 = t.n0 + wave * 64 + c32 * NF, half = (c32 >> 3) & 1;
  if (cdna4) {   // ws_off[0]: groups h and 2 + h of both columns lie 128 bytes apart
    const int KSP = (G + 7) / 8 * 8, last = (N - 1) / 32, blk = col0 / 32;
    ws_off[0] = (uint32_t)((blk < last ? blk : last) * KSP * 32 + 64 * h + 4 * (col0 % 16));
    ws_off[1] = ws_off[0] + 128;
  } else {
#pragma unroll
    for (int f = 0; f < NF; ++f) ws_off[f] = (uint32_t)(col0 + f < N ? col0 + f : N - 1) * (uint32_t)a.w_mx_stride_n;
  }
  uint64_t as_raw[NFR], ws_raw[NF];
  auto issue_sc = [&](int p) {
    p = p < n_k ? p : n_k - 1;
    const int at = 8 * p < G - 8 ? 8 * p : G - 8;
#pragma unroll
    for (int i = 0; i < NFR; ++i) as_raw[i] = load_scales(xs_base + at, as_off[i]);
    const uint8_t *w = ws_base + (cdna4 ? 256 * p : at);
#pragma unroll
    for (int f = 0; f < NF; ++f) ws_raw[f] = load_scales(w, ws_off[f]);
  };
  uint32_t sa[NFR], sw[NF];   // byte q: the scale of step q
  auto take_sc = [&](int p) {
    const int shift = 8 * (8 * p < G - 8 ? 0 : 8 * p - (G - 8));
    const uint32_t sel = 0x06040200u + (uint32_t)h * 0x01010101u;
    auto pick = [&](uint64_t v) {
      const uint64_t x = v >> shift;
      return __builtin_amdgcn_perm((uint32_t)(x >> 32), (uint32_t)x, sel);
    };
#pragma unroll
    for (int i = 0; i < NFR; ++i) sa[i] = pick(as_raw[i]);
    if (cdna4) {
      const uint32_t s2 = 0x06020400u + (uint32_t)half * 0x01010101u;
#pragma unroll
      for (int f = 0; f < NF; ++f) sw[f] = __builtin_amdgcn_perm((uint32_t)(ws_raw[1] >> (32 * f)), (uint32_t)(ws_raw[0] >> (32 * f)), s2);
    } else {
#pragma unroll
      for (int f = 0; f < NF; ++f) sw[f] = pick(ws_raw[f]);
    }
    // (made before the next stage's are requested, which then come to the same registers)
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

  uint32_t a_off[NFR];
  auto issue_a = [&](int p) {   // (chunks past K are not read: zeros)
    const int kb = p * KA;
    const uint32_t kill = kb + a_chunk * 32 < K ? 0u : kOob;
    const uint32_t to = lds_base + (p & 1) * A_STAGE + wave * 8 * A_ROW_BYTES;
#pragma unroll
    for (int i = 0; i < NFR; ++i) dma16(rx, to + i * 32 * A_ROW_BYTES, a_off[i] | kill, kb >> 1);
  };

  issue_b(0);
  await_dwords<8>(row_idx);
#pragma unroll
  for (int i = 0; i < NFR; ++i) {
    const int r = i * 32 + a_rin, rs = i * 32 + c32, row0 = t.start_m + t.off_m;
    const uint32_t src = a.gather_indx ? row_idx[i] : (uint32_t)(row0 + r);
    const uint32_t srs = a.gather_indx ? row_idx[NFR + i] : (uint32_t)(row0 + (rs < t.rows ? rs : t.rows - 1));
    a_off[i] = r < t.rows ? src * (uint32_t)a.x_stride_m + a_chunk * 16 : kOob;   // (rows past the end: zeros)
    as_off[i] = srs * (uint32_t)a.x_mx_stride_m;
  }
  issue_a(0);
  issue_sc(0);
  const int swz = (c32 >> 1) & 7;
  for (int p = 0; p < n_k; ++p) {
    wait_vmcnt<0>();   // (everything requested so far belongs to this stage)
    __syncthreads();   // stage p is visible; every wave is done with the buffer that stage p + 1 goes to
    const uint8_t *buf = lds + (p & 1) * A_STAGE;
    uint4 raw[4][NF];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const int pos = f * 32 + c32, rot = ((pos >> 2) & 3) ^ (f << 1);
        raw[q][f] = wnat ? *(const uint4 *)(bbuf + (q >> 1) * 4096 + pos * 64 + (((2 * (q & 1) + h) ^ rot) * 16))
                         : *(const uint4 *)(bbuf + pos * 128 + (((2 * q + h) ^ ((pos >> 1) & 7)) * 16));
      }
    auto read_a = [&](int q, int i) { return *(const uint4 *)(buf + (i * 32 + c32) * A_ROW_BYTES + (((2 * q + h) ^ swz) * 16)); };
    uint4 af[2][NFR];
#pragma unroll
    for (int i = 0; i < NFR; ++i) af[0][i] = read_a(0, i);
    take_sc(p);
    issue_a(p + 1);
    issue_sc(p + 1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the weights are in registers: their buffer may be refilled
    issue_b(p + 1);
    if (wave_live) {
      auto operand = [](const uint4 &v) { return i32x8_t{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0}; };
#define TAMD_STEP(q)                                                                                                      \
  {                                                                                                                       \
    if constexpr (q < 3)                                                                                                  \
      _Pragma("unroll") for (int i = 0; i < NFR; ++i) af[(q + 1) & 1][i] = read_a(q + 1, i);                              \
    _Pragma("unroll") for (int f = 0; f < NF; ++f) _Pragma("unroll") for (int i = 0; i < NFR; ++i)                        \
        acc[i][f] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(operand(af[q & 1][i]), operand(raw[q][f]), acc[i][f], \
                                                                  4, 4, q, (int)sa[i], q, (int)sw[f]);                  \
  }
      TAMD_STEP(0) TAMD_STEP(1) TAMD_STEP(2) TAMD_STEP(3)
#undef TAMD_STEP
    }
  }
  wait_vmcnt<0>();
  // (the wave's own weight region is free by now: its table goes there)
  tile_epilogue<NFR, ACT, TAMD_BF16, true>(kernel_args_late(), t, acc, lds + 2 * A_STAGE + wave * 8192);
}

template <int BM, int ACT>
__global__ __launch_bounds__(256, X4Shape<BM>::WGS) void mm_x4_mxfp4_kernel(tamd_matmul_args a, int grid_n, int64_t grid_total,
                                                                            int group_m) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  typedef X4Shape<BM> S;
  Tile t;
  if (group_m < 0) {
    if (!locate_tile_live<BM, 0>(a, grid_n, -group_m, t)) return;
  } else if (!locate_tile<BM, 0>(a, grid_n, grid_total, group_m, t)) return;
  const int nfr = (t.rows + 31) / 32;
#define TAMD_CASE(n)                                                   \
  case n:                                                              \
    if constexpr (n <= S::MF) run_tile_x4<n, BM, ACT>(a, t, lds);      \
    break;
  switch (nfr) { TAMD_CASE(1) TAMD_CASE(2) TAMD_CASE(3) TAMD_CASE(4) }
#undef TAMD_CASE
}

template <int BM, int ACT>
int launch_x4(const tamd_matmul_args &a, int grid_m, hipStream_t st) {
  const int grid_n = (a.N + BLOCK_N - 1) / BLOCK_N;
  const int64_t total = (int64_t)grid_m * grid_n;
  if (total <= 0) return 0;
  const int64_t launch = ((total + 7) / 8) * 8;
  if (launch > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
  // row blocks walked together (see launch_x16_act)
  const int64_t rows_per_slice = a.block_schedule ? a.M / a.n_experts : a.M;
  const int64_t fit = (int64_t)(2.5 * 1024 * 1024) / ((int64_t)BM * a.K / 2);
  int64_t group_m = rows_per_slice / BM;
  group_m = group_m > fit ? fit : group_m;
  group_m = group_m < 1 ? 1 : (group_m > 16 ? 16 : group_m);
  auto kern = mm_x4_mxfp4_kernel<BM, ACT>;
  if (int rc = raise_lds_limit_once((const void *)kern)) return rc;
  kern<<<dim3((unsigned)launch), 256, X4Shape<BM>::LDS, st>>>(a, grid_n, total, (int)(counts_live_blocks(a) ? -group_m : group_m));
  return launch_status();
}

template <int ACT>
int dispatch_x4_act(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st) {
  if (a.K < 256) return TAMD_E_UNSUPPORTED;   // (a stage's eight scales of a row are read at once)
  dense_grid(a, block_m, grid_m);
  switch (block_m) {
    case 16: return launch_x4<16, ACT>(a, grid_m, st);
    case 32: return launch_x4<32, ACT>(a, grid_m, st);
    case 64: return launch_x4<64, ACT>(a, grid_m, st);
    case 128: return launch_x4<128, ACT>(a, grid_m, st);
    default: return TAMD_E_UNSUPPORTED;
  }
}
int tiled_mm_swiglu_fp4(const tamd_matmul_args &a, int block_m, int grid_m, hipStream_t st);

}  // namespace tamd
