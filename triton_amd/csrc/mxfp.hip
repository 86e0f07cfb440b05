// MXFP4 / MXFP8 quantise / dequantise for gfx950.  Bandwidth kernels: 128-bit global
// accesses, one 32-element group handled by 4 lanes (quantised axis contiguous)
// or by one lane per column set (quantised axis strided, i.e. the weight layout: tiles
// of 8, 16 or 32 groups x 128 or 256 columns that pass through LDS).
//
// Arithmetic follows numerics_details/mxfp.py:212-363 and :384-449 of the
// reference: scale = 2^ceil(log2(max/6)) taken from the float32 bit pattern,
// q = x * (1/scale), round-to-nearest-even onto {0,.5,1,1.5,2,3,4,6}, saturate.
#include "common.h"
#include <type_traits>

namespace tamd {

// Two e2m1 codes (q0 in the low nibble) by the hardware conversion: round to nearest even onto the e2m1 grid,
// saturating at 6 (v_cvt_scalef32_pk_fp4_f32 with a unit scale).  NaN has no e2m1 code: it becomes the largest
// magnitude with the sign bit of the NaN's pattern.
TAMD_DEVICE uint32_t e2m1_pair(float q0, float q1) {
  uint32_t c = (uint32_t)__builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, q0, q1, 1.0f, 0) & 0xFFu;
  if (q0 != q0) c = (c & 0xF0u) | 7u | ((f32_to_bits(q0) >> 28) & 8u);
  if (q1 != q1) c = (c & 0x0Fu) | ((7u | ((f32_to_bits(q1) >> 28) & 8u)) << 4);
  return c;
}

// The same conversion with the division by the group's scale (a power of two, `ds`) done by the instruction:
// writes the code pair of (a / ds, b / ds) into byte BS of `old`.  Exact wherever a / ds is: callers keep to
// scales whose reciprocal is a normal float and to groups without NaN.
template <int BS>
TAMD_DEVICE uint32_t e2m1_pair_scaled(uint32_t old, float a, float b, float ds) {
  return (uint32_t)__builtin_amdgcn_cvt_scalef32_pk_fp4_f32(old, a, b, ds, BS);
}
// 8 e2m1 codes of one column (rows l0 .. l0+7, v[i] = row l0 + i) -> one 32-bit word
TAMD_DEVICE uint32_t e2m1_word_scaled(const float (&v)[8], float ds) {
  uint32_t w = 0;
  w = e2m1_pair_scaled<0>(w, v[0], v[1], ds);
  w = e2m1_pair_scaled<1>(w, v[2], v[3], ds);
  w = e2m1_pair_scaled<2>(w, v[4], v[5], ds);
  w = e2m1_pair_scaled<3>(w, v[6], v[7], ds);
  return w;
}

// 16-byte accesses to memory that is touched once (non-temporal).  Measured on the two tile kernels below: the
// quantiser is fastest with non-temporal loads of its source and ordinary stores of the codes (110 us; 130 with
// ordinary loads), the dequantiser with ordinary loads of the codes and non-temporal stores of its rows (61 us; 67 with
// ordinary stores, 71 with both non-temporal).
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
TAMD_DEVICE uint4 load_once(const void *p) {
  u32x4_t q = __builtin_nontemporal_load((const u32x4_t *)p);
  return make_uint4(q.x, q.y, q.z, q.w);
}
TAMD_DEVICE void store_once(void *p, uint4 v) {
  __builtin_nontemporal_store(u32x4_t{v.x, v.y, v.z, v.w}, (u32x4_t *)p);
}
// the same as ordinary accesses; through the vector type so that they stay one 16-byte instruction (a 16-byte access
// through a pointer derived from char * is split into four 4-byte ones otherwise, a quarter of the bandwidth)
TAMD_DEVICE uint4 load16(const void *p) {
  u32x4_t q = *(const u32x4_t *)p;
  return make_uint4(q.x, q.y, q.z, q.w);
}
TAMD_DEVICE void store16(void *p, uint4 v) { *(u32x4_t *)p = u32x4_t{v.x, v.y, v.z, v.w}; }

// Value kinds of a microscaled tensor: e2m1 codes (two per byte), or fp8 bytes.  Largest magnitude and
// largest power of two of each (mxfp.py:206-209, mxfp_details/_downcast_to_mxfp.py:24-31).
constexpr int QK_E2M1 = 0, QK_E4M3 = 1, QK_E5M2 = 2;
template <int QK>
constexpr float kMaxQ = QK == QK_E2M1 ? 6.0f : (QK == QK_E4M3 ? 448.0f : 57344.0f);
template <int QK>
constexpr float kInvPow2Q = QK == QK_E2M1 ? 0.25f : (QK == QK_E4M3 ? 1.0f / 256.0f : 1.0f / 32768.0f);

// e8m0 byte of a group with the largest magnitude gmax.
template <int QK>
TAMD_DEVICE uint32_t group_scale_byte(float gmax, int mode) {
  constexpr int DT = QK == QK_E2M1 ? TAMD_MXFP4 : (QK == QK_E4M3 ? TAMD_FP8_E4M3 : TAMD_FP8_E5M2);
  return mode == TAMD_ROUND_UP ? ceil_scale_byte<DT>(gmax) : f32_to_bits(gmax * kInvPow2Q<QK>) >> 23;
}
// 1 / 2^(e-127): 2^(127-e), of which the one for e = 254 is a subnormal; 0 for e = 0 (an empty group) and for infinity
TAMD_DEVICE float scale_reciprocal(uint32_t e) {
  return bits_to_f32(e == 0u || e == 255u ? 0u : (e == 254u ? 0x00400000u : (254u - e) << 23));
}
// Returns the multiplier 1/scale and writes the e8m0 byte.
template <int QK = QK_E2M1>
TAMD_DEVICE float group_scale(float gmax, int mode, uint32_t &scale_byte) {
  scale_byte = group_scale_byte<QK>(gmax, mode);
  return scale_reciprocal(scale_byte);
}

TAMD_DEVICE float e2m1_value(uint32_t code) {
  uint32_t m = code & 7u;
  uint32_t bits = m < 2u ? (m ? 0x3F000000u : 0u) : ((((m >> 1) + 126u) << 23) | ((m & 1u) << 22));
  return bits_to_f32(bits | ((code & 8u) << 28));
}

// q (already multiplied by 1/scale) -> fp8 byte: clamp to the finite range, round to nearest even (mxfp.py:313-316)
template <int QK>
TAMD_DEVICE uint32_t fp8_code(float q) {
  if (q != q) return 0x7Fu;
  const float c = __builtin_fminf(__builtin_fmaxf(q, -kMaxQ<QK>), kMaxQ<QK>);
  if constexpr (QK == QK_E4M3) return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, c, 0, false) & 0xFFu;
  return (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(c, c, 0, false) & 0xFFu;
}
template <int QK>
TAMD_DEVICE float fp8_value(uint32_t byte) {
  if constexpr (QK == QK_E4M3) return __builtin_amdgcn_cvt_f32_fp8((int)byte, 0);
  return __builtin_amdgcn_cvt_f32_bf8((int)byte, 0);
}

template <int DT>
constexpr float kMaxFinite =
    DT == TAMD_F32 ? 3.4028234663852886e+38f : (DT == TAMD_BF16 ? 3.3895313892515355e+38f : 65504.f);

template <int DT, int QK = QK_E2M1>
TAMD_DEVICE float dequant_one(uint32_t code, float mult, bool is_nan) {
  float v = (QK == QK_E2M1 ? e2m1_value(code) : fp8_value<QK>(code)) * mult;
  constexpr float mf = kMaxFinite<DT>;
  v = v != v ? v : __builtin_fminf(__builtin_fmaxf(v, -mf), mf);
  // e5m2 has infinities: they pass through whatever the scale is (mxfp.py:438-440 of the reference)
  if (QK == QK_E5M2 && (code & 0x7Fu) == 0x7Cu) v = bits_to_f32(0x7F800000u | ((code & 0x80u) << 24));
  return is_nan ? bits_to_f32(0x7FC00000u) : v;
}

template <int DT>
TAMD_DEVICE uint32_t pack2(float a, float b) {
  if constexpr (DT == TAMD_BF16) return f32_to_bf16_bits(a) | (f32_to_bf16_bits(b) << 16);
  return f32_to_f16_bits(a) | (f32_to_f16_bits(b) << 16);
}

// Division of an index below 2^31 by a divisor fixed for the launch: q = (mulhi(n, mul) + n) >> shift (Granlund and
// Montgomery, "Division by invariant integers using multiplication").  The row kernels below have 16 bytes of work per
// thread, and the two 64-bit divisions that placed a group were most of their instructions.
struct FastDiv {
  uint32_t d, mul, shift;
};
inline FastDiv fast_div(int64_t d) {
  if (d < 1 || d >= ((int64_t)1 << 31)) return FastDiv{0, 0, 0};   // (not used: the launch takes 64-bit divisions)
  uint32_t sh = 0;
  while (((uint64_t)1 << sh) < (uint64_t)d) ++sh;
  return FastDiv{(uint32_t)d, (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << sh) - (uint64_t)d)) / (uint64_t)d + 1), sh};
}
TAMD_DEVICE uint32_t div_by(uint32_t n, const FastDiv &f) { return (__umulhi(n, f.mul) + n) >> f.shift; }

// Where group number `gid` of `total` lies: (batch entry, row, group of the row).
struct GroupDiv {
  int64_t total, G, nr;
  FastDiv by_g, by_nr;
  int wide;    // 2^31 groups or more
};
inline GroupDiv group_div(int64_t nb, int64_t nr, int64_t G) {
  const int64_t total = nb * nr * G;
  return GroupDiv{total, G, nr, fast_div(G), fast_div(nr), total >= ((int64_t)1 << 31)};
}
TAMD_DEVICE void place_group(const GroupDiv &d, int64_t gid, int64_t &b, int64_t &r, int64_t &g) {
  if (d.wide) {
    const int64_t run = gid / d.G;
    g = gid - run * d.G;
    b = run / d.nr;
    r = run - b * d.nr;
  } else {
    const uint32_t run = div_by((uint32_t)gid, d.by_g);
    g = (uint32_t)gid - run * d.by_g.d;
    const uint32_t bb = div_by(run, d.by_nr);
    b = bb;
    r = run - bb * d.by_nr.d;
  }
}

// ---------------------------------------------------------------------------
// downcast, quantised axis contiguous in the source: 4 lanes x 8 elements per group, U groups per thread (64 apart,
// their loads requested together).  Bound by the latency of its loads; with a 64-bit division per index and codes made
// pair by pair it was bound by its instructions (8192 x 2880 bf16 -> e2m1: 20.4 us, now 14.5; 59 MB).
// ---------------------------------------------------------------------------
template <int DT, bool VEC, int QK, int U>
__global__ __launch_bounds__(256) void downcast_rows_kernel(
    const void *__restrict__ src, GroupDiv div, int64_t ssb, int64_t ssr, uint8_t *__restrict__ vals, int64_t vsb, int64_t vsr,
    uint8_t *__restrict__ scales, int64_t csb, int64_t csr, int mode) {
  const int sub = threadIdx.x & 3;
  const int64_t gid0 = (int64_t)blockIdx.x * (64 * U) + (threadIdx.x >> 2);
  int64_t b[U], r[U], g[U];
  constexpr int NQ = DT == TAMD_F32 ? 2 : 1;   // 16-byte pieces of a thread's 8 elements
  uint4 raw[VEC ? U : 1][NQ];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t gid = gid0 + u * 64;
    place_group(div, gid < div.total ? gid : 0, b[u], r[u], g[u]);
    if constexpr (VEC) {
      const char *p = (const char *)src + (b[u] * ssb + r[u] * ssr + g[u] * 32 + sub * 8) * (DT == TAMD_F32 ? 4 : 2);
#pragma unroll
      for (int q = 0; q < NQ; ++q) raw[u][q] = load16(p + q * 16);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float v[8];
    if constexpr (VEC) {
      const uint4 a = raw[u][0];
      if constexpr (DT == TAMD_F32) {
        const uint4 c = raw[u][1];
        v[0] = bits_to_f32(a.x); v[1] = bits_to_f32(a.y); v[2] = bits_to_f32(a.z); v[3] = bits_to_f32(a.w);
        v[4] = bits_to_f32(c.x); v[5] = bits_to_f32(c.y); v[6] = bits_to_f32(c.z); v[7] = bits_to_f32(c.w);
      } else {
        const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[2 * j] = DT == TAMD_BF16 ? bf16_bits_to_f32(w[j] & 0xFFFFu) : f16_bits_to_f32(w[j] & 0xFFFFu);
          v[2 * j + 1] = DT == TAMD_BF16 ? bf16_bits_to_f32(w[j] >> 16) : f16_bits_to_f32(w[j] >> 16);
        }
      }
    } else {
      const int64_t off = b[u] * ssb + r[u] * ssr + g[u] * 32 + sub * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = load_as_f32<DT>(src, off + j);
    }
    float m = 0.f;
    bool any_nan = false;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      m = __builtin_fmaxf(m, __builtin_fabsf(v[j]));
      any_nan |= v[j] != v[j];
    }
    // (the group's four lanes are a quad: swaps inside it are moves in the register file)
    m = __builtin_fmaxf(m, bits_to_f32((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f32_to_bits(m), 0xB1, 0xF, 0xF, true)));
    m = __builtin_fmaxf(m, bits_to_f32((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f32_to_bits(m), 0x4E, 0xF, 0xF, true)));
    uint32_t sbyte;
    const float qs = group_scale<QK>(m, mode, sbyte);
    float q[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] = v[j] * qs;
    any_nan |= sbyte >= 0xFEu;   // an infinite magnitude times a zero multiplier
    uint32_t lo = 0, hi = 0;
    if constexpr (QK == QK_E2M1) {
      if (!any_nan) {
        lo = e2m1_word_scaled(q, 1.0f);
      } else {
#pragma unroll
        for (int j = 0; j < 8; j += 2) lo |= e2m1_pair(q[j], q[j + 1]) << (4 * j);
      }
    } else if (!any_nan) {
      float c[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) c[j] = __builtin_amdgcn_fmed3f(q[j], -kMaxQ<QK>, kMaxQ<QK>);
      if constexpr (QK == QK_E4M3) {
        lo = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], 0, false), true);
        hi = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c[6], c[7], __builtin_amdgcn_cvt_pk_fp8_f32(c[4], c[5], 0, false), true);
      } else {
        lo = (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(c[2], c[3], __builtin_amdgcn_cvt_pk_bf8_f32(c[0], c[1], 0, false), true);
        hi = (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(c[6], c[7], __builtin_amdgcn_cvt_pk_bf8_f32(c[4], c[5], 0, false), true);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lo |= fp8_code<QK>(q[j]) << (8 * j);
        hi |= fp8_code<QK>(q[4 + j]) << (8 * j);
      }
    }
    if (gid0 + u * 64 < div.total) {
      uint8_t *vp = vals + b[u] * vsb + r[u] * vsr;
      if constexpr (QK == QK_E2M1) *(uint32_t *)(vp + g[u] * 16 + sub * 4) = lo;
      else *(uint2 *)(vp + g[u] * 32 + sub * 8) = make_uint2(lo, hi);
      if (sub == 0) scales[b[u] * csb + r[u] * csr + g[u]] = (uint8_t)sbyte;
    }
  }
}

// ---------------------------------------------------------------------------
// downcast, source contiguous along r (quantised axis strided), any alignment: a thread owns one column and
// walks the 32 rows of one group.  The aligned case has the tile kernel below.
// ---------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(256) void downcast_cols_kernel(
    const void *__restrict__ src, int64_t nb, int64_t G, int64_t nr, int64_t ssb, int64_t ssl,
    uint8_t *__restrict__ vals, int64_t vsb, int64_t vsr, uint8_t *__restrict__ scales, int64_t csb,
    int64_t csr, int mode) {
  // a workgroup covers 8 consecutive groups of 32 columns: the 8 lanes that share a column write 8 x 16
  // consecutive bytes of its codes (one 128-byte line) and 8 consecutive scale bytes.  The grid is
  // ceil(nr / 32) * ceil(G / 8) * nb workgroups (launch_downcast).
  int64_t blocks_r = (nr + 31) / 32;
  int64_t g_chunks = (G + 7) / 8;
  int64_t bid = blockIdx.x;
  int64_t br = bid % blocks_r;
  int64_t t = bid / blocks_r;
  int64_t g = (t % g_chunks) * 8 + threadIdx.x % 8;
  int64_t b = t / g_chunks;
  int64_t r0 = br * 32 + threadIdx.x / 8;
  if (r0 >= nr || g >= G || b >= nb) return;
  constexpr int ES = DT == TAMD_F32 ? 4 : 2;
  const char *base = (const char *)src + (b * ssb + g * 32 * ssl + r0) * ES;
  float mx = 0.f;
  float v[32];
#pragma unroll
  for (int l = 0; l < 32; ++l) {
    v[l] = load_as_f32<DT>(base, l * ssl);
    mx = __builtin_fmaxf(mx, __builtin_fabsf(v[l]));
  }
  uint32_t sbyte;
  float qs = group_scale(mx, mode, sbyte);
  uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
  for (int l = 0; l < 32; l += 2) w[l >> 3] |= e2m1_pair(v[l] * qs, v[l + 1] * qs) << (4 * (l & 7));
  *(uint4 *)(vals + b * vsb + r0 * vsr + g * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  scales[b * csb + r0 * csr + g] = (uint8_t)sbyte;
}

// ---------------------------------------------------------------------------
// downcast, source contiguous along r, 16-byte aligned: a workgroup quantises a tile of GT groups x 32*NV
// columns.  A load instruction of a wave reads 512 contiguous bytes of two source rows (a thread keeps the 32
// rows of its NV columns in registers, as above); the codes pass through LDS so that they leave as GT x 16
// contiguous bytes per column.  ONCE: the source's loads are non-temporal, since each is read once (a line too).
// ---------------------------------------------------------------------------
template <int DT>
constexpr int kTileCols = 32 * (DT == TAMD_F32 ? 4 : 8);
template <int DT, int GT>
constexpr size_t kTileLds = (size_t)kTileCols<DT> * GT * 17;

template <int DT, int GT, bool ONCE>
__global__ __launch_bounds__(256) void downcast_cols_tile_kernel(
    const void *__restrict__ src, int64_t nb, int64_t G, int64_t nr, int64_t ssb, int64_t ssl,
    uint8_t *__restrict__ vals, int64_t vsb, int64_t vsr, uint8_t *__restrict__ scales, int64_t csb,
    int64_t csr, int mode) {
  constexpr int ES = DT == TAMD_F32 ? 4 : 2;
  constexpr int NV = 16 / ES;
  constexpr int CW = kTileCols<DT>;
  // s_codes[column][slot]: slot = group ^ (column / NV) % 8 keeps both the writes (two groups, 32 column sets
  // per wave) and the reads (GT groups of 256 / GT columns per workgroup) spread over the banks
  extern __shared__ uint4 s_tile[];
  uint4 *s_codes = s_tile;
  uint8_t *s_sc = (uint8_t *)(s_tile + CW * GT);
  const int64_t tiles_r = (nr + CW - 1) / CW;
  const int64_t g_chunks = (G + GT - 1) / GT;
  const int64_t bid = blockIdx.x;
  const int64_t br = bid % tiles_r;
  const int64_t t = bid / tiles_r;
  const int64_t gc = t % g_chunks;
  const int64_t b = t / g_chunks;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int cs = lane % 32;  // the thread's column set
  const int64_t col0 = br * CW + cs * NV;
#pragma unroll 1
  for (int pass = 0; pass < GT / 8; ++pass) {
    const int gl = pass * 8 + wave * 2 + lane / 32;
    const int64_t g = gc * GT + gl;
    if (g >= G || col0 >= nr) continue;
    const char *base = (const char *)src + (b * ssb + g * 32 * ssl + col0) * ES;
    uint4 raw[32];
#pragma unroll
    for (int l = 0; l < 32; ++l) raw[l] = ONCE ? load_once(base + (int64_t)l * ssl * ES) : load16((const uint8_t *)base + (int64_t)l * ssl * ES);
    auto elem = [&](int l, int c) -> float {
      const uint4 &q = raw[l];
      uint32_t w[4] = {q.x, q.y, q.z, q.w};
      if constexpr (DT == TAMD_F32) return bits_to_f32(w[c]);
      uint32_t h = (c & 1) ? (w[c >> 1] >> 16) : (w[c >> 1] & 0xFFFFu);
      if constexpr (DT == TAMD_BF16) return bf16_bits_to_f32(h);
      return f16_bits_to_f32(h);
    };
    float mx[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) mx[c] = 0.f;
#pragma unroll
    for (int l = 0; l < 32; ++l)
#pragma unroll
      for (int c = 0; c < NV; ++c) mx[c] = __builtin_fmaxf(mx[c], __builtin_fabsf(elem(l, c)));
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      bool has_nan = false;
#pragma unroll
      for (int l = 0; l < 32; l += 2) has_nan |= __builtin_isunordered(elem(l, c), elem(l + 1, c));
      const uint32_t sbyte = group_scale_byte<QK_E2M1>(mx[c], mode);
      uint32_t w[4] = {0, 0, 0, 0};
      if (!has_nan && sbyte - 2u <= 251u) {
        // the usual case: the instruction divides by the scale and packs, 1.5 operations per element
        const float ds = bits_to_f32(sbyte << 23);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v[8] = {elem(8 * j, c),     elem(8 * j + 1, c), elem(8 * j + 2, c), elem(8 * j + 3, c),
                              elem(8 * j + 4, c), elem(8 * j + 5, c), elem(8 * j + 6, c), elem(8 * j + 7, c)};
          w[j] = e2m1_word_scaled(v, ds);
        }
      } else {
        const float qs = scale_reciprocal(sbyte);
#pragma unroll
        for (int l = 0; l < 32; l += 2)
          w[l >> 3] |= e2m1_pair(elem(l, c) * qs, elem(l + 1, c) * qs) << (4 * (l & 7));
      }
      const int cl = cs * NV + c;
      s_codes[cl * GT + (gl ^ (cs & 7))] = make_uint4(w[0], w[1], w[2], w[3]);
      s_sc[cl * GT + gl] = (uint8_t)sbyte;
    }
  }
  sync_threads();
  const int64_t n_g = G - gc * GT < GT ? G - gc * GT : GT;
  const int64_t n_c = nr - br * CW < CW ? nr - br * CW : CW;
  uint8_t *vbase = vals + b * vsb + br * CW * vsr + gc * GT * 16;
  uint8_t *sbase = scales + b * csb + br * CW * csr + gc * GT;
  const int part = threadIdx.x % GT;
  if (part < n_g) {
#pragma unroll 4
    for (int c = threadIdx.x / GT; c < n_c; c += 256 / GT) {
      store16(vbase + (int64_t)c * vsr + part * 16, s_codes[c * GT + (part ^ ((c / NV) & 7))]);
      sbase[(int64_t)c * csr + part] = s_sc[c * GT + part];
    }
  }
}

// ---------------------------------------------------------------------------
// upcast, destination contiguous along the quantised axis
// ---------------------------------------------------------------------------
// Scale bytes for which 0.5 * 2^(s-127) and 6 * 2^(s-127) are normal numbers of the destination type: there the
// product needs neither the clamp to the largest finite value nor any care about denormals.
template <int DT>
constexpr uint32_t kFastLo = DT == TAMD_F16 ? 127u - 13u : 3u;
template <int DT>
constexpr uint32_t kFastHi = DT == TAMD_F16 ? 127u + 13u : 252u;

template <int DT, int QK, int U>
__global__ __launch_bounds__(256) void upcast_rows_kernel(
    const uint8_t *__restrict__ vals, int64_t vsb, int64_t vsr, const uint8_t *__restrict__ scales,
    int64_t csb, int64_t csr, void *__restrict__ dst, GroupDiv div, int64_t dsb, int64_t dsr, int vec_ok) {
  const int sub = threadIdx.x & 3;
  const int64_t gid0 = (int64_t)blockIdx.x * (64 * U) + (threadIdx.x >> 2);
  int64_t b[U], r[U], g[U];
  uint32_t sc[U], w0[U], w1[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t gid = gid0 + u * 64;
    place_group(div, gid < div.total ? gid : 0, b[u], r[u], g[u]);
    const uint8_t *vp = vals + b[u] * vsb + r[u] * vsr;
    sc[u] = scales[b[u] * csb + r[u] * csr + g[u]];
    if constexpr (QK == QK_E2M1) {
      w0[u] = *(const uint32_t *)(vp + g[u] * 16 + sub * 4);
      w1[u] = 0;
    } else {
      const uint2 w = *(const uint2 *)(vp + g[u] * 32 + sub * 8);
      w0[u] = w.x, w1[u] = w.y;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (gid0 + u * 64 >= div.total) return;
    const uint32_t s = sc[u];
    const float mult = bits_to_f32(s << 23);
    float o[8];
    if (QK == QK_E2M1 && s - kFastLo<DT> <= kFastHi<DT> - kFastLo<DT>) {
      // the usual case: the conversion instruction yields every product (see upcast_rows2_regs); float32 products of
      // 16-bit normal numbers round to themselves below
      typedef float f32x2v_t __attribute__((ext_vector_type(2)));
      const f32x2v_t p0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w0[u], mult, 0);
      const f32x2v_t p1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w0[u], mult, 1);
      const f32x2v_t p2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w0[u], mult, 2);
      const f32x2v_t p3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w0[u], mult, 3);
      o[0] = p0.x, o[1] = p0.y, o[2] = p1.x, o[3] = p1.y, o[4] = p2.x, o[5] = p2.y, o[6] = p3.x, o[7] = p3.y;
    } else if constexpr (QK == QK_E2M1) {
      const bool is_nan = s == 0xFFu;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = dequant_one<DT>((w0[u] >> (4 * j)) & 0xFu, mult, is_nan);
    } else {
      const bool is_nan = s == 0xFFu;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        o[j] = dequant_one<DT, QK>((w0[u] >> (8 * j)) & 0xFFu, mult, is_nan);
        o[4 + j] = dequant_one<DT, QK>((w1[u] >> (8 * j)) & 0xFFu, mult, is_nan);
      }
    }
    const int64_t off = b[u] * dsb + r[u] * dsr + g[u] * 32 + sub * 8;
    if (vec_ok) {
      if constexpr (DT == TAMD_F32) {
        char *p = (char *)((float *)dst + off);
        store16(p, make_uint4(f32_to_bits(o[0]), f32_to_bits(o[1]), f32_to_bits(o[2]), f32_to_bits(o[3])));
        store16(p + 16, make_uint4(f32_to_bits(o[4]), f32_to_bits(o[5]), f32_to_bits(o[6]), f32_to_bits(o[7])));
      } else {
        store16((uint16_t *)dst + off,
                make_uint4(pack2<DT>(o[0], o[1]), pack2<DT>(o[2], o[3]), pack2<DT>(o[4], o[5]), pack2<DT>(o[6], o[7])));
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) store_from_f32<DT>(dst, off + j, o[j]);
    }
  }
}

// ---------------------------------------------------------------------------
// upcast, destination contiguous along r, any alignment: a thread owns one column of one group.  The aligned
// case has the tile kernel below.
// ---------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(256) void upcast_cols_kernel(
    const uint8_t *__restrict__ vals, int64_t vsb, int64_t vsr, const uint8_t *__restrict__ scales,
    int64_t csb, int64_t csr, void *__restrict__ dst, int64_t nb, int64_t G, int64_t nr, int64_t dsb,
    int64_t dsl) {
  // a workgroup covers 8 consecutive groups of 32 columns: the 8 lanes that share a column read 8 x 16
  // consecutive bytes of its codes (one 128-byte line) and 8 consecutive scale bytes.  The grid is
  // ceil(nr / 32) * ceil(G / 8) * nb workgroups (launch_upcast).
  int64_t blocks_r = (nr + 31) / 32;
  int64_t g_chunks = (G + 7) / 8;
  int64_t bid = blockIdx.x;
  int64_t br = bid % blocks_r;
  int64_t t = bid / blocks_r;
  int64_t g = (t % g_chunks) * 8 + threadIdx.x % 8;
  int64_t b = t / g_chunks;
  int64_t r0 = br * 32 + threadIdx.x / 8;
  if (r0 >= nr || g >= G || b >= nb) return;
  const uint4 code = *(const uint4 *)(vals + b * vsb + r0 * vsr + g * 16);
  const uint32_t s = scales[b * csb + r0 * csr + g];
  const float mult = bits_to_f32(s << 23);
  const bool isn = s == 0xFFu;
  constexpr int ES = DT == TAMD_F32 ? 4 : 2;
  char *base = (char *)dst + (b * dsb + g * 32 * dsl + r0) * ES;
  const uint32_t w[4] = {code.x, code.y, code.z, code.w};
#pragma unroll
  for (int l = 0; l < 32; ++l)
    store_from_f32<DT>(base + (int64_t)l * dsl * ES, 0, dequant_one<DT>((w[l >> 3] >> (4 * (l & 7))) & 0xFu, mult, isn));
}

// Rows l and l+1 (the code pairs in byte BS of w[c]) of a thread's 16 / sizeof(element) columns, dequantised by the
// conversion instruction and stored as two 16-byte pieces `pitch` bytes apart.
template <int DT, int BS>
TAMD_DEVICE void upcast_rows2_regs(const uint32_t *w, const float *mult, uint4 &r0, uint4 &r1) {
  if constexpr (DT == TAMD_F32) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    f32x2_t v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[c], mult[c], BS);
    r0 = make_uint4(f32_to_bits(v[0].x), f32_to_bits(v[1].x), f32_to_bits(v[2].x), f32_to_bits(v[3].x));
    r1 = make_uint4(f32_to_bits(v[0].y), f32_to_bits(v[1].y), f32_to_bits(v[2].y), f32_to_bits(v[3].y));
  } else {
    uint32_t u[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if constexpr (DT == TAMD_BF16) {
        typedef __bf16 bf16x2v_t __attribute__((ext_vector_type(2)));
        bf16x2v_t t = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[c], mult[c], BS);
        u[c] = __builtin_bit_cast(uint32_t, t);
      } else {
        typedef _Float16 f16x2v_t __attribute__((ext_vector_type(2)));
        f16x2v_t t = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w[c], mult[c], BS);
        u[c] = __builtin_bit_cast(uint32_t, t);
      }
    }
    // u[c] = (row l, row l+1) of column c; a stored word is (column 2i, column 2i+1) of one row
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      lo[i] = __builtin_amdgcn_perm(u[2 * i + 1], u[2 * i], 0x05040100u);
      hi[i] = __builtin_amdgcn_perm(u[2 * i + 1], u[2 * i], 0x07060302u);
    }
    r0 = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    r1 = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  }
}
template <bool ONCE>
TAMD_DEVICE void store_row(char *p, const uint4 &v) {
  if (ONCE) store_once(p, v);
  else store16((uint8_t *)p, v);
}
template <int DT, int BS, bool ONCE = true>
TAMD_DEVICE void upcast_rows2(const uint32_t *w, const float *mult, char *p, int64_t pitch) {
  uint4 r0, r1;
  upcast_rows2_regs<DT, BS>(w, mult, r0, r1);
  store_row<ONCE>(p, r0);
  store_row<ONCE>(p + pitch, r1);
}

// ---------------------------------------------------------------------------
// upcast, destination contiguous along r, 16-byte aligned: the mirror image of downcast_cols_tile_kernel.  The
// codes and scales of a tile of GT groups x 32*NV columns come in as GT x 16 contiguous bytes per column, pass
// through LDS, and a store instruction of a wave writes 512 contiguous bytes of two destination rows (ONCE: past the caches).
// ---------------------------------------------------------------------------
template <int DT, int GT, bool ONCE>
__global__ __launch_bounds__(256) void upcast_cols_tile_kernel(
    const uint8_t *__restrict__ vals, int64_t vsb, int64_t vsr, const uint8_t *__restrict__ scales,
    int64_t csb, int64_t csr, void *__restrict__ dst, int64_t nb, int64_t G, int64_t nr, int64_t dsb,
    int64_t dsl) {
  constexpr int ES = DT == TAMD_F32 ? 4 : 2;
  constexpr int NV = 16 / ES;
  constexpr int CW = kTileCols<DT>;
  extern __shared__ uint4 s_tile[];
  uint4 *s_codes = s_tile;
  uint8_t *s_sc = (uint8_t *)(s_tile + CW * GT);
  const int64_t tiles_r = (nr + CW - 1) / CW;
  const int64_t g_chunks = (G + GT - 1) / GT;
  const int64_t bid = blockIdx.x;
  const int64_t br = bid % tiles_r;
  const int64_t t = bid / tiles_r;
  const int64_t gc = t % g_chunks;
  const int64_t b = t / g_chunks;
  const int64_t n_g = G - gc * GT < GT ? G - gc * GT : GT;
  const int64_t n_c = nr - br * CW < CW ? nr - br * CW : CW;
  const uint8_t *vbase = vals + b * vsb + br * CW * vsr + gc * GT * 16;
  const uint8_t *sbase = scales + b * csb + br * CW * csr + gc * GT;
  const int part = threadIdx.x % GT;
  if (part < n_g) {
#pragma unroll 4
    for (int c = threadIdx.x / GT; c < n_c; c += 256 / GT) {
      s_codes[c * GT + (part ^ ((c / NV) & 7))] = load16(vbase + (int64_t)c * vsr + part * 16);
      s_sc[c * GT + part] = sbase[(int64_t)c * csr + part];
    }
  }
  sync_threads();
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int cs = lane % 32;
  const int64_t col0 = br * CW + cs * NV;
#pragma unroll 1
  for (int pass = 0; pass < GT / 8; ++pass) {
    const int gl = pass * 8 + wave * 2 + lane / 32;
    const int64_t g = gc * GT + gl;
    if (g >= G || col0 >= nr) continue;
    uint4 code[NV];
    float mult[NV];
    bool isn[NV];
    bool fast = true;
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      const int cl = cs * NV + c;
      code[c] = s_codes[cl * GT + (gl ^ (cs & 7))];
      uint32_t s = s_sc[cl * GT + gl];
      mult[c] = bits_to_f32(s << 23);
      isn[c] = s == 0xFFu;
      fast &= s - kFastLo<DT> <= kFastHi<DT> - kFastLo<DT>;
    }
    char *base = (char *)dst + (b * dsb + g * 32 * dsl + col0) * ES;
    if (fast) {
      // the usual case: every product code * scale is a normal number of the destination type, and the
      // conversion instruction yields it for two rows of a column at once
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t w[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) w[c] = j == 0 ? code[c].x : (j == 1 ? code[c].y : (j == 2 ? code[c].z : code[c].w));
        upcast_rows2<DT, 0, ONCE>(w, mult, base + (int64_t)(8 * j + 0) * dsl * ES, dsl * ES);
        upcast_rows2<DT, 1, ONCE>(w, mult, base + (int64_t)(8 * j + 2) * dsl * ES, dsl * ES);
        upcast_rows2<DT, 2, ONCE>(w, mult, base + (int64_t)(8 * j + 4) * dsl * ES, dsl * ES);
        upcast_rows2<DT, 3, ONCE>(w, mult, base + (int64_t)(8 * j + 6) * dsl * ES, dsl * ES);
      }
      continue;
    }
#pragma unroll
    for (int l = 0; l < 32; ++l) {
      float o[NV];
#pragma unroll
      for (int c = 0; c < NV; ++c) {
        uint32_t w[4] = {code[c].x, code[c].y, code[c].z, code[c].w};
        o[c] = dequant_one<DT>((w[l >> 3] >> (4 * (l & 7))) & 0xFu, mult[c], isn[c]);
      }
      char *p = base + (int64_t)l * dsl * ES;
      if constexpr (DT == TAMD_F32) {
        store_row<ONCE>(p, make_uint4(f32_to_bits(o[0]), f32_to_bits(o[1]), f32_to_bits(o[2]), f32_to_bits(o[3])));
      } else {
        store_row<ONCE>(p, make_uint4(pack2<DT>(o[0], o[1]), pack2<DT>(o[2], o[3]), pack2<DT>(o[4], o[5]),
                                      pack2<DT>(o[6], o[7])));
      }
    }
  }
}

// Up to how many tiles of 8 groups a tensor whose quantised axis is strided goes to the kernels of one column per thread instead of the tile
// kernels, given for 256 CUs.  Tiles of 32 groups (float32) and 16 left most of a last round empty on all but the largest tensors: 160
// of [1 .. 8, 512 .. 2880, 512 .. 5760], time with tiles of 8 over the time before: quantising float32 0.927, bf16 0.911, dequantising to
// float32 0.87, to bf16 0.855.  If rows start on lines the larger tiles, whose runs are longer, are as fast or faster again above some rounds over
// the CUs (kWideAbove*, in quarters): quantising float32 and dequantising to 16 bits about four (8 x 2880 x 5760: 109.5 us in tiles of 32,
// 109.8 of 8), quantising 16-bit types above one and a quarter (8 x 2336 x 2688 29 us, 37 in tiles of 8; 8 x 2400 x 5760 72 and 79, but where the
// larger ones end in half a round, 8 x 2048 x 5120, 49 and 44), dequantising to float32 above two and a half (0.94 to 1.0 of the time in tiles
// of 32, 1.05 in those of 8).  With the merged halves below, float32 and back to bf16: 8 x 2304 x 3032 55.9 + 43.2 -> 48.9 + 24.1 us,
// 8 x 2432 x 1432 39.9 + 23.3 -> 24.5 + 14.7; 200 others 0.86 and 0.82 over the same memory again and again, 0.87 and 0.87 into memory that no cache
// holds (the worst 1.09 and 1.19).  Just above the lines columns and tiles take about as long: quantising 7.5 us and 7.8 at 130 tiles
// (float32), 8.6 and 8.7 at 105 (bf16), dequantising 4.9 and 5.7 at 33, 5.3 and 5.6 at 45.
constexpr int64_t kColumnsUpToDown = 96, kColumnsUpToUp = 40;
constexpr int kWideAboveDown32 = 15, kWideAboveDown16 = 5, kWideAboveUp32 = 10, kWideAboveUp16 = 15;
// Rows that do not start on a line of 128 bytes: a line that two tiles share is read, or written in part, by both.  Non-temporal loads fetch
// it from memory for each (plain loads 0.86 to 0.98 of the time); non-temporal stores send it out in halves.  Plain ones let the caches
// merge these, which pays if they hold the destination's lines from an earlier use: dequantising over the same memory, time with plain
// stores over that with the others, by tiles: to 320 0.91 (16-bit) and 0.98 (float32), to 640 0.76 and 0.80, beyond 0.66 to 0.83; into
// memory that no cache holds 1.20 and 1.26, 1.13 and 1.12, 0.99 to 1.08.  Hence plain from 320 tiles on.  With rows on lines plain
// loads and stores take 1.04 to 1.2.
constexpr int64_t kMergedFromUp = 320;

// Groups from which a thread of the row kernels takes two: below, the grid would no longer give every SIMD a few waves.
constexpr int64_t kRowsUnrolled = 64 * 2048;

template <int DT, int QK>
int launch_downcast(const void *src, int64_t nb, int64_t L, int64_t nr, int64_t ssb, int64_t ssl, int64_t ssr,
                    uint8_t *vals, int64_t vsb, int64_t vsr, uint8_t *scales, int64_t csb, int64_t csr,
                    int mode, hipStream_t st) {
  const int64_t G = L / 32;
  constexpr int ES = DT == TAMD_F32 ? 4 : 2;
  if (ssl == 1) {
    const GroupDiv div = group_div(nb, nr, G);
    bool vec = aligned(src, 16) && (ssb * ES) % 16 == 0 && (ssr * ES) % 16 == 0;
    if ((div.total + 63) / 64 > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
    const int u = div.total >= kRowsUnrolled ? 2 : 1;
    const unsigned blocks = (unsigned)((div.total + 64 * u - 1) / (64 * u));
    auto kern = vec ? (u == 2 ? downcast_rows_kernel<DT, true, QK, 2> : downcast_rows_kernel<DT, true, QK, 1>)
                    : downcast_rows_kernel<DT, false, QK, 1>;
    kern<<<dim3(vec ? blocks : (unsigned)((div.total + 63) / 64)), 256, 0, st>>>(src, div, ssb, ssr, vals, vsb, vsr, scales, csb,
                                                                                 csr, mode);
    return launch_status();
  }
  if (ssr != 1) return TAMD_E_INVALID;
  if constexpr (QK != QK_E2M1) return TAMD_E_UNSUPPORTED;  // fp8 values: quantised axis contiguous only
  constexpr int NV = 16 / ES;
  bool vec = nr % NV == 0 && aligned(src, 16) && (ssb * ES) % 16 == 0 && (ssl * ES) % 16 == 0;
  constexpr int CW = kTileCols<DT>;
  constexpr int WIDE = DT == TAMD_F32 ? 32 : 16;   // 64 KiB of codes
  const int64_t cols = (nr + CW - 1) / CW * nb, tiles = cols * ((G + 7) / 8);
  int cus = 0;
  if (int rc = cu_count(cus)) return rc;
  if (vec && tiles * 256 > kColumnsUpToDown * cus) {
    const bool lines = aligned(src, 128) && (ssb * ES) % 128 == 0 && (ssl * ES) % 128 == 0;
    const bool wide = lines && 4 * cols * ((G + WIDE - 1) / WIDE) > (ES == 4 ? kWideAboveDown32 : kWideAboveDown16) * (int64_t)cus;
    const int64_t blocks = wide ? cols * ((G + WIDE - 1) / WIDE) : tiles;
    if (blocks > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
    auto kern = wide ? downcast_cols_tile_kernel<DT, WIDE, true> : (lines ? downcast_cols_tile_kernel<DT, 8, true> : downcast_cols_tile_kernel<DT, 8, false>);
    if (int rc = raise_lds_limit_once((const void *)kern)) return rc;
    kern<<<dim3((unsigned)blocks), 256, wide ? kTileLds<DT, WIDE> : kTileLds<DT, 8>, st>>>(src, nb, G, nr, ssb, ssl, vals, vsb, vsr, scales, csb, csr,
                                                                               mode);
  } else {
    int64_t blocks = ((nr + 31) / 32) * ((G + 7) / 8) * nb;
    if (blocks > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
    downcast_cols_kernel<DT><<<dim3((unsigned)blocks), 256, 0, st>>>(src, nb, G, nr, ssb, ssl, vals, vsb, vsr,
                                                                       scales, csb, csr, mode);
  }
  return launch_status();
}

template <int DT, int QK>
int launch_upcast(const uint8_t *vals, int64_t vsb, int64_t vsr, const uint8_t *scales, int64_t csb, int64_t csr,
                  void *dst, int64_t nb, int64_t L, int64_t nr, int64_t dsb, int64_t dsl, int64_t dsr,
                  hipStream_t st) {
  const int64_t G = L / 32;
  constexpr int ES = DT == TAMD_F32 ? 4 : 2;
  if (dsl == 1) {
    const GroupDiv div = group_div(nb, nr, G);
    int vec = aligned(dst, 16) && (dsb * ES) % 16 == 0 && (dsr * ES) % 16 == 0;
    if ((div.total + 63) / 64 > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
    const int u = div.total >= kRowsUnrolled ? 2 : 1;
    auto kern = u == 2 ? upcast_rows_kernel<DT, QK, 2> : upcast_rows_kernel<DT, QK, 1>;
    kern<<<dim3((unsigned)((div.total + 64 * u - 1) / (64 * u))), 256, 0, st>>>(vals, vsb, vsr, scales, csb, csr, dst, div, dsb,
                                                                              dsr, vec);
    return launch_status();
  }
  if (dsr != 1) return TAMD_E_INVALID;
  if constexpr (QK != QK_E2M1) return TAMD_E_UNSUPPORTED;  // fp8 values: quantised axis contiguous only
  constexpr int NV = 16 / ES;
  bool vec = nr % NV == 0 && aligned(dst, 16) && (dsb * ES) % 16 == 0 && (dsl * ES) % 16 == 0;
  constexpr int CW = kTileCols<DT>;
  const int64_t cols = (nr + CW - 1) / CW * nb, tiles = cols * ((G + 7) / 8);
  int cus = 0;
  if (int rc = cu_count(cus)) return rc;
  if (vec && tiles * 256 > kColumnsUpToUp * cus) {
    const bool lines = aligned(dst, 128) && (dsb * ES) % 128 == 0 && (dsl * ES) % 128 == 0;
    const bool wide = lines && 4 * cols * ((G + 15) / 16) > (ES == 4 ? kWideAboveUp32 : kWideAboveUp16) * (int64_t)cus;
    const int64_t blocks = wide ? cols * ((G + 15) / 16) : tiles;
    if (blocks > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
    auto kern = wide ? upcast_cols_tile_kernel<DT, 16, true>
                     : (lines || tiles * 256 <= kMergedFromUp * cus ? upcast_cols_tile_kernel<DT, 8, true> : upcast_cols_tile_kernel<DT, 8, false>);
    if (int rc = raise_lds_limit_once((const void *)kern)) return rc;
    kern<<<dim3((unsigned)blocks), 256, wide ? kTileLds<DT, 16> : kTileLds<DT, 8>, st>>>(vals, vsb, vsr, scales, csb, csr, dst, nb, G, nr, dsb, dsl);
  } else {
    int64_t blocks = ((nr + 31) / 32) * ((G + 7) / 8) * nb;
    if (blocks > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
    upcast_cols_kernel<DT><<<dim3((unsigned)blocks), 256, 0, st>>>(vals, vsb, vsr, scales, csb, csr, dst, nb, G,
                                                                     nr, dsb, dsl);
  }
  return launch_status();
}

// e2m1 codes -> float8_e4m3fn bytes, exactly: every e2m1 number (0, .5, 1, 1.5, 2, 3, 4, 6 and their negatives) is an
// e4m3 number.  The eight magnitudes' bytes are a table of two 32-bit words, out of which one byte permutation takes
// four codes at a time.
TAMD_DEVICE uint2 widen_e2m1_word(uint32_t w) {   // eight codes, low nibble first
  constexpr uint32_t kLo = 0x3C383000u, kHi = 0x4C484440u;  // {0x00, 0x30, 0x38, 0x3C}, {0x40, 0x44, 0x48, 0x4C}
  const uint32_t even = __builtin_amdgcn_perm(kHi, kLo, w & 0x07070707u) | ((w & 0x08080808u) << 4);
  const uint32_t odd = __builtin_amdgcn_perm(kHi, kLo, (w >> 4) & 0x07070707u) | (w & 0x80808080u);
  return make_uint2(__builtin_amdgcn_perm(odd, even, 0x05010400u), __builtin_amdgcn_perm(odd, even, 0x07030602u));
}
// A thread widens U pieces, a workgroup's width apart, of 8 packed bytes of a row to 16 bytes each: a wave reads 512 and
// writes 1024 contiguous bytes (8192 x 2880 codes: 9.2 us; 12.9 code by code).  div: a "group" is such a piece.
template <int U>
__global__ __launch_bounds__(256) void widen_e2m1_rows_kernel(const uint8_t *__restrict__ src, GroupDiv div, int64_t row_bytes,
                                                              int64_t src_stride, uint8_t *__restrict__ dst, int64_t dst_stride,
                                                              int vec) {
  const int64_t i0 = (int64_t)blockIdx.x * (256 * U) + threadIdx.x;
  int64_t b, r[U], c[U];
  uint2 q[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = i0 + u * 256;
    place_group(div, i < div.total ? i : 0, b, r[u], c[u]);
    c[u] *= 8;
    if (vec) q[u] = *(const uint2 *)(src + r[u] * src_stride + c[u]);   // (whole 8-byte pieces)
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (i0 + u * 256 >= div.total) return;
    uint8_t *dp = dst + r[u] * dst_stride + 2 * c[u];
    if (vec) {
      const uint2 lo = widen_e2m1_word(q[u].x), hi = widen_e2m1_word(q[u].y);
      store16(dp, make_uint4(lo.x, lo.y, hi.x, hi.y));
    } else {
      const uint8_t *sp = src + r[u] * src_stride + c[u];
      for (int64_t j = 0; j < 8 && c[u] + j < row_bytes; ++j) {
        const uint32_t two = widen_e2m1_word(sp[j]).x;
        dp[2 * j] = (uint8_t)two;
        dp[2 * j + 1] = (uint8_t)(two >> 8);
      }
    }
  }
}

}  // namespace tamd

using namespace tamd;

extern "C" int tamd_widen_mxfp4_rows(const uint8_t *src, int64_t rows, int64_t row_bytes, int64_t src_stride, uint8_t *dst,
                                     int64_t dst_stride, void *stream) {
  if (rows < 0 || row_bytes < 0) return TAMD_E_INVALID;
  if (rows == 0 || row_bytes == 0) return 0;
  if (!src || !dst) return TAMD_E_INVALID;
  const int vec = aligned(src, 8) && aligned(dst, 16) && src_stride % 8 == 0 && dst_stride % 16 == 0 && row_bytes % 8 == 0;
  const GroupDiv div = group_div(1, rows, (row_bytes + 7) / 8);
  const int u = div.total >= 4 * kRowsUnrolled ? 2 : 1;
  if ((div.total + 255) / 256 > 0x7FFFFFFF) return TAMD_E_UNSUPPORTED;
  auto kern = u == 2 ? widen_e2m1_rows_kernel<2> : widen_e2m1_rows_kernel<1>;
  kern<<<dim3((unsigned)((div.total + 256 * u - 1) / (256 * u))), 256, 0, (hipStream_t)stream>>>(src, div, row_bytes, src_stride, dst,
                                                                                              dst_stride, vec);
  return launch_status();
}

extern "C" int tamd_downcast_mxfp(const void *src, int src_dtype, int64_t nb, int64_t L, int64_t nr,
                                  int64_t src_stride_b, int64_t src_stride_l, int64_t src_stride_r,
                                  void *out_vals, int out_dtype, int64_t val_stride_b, int64_t val_stride_r,
                                  uint8_t *out_scales, int64_t scale_stride_b, int64_t scale_stride_r,
                                  int rounding_mode, void *stream) {
  if (nb < 0 || L < 0 || nr < 0 || L % 32 != 0) return TAMD_E_INVALID;
  if (rounding_mode != TAMD_ROUND_UP && rounding_mode != TAMD_ROUND_DOWN) return TAMD_E_INVALID;
  if (out_dtype != TAMD_MXFP4 && out_dtype != TAMD_FP8_E4M3 && out_dtype != TAMD_FP8_E5M2) return TAMD_E_INVALID;
  if (nb == 0 || L == 0 || nr == 0) return 0;
  if (!src || !out_vals || !out_scales) return TAMD_E_INVALID;
  if (!aligned(out_vals, 16) || val_stride_b % 16 != 0 || val_stride_r % 16 != 0) return TAMD_E_ALIGNMENT;
  hipStream_t st = (hipStream_t)stream;
  uint8_t *v = (uint8_t *)out_vals;
#define TAMD_DOWN(DT, QK)                                                                                          \
  return launch_downcast<DT, QK>(src, nb, L, nr, src_stride_b, src_stride_l, src_stride_r, v, val_stride_b,          \
                                 val_stride_r, out_scales, scale_stride_b, scale_stride_r, rounding_mode, st)
#define TAMD_DOWN_SRC(QK)                      \
  switch (src_dtype) {                         \
    case TAMD_F32: TAMD_DOWN(TAMD_F32, QK);    \
    case TAMD_BF16: TAMD_DOWN(TAMD_BF16, QK);  \
    case TAMD_F16: TAMD_DOWN(TAMD_F16, QK);    \
    default: return TAMD_E_INVALID;            \
  }
  if (out_dtype == TAMD_MXFP4) TAMD_DOWN_SRC(QK_E2M1)
  if (out_dtype == TAMD_FP8_E4M3) TAMD_DOWN_SRC(QK_E4M3)
  TAMD_DOWN_SRC(QK_E5M2)
#undef TAMD_DOWN_SRC
#undef TAMD_DOWN
}

extern "C" int tamd_upcast_mxfp(const void *vals, int val_dtype, int64_t val_stride_b, int64_t val_stride_r,
                                const uint8_t *scales, int64_t scale_stride_b, int64_t scale_stride_r, void *dst,
                                int dst_dtype, int64_t nb, int64_t L, int64_t nr, int64_t dst_stride_b,
                                int64_t dst_stride_l, int64_t dst_stride_r, void *stream) {
  if (nb < 0 || L < 0 || nr < 0 || L % 32 != 0) return TAMD_E_INVALID;
  if (val_dtype != TAMD_MXFP4 && val_dtype != TAMD_FP8_E4M3 && val_dtype != TAMD_FP8_E5M2) return TAMD_E_INVALID;
  if (nb == 0 || L == 0 || nr == 0) return 0;
  if (!vals || !scales || !dst) return TAMD_E_INVALID;
  if (!aligned(vals, 16) || val_stride_b % 16 != 0 || val_stride_r % 16 != 0) return TAMD_E_ALIGNMENT;
  hipStream_t st = (hipStream_t)stream;
  const uint8_t *v = (const uint8_t *)vals;
#define TAMD_UP(DT, QK)                                                                                              \
  return launch_upcast<DT, QK>(v, val_stride_b, val_stride_r, scales, scale_stride_b, scale_stride_r, dst, nb, L, nr, \
                               dst_stride_b, dst_stride_l, dst_stride_r, st)
#define TAMD_UP_DST(QK)                      \
  switch (dst_dtype) {                       \
    case TAMD_F32: TAMD_UP(TAMD_F32, QK);    \
    case TAMD_BF16: TAMD_UP(TAMD_BF16, QK);  \
    case TAMD_F16: TAMD_UP(TAMD_F16, QK);    \
    default: return TAMD_E_INVALID;          \
  }
  if (val_dtype == TAMD_MXFP4) TAMD_UP_DST(QK_E2M1)
  if (val_dtype == TAMD_FP8_E4M3) TAMD_UP_DST(QK_E4M3)
  TAMD_UP_DST(QK_E5M2)
#undef TAMD_UP_DST
#undef TAMD_UP
}
