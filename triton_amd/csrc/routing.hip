// Routing kernels for gfx950: top-k (+softmax, bit matrix), expert histogram with a
// stable expert-major ordering of the (token, slot) pairs, and the ragged-tensor
// block metadata.  Integer work only; wave64 ballots / shuffles, no float atomics,
// results independent of scheduling.
#include <atomic>

#include "common.h"

namespace tamd {

// Workspace of tamd_routing_metadata_static: lives in the code object instead of an allocation.  Every GPU that
// loads the library holds its own copy (4 MiB) until the process ends.
constexpr int64_t kStaticWorkspaceInts = 1 << 20;
static __device__ __align__(256) int32_t scratch[kStaticWorkspaceInts];

// ---------------------------------------------------------------------------
// top-k
// ---------------------------------------------------------------------------
// Order-preserving map of a logit's bits.  -0.0 counts as +0.0, so that both zeros tie, as they do under the reference's
// stable argsort of -x (topk_details/_topk_forward.py:15-30; the sum with +0.0 takes the sign).
TAMD_DEVICE uint32_t ordered_bits(float x) {
  const uint32_t u = f32_to_bits(x + 0.0f);
  return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
// Its inverse (a -0.0 logit comes back as +0.0).
TAMD_DEVICE float logit_of(uint32_t u) { return bits_to_f32(u ^ (~(uint32_t)((int32_t)u >> 31) | 0x80000000u)); }

// Sort key of a logit and its column, all different: the higher logit first, the lower column among equals
// (_topk_forward.py:15-30).  A 16-bit logit and its column are one 32-bit integer, a float32 and its column two.  (As one double
// between 1 and 2 the latter would need one instruction to find the larger of two keys, but v_max_f64 takes a quarter of the lanes
// at a time; a 64-bit integer comparison likewise.)
template <int DT>
struct SortKey {
  uint32_t v;  // logit in the high half, 0xFFFF - column in the low half
  TAMD_DEVICE static SortKey of(float x, int col) {
    const uint32_t u = (DT == TAMD_F16 ? f32_to_f16_bits(x + 0.0f) : f32_to_bf16_bits(x + 0.0f)) << 16;  // exact: x was loaded from such bits
    return {((u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u)) & 0xFFFF0000u) | (0xFFFFu - (uint32_t)col)};
  }
  TAMD_DEVICE static SortKey none(int col) { return {0xFFFFu - (uint32_t)col}; }
  TAMD_DEVICE uint32_t column_field() const { return v & 0xFFFFu; }
  TAMD_DEVICE bool same(SortKey o) const { return v == o.v; }
  TAMD_DEVICE float logit() const {
    const uint32_t u = f32_to_bits(logit_of(v & 0xFFFF0000u)) >> 16;
    return DT == TAMD_F16 ? f16_bits_to_f32(u) : bf16_bits_to_f32(u);
  }
  TAMD_DEVICE static void order(SortKey &a, SortKey &b) {
    const uint32_t x = a.v, y = b.v;
    a.v = x > y ? x : y;
    b.v = x > y ? y : x;
  }
  TAMD_DEVICE static SortKey pick(bool first, SortKey a, SortKey b) { return {first ? a.v : b.v}; }
  template <int L>
  TAMD_DEVICE static SortKey group_largest(SortKey q);
};
template <>
struct SortKey<TAMD_F32> {
  uint32_t u, c;  // logit, 0xFFFF - column
  TAMD_DEVICE static SortKey of(float x, int col) { return {ordered_bits(x), 0xFFFFu - (uint32_t)col}; }
  TAMD_DEVICE static SortKey none(int col) { return {0u, 0xFFFFu - (uint32_t)col}; }
  TAMD_DEVICE uint32_t column_field() const { return c; }
  TAMD_DEVICE bool same(SortKey o) const { return c == o.c; }
  TAMD_DEVICE float logit() const { return logit_of(u); }
  TAMD_DEVICE static void order(SortKey &a, SortKey &b) {
    const SortKey x = a, y = b;
    const bool less = x.u < y.u;  // (equal ones stay as they are: the lower column is in front)
    a = {x.u > y.u ? x.u : y.u, less ? y.c : x.c};
    b = {x.u > y.u ? y.u : x.u, less ? x.c : y.c};
  }
  TAMD_DEVICE static SortKey pick(bool first, SortKey a, SortKey b) { return {first ? a.u : b.u, first ? a.c : b.c}; }
  template <int L>
  TAMD_DEVICE static SortKey group_largest(SortKey q);
};

// Reductions over aligned groups of L lanes; every lane gets the result.  Step O (1, 2, 4, ...) of the butterfly combines a lane with
// one of the other aligned block of O lanes.  All lanes of a block of O hold the same value by then, so for O = 4 and 8 the
// partner may be the mirrored lane, which, like the swaps inside a quad, the data-parallel move does in the register
// file; for 16 and 32 rows of lanes change places, and the two registers that hold the halves then are combined.
template <int O>
TAMD_DEVICE void butterfly(uint32_t v, uint32_t &a, uint32_t &b) {
  a = v;
  if constexpr (O == 1) b = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true);        // quad_perm [1,0,3,2]
  else if constexpr (O == 2) b = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
  else if constexpr (O == 4) b = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true);  // row_half_mirror
  else if constexpr (O == 8) b = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true);  // row_mirror
  else if constexpr (O == 16) { const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false); a = r[0]; b = r[1]; }
  else { const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false); a = r[0]; b = r[1]; }
}
template <int L, int O = 1, typename OP>
TAMD_DEVICE uint32_t group_reduce(uint32_t v, OP op) {
  if constexpr (O >= L) {
    return v;
  } else {
    uint32_t a, b;
    butterfly<O>(v, a, b);
    return group_reduce<L, O * 2>(op(a, b), op);
  }
}
template <int L>
TAMD_DEVICE uint32_t group_max_u32(uint32_t v) {
  return group_reduce<L>(v, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}
template <int L>
TAMD_DEVICE uint32_t group_min_u32(uint32_t v) {
  return group_reduce<L>(v, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
}
template <int DT>
template <int L>
TAMD_DEVICE SortKey<DT> SortKey<DT>::group_largest(SortKey q) { return {group_max_u32<L>(q.v)}; }
template <int L>
TAMD_DEVICE SortKey<TAMD_F32> SortKey<TAMD_F32>::group_largest(SortKey q) {
  const uint32_t m = group_max_u32<L>(q.u);
  return {m, group_max_u32<L>(q.u == m ? q.c : 0u)};
}
template <int L>
TAMD_DEVICE float group_sum_f32(float v) {
  return bits_to_f32(group_reduce<L>(f32_to_bits(v), [](uint32_t a, uint32_t b) { return f32_to_bits(bits_to_f32(a) + bits_to_f32(b)); }));
}
template <int L>
TAMD_DEVICE float group_max_f32(float v) {
  return bits_to_f32(group_reduce<L>(f32_to_bits(v), [](uint32_t a, uint32_t b) { return f32_to_bits(__builtin_fmaxf(bits_to_f32(a), bits_to_f32(b))); }));
}

// The logits of a row, EPL of its L lanes' columns `sub + j * L` each, requested together: every lane loads (columns past the
// end re-read the last one), and `take` pins the values before they are selected: a load that the compiler may move under
// the per-lane condition is awaited before the next one is issued, EPL round trips to memory instead of one.
template <int DT, int L, int EPL>
struct RowLogits {
  float x[EPL];
  TAMD_DEVICE void request(const void *p, int64_t off, int n_cols, int sub) {
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      const int c = sub + j * L;
      x[j] = load_as_f32<DT>(p, off + (c < n_cols ? c : n_cols - 1));
    }
  }
  TAMD_DEVICE void take(SortKey<DT> *keys, int n_cols, int sub) {
#pragma unroll
    for (int j = 0; j < EPL; ++j) asm volatile("" : "+v"(x[j]));
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      keys[j] = SortKey<DT>::pick(sub + j * L < n_cols, SortKey<DT>::of(x[j], sub + j * L), SortKey<DT>::none(sub + j * L));
  }
};

// What a lane of a row's group knows of the k picked columns: the column and the key of the pick that its own place in the
// group stands for, the largest key, and the picked columns among 32 * sub .. 32 * sub + 31 as bits.
template <int DT>
struct Picks {
  SortKey<DT> key, top;
  uint32_t word;
  TAMD_DEVICE int col() const { return (int)(0xFFFFu - key.column_field()); }
};

// Every lane sorts its own keys; then k rounds of: the largest of the lanes' first keys, taken out of its lane's list.  What it costs is
// the number of instructions, about six cycles each to a wave that has its SIMD to itself: one row of 128 float32
// logits and four picks 2200 cycles, 3200 when every round compared all keys as 64-bit integers.  (Two 32-bit searches of all
// keys per round 2100 and, with eight picks of 16-bit logits, 64 rows of 256 9.2 us instead of 8.4; as doubles 2100.)
template <int L, int EPL, int DT>
TAMD_DEVICE Picks<DT> pick_columns(SortKey<DT> *q, int k, int sub) {
  // Only neighbours change places: equal logits never pass each other, so one comparison of 32 bits decides (28 exchanges for 8 keys, where
  // the 19 of a shorter network would have to compare the columns too).  Of up to four picks a lane gives no more than its four
  // largest: these to the front, two at a time, whose exchanges overlap (13 for two, 22 for four; more than four 1 to 3 % slower so than
  // all of them in rounds).  With all keys sorted throughout, 65000 rows of 384 float32 logits took 39.9 us with one pick, 33 with
  // every round comparing all keys, 30.1 now; 43.5, 39 and 34.0 with two; 49.9, 52 and 47.9 with four.
  if (EPL > 4 && k <= 4) {
#pragma unroll
    for (int front = 0; front < 4; front += 2) {
      if (front >= k) break;
#pragma unroll
      for (int f = front; f < front + 2; ++f)
#pragma unroll
        for (int j = EPL - 2; j >= f; --j) SortKey<DT>::order(q[j], q[j + 1]);
    }
  } else {
#pragma unroll
    for (int round = 0; round < EPL; ++round)
#pragma unroll
      for (int j = round & 1; j + 1 < EPL; j += 2) SortKey<DT>::order(q[j], q[j + 1]);
  }
  Picks<DT> r{q[0], q[0], 0u};
#pragma clang loop unroll(disable)
  for (int pass = 0; pass < k; ++pass) {
    const SortKey<DT> m = SortKey<DT>::template group_largest<L>(q[0]);
    const bool mine = q[0].same(m);
#pragma unroll
    for (int j = 0; j < 3; ++j) q[j] = SortKey<DT>::pick(mine, q[j + 1], q[j]);
    if (EPL > 4 && k > 4) {  // (of four picks no lane gives more than its first four)
#pragma unroll
      for (int j = 3; j < EPL - 1; ++j) q[j] = SortKey<DT>::pick(mine, q[j + 1], q[j]);
    }
    if (mine && (EPL == 4 || k > 4)) q[EPL - 1] = SortKey<DT>::none(0xFFFF);  // the list's end
    r.top = SortKey<DT>::pick(pass == 0, m, r.top);
    r.key = SortKey<DT>::pick(sub == pass, m, r.key);
    const uint32_t f = m.column_field();
    r.word |= f >> 5 == 0x7FFu - (uint32_t)sub ? 0x80000000u >> (f & 31u) : 0u;
  }
  return r;
}

// The softmax over the picked logits, of this lane's slot (lanes past the last slot: 0).
template <int L, int DT>
TAMD_DEVICE float pick_softmax(const Picks<DT> &r, bool slot) {
  const float e = slot ? expf(r.key.logit() - r.top.logit()) : 0.f;
  return e / group_sum_f32<L>(e);
}

// Bits of a gate weight as stored.
template <int DT>
TAMD_DEVICE uint32_t stored_bits(float v) {
  return DT == TAMD_F32 ? f32_to_bits(v) : DT == TAMD_BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v);
}

// L lanes cooperate on one row; EPL > 0 keeps ceil(n_cols/L) <= EPL keys in registers.  `row` is the row of this
// thread's group of L lanes (any row >= n_rows: a group that only takes part in the shuffles).
template <int DT, int L, int EPL>
TAMD_DEVICE void topk_row(const void *__restrict__ x, int64_t x_stride, int n_rows, int n_cols, int k,
                          int apply_softmax, int use_provided, void *__restrict__ y_vals,
                          int16_t *__restrict__ y_indx, int64_t y_stride, uint32_t *__restrict__ bits,
                          int64_t bits_stride_row, int64_t bits_stride_word, int64_t row) {
  const int sub = threadIdx.x % L;
  const bool live = row < n_rows;
  const int64_t rrow = live ? row : 0;
  const int64_t xoff = rrow * x_stride;
  int my_idx = 0;
  uint32_t words = 0u;  // (EPL > 0)
  float v = 0.f, top = 0.f;
  const bool slot = sub < k;
  if (use_provided) {
    if (slot) my_idx = y_indx[rrow * y_stride + sub];
  } else if constexpr (EPL > 0) {
    RowLogits<DT, L, EPL> logits;
    SortKey<DT> keys[EPL];
    logits.request(x, xoff, n_cols, sub);
    logits.take(keys, n_cols, sub);
    const Picks<DT> r = pick_columns<L, EPL, DT>(keys, k, sub);
    my_idx = r.col();
    words = r.word;
    v = r.key.logit();  // a zero's sign is lost in the key and makes no difference to the softmax
    top = r.top.logit();
  } else {
    // bits and column of the last pick: what comes after it in the order has lower bits, or the same and a higher column
    uint32_t prev = 0u, prev_c = 0u;
    for (int pass = 0; pass < k; ++pass) {
      uint32_t m = 0u, mc = 0xFFFFu;
      for (int c = sub; c < n_cols; c += L) {
        const uint32_t q = ordered_bits(load_as_f32<DT>(x, xoff + c));
        const bool left = pass == 0 || q < prev || (q == prev && (uint32_t)c > prev_c);
        if (left && (mc == 0xFFFFu || q > m)) {
          m = q;
          mc = (uint32_t)c;
        }
      }
      const uint32_t best = group_max_u32<L>(mc == 0xFFFFu ? 0u : m);
      prev_c = group_min_u32<L>(m == best ? mc : 0xFFFFu);
      prev = best;
      if (pass == 0) top = logit_of(best);
      if (sub == pass) {
        v = logit_of(best);
        my_idx = (int)prev_c;
      }
    }
  }
  if (!apply_softmax || use_provided) v = slot ? load_as_f32<DT>(x, xoff + my_idx) : 0.f;
  if (apply_softmax) {
    const float mx = use_provided ? group_max_f32<L>(slot ? v : -__builtin_inff()) : top;
    const float e = slot ? expf(v - mx) : 0.f;
    v = e / group_sum_f32<L>(e);
  }
  if (live && slot) {
    store_from_f32<DT>(y_vals, rrow * y_stride + sub, v);
    if (!use_provided) y_indx[rrow * y_stride + sub] = (int16_t)my_idx;
  }
  const int n_words = (n_cols + 31) / 32;
  if (EPL > 0 && !use_provided) {
    if (live && sub < n_words) bits[rrow * bits_stride_row + (int64_t)sub * bits_stride_word] = words;
    return;
  }
  const int base_lane = (threadIdx.x % kWave) - sub;
  for (int w0 = 0; w0 < n_words; w0 += L) {
    int w = w0 + sub;
    uint32_t word = 0;
    for (int j = 0; j < k; ++j) {
      int ij = __shfl(my_idx, base_lane + j);
      word |= ((ij >> 5) == w) ? (1u << (ij & 31)) : 0u;
    }
    if (live && w < n_words) bits[rrow * bits_stride_row + (int64_t)w * bits_stride_word] = word;
  }
}

template <int DT, int L, int EPL>
__global__ __launch_bounds__(256) void topk_kernel(const void *__restrict__ x, int64_t x_stride, int n_rows,
                                                   int n_cols, int k, int apply_softmax, int use_provided,
                                                   void *__restrict__ y_vals, int16_t *__restrict__ y_indx,
                                                   int64_t y_stride, uint32_t *__restrict__ bits,
                                                   int64_t bits_stride_row, int64_t bits_stride_word) {
  constexpr int ROWS_PER_BLOCK = 256 / L;
  topk_row<DT, L, EPL>(x, x_stride, n_rows, n_cols, k, apply_softmax, use_provided, y_vals, y_indx, y_stride, bits,
                       bits_stride_row, bits_stride_word, (int64_t)blockIdx.x * ROWS_PER_BLOCK + threadIdx.x / L);
}

template <int DT>
int launch_topk(const void *x, int64_t xs, int n_rows, int n_cols, int k, int sm, int prov, void *yv, int16_t *yi,
                int64_t ys, uint32_t *bits, int64_t bsr, int64_t bsw, hipStream_t st) {
  int need = (n_cols + 7) / 8;
  if (need < k) need = k;
#define TAMD_TOPK(LL, EE)                                                                                    \
  topk_kernel<DT, LL, EE><<<dim3((unsigned)((n_rows + (256 / LL) - 1) / (256 / LL))), 256, 0, st>>>(          \
      x, xs, n_rows, n_cols, k, sm, prov, yv, yi, ys, bits, bsr, bsw)
  if (need <= 8) {
    if (n_cols <= 32) TAMD_TOPK(8, 4);
    else TAMD_TOPK(8, 8);
  } else if (need <= 16) TAMD_TOPK(16, 8);
  else if (need <= 32) TAMD_TOPK(32, 8);
  else if (n_cols <= 512) TAMD_TOPK(64, 8);
  else TAMD_TOPK(64, 0);
#undef TAMD_TOPK
  return launch_status();
}

// ---------------------------------------------------------------------------
// histogram + stable expert-major ordering
// ---------------------------------------------------------------------------
// Entries are processed in chunks of 64 (one wave, one entry per lane).  Inside a
// chunk the rank of an entry among the entries with the same expert is a popcount
// of the lanes below it that hold the same id; the set of such lanes is built
// from one ballot per bit of the id.  Per-chunk counts are prefix-summed inside a
// block (CH chunks), per-block totals across blocks, expert totals across
// experts; the position of an entry is the sum of those three prefixes and its
// in-chunk rank.  No atomics, so the order is the flat (token, slot) order.

TAMD_DEVICE int load_indx(const void *p, int is16, int64_t i) {
  return is16 ? (int)((const int16_t *)p)[i] : ((const int32_t *)p)[i];
}

// Gate weights in expert-sorted order (what the down projection takes as its per-row factors): entry i of the flat
// (token, slot) array goes to the place its index goes to.  Bits are moved as they are; `esz` is 4 or 2, 0 when no
// sorted copy is asked for.
struct Gates {
  const void *vals;
  void *sorted;
  int esz;
};
TAMD_DEVICE uint32_t load_gate(const Gates &g, int64_t i) {
  if (g.esz == 4) return ((const uint32_t *)g.vals)[i];
  if (g.esz == 2) return ((const uint16_t *)g.vals)[i];
  return 0;
}
TAMD_DEVICE void store_gate(const Gates &g, int64_t pos, uint32_t bits) {
  if (g.esz == 4) ((uint32_t *)g.sorted)[pos] = bits;
  else if (g.esz == 2) ((uint16_t *)g.sorted)[pos] = (uint16_t)bits;
}

TAMD_DEVICE uint64_t same_id_mask(int e, bool valid, int nbits) {
  uint64_t same = __ballot(valid);
  for (int b = 0; b < nbits; ++b) {
    bool bit = (e >> b) & 1;
    uint64_t m = __ballot(valid && bit);
    same &= bit ? m : ~m;
  }
  return same;
}

TAMD_DEVICE uint64_t lanemask_lt() {
  int lane = threadIdx.x % kWave;
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

__global__ __launch_bounds__(1024) void hist_kernel(const void *__restrict__ indx, int is16, int64_t n, int E,
                                                   int CH, int nbits, int32_t *__restrict__ chunk_pref,
                                                   int32_t *__restrict__ block_tot) {
  extern __shared__ int32_t hist[];  // [CH][E]
  const int blk = blockIdx.x;
  for (int i = threadIdx.x; i < CH * E; i += 1024) hist[i] = 0;
  sync_threads();
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  for (int c = wave; c < CH; c += 16) {  // CH <= 16: one chunk per wave, so a workgroup waits for memory once
    int64_t i = ((int64_t)blk * CH + c) * 64 + lane;
    int e = i < n ? load_indx(indx, is16, i) : -1;
    bool valid = e >= 0 && e < E;
    uint64_t same = same_id_mask(e, valid, nbits);
    if (valid && (same & lanemask_lt()) == 0) hist[c * E + e] = __popcll(same);
  }
  sync_threads();
  for (int e = threadIdx.x; e < E; e += 1024) {
    int run = 0;
    for (int c = 0; c < CH; ++c) {
      int t = hist[c * E + e];
      if (chunk_pref) chunk_pref[((int64_t)blk * CH + c) * E + e] = run;  // (not needed by order_scan_kernel)
      run += t;
    }
    block_tot[(int64_t)blk * E + e] = run;
  }
}

// Exclusive scan of up to 1024 ints held one per thread; returns the total.
TAMD_DEVICE int block_excl_scan_1024(int v, int &total, int *lds /* >= 17 ints */) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int inc = wave_incl_scan(v);
  sync_threads();
  if (lane == kWave - 1) lds[wave] = inc;
  sync_threads();
  if (threadIdx.x == 0) {
    int run = 0;
    for (int w = 0; w < 16; ++w) {
      int t = lds[w];
      lds[w] = run;
      run += t;
    }
    lds[16] = run;
  }
  sync_threads();
  total = lds[16];
  return inc - v + lds[wave];
}

// Exclusive prefix over the workgroups' totals of expert e (written to `out` when given; it may be `tot` itself);
// returns the expert's total.  Sixteen totals are loaded before any of them is used or stored, so that a thread
// waits for memory once per sixteen blocks and not once per block.
TAMD_DEVICE int scan_block_totals(const int32_t *tot, int32_t *out, int n_blocks, int E, int e) {
  int run = 0;
  for (int b0 = 0; b0 < n_blocks; b0 += 16) {
    int t[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) t[u] = tot[(int64_t)(b0 + u < n_blocks ? b0 + u : n_blocks - 1) * E + e];
#pragma unroll
    for (int u = 0; u < 16; ++u) asm volatile("" : "+v"(t[u]));
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (b0 + u < n_blocks) {
        if (out) out[(int64_t)(b0 + u) * E + e] = run;
        run += t[u];
      }
    }
  }
  return run;
}

__global__ __launch_bounds__(1024) void scan_kernel(int E, int n_blocks, int32_t *__restrict__ block_tot,
                                                    int32_t *__restrict__ col_sum, int32_t *__restrict__ col_offs,
                                                    int32_t *__restrict__ n_valid) {
  __shared__ int lds[17];
  int carry = 0;
  for (int e0 = 0; e0 < E; e0 += 1024) {
    int e = e0 + threadIdx.x;
    int run = 0;
    if (e < E) {
      run = scan_block_totals(block_tot, block_tot, n_blocks, E, e);
      col_sum[e] = run;
    }
    int total;
    int ex = block_excl_scan_1024(run, total, lds);
    if (e < E) col_offs[e] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) *n_valid = carry;
}

__global__ __launch_bounds__(1024) void order_kernel(const void *__restrict__ indx, int is16, int64_t n, int E,
                                                    int CH, int nbits, int k, const int32_t *__restrict__ chunk_pref,
                                                    const int32_t *__restrict__ block_off,
                                                    const int32_t *__restrict__ col_offs,
                                                    const int32_t *__restrict__ n_valid,
                                                    int32_t *__restrict__ col_sorted, int32_t *__restrict__ row_sorted,
                                                    int32_t *__restrict__ gather, Gates gates) {
  const int blk = blockIdx.x;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int nv = *n_valid;
  for (int c = wave; c < CH; c += 16) {
    int64_t chunk = (int64_t)blk * CH + c;
    int64_t i = chunk * 64 + lane;
    int e = i < n ? load_indx(indx, is16, i) : -1;
    bool valid = e >= 0 && e < E;
    uint64_t same = same_id_mask(e, valid, nbits);
    if (valid) {
      int pos = col_offs[e] + block_off[(int64_t)blk * E + e] + chunk_pref[chunk * E + e] +
                __popcll(same & lanemask_lt());
      row_sorted[i] = pos;
      col_sorted[pos] = (int32_t)i;
      if (gather) gather[pos] = (int32_t)(i / k);
      store_gate(gates, pos, load_gate(gates, i));
    } else if (i < n) {
      row_sorted[i] = -1;
    }
    if (i >= nv && i < n) {
      col_sorted[i] = -1;
      if (gather) gather[i] = 0;  // trunc(-1 / k)
    }
  }
}

struct MetaPlan {
  int CH;
  int nbits;
  int64_t n_chunks, n_blocks;
  int64_t off_chunk_pref, off_block_tot, off_block_off, off_col_offs, off_n_valid, total;
};

inline MetaPlan make_meta_plan(int64_t n_indx, int E) {
  MetaPlan p;
  // LDS histogram of CH*E ints, at most 64 KiB
  int ch = 16;
  while (ch > 1 && (int64_t)ch * E * 4 > 65536) ch >>= 1;
  p.CH = ch;
  p.nbits = 0;
  while ((1 << p.nbits) < E) ++p.nbits;
  p.n_chunks = (n_indx + 63) / 64;
  p.n_blocks = (p.n_chunks + ch - 1) / ch;
  if (p.n_blocks < 1) p.n_blocks = 1;
  p.off_chunk_pref = 0;
  p.off_block_tot = p.n_blocks * ch * (int64_t)E;
  p.off_block_off = p.off_block_tot + p.n_blocks * (int64_t)E;
  p.off_col_offs = p.off_block_off + p.n_blocks * (int64_t)E;
  p.off_n_valid = p.off_col_offs + E;
  p.total = p.off_n_valid + 1;
  return p;
}

inline int launch_bitmatrix_metadata(const void *indx, int is16, int64_t n, int E, int k, int32_t *col_sum,
                                     int32_t *col_sorted, int32_t *row_sorted, int32_t *gather, Gates gates, int32_t *ws,
                                     hipStream_t st, bool before_order(void *), void *ctx) {
  MetaPlan p = make_meta_plan(n, E);
  size_t lds = (size_t)p.CH * E * 4;
  hist_kernel<<<dim3((unsigned)p.n_blocks), 1024, lds, st>>>(indx, is16, n, E, p.CH, p.nbits, ws + p.off_chunk_pref,
                                                           ws + p.off_block_tot);
  scan_kernel<<<1, 1024, 0, st>>>(E, (int)p.n_blocks, ws + p.off_block_tot, col_sum, ws + p.off_col_offs,
                                  ws + p.off_n_valid);
  if (before_order && !before_order(ctx)) return launch_status();
  order_kernel<<<dim3((unsigned)p.n_blocks), 1024, 0, st>>>(indx, is16, n, E, p.CH, p.nbits, k, ws + p.off_chunk_pref,
                                                          ws + p.off_block_tot, ws + p.off_col_offs,
                                                          ws + p.off_n_valid, col_sorted, row_sorted, gather, gates);
  return launch_status();
}

// ---------------------------------------------------------------------------
// ragged tensor metadata
// ---------------------------------------------------------------------------
// Row r of the offsets table: r = 0 slice offsets, r >= 1 block offsets for block size 8 << r.
// Wave r < 6 of a workgroup scans row r (64 slices per step with a running carry) into `tab`
// (pitch S + 1) and, when `offs` is given, into global memory.
TAMD_DEVICE void ragged_scan_rows(const int32_t *sizes, int S, int32_t *tab, int32_t *offs, int64_t offs_pitch) {
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (wave >= 6) return;
  const int sh = wave == 0 ? 0 : wave + 3;
  int32_t *trow = tab + (int64_t)wave * (S + 1);
  int32_t *grow = offs ? offs + (int64_t)wave * offs_pitch : nullptr;
  int carry = 0;
  for (int s0 = 0; s0 < S; s0 += kWave) {
    const int s = s0 + lane;
    const int v = s < S ? ((sizes[s] + ((1 << sh) - 1)) >> sh) : 0;
    const int inc = wave_incl_scan(v);
    if (s < S) {
      trow[s] = carry + inc - v;
      if (grow) grow[s] = carry + inc - v;
    }
    carry += __shfl(inc, kWave - 1);
  }
  if (lane == 0) {
    trow[S] = carry;
    if (grow) grow[S] = carry;
  }
}

// Schedule entry j of block size index b is ((j - block_offs[s]) << 16) | s for the slice s whose block
// range holds j (binary search in the scanned row; empty slices are skipped by the search), -1 past
// the last block.  Entries [first, first + count) of the flattened [5][max_blocks] table.
TAMD_DEVICE void ragged_fill_schedule(const int32_t *tab, int S, int32_t *sched, int64_t sched_pitch, int max_blocks,
                                      int64_t first, int64_t count) {
  const bool narrow = first + count <= 0x7FFFFFFF;  // then the table index is found with a 32-bit division
  for (int64_t idx = first + threadIdx.x; idx < first + count; idx += blockDim.x) {
    const int b = narrow ? (int)((uint32_t)idx / (uint32_t)max_blocks) : (int)(idx / max_blocks);
    const int j = (int)(idx - (int64_t)b * max_blocks);
    const int32_t *row = tab + (int64_t)(b + 1) * (S + 1);
    int val = -1;
    if (j < row[S]) {
      int lo = 0, hi = S - 1;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (row[mid + 1] <= j) lo = mid + 1;
        else hi = mid;
      }
      val = ((j - row[lo]) << 16) + lo;
    }
    sched[(int64_t)b * sched_pitch + j] = val;
  }
}

// Every workgroup scans the (small) size vector into its own LDS copy of the table, workgroup 0 also
// writes it out, and the schedule entries are split evenly over the workgroups.
__global__ __launch_bounds__(1024) void ragged_kernel(const int32_t *__restrict__ sizes, int S,
                                                      int32_t *__restrict__ offs, int64_t offs_pitch,
                                                      int32_t *__restrict__ sched, int64_t sched_pitch, int max_blocks) {
  extern __shared__ int32_t tab[];  // [6][S + 1]
  ragged_scan_rows(sizes, S, tab, blockIdx.x == 0 ? offs : nullptr, offs_pitch);
  sync_threads();
  const int64_t total = 5 * (int64_t)max_blocks;
  const int64_t per = (total + gridDim.x - 1) / gridDim.x;
  const int64_t first = per * blockIdx.x;
  if (first < total) ragged_fill_schedule(tab, S, sched, sched_pitch, max_blocks, first, per < total - first ? per : total - first);
}

// Second of three launches for larger index arrays: the prefix sums over the per-workgroup histograms
// (as scan_kernel) merged with the ragged tables.  Every workgroup repeats the small scans into its own
// LDS and fills its share of the schedule; workgroup 0 alone writes the scan results.  The prefix over
// workgroups goes to `block_off` (not in place: the other workgroups still read `block_tot`).
__global__ __launch_bounds__(1024) void scan_ragged_kernel(int E, int n_blocks, const int32_t *__restrict__ block_tot,
                                                           int32_t *__restrict__ block_off, int32_t *__restrict__ col_sum,
                                                           int32_t *__restrict__ col_offs, int32_t *__restrict__ n_valid,
                                                           int32_t *__restrict__ offs, int64_t offs_pitch,
                                                           int32_t *__restrict__ sched, int64_t sched_pitch, int max_blocks) {
  extern __shared__ int32_t sm[];
  int32_t *csum = sm;             // [E]
  int32_t *tab = csum + E;        // [6][E + 1]
  int32_t *scr = tab + 6 * (E + 1);
  const bool lead = blockIdx.x == 0;
  int carry = 0;
  for (int e0 = 0; e0 < E; e0 += 1024) {
    const int e = e0 + threadIdx.x;
    int run = 0;
    if (e < E) {
      run = scan_block_totals(block_tot, lead ? block_off : nullptr, n_blocks, E, e);
      csum[e] = run;
      if (lead) col_sum[e] = run;
    }
    int total;
    const int ex = block_excl_scan_1024(run, total, scr);
    if (lead && e < E) col_offs[e] = carry + ex;
    carry += total;
    sync_threads();
  }
  if (lead && threadIdx.x == 0) *n_valid = carry;
  ragged_scan_rows(csum, E, tab, lead ? offs : nullptr, offs_pitch);
  sync_threads();
  const int64_t total_e = 5 * (int64_t)max_blocks;
  const int64_t per = (total_e + gridDim.x - 1) / gridDim.x;
  const int64_t first = per * blockIdx.x;
  if (first < total_e)
    ragged_fill_schedule(tab, E, sched, sched_pitch, max_blocks, first, per < total_e - first ? per : total_e - first);
}

// ---------------------------------------------------------------------------
// metadata in two launches (up to kMaxTableBlocks blocks of chunks)
// ---------------------------------------------------------------------------
// The first launch leaves one histogram per block of CH chunks (hist_kernel).  In the second, every workgroup reduces that small table by itself -- the experts' totals, their prefix and,
// for the workgroup that orders block `blk`, the counts of the blocks before it -- instead of waiting for a scan kernel
// in between: workgroups 0..nb-1 recount their own chunks and place their entries, the remaining ones build the ragged
// tables and fill the block schedule.
constexpr int kMaxTableBlocks = 128;

// Sums of tot[b][e] over the blocks b of [b_lo, b_hi): all of them, and those before block `blk`.  Sixteen loads are
// in flight together.
TAMD_DEVICE void sum_block_range(const int32_t *__restrict__ tot, int E, int e, int b_lo, int b_hi, int blk, int &all,
                                 int &below) {
  all = 0;
  below = 0;
  for (int b0 = b_lo; b0 < b_hi; b0 += 16) {
    int t[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) t[u] = tot[(int64_t)(b0 + u < b_hi ? b0 + u : b_hi - 1) * E + e];
#pragma unroll
    for (int u = 0; u < 16; ++u) asm volatile("" : "+v"(t[u]));
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      all += b0 + u < b_hi ? t[u] : 0;
      below += b0 + u < b_hi && b0 + u < blk ? t[u] : 0;
    }
  }
}

__global__ __launch_bounds__(1024) void order_scan_kernel(const void *__restrict__ indx, int is16, int n, int E, int CH,
                                                          int nbits, int k, const int32_t *__restrict__ block_tot, int nb,
                                                          int P, int32_t *__restrict__ col_sum,
                                                          int32_t *__restrict__ col_sorted, int32_t *__restrict__ row_sorted,
                                                          int32_t *__restrict__ gather, int32_t *__restrict__ offs,
                                                          int64_t offs_pitch, int32_t *__restrict__ sched,
                                                          int64_t sched_pitch, int max_blocks, Gates gates) {
  extern __shared__ int32_t sm[];
  int32_t *hist = sm;                          // [CH][E]  counts of this block's chunks, then their exclusive prefix
  int32_t *tot = hist + (int64_t)CH * E;       // [E]      entries per expert
  int32_t *boff = tot + E;                     // [E]      entries per expert in the blocks before this one
  int32_t *psum = boff + E;                    // [P][E]   partial sums over ranges of blocks
  int32_t *pbel = psum + (int64_t)P * E;       // [P][E]
  int32_t *tab = pbel + (int64_t)P * E;        // [6][E + 1]
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int blk = blockIdx.x;
  const bool orders = blk < nb;
  // this wave's chunk of the index array: requested first, used after the table has been reduced
  const int i = (blk * CH + wave) * 64 + lane;
  const bool has = orders && wave < CH && i < n;
  int ev = 0;
  uint32_t gate = 0;
  if (n > 0) {
    ev = load_indx(indx, is16, has ? i : 0);
    gate = load_gate(gates, has ? i : 0);
  }
  if (orders)
    for (int j = tid; j < CH * E; j += 1024) hist[j] = 0;
  // 1. partial sums of the table: thread (part, e) takes the blocks [part * per, (part + 1) * per)
  {
    const int part = tid / E, e = tid - part * E;
    if (part < P) {
      const int per = (nb + P - 1) / P;
      const int b_hi = (part + 1) * per < nb ? (part + 1) * per : nb;
      int all, below;
      sum_block_range(block_tot, E, e, part * per, b_hi, blk, all, below);
      psum[part * E + e] = all;
      pbel[part * E + e] = below;
    }
  }
  asm volatile("" : "+v"(ev), "+v"(gate));
  ev = has ? ev : -1;
  sync_threads();
  // 2. totals per expert; counts of this wave's chunk
  for (int e = tid; e < E; e += 1024) {
    int all = 0, below = 0;
    for (int q = 0; q < P; ++q) {
      all += psum[q * E + e];
      below += pbel[q * E + e];
    }
    tot[e] = all;
    boff[e] = below;
    if (blk == 0) col_sum[e] = all;
  }
  const bool valid = ev >= 0 && ev < E;
  const uint64_t same = same_id_mask(ev, valid, nbits);
  if (valid && (same & lanemask_lt()) == 0) hist[wave * E + ev] = __popcll(same);
  sync_threads();
  // 3. exclusive prefix over this block's chunks; the ragged tables (row 0: exclusive prefix over the experts)
  if (orders) {
    for (int e = tid; e < E; e += 1024) {
      int run = 0;
      for (int c = 0; c < CH; ++c) {
        const int v = hist[c * E + e];
        hist[c * E + e] = run;
        run += v;
      }
    }
  }
  ragged_scan_rows(tot, E, tab, blk == nb ? offs : nullptr, offs_pitch);
  sync_threads();
  if (orders) {
    // 4. placement
    const int nv = tab[E];
    if (valid) {
      const int pos = tab[ev] + boff[ev] + hist[wave * E + ev] + __popcll(same & lanemask_lt());
      row_sorted[i] = pos;
      col_sorted[pos] = i;
      if (gather) gather[pos] = i / k;
      store_gate(gates, pos, gate);
    } else if (wave < CH && i < n) {
      row_sorted[i] = -1;
    }
    if (wave < CH && i >= nv && i < n) {
      col_sorted[i] = -1;
      if (gather) gather[i] = 0;  // trunc(-1 / k)
    }
  } else {
    // 4'. this workgroup's share of the block schedule
    const int64_t total = 5 * (int64_t)max_blocks;
    const int64_t shares = (int64_t)gridDim.x - nb;
    const int64_t per = (total + shares - 1) / shares;
    const int64_t first = per * (blk - nb);
    if (first < total) ragged_fill_schedule(tab, E, sched, sched_pitch, max_blocks, first, per < total - first ? per : total - first);
  }
}

// Second launch of the two: the grid, the LDS size and the limits of order_scan_kernel.
inline bool order_scan_applicable(int64_t n, int E, int CH, int64_t nb) {
  if (E > 1024 || nb < 1 || nb > kMaxTableBlocks || n > 0x7FFFFFFF - 64 * 1024) return false;
  int P = 1024 / E;
  P = P > 16 ? 16 : P;
  const int64_t ints = (int64_t)CH * E + 2 * (int64_t)E + 2 * (int64_t)P * E + 6 * ((int64_t)E + 1);
  return ints * 4 <= 150 * 1024;
}

inline int launch_order_scan(const void *indx, int is16, int64_t n, int E, int CH, int nbits, int k, const int32_t *block_tot,
                             int64_t nb, int32_t *col_sum, int32_t *col_sorted, int32_t *row_sorted, int32_t *gather,
                             int32_t *offs, int64_t offs_pitch, int32_t *sched, int64_t sched_pitch, int max_blocks,
                             Gates gates, hipStream_t st) {
  int P = 1024 / E;
  P = P > 16 ? 16 : P;
  P = P > nb ? (int)nb : P;
  const int64_t ints = (int64_t)CH * E + 2 * (int64_t)E + 2 * (int64_t)P * E + 6 * ((int64_t)E + 1);
  int64_t shares = (5 * (int64_t)max_blocks + 4095) / 4096;  // about four schedule entries per thread
  shares = shares < 1 ? 1 : (shares > 64 ? 64 : shares);
  if (int rc = raise_lds_limit_once((const void *)order_scan_kernel)) return rc;
  order_scan_kernel<<<dim3((unsigned)(nb + shares)), 1024, (size_t)ints * 4, st>>>(
      indx, is16, (int)n, E, CH, nbits, k, block_tot, (int)nb, P, col_sum, col_sorted, row_sorted, gather, offs, offs_pitch,
      sched, sched_pitch, max_blocks, gates);
  return launch_status();
}

// ---------------------------------------------------------------------------
// routing from the logits in two launches
// ---------------------------------------------------------------------------
// A row picks an expert at most once.  So a block of rows (kMaxRowsPerBlock) counts its entries per expert in a byte, and the place of
// an entry among those of its expert is the number of earlier rows that picked it: bits of a mask with one bit per row
// and expert, set in LDS in any order, and counted.  No ballots per chunk, no prefix sums over chunks.

// i / k for i * k < 2^19, k <= 64: i * reciprocal_of(k) >> 19 (the reciprocal is too large by at most k / 2^19).
inline uint32_t reciprocal_of(int k) { return (1u << 19) / (uint32_t)k + 1u; }
TAMD_DEVICE int over_k(int i, uint32_t inv) { return (int)((uint32_t)i * inv >> 19); }

// Rows of `members` [E][W]: the rows before row r that picked expert e.
TAMD_DEVICE int rows_before(const uint32_t *members, int W, int e, int r) {
  const int rw = r >> 5;
  int n = 0;
  for (int w = 0; w < W; ++w) {
    const uint32_t m = members[e * W + w];
    n += __popc(w < rw ? m : (w == rw ? m & ((1u << (r & 31)) - 1u) : 0u));
  }
  return n;
}

// First launch: the experts of RB rows per workgroup, TH / L at a time, and the bytes of their counts: row `blockIdx.x` of
// the table, `pitch` bytes.  The workgroups are as small as a short table allows, since a row is a chain of
// instructions that the waves of a SIMD share.  (Both launches in a graph, with 32-bit tables and a histogram per 64 entries before:
// 4096 rows of 128, top-4: 12.0 -> 8.3 us; 333 of 32: 9.0 -> 6.8; 9350 of 256, bf16, top-8: 22.8 -> 16.2, four launches
// before; 32768 of 256, top-8: 52 -> 36.)
template <int DT, int L, int EPL, int TH>
__global__ __launch_bounds__(TH) void topk_hist_kernel(const void *__restrict__ x, int64_t x_stride, int n_rows, int E,
                                                         int k, void *__restrict__ y_vals, int16_t *__restrict__ y_indx,
                                                         uint32_t *__restrict__ bits, int64_t bits_stride_row,
                                                         int64_t bits_stride_word, int RB, int pitch,
                                                         uint32_t *__restrict__ table) {
  __shared__ int32_t hist[512];
  constexpr int ROWS = TH / L;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), sub = tid % L, n_words = (E + 31) / 32;
  const int64_t end = (int64_t)(blockIdx.x + 1) * RB < n_rows ? (int64_t)(blockIdx.x + 1) * RB : n_rows;
  int64_t row = (int64_t)blockIdx.x * RB + tid / L;
  RowLogits<DT, L, EPL> logits;
  logits.request(x, (row < end ? row : end - 1) * x_stride, E, sub);
  for (int j = tid; j < pitch; j += TH) hist[j] = 0;
  sync_threads();
  // (a wave without a row of its own stays out)
  for (int64_t row0 = (int64_t)blockIdx.x * RB + wave * (kWave / L); row0 < end; row0 += ROWS, row += ROWS) {
    SortKey<DT> keys[EPL];
    logits.take(keys, E, sub);
    if (row0 + ROWS < end) logits.request(x, (row + ROWS < end ? row + ROWS : end - 1) * x_stride, E, sub);
    const Picks<DT> r = pick_columns<L, EPL, DT>(keys, k, sub);
    const bool slot = sub < k;
    if (row < end && slot) atomicAdd(&hist[r.col()], 1);
    const float v = pick_softmax<L, DT>(r, slot);
    if (row < end) {
      if (slot) {
        store_from_f32<DT>(y_vals, row * k + sub, v);
        y_indx[row * k + sub] = (int16_t)r.col();
      }
      if (sub < n_words) bits[row * bits_stride_row + (int64_t)sub * bits_stride_word] = r.word;
    }
  }
  sync_threads();
  for (int j = tid; j < pitch / 4; j += TH)
    table[(int64_t)blockIdx.x * (pitch / 4) + j] =
        (uint32_t)hist[4 * j] | (uint32_t)hist[4 * j + 1] << 8 | (uint32_t)hist[4 * j + 2] << 16 | (uint32_t)hist[4 * j + 3] << 24;
}

// Second launch: every workgroup sums the bytes of the table by itself (all blocks, and those before its own rows: two
// experts to a register, sixteen bits each, so up to 65535 rows).  The first `nbo` place the entries of `sub` blocks
// each; the others build the ragged tables and fill the block schedule, about an entry per thread (a search of the
// table's row is a chain of LDS reads, and four of them in a row were the longest path of the launch).
__global__ __launch_bounds__(1024) void order_rows_kernel(const int16_t *__restrict__ indx, int n, int E, int k, uint32_t inv_k,
                                                          const uint32_t *__restrict__ table, int lg_cols, int nb, int RB,
                                                          int sub, int nbo, int W, int32_t *__restrict__ col_sum,
                                                          int32_t *__restrict__ col_sorted, int32_t *__restrict__ row_sorted,
                                                          int32_t *__restrict__ gather, int32_t *__restrict__ offs,
                                                          int64_t offs_pitch, int32_t *__restrict__ sched,
                                                          int64_t sched_pitch, int max_blocks, Gates gates) {
  extern __shared__ int32_t sm[];
  const int cols = 1 << lg_cols;                       // dwords of a table row
  uint32_t *sums = (uint32_t *)sm;                     // [4][cols]  experts 4c, 4c + 2 | 4c + 1, 4c + 3: all blocks, then the earlier ones
  uint32_t *members = sums + 4 * cols;                 // [E][W]
  int32_t *place = (int32_t *)members + E * W;         // [waves][E] first entry of each expert (a copy per wave) or [6][E + 1]
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, blk = blockIdx.x;
  const bool orders = blk < nbo;
  const int first = blk * sub * RB * k;                // this workgroup's entries
  const int count = orders ? (sub * RB * k < n - first ? sub * RB * k : n - first) : 0;
  // entries and table are requested together; LDS is cleared meanwhile
  const int i0 = tid < count ? tid : 0;
  int ev = indx[first < n ? first + i0 : 0];
  uint32_t gate = load_gate(gates, first < n ? first + i0 : 0);
  const int c = tid & (cols - 1), r0 = tid >> lg_cols, step = 1024 >> lg_cols;
  uint32_t t[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) t[u] = table[(int64_t)(r0 + u * step < nb ? r0 + u * step : nb - 1) * cols + c];
  for (int j = tid; j < 4 * cols + E * W; j += 1024) sm[j] = 0;
  sync_threads();
  uint32_t all0 = 0, all1 = 0, bel0 = 0, bel1 = 0;
  for (int b0 = r0;;) {
#pragma unroll
    for (int u = 0; u < 8; ++u) asm volatile("" : "+v"(t[u]));
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int b = b0 + u * step;
      const uint32_t even = b < nb ? t[u] & 0x00FF00FFu : 0u, odd = b < nb ? t[u] >> 8 & 0x00FF00FFu : 0u;
      all0 += even;
      all1 += odd;
      bel0 += b < blk * sub ? even : 0u;
      bel1 += b < blk * sub ? odd : 0u;
    }
    b0 += 8 * step;
    if (b0 - r0 >= nb) break;
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = table[(int64_t)(b0 + u * step < nb ? b0 + u * step : nb - 1) * cols + c];
  }
  if (r0 < nb) {
    atomicAdd(&sums[c], all0);
    atomicAdd(&sums[cols + c], all1);
    if (orders) {
      atomicAdd(&sums[2 * cols + c], bel0);
      atomicAdd(&sums[3 * cols + c], bel1);
    }
  }
  for (int i = tid; i < count; i += 1024) {
    const int e = i == tid ? ev : indx[first + i], r = over_k(i, inv_k);
    atomicOr(&members[e * W + (r >> 5)], 1u << (r & 31));
  }
  sync_threads();
  const auto total_of = [&](const uint32_t *part, int e) { return (int)(part[(e & 1) * cols + (e >> 2)] >> ((e & 2) * 8) & 0xFFFFu); };
  if (orders) {
    // a wave with entries scans the totals into a copy of its own: no barrier in between
    if (wave * kWave < count) {
      int32_t *mine = place + wave * E;
      int carry = 0;
      for (int s0 = 0; s0 < E; s0 += kWave) {
        const int s = s0 + lane, v = s < E ? total_of(sums, s) : 0, inc = wave_incl_scan(v);
        if (s < E) mine[s] = carry + inc - v;
        if (s < E && blk == 0 && wave == 0) col_sum[s] = v;
        carry += __builtin_amdgcn_readlane(inc, kWave - 1);
      }
      for (int i = tid; i < count; i += 1024) {
        const int e = i == tid ? ev : indx[first + i], r = over_k(i, inv_k);
        const int pos = mine[e] + total_of(sums + 2 * cols, e) + rows_before(members, W, e, r);
        row_sorted[first + i] = pos;
        col_sorted[pos] = first + i;
        if (gather) gather[pos] = blk * sub * RB + r;
        store_gate(gates, pos, i == tid ? gate : load_gate(gates, first + i));
      }
    }
  } else {
    int32_t *sizes = (int32_t *)members, *tab = place;  // (E * W >= E)
    for (int e = tid; e < E; e += 1024) sizes[e] = total_of(sums, e);
    sync_threads();
    ragged_scan_rows(sizes, E, tab, blk == nbo ? offs : nullptr, offs_pitch);
    sync_threads();
    const int64_t total = 5 * (int64_t)max_blocks;
    const int64_t shares = (int64_t)gridDim.x - nbo;
    const int64_t per = (total + shares - 1) / shares;
    const int64_t begin = per * (blk - nbo);
    if (begin < total) ragged_fill_schedule(tab, E, sched, sched_pitch, max_blocks, begin, per < total - begin ? per : total - begin);
  }
}

template <int DT>
int launch_topk_hist(const void *x, int64_t xs, int n_rows, int E, int k, void *yv, int16_t *yi, uint32_t *bits, int64_t bsr,
                     int64_t bsw, int L, const RowPlan &p, uint32_t *table, hipStream_t st) {
#define TAMD_TH(LL, EE)                                                                                                 \
  do {                                                                                                                  \
    auto kern = p.TH == 256 ? topk_hist_kernel<DT, LL, EE, 256>                                                         \
                            : (p.TH == 512 ? topk_hist_kernel<DT, LL, EE, 512> : topk_hist_kernel<DT, LL, EE, 1024>);   \
    kern<<<(unsigned)p.nb, p.TH, 0, st>>>(x, xs, n_rows, E, k, yv, yi, bits, bsr, bsw, p.RB, p.pitch, table);           \
  } while (0)
  if (L == 8 && E <= 32) TAMD_TH(8, 4);
  else if (L == 8) TAMD_TH(8, 8);
  else if (L == 16) TAMD_TH(16, 8);
  else if (L == 32) TAMD_TH(32, 8);
  else TAMD_TH(64, 8);
#undef TAMD_TH
  return launch_status();
}

inline int launch_order_rows(const int16_t *indx, int64_t n, int E, int k, const RowPlan &p, const uint32_t *table, int32_t *col_sum,
                             int32_t *col_sorted, int32_t *row_sorted, int32_t *gather, int32_t *offs, int64_t offs_pitch,
                             int32_t *sched, int64_t sched_pitch, int max_blocks, Gates gates, hipStream_t st) {
  int64_t shares = (5 * (int64_t)max_blocks + 1023) / 1024;
  shares = shares < 1 ? 1 : (shares > 64 ? 64 : shares);
  if (int rc = raise_lds_limit_once((const void *)order_rows_kernel)) return rc;
  order_rows_kernel<<<(unsigned)(p.nbo + shares), 1024, p.lds, st>>>(indx, (int)n, E, k, reciprocal_of(k), table, p.lg_cols, p.nb, p.RB,
                                                                    p.sub, p.nbo, p.W, col_sum, col_sorted, row_sorted, gather, offs,
                                                                    offs_pitch, sched, sched_pitch, max_blocks, gates);
  return launch_status();
}

// ---------------------------------------------------------------------------
// all routing metadata in one workgroup
// ---------------------------------------------------------------------------
// For index arrays small enough that the per-chunk histogram fits LDS (n/64 * E ints): histogram,
// the three prefix sums, the ordering and the ragged tables without leaving the workgroup --
// one launch instead of four, which is what the cost of routing is made of at these sizes.
__global__ __launch_bounds__(1024) void meta_fused_kernel(const void *__restrict__ indx, int is16, int n, int E, int k,
                                                          int nbits, int NC, int P, int32_t *__restrict__ col_sum,
                                                          int32_t *__restrict__ col_sorted, int32_t *__restrict__ row_sorted,
                                                          int32_t *__restrict__ gather, int32_t *__restrict__ offs,
                                                          int64_t offs_pitch, int32_t *__restrict__ sched,
                                                          int64_t sched_pitch, int max_blocks, Gates gates) {
  extern __shared__ int32_t sm[];
  int32_t *hist = sm;                         // [NC][E]  counts, then exclusive prefix over chunks
  int32_t *csum = hist + (int64_t)NC * E;     // [E]
  int32_t *psum = csum + E;                   // [P][E]   partial sums of chunk ranges
  int32_t *tab = psum + (int64_t)P * E;       // [6][E + 1]
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  for (int i = tid; i < NC * E; i += 1024) hist[i] = 0;
  sync_threads();
  // 1. per-chunk histogram.  A wave takes its chunks eight at a time so that eight index loads are in
  // flight together (one workgroup has nothing else to hide their latency with).
  for (int c0 = wave; c0 < NC && n > 0; c0 += 16 * 8) {
    int ev[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {  // unconditional loads (entries past the end re-read entry 0), so all eight are in flight
      const int i = (c0 + 16 * u) * 64 + lane;
      const bool ok = c0 + 16 * u < NC && i < n;
      ev[u] = load_indx(indx, is16, ok ? i : 0);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) asm volatile("" : "+v"(ev[u]));  // pinned: the loads stay outside the selection below
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = (c0 + 16 * u) * 64 + lane;
      ev[u] = (c0 + 16 * u < NC && i < n) ? ev[u] : -1;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = c0 + 16 * u;
      if (c >= NC) break;
      const int e = ev[u];
      const bool valid = e >= 0 && e < E;
      const uint64_t same = same_id_mask(e, valid, nbits);
      if (valid && (same & lanemask_lt()) == 0) hist[c * E + e] = __popcll(same);
    }
  }
  sync_threads();
  // 2. exclusive prefix over chunks for every expert: a few chunks in one go, else P chunk ranges per expert in two passes
  const int per = (NC + P - 1) / P;
  if (NC <= 8) {
    for (int e = tid; e < E; e += 1024) {
      int run = 0;
      for (int c = 0; c < NC; ++c) {
        const int v = hist[c * E + e];
        hist[c * E + e] = run;
        run += v;
      }
      csum[e] = run;
      col_sum[e] = run;
    }
  } else {
  for (int t = tid; t < P * E; t += 1024) {
    const int part = t / E, e = t - part * E;
    int run = 0;
    for (int c = part * per; c < NC && c < (part + 1) * per; ++c) run += hist[c * E + e];
    psum[part * E + e] = run;
  }
  sync_threads();
  for (int t = tid; t < P * E; t += 1024) {
    const int part = t / E, e = t - part * E;
    int run = 0;
    for (int q = 0; q < part; ++q) run += psum[q * E + e];
    for (int c = part * per; c < NC && c < (part + 1) * per; ++c) {
      const int v = hist[c * E + e];
      hist[c * E + e] = run;
      run += v;
    }
    if (part == P - 1) {
      csum[e] = run;
      col_sum[e] = run;
    }
  }
  }
  sync_threads();
  // 3. ragged tables of the histogram; the first one is the exclusive prefix over experts that places the entries
  ragged_scan_rows(csum, E, tab, offs, offs_pitch);
  sync_threads();
  const int32_t *coff = tab;
  const int nv = tab[E];
  // 4. placement
  for (int c0 = wave; c0 < NC && n > 0; c0 += 16 * 8) {
    int ev[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {  // unconditional loads (entries past the end re-read entry 0), so all eight are in flight
      const int i = (c0 + 16 * u) * 64 + lane;
      const bool ok = c0 + 16 * u < NC && i < n;
      ev[u] = load_indx(indx, is16, ok ? i : 0);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) asm volatile("" : "+v"(ev[u]));  // pinned: the loads stay outside the selection below
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = (c0 + 16 * u) * 64 + lane;
      ev[u] = (c0 + 16 * u < NC && i < n) ? ev[u] : -1;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = c0 + 16 * u;
      if (c >= NC) break;
      const int i = c * 64 + lane;
      const int e = ev[u];
      const bool valid = e >= 0 && e < E;
      const uint64_t same = same_id_mask(e, valid, nbits);
      if (valid) {
        const int pos = coff[e] + hist[c * E + e] + __popcll(same & lanemask_lt());
        row_sorted[i] = pos;
        col_sorted[pos] = i;
        if (gather) gather[pos] = i / k;
        store_gate(gates, pos, load_gate(gates, i));
      } else if (i < n) {
        row_sorted[i] = -1;
      }
      if (i >= nv && i < n) {
        col_sorted[i] = -1;
        if (gather) gather[i] = 0;  // trunc(-1 / k)
      }
    }
  }
  // 5. block schedule (reads the tables only: no barrier after the placement)
  ragged_fill_schedule(tab, E, sched, sched_pitch, max_blocks, 0, 5 * (int64_t)max_blocks);
}

// ---------------------------------------------------------------------------
// top-k and all routing metadata in one workgroup (decode sizes)
// ---------------------------------------------------------------------------
// With a few dozen tokens two launches of routing cost more than their work.  Here 1024 threads pick the experts of as many
// rows as they hold and set the rows' bits per expert (`members`, as above); six waves sum and scan those bits into the
// ragged tables, each the row of one block size, and write their entries of the block schedule from the scan's registers;
// then every entry is placed by the lane that picked it.  What such a workgroup is made of is the length of its chains, not its work:
// with a histogram per 64 entries, prefix sums over them and a search per schedule entry one row of 128 logits took 6.4 us
// (14 500 cycles; 64 rows 9.5), now 3.4 and 5.2.
template <int DT, int L, int EPL>
__global__ __launch_bounds__(1024) void routing_fused_kernel(const void *__restrict__ x, int64_t x_stride, int n_rows,
                                                             int E, int k, int W, void *__restrict__ y_vals,
                                                             int16_t *__restrict__ y_indx, uint32_t *__restrict__ bits,
                                                             int64_t bits_stride_row, int64_t bits_stride_word,
                                                             int32_t *__restrict__ col_sum,
                                                             int32_t *__restrict__ col_sorted,
                                                             int32_t *__restrict__ row_sorted, int32_t *__restrict__ gather,
                                                             int32_t *__restrict__ offs, int64_t offs_pitch,
                                                             int32_t *__restrict__ sched, int64_t sched_pitch,
                                                             int max_blocks, Gates gates) {
  extern __shared__ int32_t sm[];
  constexpr int PER = L * EPL > kWave ? L * EPL / kWave : 1;  // neighbouring experts to a lane of the scans
  uint32_t *members = (uint32_t *)sm;              // [E][W]
  int32_t *place = sm + E * W;                     // [E]  first entry of each expert
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave, sub = tid % L;
  const int row = tid / L;
  const bool busy = wave * (kWave / L) < n_rows;   // (a wave without a row stays out of the way of those that have one)
  const bool slot = sub < k && row < n_rows;
  RowLogits<DT, L, EPL> logits;
  if (busy) logits.request(x, (int64_t)(row < n_rows ? row : n_rows - 1) * x_stride, E, sub);
  for (int i = tid; i < E * W; i += 1024) members[i] = 0;
  sync_threads();
  Picks<DT> r{};
  if (busy) {
    SortKey<DT> keys[EPL];
    logits.take(keys, E, sub);
    r = pick_columns<L, EPL, DT>(keys, k, sub);
    if (slot) atomicOr(&members[r.col() * W + (row >> 5)], 1u << (row & 31));
  }
  sync_threads();
  const int t = wave - 10;  // the last six waves: row t of the tables
  if (t >= 0) {
    const int sh = t == 0 ? 0 : t + 3;
    int32_t *orow = offs + (int64_t)t * offs_pitch, *srow = sched + (int64_t)(t - 1) * sched_pitch;
    int size[PER], v[PER], sum = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int s = lane * PER + u;
      size[u] = 0;
      for (int w = 0; w < W; ++w) size[u] += __popc(members[(s < E ? s : 0) * W + w]);
      size[u] = s < E ? size[u] : 0;
      v[u] = (size[u] + ((1 << sh) - 1)) >> sh;
      sum += v[u];
    }
    const int inc = wave_incl_scan(sum), total = __builtin_amdgcn_readlane(inc, kWave - 1);
    int ex = inc - sum;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int s = lane * PER + u;
      if (s < E) {
        if (t == 0) {
          place[s] = ex;
          col_sum[s] = size[u];
        }
        orow[s] = ex;
        if (t > 0)
          for (int q = 0; q < v[u] && ex + q < max_blocks; ++q) srow[ex + q] = (q << 16) + s;
      }
      ex += v[u];
    }
    if (lane == 0) orow[E] = total;
    if (t > 0)
      for (int j = total + lane; j < max_blocks; j += kWave) srow[j] = -1;
  }
  uint32_t gate = 0;
  int rank = 0;
  if (busy) {
    const float p = pick_softmax<L, DT>(r, sub < k);
    gate = stored_bits<DT>(p);
    if (slot) {
      rank = rows_before(members, W, r.col(), row);
      store_from_f32<DT>(y_vals, (int64_t)row * k + sub, p);
      y_indx[(int64_t)row * k + sub] = (int16_t)r.col();
    }
    if (row < n_rows && sub < (E + 31) / 32) bits[row * bits_stride_row + (int64_t)sub * bits_stride_word] = r.word;
  }
  sync_threads();
  if (busy && slot) {
    const int i = row * k + sub, pos = place[r.col()] + rank;
    row_sorted[i] = pos;
    col_sorted[pos] = i;
    if (gather) gather[pos] = row;
    store_gate(gates, pos, gate);
  }
}

template <int DT>
int launch_routing_fused(const void *x, int64_t xs, int n_rows, int E, int k, int L, void *yv, int16_t *yi, uint32_t *bits,
                         int64_t bsr, int64_t bsw, int W, size_t lds, int32_t *col_sum,
                         int32_t *col_sorted, int32_t *row_sorted, int32_t *gather, int32_t *offs, int64_t offs_pitch,
                         int32_t *sched, int64_t sched_pitch, int max_blocks, Gates gates, hipStream_t st) {
#define TAMD_RF(LL, EE)                                                                                              \
  do {                                                                                                               \
    auto kern = routing_fused_kernel<DT, LL, EE>;                                                                    \
    if (int rc = raise_lds_limit_once((const void *)kern)) return rc;                                                \
    kern<<<1, 1024, lds, st>>>(x, xs, n_rows, E, k, W, yv, yi, bits, bsr, bsw, col_sum, col_sorted, \
                               row_sorted, gather, offs, offs_pitch, sched, sched_pitch, max_blocks, gates);         \
  } while (0)
  if (L == 8 && E <= 32) TAMD_RF(8, 4);
  else if (L == 8) TAMD_RF(8, 8);
  else if (L == 16) TAMD_RF(16, 8);
  else if (L == 32) TAMD_RF(32, 8);
  else TAMD_RF(64, 8);
#undef TAMD_RF
  return launch_status();
}

}  // namespace tamd

using namespace tamd;

extern "C" int tamd_topk_forward(const void *x, int x_dtype, int64_t x_stride, int n_rows, int n_cols, int k,
                                 int apply_softmax, int use_provided_indx, void *y_vals, int16_t *y_indx,
                                 int64_t y_stride, uint32_t *bits, int64_t bits_stride_row,
                                 int64_t bits_stride_word, void *stream) {
  if (n_rows < 0 || n_cols <= 0 || n_cols >= 32768 || k < 1 || k > 64 || k > n_cols) return TAMD_E_INVALID;
  if (n_rows == 0) return 0;
  if (!x || !y_vals || !y_indx || !bits) return TAMD_E_INVALID;
  hipStream_t st = (hipStream_t)stream;
  switch (x_dtype) {
    case TAMD_F32:
      return launch_topk<TAMD_F32>(x, x_stride, n_rows, n_cols, k, apply_softmax, use_provided_indx, y_vals, y_indx,
                                   y_stride, bits, bits_stride_row, bits_stride_word, st);
    case TAMD_BF16:
      return launch_topk<TAMD_BF16>(x, x_stride, n_rows, n_cols, k, apply_softmax, use_provided_indx, y_vals, y_indx,
                                    y_stride, bits, bits_stride_row, bits_stride_word, st);
    case TAMD_F16:
      return launch_topk<TAMD_F16>(x, x_stride, n_rows, n_cols, k, apply_softmax, use_provided_indx, y_vals, y_indx,
                                   y_stride, bits, bits_stride_row, bits_stride_word, st);
    default:
      return TAMD_E_INVALID;
  }
}

extern "C" int64_t tamd_bitmatrix_metadata_workspace(int64_t n_indx, int n_cols) {
  if (n_indx < 0 || n_cols <= 0) return 0;
  return make_meta_plan(n_indx, n_cols).total;
}

extern "C" int tamd_bitmatrix_metadata(const void *indx, int indx_is_int16, int64_t n_indx, int n_cols,
                                       int32_t *col_sum, int32_t *col_sorted_indx, int32_t *row_sorted_indx,
                                       int32_t *workspace, void *stream) {
  if (n_indx < 0 || n_cols <= 0 || n_cols > 16384 || n_indx > 0x7FFFFFFF) return TAMD_E_INVALID;
  if (!col_sum || !workspace || (n_indx > 0 && (!indx || !col_sorted_indx || !row_sorted_indx))) return TAMD_E_INVALID;
  return launch_bitmatrix_metadata(indx, indx_is_int16, n_indx, n_cols, 1, col_sum, col_sorted_indx, row_sorted_indx,
                                   nullptr, Gates{nullptr, nullptr, 0}, workspace, (hipStream_t)stream, nullptr, nullptr);
}

static int ragged_launch(const int32_t *slice_sizes, int n_slices, int32_t *offs, int64_t offs_pitch,
                         int32_t *schedule, int64_t sched_pitch, int max_n_blocks, hipStream_t st) {
  const size_t lds = 6 * (size_t)(n_slices + 1) * 4;
  if (lds > 150 * 1024) return TAMD_E_UNSUPPORTED;  // more than ~6000 slices
  if (int rc = raise_lds_limit_once((const void *)ragged_kernel)) return rc;
  int64_t wgs = (5 * (int64_t)max_n_blocks + 4095) / 4096;  // about four entries per thread
  wgs = wgs < 1 ? 1 : (wgs > 256 ? 256 : wgs);
  ragged_kernel<<<dim3((unsigned)wgs), 1024, lds, st>>>(slice_sizes, n_slices, offs, offs_pitch, schedule, sched_pitch,
                                                      max_n_blocks);
  return launch_status();
}

extern "C" int tamd_ragged_metadata(const int32_t *slice_sizes, int n_slices, int32_t *offs, int64_t offs_pitch,
                                    int32_t *schedule, int64_t sched_pitch, int max_n_blocks, void *stream) {
  if (n_slices < 0 || n_slices > 65535 || max_n_blocks < 0 || offs_pitch < n_slices + 1 ||
      sched_pitch < max_n_blocks)
    return TAMD_E_INVALID;
  if (!offs || (n_slices > 0 && !slice_sizes) || (max_n_blocks > 0 && !schedule)) return TAMD_E_INVALID;
  return ragged_launch(slice_sizes, n_slices, offs, offs_pitch, schedule, sched_pitch, max_n_blocks,
                       (hipStream_t)stream);
}

namespace {
struct RaggedCtx {
  const int32_t *sizes;
  int n_slices;
  int32_t *offs;
  int64_t offs_pitch;
  int32_t *sched;
  int64_t sched_pitch;
  int max_blocks;
  hipStream_t st;
};
bool ragged_between(void *p) {
  RaggedCtx *c = (RaggedCtx *)p;
  return ragged_launch(c->sizes, c->n_slices, c->offs, c->offs_pitch, c->sched, c->sched_pitch, c->max_blocks,
                       c->st) == 0;
}
}  // namespace

// One workgroup does it all, without a workspace, where the per-chunk histogram fits its LDS; false where it does not.  (Beyond about 4096
// entries one CU is slower than three launches.)
static bool metadata_by_one_workgroup(const void *indx, int indx_is_int16, int64_t n_indx, int n_cols, int k, int32_t *col_sum,
                                      int32_t *col_sorted_indx, int32_t *row_sorted_indx, int32_t *gather_indx, int32_t *offs,
                                      int64_t offs_pitch, int32_t *schedule, int64_t sched_pitch, int max_n_blocks, Gates gates,
                                      hipStream_t st, int &rc) {
  const int64_t NC = (n_indx + 63) / 64 > 0 ? (n_indx + 63) / 64 : 1;
  int64_t P = 1024 / n_cols;
  P = P < 1 ? 1 : (P > NC ? NC : P);
  const int64_t ints = NC * n_cols + (int64_t)n_cols + P * n_cols + 6 * (int64_t)(n_cols + 1);
  if (NC > 64 || ints * 4 > 156 * 1024) return false;
  int nbits = 0;
  while ((1 << nbits) < n_cols) ++nbits;
  rc = raise_lds_limit_once((const void *)meta_fused_kernel);
  if (rc != 0) return true;
  meta_fused_kernel<<<1, 1024, (size_t)ints * 4, st>>>(indx, indx_is_int16, (int)n_indx, n_cols, k, nbits, (int)NC, (int)P, col_sum,
                                                       col_sorted_indx, row_sorted_indx, gather_indx, offs, offs_pitch, schedule,
                                                       sched_pitch, max_n_blocks, gates);
  rc = launch_status();
  return true;
}

static int routing_metadata_impl(const void *indx, int indx_is_int16, int64_t n_indx, int n_cols, int k,
                                 int32_t *col_sum, int32_t *col_sorted_indx, int32_t *row_sorted_indx,
                                 int32_t *gather_indx, int32_t *offs, int64_t offs_pitch, int32_t *schedule,
                                 int64_t sched_pitch, int max_n_blocks, int32_t *workspace, Gates gates, void *stream) {
  if (n_indx < 0 || n_cols <= 0 || n_cols > 16384 || n_indx > 0x7FFFFFFF || k < 1) return TAMD_E_INVALID;
  if (max_n_blocks < 0 || offs_pitch < n_cols + 1 || sched_pitch < max_n_blocks) return TAMD_E_INVALID;
  if (!col_sum || !workspace || !offs || (max_n_blocks > 0 && !schedule)) return TAMD_E_INVALID;
  if (n_indx > 0 && (!indx || !col_sorted_indx || !row_sorted_indx)) return TAMD_E_INVALID;
  int one_rc = 0;
  if (metadata_by_one_workgroup(indx, indx_is_int16, n_indx, n_cols, k, col_sum, col_sorted_indx, row_sorted_indx, gather_indx, offs,
                                offs_pitch, schedule, sched_pitch, max_n_blocks, gates, (hipStream_t)stream, one_rc))
    return one_rc;
  {
    // two launches while the table of block histograms is small enough for every workgroup to reduce by itself
    const MetaPlan p = make_meta_plan(n_indx, n_cols);
    if (order_scan_applicable(n_indx, n_cols, p.CH, p.n_blocks)) {
      hipStream_t st = (hipStream_t)stream;
      hist_kernel<<<dim3((unsigned)p.n_blocks), 1024, (size_t)p.CH * n_cols * 4, st>>>(
          indx, indx_is_int16, n_indx, n_cols, p.CH, p.nbits, nullptr, workspace + p.off_block_tot);
      return launch_order_scan(indx, indx_is_int16, n_indx, n_cols, p.CH, p.nbits, k, workspace + p.off_block_tot, p.n_blocks,
                               col_sum, col_sorted_indx, row_sorted_indx, gather_indx, offs, offs_pitch, schedule, sched_pitch,
                               max_n_blocks, gates, st);
    }
  }
  const size_t sr_lds = ((size_t)n_cols + 6 * ((size_t)n_cols + 1) + 17) * 4;
  if (sr_lds <= 150 * 1024) {
    // three launches: histograms per workgroup, scans + ragged tables, placement
    hipStream_t st = (hipStream_t)stream;
    MetaPlan p = make_meta_plan(n_indx, n_cols);
    hist_kernel<<<dim3((unsigned)p.n_blocks), 1024, (size_t)p.CH * n_cols * 4, st>>>(
        indx, indx_is_int16, n_indx, n_cols, p.CH, p.nbits, workspace + p.off_chunk_pref, workspace + p.off_block_tot);
    if (int rc = raise_lds_limit_once((const void *)scan_ragged_kernel)) return rc;
    int64_t wgs = (5 * (int64_t)max_n_blocks + 4095) / 4096;
    wgs = wgs < 1 ? 1 : (wgs > 64 ? 64 : wgs);
    scan_ragged_kernel<<<dim3((unsigned)wgs), 1024, sr_lds, st>>>(
        n_cols, (int)p.n_blocks, workspace + p.off_block_tot, workspace + p.off_block_off, col_sum,
        workspace + p.off_col_offs, workspace + p.off_n_valid, offs, offs_pitch, schedule, sched_pitch, max_n_blocks);
    order_kernel<<<dim3((unsigned)p.n_blocks), 1024, 0, st>>>(
        indx, indx_is_int16, n_indx, n_cols, p.CH, p.nbits, k, workspace + p.off_chunk_pref, workspace + p.off_block_off,
        workspace + p.off_col_offs, workspace + p.off_n_valid, col_sorted_indx, row_sorted_indx, gather_indx, gates);
    return launch_status();
  }
  RaggedCtx ctx{col_sum, n_cols, offs, offs_pitch, schedule, sched_pitch, max_n_blocks, (hipStream_t)stream};
  return launch_bitmatrix_metadata(indx, indx_is_int16, n_indx, n_cols, k, col_sum, col_sorted_indx,
                                   row_sorted_indx, gather_indx, gates, workspace, (hipStream_t)stream, ragged_between, &ctx);
}

extern "C" int tamd_routing_metadata(const void *indx, int indx_is_int16, int64_t n_indx, int n_cols, int k,
                                     int32_t *col_sum, int32_t *col_sorted_indx, int32_t *row_sorted_indx,
                                     int32_t *gather_indx, int32_t *offs, int64_t offs_pitch, int32_t *schedule,
                                     int64_t sched_pitch, int max_n_blocks, int32_t *workspace, void *stream) {
  return routing_metadata_impl(indx, indx_is_int16, n_indx, n_cols, k, col_sum, col_sorted_indx, row_sorted_indx,
                               gather_indx, offs, offs_pitch, schedule, sched_pitch, max_n_blocks, workspace,
                               Gates{nullptr, nullptr, 0}, stream);
}

extern "C" int tamd_routing(const void *logits, int dtype, int64_t stride, int n_rows, int n_cols, int k, void *y_vals,
                            int16_t *y_indx, uint32_t *bits, int64_t bits_stride_row, int64_t bits_stride_word,
                            int32_t *col_sum, int32_t *col_sorted_indx, int32_t *row_sorted_indx, int32_t *gather_indx,
                            int32_t *offs, int64_t offs_pitch, int32_t *schedule, int64_t sched_pitch, int max_n_blocks,
                            int32_t *workspace, void *stream) {
  return tamd_routing_gates(logits, dtype, stride, n_rows, n_cols, k, y_vals, y_indx, bits, bits_stride_row, bits_stride_word,
                            col_sum, col_sorted_indx, row_sorted_indx, gather_indx, nullptr, offs, offs_pitch, schedule,
                            sched_pitch, max_n_blocks, workspace, stream);
}

extern "C" int tamd_routing_gates(const void *logits, int dtype, int64_t stride, int n_rows, int n_cols, int k, void *y_vals,
                                  int16_t *y_indx, uint32_t *bits, int64_t bits_stride_row, int64_t bits_stride_word,
                                  int32_t *col_sum, int32_t *col_sorted_indx, int32_t *row_sorted_indx, int32_t *gather_indx,
                                  void *sorted_vals, int32_t *offs, int64_t offs_pitch, int32_t *schedule,
                                  int64_t sched_pitch, int max_n_blocks, int32_t *workspace, void *stream) {
  const Gates gates{y_vals, sorted_vals, sorted_vals ? dtype_size(dtype) : 0};
  if (n_rows > 0 && n_cols > 0 && n_cols <= 512 && k >= 1 && k <= 64 && k <= n_cols && logits && y_vals && y_indx && bits &&
      (dtype == TAMD_F32 || dtype == TAMD_BF16 || dtype == TAMD_F16) && col_sum && offs && col_sorted_indx &&
      row_sorted_indx && max_n_blocks >= 0 && offs_pitch >= n_cols + 1 && sched_pitch >= max_n_blocks &&
      (max_n_blocks == 0 || schedule)) {
    const int L = lanes_per_row(n_cols, k);
    const int64_t n = (int64_t)n_rows * k;
    hipStream_t st = (hipStream_t)stream;
    // One launch where 1024 threads hold the rows: also at the line it is the faster (64 rows of 128: 5.6 us against 7.5 in
    // two launches, which take 2.8 us longer to launch; 128 of 32: 4.7 and 6.5).
    if (n_rows <= 1024 / L) {
      const int W = (n_rows + 31) / 32;
      const size_t lds = (size_t)n_cols * (W + 1) * 4;
#define TAMD_RFD(DT)                                                                                                  \
  return launch_routing_fused<DT>(logits, stride, n_rows, n_cols, k, L, y_vals, y_indx, bits, bits_stride_row,         \
                                  bits_stride_word, W, lds, col_sum, col_sorted_indx, row_sorted_indx, gather_indx,    \
                                  offs, offs_pitch, schedule, sched_pitch, max_n_blocks, gates, st)
      if (dtype == TAMD_F32) TAMD_RFD(TAMD_F32);
      if (dtype == TAMD_BF16) TAMD_RFD(TAMD_BF16);
      TAMD_RFD(TAMD_F16);
#undef TAMD_RFD
    }
    // Up to twice as many rows a caller may leave the workspace out.
    if (!workspace && n_rows <= 2 * (1024 / L)) {
      int rc = tamd_topk_forward(logits, dtype, stride, n_rows, n_cols, k, 1, 0, y_vals, y_indx, k, bits, bits_stride_row, bits_stride_word, stream);
      if (rc != 0) return rc;
      return metadata_by_one_workgroup(y_indx, 1, n, n_cols, k, col_sum, col_sorted_indx, row_sorted_indx, gather_indx, offs, offs_pitch,
                                       schedule, sched_pitch, max_n_blocks, gates, st, rc) ? rc : TAMD_E_INVALID;
    }
    RowPlan plan;
    if (workspace && make_row_plan(n_rows, n_cols, k, L, tamd_bitmatrix_metadata_workspace(n, n_cols), plan)) {
      uint32_t *table = (uint32_t *)workspace;
      int rc;
      if (dtype == TAMD_F32)
        rc = launch_topk_hist<TAMD_F32>(logits, stride, n_rows, n_cols, k, y_vals, y_indx, bits, bits_stride_row, bits_stride_word, L, plan, table, st);
      else if (dtype == TAMD_BF16)
        rc = launch_topk_hist<TAMD_BF16>(logits, stride, n_rows, n_cols, k, y_vals, y_indx, bits, bits_stride_row, bits_stride_word, L, plan, table, st);
      else
        rc = launch_topk_hist<TAMD_F16>(logits, stride, n_rows, n_cols, k, y_vals, y_indx, bits, bits_stride_row, bits_stride_word, L, plan, table, st);
      if (rc != 0) return rc;
      return launch_order_rows(y_indx, n, n_cols, k, plan, table, col_sum, col_sorted_indx, row_sorted_indx, gather_indx, offs,
                               offs_pitch, schedule, sched_pitch, max_n_blocks, gates, st);
    }
  }
  const int rc = tamd_topk_forward(logits, dtype, stride, n_rows, n_cols, k, 1, 0, y_vals, y_indx, k, bits, bits_stride_row,
                                   bits_stride_word, stream);
  if (rc != 0) return rc;
  return routing_metadata_impl(y_indx, 1, (int64_t)n_rows * k, n_cols, k, col_sum, col_sorted_indx, row_sorted_indx,
                               gather_indx, offs, offs_pitch, schedule, sched_pitch, max_n_blocks, workspace, gates, stream);
}

// Device address of `scratch` on the current device.  In host code the array's name only stands for the symbol: its
// memory is reached through the address the runtime reports, which differs from GPU to GPU and is looked up once
// per device (with that device current) and kept.
static int static_workspace(int32_t **out) {
  constexpr int kMaxDevices = 64;
  static std::atomic<int32_t *> ptr_of_device[kMaxDevices];
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return TAMD_E_UNSUPPORTED;
  int32_t *p = ptr_of_device[dev].load(std::memory_order_acquire);
  if (!p) {
    e = hipGetSymbolAddress((void **)&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return TAMD_E_INVALID;
    ptr_of_device[dev].store(p, std::memory_order_release);  // two racing first calls store the same address
  }
  *out = p;
  return 0;
}

extern "C" int64_t tamd_routing_metadata_static_max_workspace(void) { return kStaticWorkspaceInts; }

// Everything tamd_routing_metadata_static does once per device on the host side -- the address of the static array
// and the raised LDS limits of the kernels the metadata path launches -- so that callers under graph capture can have
// it done beforehand.  (tamd_routing_metadata_static does the same by itself on a device's first call.)
extern "C" int tamd_routing_metadata_static_init(void) {
  int32_t *ws = nullptr;
  if (int rc = static_workspace(&ws)) return rc;
  if (int rc = raise_lds_limit_once((const void *)meta_fused_kernel)) return rc;
  if (int rc = raise_lds_limit_once((const void *)order_scan_kernel)) return rc;
  if (int rc = raise_lds_limit_once((const void *)scan_ragged_kernel)) return rc;
  return 0;
}

extern "C" int tamd_routing_metadata_static(const void *indx, int indx_is_int16, int64_t n_indx, int n_cols, int k,
                                            int32_t *col_sum, int32_t *col_sorted_indx, int32_t *row_sorted_indx,
                                            int32_t *gather_indx, int32_t *offs, int64_t offs_pitch,
                                            int32_t *schedule, int64_t sched_pitch, int max_n_blocks, void *stream) {
  if (n_indx < 0 || n_cols <= 0) return TAMD_E_INVALID;
  if (make_meta_plan(n_indx, n_cols).total > kStaticWorkspaceInts) return TAMD_E_TOO_LARGE;
  int32_t *ws = nullptr;
  const int rc = static_workspace(&ws);
  if (rc != 0) return rc;
  // every entry of the workspace that a launch reads is written earlier by the same call (per-chunk prefixes and
  // per-workgroup totals by the histogram kernel, the prefix tables by the scan kernel): nothing has to start at zero
  return routing_metadata_impl(indx, indx_is_int16, n_indx, n_cols, k, col_sum, col_sorted_indx, row_sorted_indx,
                               gather_indx, offs, offs_pitch, schedule, sched_pitch, max_n_blocks, ws,
                               Gates{nullptr, nullptr, 0}, stream);
}
