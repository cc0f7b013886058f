// What the attention kernels share: the rows a query sees, where a logical row
// sits in the table, the output gate, and the parts a key range is split into.
#pragma once

#include "wptv_common.h"

#include <algorithm>
#include <climits>

namespace wptv {
namespace {

constexpr float kNegInf = -__builtin_inff();

struct Bounds {
  int lo, hi;  // inclusive key-row range a query sees (hi < lo: none)
};

// p[i] of an input that no kernel of the launch writes, read as constant
// memory: a scalar load where i is uniform (on the scalar counter, apart from
// the vector-memory counter the kernels' DMA runs on, which the compiler's own
// waits cannot count), a vector load where it is not.
template <typename T>
__device__ __forceinline__ T const_load(const T* p, int64_t i) {
  return ((const __attribute__((address_space(4))) T*)(uintptr_t)p)[i];
}

// A batch row's query positions: p[t], or (a draft tree given without
// positions) node t at base + t.
struct QueryPos {
  const int64_t* p;
  int64_t base;
  __device__ __forceinline__ int64_t at(int t) const { return p ? const_load(p, t) : base + t; }
};

__device__ __forceinline__ QueryPos query_pos(const int64_t* positions, const int64_t* tree_base, int b, int T) {
  return positions ? QueryPos{positions + (int64_t)b * T, 0} : QueryPos{nullptr, tree_base[b]};
}

// The key rows query position t sees, before the tree mask.
__device__ __forceinline__ Bounds query_bounds(const QueryPos& pos_b, int t, int window, int N) {
  const int64_t p = pos_b.at(t);
  int64_t hi = p < (int64_t)N - 1 ? p : (int64_t)N - 1;
  int64_t lo = window > 0 ? p - window + 1 : 0;
  if (lo < 0) lo = 0;
  Bounds r;
  r.lo = (int)lo;
  r.hi = hi < lo ? (int)lo - 1 : (int)hi;
  return r;
}

// The union [u_lo, u_hi] of the key rows that positions t_first .. t_last
// see (u_hi < u_lo: none), uniform.  A lane per position, so the positions
// come in by one vector load instead of one dependent scalar load each; every
// lane of the wavefront must be active.
__device__ __forceinline__ void union_bounds(const QueryPos& pos_b, int t_first, int t_last, int window, int N,
                                             int lane, int& u_lo, int& u_hi) {
  int lo_l = INT_MAX, hi_l = -1;
  for (int t0 = t_first; t0 <= t_last; t0 += 64) {
    if (t0 + lane <= t_last) {
      const Bounds bt = query_bounds(pos_b, t0 + lane, window, N);
      if (bt.hi >= bt.lo) {
        lo_l = min(lo_l, bt.lo);
        hi_l = max(hi_l, bt.hi);
      }
    }
  }
  u_lo = __builtin_amdgcn_readfirstlane(wave_min_i32(lo_l));
  u_hi = __builtin_amdgcn_readfirstlane(wave_max_i32(hi_l));
}

__device__ __forceinline__ bool tree_visible(int n, int64_t tbase, uint64_t anc) {
  if ((int64_t)n < tbase) return true;
  const int64_t node = (int64_t)n - tbase;
  return node < 64 && ((anc >> node) & 1ull);
}

// Where logical row n (a token's position) of batch row b sits in the table:
// physical row (n - base[b]) & mask.  The default (base NULL, mask all ones)
// is token p at row p; a window layer's ring of 2^r rows per batch row has
// mask 2^r - 1; a table that starts at a later token has base[b] = that
// token's position.
struct RowMap {
  const int64_t* base;
  uint32_t mask;
};

// The table row of batch row b's first ring slot (a scalar load).
__device__ __forceinline__ int row_base(const RowMap& m, int b) { return m.base ? (int)const_load(m.base, b) : 0; }

// A window or sparse layer's output gate (attention.py:128-130): the output
// o (rounded to bf16, the attention's dtype) times sigmoid(gate) (rounded to
// bf16, as torch.sigmoid of a bf16 tensor), rounded again.  Row (b*T + t) of
// the gate at g + (b*T + t)*stride, head h's columns at + h*c; g NULL: none.
struct OutGate {
  const void* g;  // in the attention's dtype
  int64_t stride;
  template <typename E>
  __device__ __forceinline__ const E* row(int b, int T, int r, int H, int C) const {
    return g ? static_cast<const E*>(g) + ((int64_t)b * T + r / H) * stride + (int64_t)(r % H) * C : nullptr;
  }
};

// Few instructions, since a call of one part has few wavefronts to gate with (a
// lane of the 32-row blocks gates 64 columns): with a division and the rounding
// in integers a window of 128 took, graph replays, us, in one part and in the two
// parts that this replaced, then in one part as here: batch 32, 5 queries of 16
// heads 15.7, 13.3, 11.1; batch 16, 31 queries 21.4, 16.1, 12.7.  The reciprocal is
// v_rcp_f32 of a quarter of the denominator, a quarter of that again, so that a
// subnormal factor is kept; each of the 65536 gates gives the division's bits.
__device__ __forceinline__ float round_bf16(float f) { return static_cast<float>(static_cast<__bf16>(f)); }

__device__ __forceinline__ float gate_factor(unsigned short g) {
  return round_bf16(0.25f * __builtin_amdgcn_rcpf(0.25f + 0.25f * __expf(-bf16_to_f32(g))));
}

// o rounded to bf16, times the gate factor, rounded again.
__device__ __forceinline__ unsigned short gated_bf16(float o, unsigned short g) {
  return __builtin_bit_cast(unsigned short, static_cast<__bf16>(round_bf16(o) * gate_factor(g)));
}

// Key-range parts of each of `units` workgroups' `tiles` 32-row tiles (at most
// max_splits).  A compute unit holds one workgroup of most of these kernels, so
// the parts run in rounds of one a compute unit, and a last round of a few parts
// costs as much as a whole one: the counts tried are those that fill one, two or
// three rounds, and no split at all.  A round costs its parts' tiles and about
// 12 tiles' time to start and merge, the combine launch `merge` more: measured, us,
// the count before (a part more than fills one round) -> the rule's: batch 47 x
// 1536 rows, 5 queries of 16 heads, 24.9 at 6 -> 16.4 at 5 (8 and 10: 23.8,
// 24.5); 39 x 4500, 37.8 at 7 -> 24.4 at 6; 23 x 2031, 26.3 at 12 -> 17.4 at 11;
// 48 x 5000, one query, 46.7 at 6 -> 29.6 at 5; prompts of 3 x 546 tokens, 31.6
// at 2 -> 21.1 at 1, of 1 x 925, 28.7 at 3 -> 23.1 at 2.
//
// merge: 6 where a program launches call by call (up to ten tiles then run in
// one part: batch 1 x 300 17.5 us in three, 13.1 in one).  Less for the bf16
// row-block kernels on the GPU alone, as in a graph (graph_merge).
//
// fp32_parts: the parts are held in FP32.  Parts of bf16 add a rounding each, so
// where one part a unit fills the compute units the range stays whole, although
// two were faster (batch 257 x 4100, 5 queries of 16 heads: 150 us, 131 in two,
// 300: 153, 134; 4 prompts of 600 tokens over 3600 rows 125, 116): outputs over
// 3600 rows are off by 0.00235 of their norm in one part, 0.0029 in two.
//
// Where a compute unit holds two workgroups of a form at once, a second one costs
// less than a round (kHalfRound; the figures at head width 64, where each form
// fits twice, are us at the counts in brackets).  One 16-row block: a part over
// one a compute unit matters so little that the parts just cover the compute
// units (39 x 4500 16.4 [7], 17.0 [6]).  Two blocks: a second workgroup adds 0.8
// of a round, in proportion to how many compute units have one (200 x 4100 49.7
// [1], 43.2 [2]; 100 x 3000 25.0 [2], 23.6 [3], 20.9 [5]; 150 x 1500 20.6 [1], 20.0
// [2], 18.2 [3]; 23 x 4100 13.6 [11], 15.0 [22]).  Three blocks and more, and the
// sparse form: their arithmetic fills a compute unit, and a second workgroup
// costs a round (three blocks, 100 x 4100 33.2 [2], 41.9 [3]; 47 x 4100 19.2 [5],
// 26.8 [6]; sparse, 160 queries 17.1 [1], 20.3 [2]).
enum class Second { kRound, kHalfRound, kFree };

inline long long pick_splits(long long units, long long tiles, long long max_splits, bool fp32_parts,
                             double merge = 6.0, Second second = Second::kRound) {
  const long long cus = compute_units();
  if (!fp32_parts && units >= cus) return 1;
  if (second == Second::kFree && tiles > 10) return std::max(1LL, std::min((cus + units - 1) / units, max_splits));
  auto rounds_of = [&](long long parts) {
    if (second == Second::kRound) return (double)((parts + cus - 1) / cus);
    const long long pairs = parts / (2 * cus), rest = parts % (2 * cus);
    const double last = rest > cus ? 1.0 + 0.8 * (double)(rest - cus) / (double)cus : rest > 0 ? 1.0 : 0.0;
    return 1.8 * (double)pairs + last;
  };
  long long best = 1;
  double best_cost = (double)(tiles + 12) * rounds_of(units);
  for (int rounds = 1; rounds <= 3; ++rounds) {
    const long long s = std::min(rounds * cus / units, max_splits);
    if (s <= 1) continue;
    const double cost = (double)((tiles + s - 1) / s + 12) * rounds_of(units * s) + merge;
    if (cost < best_cost) {
      best = s;
      best_cost = cost;
    }
  }
  return best;
}

}  // namespace
}  // namespace wptv
