// Exact attention's choice of rows for gfx950: for each query, the top_k
// table rows it weighs most among those at least `window` tokens back
// (HySparse's oracle selection), which the sparse layers after an exact
// layer read.
//
// Semantics follow the reference's PyTorch form
// (packages/wpt-model/src/wpt_model/pytorch_kernels.py:112-117): a row's
// score for a query is its largest log-weight over the heads,
//   score(n) = max_h (q_h . k_n * scale - lse_h),
// lse_h the head's log-sum-exp over every row the query sees; the rows
// n > p - window are not candidates; the query keeps the K highest-scoring
// candidates, K = max(0, min(top_k, N - window)), or every candidate and -1
// after them when it has fewer.  The reference leaves the order of equal
// scores to torch.topk ("whichever row topk returns first"); here the rows
// strictly above the K-th largest score come first in row order, then the
// rows equal to it, lowest rows first, up to K.
//
// Two passes (the Triton kernel instead re-streams the keys in up to 16
// counting passes, triton_kernels.py:393-508):
//   choice_scores_*  one workgroup per (batch row, block of query positions,
//                    64 table rows): the scores of the 64 rows for every
//                    query of the block, written once (4 bytes per row and
//                    query, against the 2c bytes of the key read once)
//                      bf16, head width 64 or 128: v_mfma_f32_16x16x32_bf16,
//                        the max over 8 or 16 heads in registers, over other
//                        counts through LDS
//                      otherwise: FP32 dot products on the VALU
//   choice_select_regs  one workgroup per query, tables up to 8192 rows: the
//                    query's scores in registers, the K-th largest found by
//                    a histogram of their range and ranks within its bin, the
//                    chosen rows written in row order after one scan
//   choice_select    longer tables: a 4-pass radix select of the K-th
//                    largest score (order-preserving keys, most significant
//                    byte first; the scores stay in L2), then one pass that
//                    compacts the chosen rows in row order with wavefront
//                    ballots
#include "wptv_common.h"

namespace wptv {
namespace {

constexpr int kKeys = 64;       // table rows per score workgroup
constexpr int kMaxRows = 128;   // query rows (positions x heads) per score workgroup
constexpr int kST = 256;        // threads of the score and select kernels
constexpr float kInf = __builtin_inff();

// The candidates of query position p: rows 0 .. far - 1.
__device__ __forceinline__ int far_rows(int64_t p, int window, int N) {
  int64_t f = p - window + 1;
  f = f < N ? f : N;
  return f > 0 ? (int)f : 0;
}

// Workgroup coordinates of the score kernels: (batch row, position block,
// row block); the first position of the block and its count.
struct ScoreBlock {
  int b, t0, tn, n0;
};

__device__ __forceinline__ ScoreBlock score_block(int T, int tb_positions, int ntb, int nkb) {
  ScoreBlock s;
  const int kb = blockIdx.x % nkb;
  const int rest = blockIdx.x / nkb;
  s.b = rest / ntb;
  s.t0 = (rest % ntb) * tb_positions;
  s.tn = min(tb_positions, T - s.t0);
  s.n0 = kb * kKeys;
  return s;
}

// Rows past every query's candidates of the block are never read: such a
// row block writes nothing.
__device__ __forceinline__ bool block_has_candidates(const ScoreBlock& s, const int64_t* pos_b, int window, int N) {
  int far = 0;
  for (int t = 0; t < s.tn; ++t) far = max(far, far_rows(pos_b[s.t0 + t], window, N));
  return s.n0 < far;
}

// xs[key][r] holds q_r . k_key * scale - lse_r in log2 units for the block's
// R = tn * H query rows; each (row, position) takes the max over the heads.
__device__ __forceinline__ void store_scores(const float (*xs)[kMaxRows + 1], const ScoreBlock& s,
                                             const int64_t* pos_b, int T, int H, int N, int window,
                                             float* __restrict__ scores, int64_t ns) {
  for (int idx = threadIdx.x; idx < kKeys * s.tn; idx += kST) {
    const int key = idx % kKeys, t = idx / kKeys;
    const int n = s.n0 + key;
    if (n >= N) continue;
    float m = -kInf;
    for (int h = 0; h < H; ++h) m = fmaxf(m, xs[key][t * H + h]);
    const int64_t p = pos_b[s.t0 + t];
    scores[((int64_t)s.b * T + s.t0 + t) * ns + n] = (int64_t)n <= p - window ? m : -kInf;
  }
}

template <int C>
__global__ __launch_bounds__(kST) void choice_scores_mfma(
    const unsigned short* __restrict__ q, const unsigned short* __restrict__ k, int64_t ksb, int64_t ksn,
    const int64_t* __restrict__ positions, const float* __restrict__ lse, int T, int H, int N, int window,
    float scale_log2, int tb_positions, int ntb, int nkb, float* __restrict__ scores, int64_t ns) {
  constexpr int S = C / 32;  // k-steps of 16x16x32
  __shared__ float xs[kKeys][kMaxRows + 1];
  const ScoreBlock blk = score_block(T, tb_positions, ntb, nkb);
  const int64_t* pos_b = positions + (int64_t)blk.b * T;
  if (!block_has_candidates(blk, pos_b, window, N)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int j = lane & 15, g = lane >> 4;
  const int R = blk.tn * H;

  // A operand: key row n0 + 16 w + j (clamped; the clamped rows are not
  // written), elements 32 s + 8 g .. + 7 of k-step s.
  int n = blk.n0 + 16 * w + j;
  n = n < N ? n : N - 1;
  const unsigned short* krow = k + (int64_t)blk.b * ksb + (int64_t)n * ksn;
  bf16x8 kop[S];
#pragma unroll
  for (int s = 0; s < S; ++s) kop[s] = *reinterpret_cast<const bf16x8*>(krow + 32 * s + 8 * g);

  // B operand: query row 16 mb + j of the block (padding rows repeat the
  // last; their scores are never read).
  const unsigned short* qb = q + ((int64_t)blk.b * T + blk.t0) * H * C;
  const float* lb = lse + ((int64_t)blk.b * T + blk.t0) * H;
  const int MB = (R + 15) / 16;
  for (int mb = 0; mb < MB; ++mb) {
    const int r = 16 * mb + j;
    const int rr = r < R ? r : R - 1;
    bf16x8 qop[S];
#pragma unroll
    for (int s = 0; s < S; ++s) qop[s] = *reinterpret_cast<const bf16x8*>(qb + (int64_t)rr * C + 32 * s + 8 * g);
    const float l2 = lb[rr] * kLog2e;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < S; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[s], qop[s], acc, 0, 0, 0);
    // acc[i] = S^T[key 4 g + i][query row r]
#pragma unroll
    for (int i = 0; i < 4; ++i) xs[16 * w + 4 * g + i][r] = fmaf(acc[i], scale_log2, -l2);
  }
  __syncthreads();
  store_scores(xs, blk, pos_b, T, H, N, window, scores, ns);
}

// 8 or 16 heads: the (position, head) query rows in 16-row MFMA blocks (two
// positions a block at 8 heads), one workgroup per (batch row, 256 table rows),
// every position of the pass.  A wavefront takes four 16-row sub-blocks with
// all its keys and queries requested before the first product: one memory round
// trip, which is what bounds it.  The queries are the A operand, so a lane ends
// with four heads of one key: their maximum takes three instructions, and the
// permlane swaps that finish it across the lane groups take the four sub-blocks
// together, leaving sub-block g in lane group g: 64 consecutive rows a store.
// Batch 32, 5 queries of 16 heads, 4100 rows: 16.4 us (2.1 TB/s of keys), 18.1
// with 128 rows a wavefront; 24.0 with the keys as A (16 DPP steps a sub-block
// and position for the maximum) and two round trips of 64 rows; 8 heads 12.3.
constexpr int kBlockRows = 256;  // table rows per workgroup

template <int C, int H, int QB>
__global__ __launch_bounds__(kST) void choice_scores_blocks(
    const unsigned short* __restrict__ q, const unsigned short* __restrict__ k, int64_t ksb, int64_t ksn,
    const int64_t* __restrict__ positions, const float* __restrict__ lse, int T, int N, int window, float scale_log2,
    int nkb, float* __restrict__ scores, int64_t ns) {
  static_assert(H == 8 || H == 16, "a lane group holds four heads of one position");
  constexpr int S = C / 32;
  constexpr int kPer = 16 / H;  // positions of a block
  const int b = blockIdx.x / nkb;
  const int n0 = (blockIdx.x % nkb) * kBlockRows;
  const int64_t* pos_b = positions + (int64_t)b * T;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int wn0 = n0 + 64 * w;
  const int R = T * H, blocks = (R + 15) / 16;
  const unsigned short* kb = k + (int64_t)b * ksb;
  bf16x8 kop[4][S];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int n = wn0 + 16 * u + j;
    n = n < N ? n : N - 1;  // clamped rows are not written
#pragma unroll
    for (int s = 0; s < S; ++s) kop[u][s] = *reinterpret_cast<const bf16x8*>(kb + (int64_t)n * ksn + 32 * s + 8 * g);
  }
  bf16x8 qop[QB][S];
  float l2[QB][4];
#pragma unroll
  for (int t = 0; t < QB; ++t) {
    const int row = min(16 * t + j, R - 1);  // padding rows repeat the last; their scores are not written
#pragma unroll
    for (int s = 0; s < S; ++s)
      qop[t][s] = *reinterpret_cast<const bf16x8*>(q + ((int64_t)b * R + row) * C + 32 * s + 8 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) l2[t][i] = lse[(int64_t)b * R + min(16 * t + 4 * g + i, R - 1)] * kLog2e;
  }
  int far = 0;
  for (int t = 0; t < T; ++t) far = max(far, far_rows(pos_b[t], window, N));
  if (wn0 >= far) return;
  const int n = wn0 + lane;
#pragma unroll
  for (int t = 0; t < QB; ++t) {
    if (t >= blocks) break;
    float x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < S; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qop[t][s], kop[u][s], acc, 0, 0, 0);
      // acc[i] = S[query row 16 t + 4 g + i][key 16 u + j]
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = fmaf(acc[i], scale_log2, -l2[t][i]);
      x[u] = fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3]));
    }
    // rows of 16 lanes: z01 = sub-blocks (0, 1, 0, 1), z23 = (2, 3, 2, 3), over lane groups
    // 0, 1 in the lower half and 2, 3 in the upper; then lo = sub-blocks 0 .. 3 over groups
    // 0, 1 (8 heads: the block's first position), hi over groups 2, 3 (its second)
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[0]), __float_as_uint(x[1]), false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[2]), __float_as_uint(x[3]), false, false);
    const float z01 = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const float z23 = fmaxf(__uint_as_float(c[0]), __uint_as_float(c[1]));
    const auto d = __builtin_amdgcn_permlane32_swap(__float_as_uint(z01), __float_as_uint(z23), false, false);
    const float lo = __uint_as_float(d[0]), hi = __uint_as_float(d[1]);
    if (n < N) {
#pragma unroll
      for (int e = 0; e < kPer; ++e) {
        const int tt = kPer * t + e;
        if (tt < T) {
          const float v = kPer == 1 ? fmaxf(lo, hi) : e == 0 ? lo : hi;
          scores[((int64_t)b * T + tt) * ns + n] = n < far_rows(pos_b[tt], window, N) ? v : -kInf;
        }
      }
    }
  }
}

template <typename E>
__global__ __launch_bounds__(kST) void choice_scores_generic(
    const E* __restrict__ q, const E* __restrict__ k, int64_t ksb, int64_t ksn, const int64_t* __restrict__ positions,
    const float* __restrict__ lse, int T, int H, int c, int N, int window, float scale_log2, int tb_positions,
    int ntb, int nkb, float* __restrict__ scores, int64_t ns) {
  __shared__ float xs[kKeys][kMaxRows + 1];
  __shared__ float ks[kKeys][256 + 1];
  const ScoreBlock blk = score_block(T, tb_positions, ntb, nkb);
  const int64_t* pos_b = positions + (int64_t)blk.b * T;
  if (!block_has_candidates(blk, pos_b, window, N)) return;
  const int R = blk.tn * H;
  for (int idx = threadIdx.x; idx < kKeys * c; idx += kST) {
    const int key = idx / c, e = idx % c;
    const int n = min(blk.n0 + key, N - 1);
    ks[key][e] = load_f32(k + (int64_t)blk.b * ksb + (int64_t)n * ksn + e);
  }
  __syncthreads();
  const E* qb = q + ((int64_t)blk.b * T + blk.t0) * H * c;
  const float* lb = lse + ((int64_t)blk.b * T + blk.t0) * H;
  // lanes of a wavefront share the query row (uniform loads) and take 64 keys
  for (int idx = threadIdx.x; idx < kKeys * R; idx += kST) {
    const int key = idx % kKeys, r = idx / kKeys;
    const E* qr = qb + (int64_t)r * c;
    float d = 0.f;
    for (int e = 0; e < c; ++e) d = fmaf(load_f32(qr + e), ks[key][e], d);
    xs[key][r] = fmaf(d, scale_log2, -lb[r] * kLog2e);
  }
  __syncthreads();
  store_scores(xs, blk, pos_b, T, H, N, window, scores, ns);
}

__global__ __launch_bounds__(kST) void choice_select(const float* __restrict__ scores, int64_t ns,
                                                     const int64_t* __restrict__ positions, int N, int window, int K,
                                                     int64_t* __restrict__ chosen) {
  __shared__ int hist[256];
  __shared__ int sel[2];
  __shared__ int wcount[2][kST / 64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t bt = blockIdx.x;
  const int nf = far_rows(positions[bt], window, N);
  int64_t* out = chosen + bt * K;
  const float* s = scores + bt * ns;
  if (nf <= K) {  // every candidate, then none
    for (int i = tid; i < K; i += kST) out[i] = i < nf ? i : -1;
    return;
  }
  // The K-th largest key.
  uint32_t prefix = 0, mask = 0;
  int remaining = K;
  for (int shift = 24; shift >= 0; shift -= 8) {
    __syncthreads();
    hist[tid] = 0;
    __syncthreads();
    for (int n = tid; n < nf; n += kST) {
      const uint32_t u = order_key(s[n]);
      if ((u & mask) == prefix) atomicAdd(&hist[(u >> shift) & 255], 1);
    }
    __syncthreads();
    if (tid < 64) {
      // lane l holds bins 4l .. 4l + 3; suffix = entries in bins >= 4l
      int cnt[4], total = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) total += (cnt[e] = hist[4 * lane + e]);
      int suffix = total;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int other = __shfl_down(suffix, o, 64);
        if (lane + o < 64) suffix += other;
      }
      const uint64_t hit = __builtin_amdgcn_ballot_w64(suffix >= remaining);
      const int top = 63 - __builtin_clzll(hit);  // the highest lane still reaching the K-th entry
      if (lane == top) {
        int above = suffix - total;
        int digit = 4 * lane;
        for (int e = 3; e >= 0; --e) {
          if (above + cnt[e] >= remaining) {
            digit = 4 * lane + e;
            break;
          }
          above += cnt[e];
        }
        sel[0] = digit;
        sel[1] = remaining - above;
      }
    }
    __syncthreads();
    prefix |= (uint32_t)sel[0] << shift;
    mask |= 255u << shift;
    remaining = sel[1];
  }
  // Rows above the K-th largest (K - remaining of them), then `remaining`
  // rows equal to it, each in row order.
  const uint32_t tau = prefix;
  const int need_eq = remaining, n_gt = K - remaining;
  const uint64_t below = (1ull << lane) - 1ull;
  int base_gt = 0, base_eq = 0;
  for (int start = 0; start < nf; start += kST) {
    const int n = start + tid;
    const uint32_t u = n < nf ? order_key(s[n]) : 0u;
    const bool gt = n < nf && u > tau, eq = n < nf && u == tau;
    const uint64_t bg = __builtin_amdgcn_ballot_w64(gt), be = __builtin_amdgcn_ballot_w64(eq);
    if (lane == 0) {
      wcount[0][w] = __builtin_popcountll(bg);
      wcount[1][w] = __builtin_popcountll(be);
    }
    __syncthreads();
    int pg = base_gt, pe = base_eq;
    for (int i = 0; i < w; ++i) {
      pg += wcount[0][i];
      pe += wcount[1][i];
    }
    pg += __builtin_popcountll(bg & below);
    pe += __builtin_popcountll(be & below);
    if (gt) out[pg] = n;
    if (eq && pe < need_eq) out[n_gt + pe] = n;
#pragma unroll
    for (int i = 0; i < kST / 64; ++i) {
      base_gt += wcount[0][i];
      base_eq += wcount[1][i];
    }
    __syncthreads();
    if (base_gt >= n_gt && base_eq >= need_eq) break;  // uniform: every thread holds the same counts
  }
}

// The sum over the lanes up to and including this one; every lane must be
// active (DPP: shifts within the rows of 16, then the rows' totals carried on).
__device__ __forceinline__ int wave_scan_i32(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return x;
}

// The select for up to 4 V THREADS candidates, one workgroup a query: with
// nv = ceil(candidates / 4 THREADS) quads each, thread t holds the keys of rows
// 4 nv t .. 4 nv t + 4 nv - 1 in registers (one memory round trip).  The K-th
// largest key is found by histograms of 1024 equal bins over the range of keys
// still open (first smallest to largest): the bin that holds it, then, when
// that holds at most kCand keys, their ranks among each other by counting, else
// a histogram of the bin's own range.  A range shrinks 2^9 times a pass at the
// least, so four passes end it whatever the keys are (equal ones end in a bin
// of width one); scores take one pass and the ranks.  The chosen rows are
// gathered in LDS in row order, after one scan of the threads' counts, and
// written out in whole lines.  A serial chain of barriers bounds it: about ten,
// where finding the key two bits at a time took eighteen, with every key compared
// three times between each two.  160 queries, 1024 of 3972 rows: 20.0 -> 6.1 us.
template <int THREADS, int V>
__global__ __launch_bounds__(THREADS) void choice_select_regs(const float* __restrict__ scores, int64_t ns,
                                                              const int64_t* __restrict__ positions, int N,
                                                              int window, int K, int64_t* __restrict__ chosen) {
  constexpr int kWaves = THREADS / 64, kBins = 1024, kCand = 256;
  constexpr int kPerLane = kBins / 64;
  static_assert(4 * V * THREADS < 65536, "packed counts hold 16 bits");
  static_assert(kBins % THREADS == 0 && kCand <= THREADS, "bins and candidates a thread");
  __shared__ __attribute__((aligned(16))) int hist[kBins];
  __shared__ __attribute__((aligned(16))) uint32_t cand[kCand];
  __shared__ int range[2][kWaves], counts[kWaves], sel[3], ncand;
  __shared__ uint32_t found;
  __shared__ int staged[4 * V * THREADS];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t bt = blockIdx.x;
  const int nf = far_rows(positions[bt], window, N);
  int64_t* out = chosen + bt * K;
  if (nf <= K) {  // every candidate, then none
    for (int i = tid; i < K; i += THREADS) out[i] = i < nf ? i : -1;
    return;
  }
  const float* s = scores + bt * ns;
  const int nv = (nf + 4 * THREADS - 1) / (4 * THREADS);  // 1 .. V: nf <= N <= 4 V THREADS
  const int base = tid * 4 * nv;
  const int valid = nf - base;  // this thread's items 0 .. valid - 1 are candidates
  uint32_t key[4 * V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    if (v >= nv) break;
    const int n = base + 4 * v;  // a multiple of 4; the scores' row stride is one of 64
    const f32x4 x = n < nf ? *reinterpret_cast<const f32x4*>(s + n) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) key[4 * v + e] = order_key(x[e]);
  }
  auto each = [&](auto&& f) {  // f(item, key) over this thread's candidates
#pragma unroll
    for (int v = 0; v < V; ++v) {
      if (v >= nv) break;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * v + e < valid) f(4 * v + e, key[4 * v + e]);
    }
  };
#pragma unroll
  for (int i = 0; i < kBins / THREADS; ++i) hist[tid + i * THREADS] = 0;
  if (tid == 0) ncand = 0;
  int kmin = INT32_MAX, kmax = INT32_MIN;  // as signed, order kept
  each([&](int, uint32_t x) {
    const int y = (int)(x ^ 0x80000000u);
    kmin = min(kmin, y);
    kmax = max(kmax, y);
  });
  kmin = wave_min_i32(kmin);
  kmax = wave_max_i32(kmax);
  if (lane == 0) {
    range[0][w] = kmin;
    range[1][w] = kmax;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    kmin = min(kmin, range[0][i]);
    kmax = max(kmax, range[1][i]);
  }
  uint32_t lo = (uint32_t)kmin ^ 0x80000000u, hi = (uint32_t)kmax ^ 0x80000000u;
  int remaining = K;  // the key sought is the remaining-th largest of those in lo .. hi
  uint32_t tau;
  for (;;) {
    const uint32_t span = hi - lo;
    const int shift = span < kBins ? 0 : 22 - __builtin_clz(span);  // span >> shift < kBins
    each([&](int, uint32_t x) {
      if (x >= lo && x <= hi) atomicAdd(&hist[(x - lo) >> shift], 1);
    });
    __syncthreads();
    if (w == 0) {
      // lane l holds bins top - 15 .. top, top = kBins - 1 - 16 l
      int cnt[kPerLane], total = 0;
      const int first = kBins - kPerLane * (lane + 1);
#pragma unroll
      for (int e = 0; e < kPerLane; ++e) total += (cnt[e] = hist[first + e]);
      const int upto = wave_scan_i32(total);
      if (upto >= remaining && upto - total < remaining) {  // one lane
        int above = upto - total, bin = first, c = 0;
#pragma unroll
        for (int e = kPerLane - 1; e >= 0; --e) {
          if (c == 0 && above + cnt[e] >= remaining) {
            bin = first + e;
            c = cnt[e];
          }
          if (c == 0) above += cnt[e];
        }
        sel[0] = bin;
        sel[1] = above;
        sel[2] = c;
      }
    }
    __syncthreads();
    const int count = sel[2];
    remaining -= sel[1];
    lo += (uint32_t)sel[0] << shift;
    if (shift == 0) {  // the bin's keys are equal
      tau = lo;
      break;
    }
    const uint32_t width = (1u << shift) - 1u;
    if (hi - lo > width) hi = lo + width;
    if (count <= kCand) {
      each([&](int, uint32_t x) {
        if (x >= lo && x <= hi) cand[atomicAdd(&ncand, 1)] = x;
      });
      __syncthreads();
      if (tid < count) {
        const uint32_t mine = cand[tid];
        int gt = 0, ge = 0;
        for (int i = 0; i < count; ++i) {
          const uint32_t x = cand[i];
          gt += x > mine ? 1 : 0;
          ge += x >= mine ? 1 : 0;
        }
        if (gt < remaining && ge >= remaining) found = mine;  // the same key from each that writes
      }
      __syncthreads();
      tau = found;
      break;
    }
#pragma unroll
    for (int i = 0; i < kBins / THREADS; ++i) hist[tid + i * THREADS] = 0;
    __syncthreads();
  }
  // rows above tau and equal to it, each in row order: one scan of both counts
  int mine = 0;
  each([&](int, uint32_t x) { mine += x > tau ? 1 : x == tau ? 65536 : 0; });
  const int upto = wave_scan_i32(mine);
  if (lane == 63) counts[w] = upto;
  __syncthreads();
  int before = upto - mine, n_gt = 0;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    if (i < w) before += counts[i];
    n_gt += counts[i] & 65535;
  }
  int pg = before & 65535, pe = n_gt + (before >> 16);
  each([&](int i, uint32_t x) {
    if (x > tau) {
      staged[pg++] = base + i;
    } else if (x == tau) {
      if (pe < K) staged[pe] = base + i;
      ++pe;
    }
  });
  __syncthreads();
  for (int i = tid; i < K; i += THREADS) out[i] = staged[i];
}

}  // namespace
}  // namespace wptv

using namespace wptv;

namespace {
int64_t score_stride(int N) { return (int64_t)align_up((size_t)N, kKeys); }
}  // namespace

extern "C" int wptv_choice_workspace(int B, int T, int N, size_t* bytes) {
  if (!bytes) return fail(WPTV_E_INVALID, "choice_workspace: bytes is NULL");
  if (B <= 0 || T <= 0 || N <= 0) return fail(WPTV_E_INVALID, "choice_workspace: B=%d T=%d N=%d must be > 0", B, T, N);
  *bytes = (size_t)B * T * score_stride(N) * sizeof(float);
  return WPTV_OK;
}

extern "C" int wptv_exact_choice(const void* q, const void* k, int64_t k_stride_b, int64_t k_stride_n, int dtype,
                                 const int64_t* positions, const float* lse, int B, int T, int H, int c, int N,
                                 float scale, int top_k, int window, int64_t* chosen, void* workspace,
                                 size_t workspace_bytes, hipStream_t stream) {
  if (B <= 0 || T <= 0 || H <= 0 || c <= 0 || N <= 0)
    return fail(WPTV_E_INVALID, "exact_choice: B=%d T=%d H=%d c=%d N=%d must be > 0", B, T, H, c, N);
  if (top_k < 0 || window < 0) return fail(WPTV_E_INVALID, "exact_choice: top_k=%d window=%d", top_k, window);
  const int K = max(0, min(top_k, N - window));
  if (K == 0) return WPTV_OK;
  if (!q || !k || !positions || !lse || !chosen || !workspace)
    return fail(WPTV_E_INVALID, "exact_choice: a required pointer is NULL");
  if (dtype != WPTV_F32 && dtype != WPTV_BF16) return fail(WPTV_E_UNSUPPORTED, "exact_choice: dtype %d", dtype);
  if (H > kMaxRows) return fail(WPTV_E_UNSUPPORTED, "exact_choice: at most %d heads (got %d)", kMaxRows, H);
  if (c > 256) return fail(WPTV_E_UNSUPPORTED, "exact_choice: head width at most 256 (got %d)", c);
  if (!(scale > 0.f)) return fail(WPTV_E_INVALID, "exact_choice: scale must be > 0 (got %g)", (double)scale);
  size_t need = 0;
  wptv_choice_workspace(B, T, N, &need);
  if (workspace_bytes < need)
    return fail(WPTV_E_INVALID, "exact_choice: workspace of %zu bytes, %zu needed", workspace_bytes, need);
  const int64_t ns = score_stride(N);
  const int tb = max(1, min(T, kMaxRows / H));
  const int ntb = (T + tb - 1) / tb;
  const int nkb = (N + kKeys - 1) / kKeys;
  const int64_t grid = (int64_t)B * ntb * nkb;
  if (grid > INT32_MAX || (int64_t)B * T > INT32_MAX) return fail(WPTV_E_INVALID, "exact_choice: grid too large");
  float* scores = static_cast<float*>(workspace);
  const float scale_log2 = scale * kLog2e;
  const bool mfma = dtype == WPTV_BF16 && (c == 64 || c == 128) && aligned(q, 16) && aligned(k, 16) &&
                    k_stride_n % 8 == 0 && k_stride_b % 8 == 0;
  // up to 128 query rows: the queries of a workgroup fit its registers
  if (mfma && (H == 8 || H == 16) && T * H <= kMaxRows) {
    const auto* qq = static_cast<const unsigned short*>(q);
    const auto* kk = static_cast<const unsigned short*>(k);
    const int blocks = (T * H + 15) / 16;
    const int nkbb = (N + kBlockRows - 1) / kBlockRows;
#define WPTV_BLOCKS(CC, HH, QB)                                                                                   \
  choice_scores_blocks<CC, HH, QB><<<B * nkbb, kST, 0, stream>>>(qq, kk, k_stride_b, k_stride_n, positions, lse, T, \
                                                                 N, window, scale_log2, nkbb, scores, ns)
#define WPTV_BLOCKS_Q(CC, HH)                       \
  (blocks <= 1   ? WPTV_BLOCKS(CC, HH, 1)           \
   : blocks <= 2 ? WPTV_BLOCKS(CC, HH, 2)           \
   : blocks <= 3 ? WPTV_BLOCKS(CC, HH, 3)           \
   : blocks <= 5 ? WPTV_BLOCKS(CC, HH, 5)           \
                 : WPTV_BLOCKS(CC, HH, 8))
    if (c == 128) {
      if (H == 16) WPTV_BLOCKS_Q(128, 16); else WPTV_BLOCKS_Q(128, 8);
    } else {
      if (H == 16) WPTV_BLOCKS_Q(64, 16); else WPTV_BLOCKS_Q(64, 8);
    }
#undef WPTV_BLOCKS_Q
#undef WPTV_BLOCKS
  } else if (mfma) {
    const auto* qq = static_cast<const unsigned short*>(q);
    const auto* kk = static_cast<const unsigned short*>(k);
    if (c == 128)
      choice_scores_mfma<128><<<(int)grid, kST, 0, stream>>>(qq, kk, k_stride_b, k_stride_n, positions, lse, T, H, N,
                                                              window, scale_log2, tb, ntb, nkb, scores, ns);
    else
      choice_scores_mfma<64><<<(int)grid, kST, 0, stream>>>(qq, kk, k_stride_b, k_stride_n, positions, lse, T, H, N,
                                                             window, scale_log2, tb, ntb, nkb, scores, ns);
  } else if (dtype == WPTV_BF16) {
    choice_scores_generic<unsigned short><<<(int)grid, kST, 0, stream>>>(
        static_cast<const unsigned short*>(q), static_cast<const unsigned short*>(k), k_stride_b, k_stride_n,
        positions, lse, T, H, c, N, window, scale_log2, tb, ntb, nkb, scores, ns);
  } else {
    choice_scores_generic<float><<<(int)grid, kST, 0, stream>>>(static_cast<const float*>(q),
                                                               static_cast<const float*>(k), k_stride_b, k_stride_n,
                                                               positions, lse, T, H, c, N, window, scale_log2, tb,
                                                               ntb, nkb, scores, ns);
  }
  int status = launched("choice_scores");
  if (status != WPTV_OK) return status;
  // the candidates of a query are at most N rows: in registers up to 8192
  if (N <= 1024)
    choice_select_regs<256, 1><<<B * T, 256, 0, stream>>>(scores, ns, positions, N, window, K, chosen);
  else if (N <= 2048)
    choice_select_regs<512, 1><<<B * T, 512, 0, stream>>>(scores, ns, positions, N, window, K, chosen);
  else if (N <= 8192)
    choice_select_regs<1024, 2><<<B * T, 1024, 0, stream>>>(scores, ns, positions, N, window, K, chosen);
  else
    choice_select<<<B * T, kST, 0, stream>>>(scores, ns, positions, N, window, K, chosen);
  return launched("choice_select");
}
