// FP32 verify attention on the matrix cores (head width 64 or 128): the FP32
// decoder's exact and window layers, whose results are held to 1e-5 of the
// reference's FP32 form (pytorch_kernels.py:98-121, 149-153; attention.py:74-82).
//
// What bounds it: the keys and values once (2 c x 4 bytes a row) while a batch
// row has few query rows (T H), the FP32 matrix rate (154 TFLOP/s) once it has
// about 40 and more; a verify step's small tables are bound by two launches and
// their memory round trips.  So the T H query rows of a batch row are stacked
// into 16-row blocks that share every key and value, and the products run on
// v_mfma_f32_16x16x4_f32, an FP32 fused multiply-add per product.
//
// One workgroup of four wavefronts per (batch row, 16 query rows, key split).
// Each wavefront holds the 16 rows and takes the 16-key tiles w, w + 4, ... of
// the split, with no barrier in the loop:
//
//   S^T[key, q] = K . Q^T       A = K, lane (g, j) = (l / 16, l % 16) holds key
//                               j at channels 16 u + 4 g + e (step 4 u + e):
//                               one 16-byte load a lane per u, straight from
//                               memory; B = Q^T in the same channel order
//                               from LDS.  Lane (g, j) ends with the
//                               scores of query j against keys 4 g + i
//   O^T[c, q] += V^T . P^T      step i multiplies the keys {4 g + i}: B is the
//                               score register i as it stands, A = V^T, lane
//                               (g, j) holds row 4 g + i at columns NCB j ..
//                               NCB j + NCB - 1 (block cb's row j is column
//                               NCB j + cb, NCB = c / 16): whole rows, 16 bytes
//                               a lane.  Lane (g, j) ends with columns 4 NCB g
//                               .. + 4 NCB - 1 of query j
//
// The wavefronts merge through LDS, the splits in a second launch
// (combine_splits_f32), both in a fixed order.
//
// The running maximum moves with every larger score, so p never exceeds 1 and
// the kernel's range is the wave-per-query kernel's.  That kernel never touches
// a row its query does not see; here a matrix product multiplies such a row's
// values by p = 0, so a tile with masked entries whose values are not all
// finite adds the visible rows alone, an entry at a time.
#include "attention_f32.h"

#include <climits>

namespace wptv {
namespace {

constexpr int kF32Waves = 4;
constexpr int kF32Tile = 16;  // keys a wavefront multiplies at once
constexpr int kF32Rows = 16;  // query rows of a workgroup

// max / sum over the four 16-lane groups of a query's scores (NaN propagates)
__device__ __forceinline__ float lanes4_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __builtin_elementwise_maximum(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __builtin_elementwise_maximum(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ float lanes4_sum(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

__device__ __forceinline__ float gated_f32(float o, const float* gate, int col) {
  return gate ? o * (1.f / (1.f + __expf(-gate[col]))) : o;
}

template <int C, bool TREE>
__global__ __launch_bounds__(kF32Waves * 64, 1) void attention_f32_mfma(
    const int64_t* __restrict__ positions, const int64_t* __restrict__ tree_base, int xcd_map, int groups, int splits,
    int T, int H, int N, int window, const float* __restrict__ q, const float* __restrict__ k, int64_t ksb,
    int64_t ksn, const float* __restrict__ v, int64_t vsb, int64_t vsn, const uint64_t* __restrict__ ancestors,
    const float* __restrict__ sink, float scale_log2, RowMap rows, OutGate gate, float* __restrict__ out,
    float* __restrict__ lse_out, float* __restrict__ part_o, float* __restrict__ part_lse) {
  constexpr int NCB = C / 16;  // 16-column blocks of O
  constexpr int U = C / 16;    // 16-channel steps of the QK product
  __shared__ f32x4 buf[2 * NCB * 64];  // Q during the loop, then two wavefronts' O
  __shared__ float stats[2][2][16];    // their m and l
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, j = lane & 15;

  // a batch row's groups and splits on one XCD, which reads its table once
  int unit, split;
  if (xcd_map) {
    const int slot = (int)blockIdx.x >> 3, per_row = groups * splits;
    unit = (((int)blockIdx.x & 7) + 8 * (slot / per_row)) * groups + slot % per_row / splits;
    split = slot % per_row % splits;
  } else {
    unit = (int)blockIdx.x / splits;
    split = (int)blockIdx.x % splits;
  }
  const int b = unit / groups;
  const int R = T * H;
  const int r_base = unit % groups * kF32Rows, r = r_base + j;
  const QueryPos pos_b = query_pos(positions, tree_base, b, T);

  // This lane's query row, the rows any query of the group sees [u_lo, u_hi]
  // and the rows all of them see [f_lo, f_hi].
  int lo = INT_MAX, hi = -1;
  uint64_t anc = 0;
  int u_lo = INT_MAX, u_hi = -1, f_lo = 0, f_hi = INT_MAX;
  const int64_t tbase = TREE ? tree_base[b] : (int64_t)INT_MAX;
  if (r < R) {
    const Bounds bt = query_bounds(pos_b, r / H, window, N);
    f_lo = lo = bt.lo;
    f_hi = hi = bt.hi;
    if constexpr (TREE) anc = ancestors[r / H];
    if (hi >= lo) {
      u_lo = lo;
      u_hi = hi;
    }
  }
  u_lo = __builtin_amdgcn_readfirstlane(wave_min_i32(u_lo));
  u_hi = __builtin_amdgcn_readfirstlane(wave_max_i32(u_hi));
  f_lo = __builtin_amdgcn_readfirstlane(wave_max_i32(f_lo));
  f_hi = __builtin_amdgcn_readfirstlane(wave_min_i32(f_hi));
  if (TREE && tbase <= (int64_t)f_hi) f_hi = (int)tbase - 1;

  // the split's tiles, as even as they go
  const int tiles = u_hi >= u_lo ? (u_hi - u_lo) / kF32Tile + 1 : 0;
  const int per = tiles / splits, more = tiles % splits;
  const int first = split * per + min(split, more);
  const int ntiles = per + (split < more ? 1 : 0);
  const int key0 = u_lo + kF32Tile * first;  // ntiles > 0 only where u_lo is a row

  const float* kb = k + (int64_t)b * ksb + 4 * g;
  const float* vb = v + (int64_t)b * vsb + NCB * j;
  const int rbase = row_base(rows, b);
  // rows past the last one any query sees are fetched as that row and masked
  auto table_row = [&](int n) { return (int64_t)((uint32_t)(min(n, u_hi) - rbase) & rows.mask); };
  f32x4 kt[U], vt[4][NCB / 4];  // the tile's operands
  auto load_k = [&](int tile) {
    const float* kp = kb + table_row(key0 + kF32Tile * tile + j) * ksn;
#pragma unroll
    for (int u = 0; u < U; ++u) kt[u] = *reinterpret_cast<const f32x4*>(kp + 16 * u);
  };
  auto load_v = [&](int tile) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* vp = vb + table_row(key0 + kF32Tile * tile + 4 * g + i) * vsn;
#pragma unroll
      for (int x = 0; x < NCB / 4; ++x) vt[i][x] = *reinterpret_cast<const f32x4*>(vp + 4 * x);
    }
  };
  if (wv < ntiles) {
    load_k(wv);
    load_v(wv);
  }

  // the group's queries into LDS in the B operand's order
  for (int i = threadIdx.x; i < U * 64; i += kF32Waves * 64) {
    const int row = min(r_base + (i & 15), R - 1);
    buf[i] = *reinterpret_cast<const f32x4*>(q + ((int64_t)b * R + row) * C + 16 * (i >> 6) + 4 * ((i >> 4) & 3));
  }
  __syncthreads();

  f32x4 o[NCB];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) o[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegInf, l_run = 0.f;

  // A tile: the next tile's keys are requested once this one's are used up,
  // its values likewise, so each load has a product and the softmax to arrive
  // in and the registers of one tile leave room for other workgroups.
  auto multiply = [&](int tile) {
    const int n0 = key0 + kF32Tile * tile;
    const bool more_tiles = tile + kF32Waves < ntiles;
    f32x4 s = {0.f, 0.f, 0.f, 0.f}, s2 = s;  // two chains: a product waits for the one before it in its chain
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const f32x4 qf = buf[u * 64 + lane];
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[u][0], qf[0], s, 0, 0, 0);
      s2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[u][1], qf[1], s2, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[u][2], qf[2], s, 0, 0, 0);
      s2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[u][3], qf[3], s2, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more_tiles) load_k(tile + kF32Waves);
    auto visible = [&](int n) {
      bool vis = n >= lo && n <= hi;
      if constexpr (TREE) vis = vis && tree_visible(n, tbase, anc);
      return vis;
    };
    const bool full = n0 >= f_lo && n0 + kF32Tile - 1 <= f_hi;  // every query sees every key
    s = (s + s2) * scale_log2;
    if (!full) {
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = visible(n0 + 4 * g + i) ? s[i] : kNegInf;
    }
    const float bm = lanes4_max(__builtin_elementwise_maximum(__builtin_elementwise_maximum(s[0], s[1]),
                                                              __builtin_elementwise_maximum(s[2], s[3])));
    if (__builtin_amdgcn_ballot_w64(bm > m_run)) {
      const float m_new = bm > m_run ? bm : m_run;
      const float alpha = m_run == kNegInf ? (m_new == kNegInf ? 1.f : 0.f) : exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) o[cb] *= alpha;
      m_run = m_new;
    }
    const float m = m_run == kNegInf ? 0.f : m_run;
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = exp2f(s[i] - m);
    l_run += (s[0] + s[1]) + (s[2] + s[3]);
    bool odd = false;  // a value that is not finite, in a tile some query sees a part of
    if (!full) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int x = 0; x < NCB / 4; ++x)
#pragma unroll
          for (int e = 0; e < 4; ++e) odd = odd || !(fabsf(vt[i][x][e]) < __builtin_inff());
    }
    if (__builtin_amdgcn_ballot_w64(odd)) {  // rare: the visible rows alone, an entry at a time
#pragma unroll 1
      for (int key = 0; key < kF32Tile; ++key) {
        const int n = n0 + key;
        const float* vp = v + (int64_t)b * vsb + table_row(n) * vsn + 4 * NCB * g;
        float p = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pi = __shfl(s[i], (key >> 2) * 16 + j, 64);
          p = (key & 3) == i ? pi : p;
        }
        if (!visible(n)) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int cb = 0; cb < NCB; ++cb) o[cb][i] = fmaf(p, vp[i * NCB + cb], o[cb][i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb)
          o[cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(vt[i][cb / 4][cb % 4], s[i], o[cb], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more_tiles) load_v(tile + kF32Waves);
  };

#pragma unroll 1
  for (int t = wv; t < ntiles; t += kF32Waves) multiply(t);
  l_run = lanes4_sum(l_run);

  // ---- the wavefronts: 2 into 0 and 3 into 1, then 1 into 0 ----
  auto give = [&](int slot) {
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) buf[(slot * NCB + cb) * 64 + lane] = o[cb];
    if (g == 0) {
      stats[slot][0][j] = m_run;
      stats[slot][1][j] = l_run;
    }
  };
  auto take = [&](int slot) {
    const float m1 = stats[slot][0][j], l1 = stats[slot][1][j];
    const float M = fmaxf(m_run, m1);
    const float a0 = m_run == kNegInf ? 0.f : exp2f(m_run - M);
    const float a1 = m1 == kNegInf ? 0.f : exp2f(m1 - M);
    l_run = l_run * a0 + l1 * a1;  // NaN sums stay NaN
    m_run = M;
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) o[cb] = o[cb] * a0 + buf[(slot * NCB + cb) * 64 + lane] * a1;
  };
  __syncthreads();  // every wavefront is done with Q
  if (wv >= 2) give(wv - 2);
  __syncthreads();
  if (wv < 2) take(wv);
  __syncthreads();
  if (wv == 1) give(0);
  __syncthreads();
  if (wv != 0) return;
  take(0);

  if (r >= R) return;
  float M = m_run, L = l_run, f = 1.f;
  if (splits == 1 && sink) {
    const float sl = sink[r % H] * kLog2e;
    const float M2 = fmaxf(M, sl);
    f = M == kNegInf ? 0.f : exp2f(M - M2);
    L = L * f + exp2f(sl - M2);
    M = M2;
  }
  const float norm = L > 0.f ? f / L : 0.f;  // L NaN: o is NaN already
  const float lse2 = L > 0.f ? M + log2f(L) : kNegInf;
  const int64_t orow = splits == 1 ? (int64_t)b * R + r : ((int64_t)unit * splits + split) * kF32Rows + j;
  float* dst = (splits == 1 ? out : part_o) + orow * C + 4 * NCB * g;
  const float* grow = splits == 1 ? gate.row<float>(b, T, r, H, C) : nullptr;
  if (grow) grow += 4 * NCB * g;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int x = 0; x < NCB; x += 4) {
      f32x4 val;
#pragma unroll
      for (int e = 0; e < 4; ++e) val[e] = gated_f32(o[x + e][i] * norm, grow, i * NCB + x + e);
      *reinterpret_cast<f32x4*>(dst + i * NCB + x) = val;
    }
  if (g == 0) {
    if (splits > 1)
      part_lse[orow] = L != L ? L : lse2;  // a NaN row stays one through the merge
    else if (lse_out)
      lse_out[orow] = lse2 * kLn2;
  }
}

// Merges the splits of each query row: one thread per (query row, 4 columns),
// eight parts' loads in flight, the sink and the gate joining here.
__global__ __launch_bounds__(256) void combine_splits_f32(const float* __restrict__ part_o,
                                                          const float* __restrict__ part_lse,
                                                          const float* __restrict__ sink, int B, int T, int H, int C,
                                                          int rows_per_group, int groups, int splits, OutGate gate,
                                                          float* __restrict__ out, float* __restrict__ lse_out) {
  constexpr int kGroup = 8;
  const int R = T * H, per_row = C / 4;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)B * R * per_row) return;
  const int64_t brow = idx / per_row;
  const int b = (int)(brow / R), r = (int)(brow % R), c4 = (int)(idx % per_row) * 4;
  const int64_t row0 =
      (int64_t)(b * groups + r / rows_per_group) * splits * rows_per_group + r % rows_per_group;  // split 0's part
  float M = kNegInf, L = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < splits; s0 += kGroup) {
    float ls[kGroup];
    f32x4 po[kGroup];
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      const int64_t prow = row0 + (int64_t)(s0 + u) * rows_per_group;
      const bool in = s0 + u < splits;
      ls[u] = in ? part_lse[prow] : kNegInf;
      po[u] = in ? *reinterpret_cast<const f32x4*>(part_o + prow * C + c4) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float m = M;
#pragma unroll
    for (int u = 0; u < kGroup; ++u) m = fmaxf(m, ls[u]);  // a NaN part joins below
    const float f = M == kNegInf ? 0.f : exp2f(M - m);
    L *= f;
    acc *= f;
    M = m;
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      if (ls[u] == kNegInf) continue;
      const float wgt = exp2f(ls[u] - M);
      L += wgt;
      acc += po[u] * wgt;
    }
  }
  if (sink) {
    const float sl = sink[r % H] * kLog2e;
    const float M2 = fmaxf(M, sl);
    const float f = M == kNegInf ? 0.f : exp2f(M - M2);
    L = L * f + exp2f(sl - M2);
    acc *= f;
    M = M2;
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  const float* grow = gate.row<float>(b, T, r, H, C);
  f32x4 res;
#pragma unroll
  for (int e = 0; e < 4; ++e) res[e] = gated_f32(acc[e] * inv, grow, c4 + e);
  *reinterpret_cast<f32x4*>(out + brow * C + c4) = res;
  if (lse_out && c4 == 0) lse_out[brow] = L > 0.f ? (M + log2f(L)) * kLn2 : kNegInf;
}

template <int C>
void launch_width(const F32Plan& p, const F32Call& a, float* part_o, float* part_lse, hipStream_t stream) {
  const dim3 grid((unsigned)(a.B * p.groups * p.splits));
  const int xcd_map = a.B % 8 == 0 ? 1 : 0;
  const RowMap rows{a.row_base, a.row_mask};
  const OutGate gate{a.gate, a.gate_stride};
  if (a.tree_base)
    hipLaunchKernelGGL((attention_f32_mfma<C, true>), grid, dim3(kF32Waves * 64), 0, stream, a.positions, a.tree_base,
                       xcd_map, p.groups, p.splits, a.T, a.H, a.N, a.window, a.q, a.k, a.ksb, a.ksn, a.v, a.vsb,
                       a.vsn, a.ancestors, a.sink, a.scale_log2, rows, gate, a.out, a.lse, part_o, part_lse);
  else
    hipLaunchKernelGGL((attention_f32_mfma<C, false>), grid, dim3(kF32Waves * 64), 0, stream, a.positions,
                       a.tree_base, xcd_map, p.groups, p.splits, a.T, a.H, a.N, a.window, a.q, a.k, a.ksb, a.ksn, a.v,
                       a.vsb, a.vsn, a.ancestors, a.sink, a.scale_log2, rows, gate, a.out, a.lse, part_o, part_lse);
}

}  // namespace

bool attention_f32_takes(int c) { return c == 64 || c == 128; }

// Whole rounds of one workgroup per compute unit (pick_splits), each wavefront
// at least one tile, so that ranges of nine 32-row tiles and more are cut.  A
// compute unit holds several workgroups of this kernel; that whole rounds serve
// is what the table says, not an occupancy.  Measured on the MI355X, graph replays, us a call (batch,
// queries, heads, width, rows): the wave-per-query kernel, this one with a
// part more than fills the round, this one
//   (8, 5, 4, 64, 1029)     366   10.2  10.2
//   (1, 5, 4, 64, 300)      103    7.7   7.7
//   (4, 6, 16, 128, 1769)         20.4  15.5
//   (8, 9, 16, 128, 2048)  1937   32.3  26.8
//   (2, 200, 8, 64, 700)    369   18.1  15.4
//   (2, 175, 4, 64, 175)           8.6   7.4
// A wavefront holding two to five row blocks (each key read by fewer
// workgroups) was slower at all of these: 12.4-50 us, one wavefront a SIMD.
F32Plan attention_f32_plan(int B, int T, int H, int c, int N, int window, int requested) {
  F32Plan p{};
  p.groups = (int)(((long long)T * H + kF32Rows - 1) / kF32Rows);
  long long span = N;
  if (window > 0 && (long long)window + T - 1 < span) span = (long long)window + T - 1;
  const long long max_splits = (span + kF32Tile * kF32Waves - 1) / (kF32Tile * kF32Waves);
  const long long units = (long long)B * p.groups;
  long long s = requested > 0 ? requested : pick_splits(units, (span + 31) / 32, max_splits, true);
  if (s > max_splits) s = max_splits;
  if (s < 1) s = 1;
  p.splits = (int)s;
  if (s > 1) {
    const size_t rows = (size_t)units * s * kF32Rows;
    p.bytes = align_up(rows * c * sizeof(float), 256) + align_up(rows * sizeof(float), 256);
  }
  return p;
}

int attention_f32(const F32Plan& p, const F32Call& a, hipStream_t stream) {
  float *part_o = nullptr, *part_lse = nullptr;
  if (p.splits > 1) {
    const size_t rows = (size_t)a.B * p.groups * p.splits * kF32Rows;
    part_o = static_cast<float*>(a.workspace);
    part_lse = reinterpret_cast<float*>(static_cast<char*>(a.workspace) + align_up(rows * a.c * sizeof(float), 256));
  }
  if (a.c == 128)
    launch_width<128>(p, a, part_o, part_lse, stream);
  else
    launch_width<64>(p, a, part_o, part_lse, stream);
  const int st = launched("attention_f32_mfma");
  if (st != WPTV_OK || p.splits == 1) return st;
  const long long items = (long long)a.B * a.T * a.H * (a.c / 4);
  const int threads = items >= 256LL * 256 ? 256 : 64;
  hipLaunchKernelGGL(combine_splits_f32, dim3((unsigned)((items + threads - 1) / threads)), dim3(threads), 0, stream,
                     part_o, part_lse, a.sink, a.B, a.T, a.H, a.c, kF32Rows, p.groups, p.splits,
                     OutGate{a.gate, a.gate_stride}, a.out, a.lse);
  return launched("combine_splits_f32");
}

}  // namespace wptv
