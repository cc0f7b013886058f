// The FP32 matrix-core attention (attention_f32.hip) as attention.hip
// dispatches to it.
#pragma once

#include "attention_common.h"

namespace wptv {

struct F32Plan {
  int groups;    // groups of 16 query rows per batch row
  int splits;    // key-range parts per batch row
  size_t bytes;  // workspace of the parts (0 with one)
};

// Whether the head width has a kernel form.
bool attention_f32_takes(int c);

// requested <= 0: the library chooses the parts.
F32Plan attention_f32_plan(int B, int T, int H, int c, int N, int window, int requested);

struct F32Call {
  const float *q, *k, *v;
  int64_t ksb, ksn, vsb, vsn;
  const int64_t* positions;
  const int64_t* tree_base;
  const uint64_t* ancestors;
  const float* sink;
  const int64_t* row_base;  // RowMap
  uint32_t row_mask;
  const float* gate;
  int64_t gate_stride;
  int B, T, H, c, N, window;
  float scale_log2;
  float *out, *lse;
  void* workspace;
};

int attention_f32(const F32Plan& p, const F32Call& call, hipStream_t stream);

}  // namespace wptv
