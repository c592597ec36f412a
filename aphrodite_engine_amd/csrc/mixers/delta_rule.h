// What the two forms of the gated delta rule (delta_rule.hip: token by token; delta_rule_chunked.hip: chunks of 64 tokens on the matrix
// cores) share: the call's arguments.
#pragma once
#include "mixers_common.h"

namespace aphro {

struct GatedDelta {
  float* out;
  const void *q, *k, *v, *b, *a;
  int64_t q_stride, k_stride, v_stride, b_stride, a_stride;
  const float *a_log, *dt_bias;
  float* state;
  const int32_t* slot_of_seq;
  int num_slots;
  const int32_t *q_start, *q_len, *ctx_len;
  int num_seqs;
  int64_t num_tokens;
  int heads, kv_heads, dim, vdim, channel_decay;
  float q_scale, norm_eps;
  int dtype;
  hipStream_t stream;
};

int gated_delta_check(const GatedDelta& p);
// The token-by-token form over the segments shorter than ``below`` tokens; ``wide``: the work split of prompt portions.
int gated_delta_scan_launch(const GatedDelta& p, int below, bool wide);

}  // namespace aphro
