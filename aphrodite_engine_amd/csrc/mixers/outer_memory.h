// What the two forms of the gated outer-product memories (outer_memory.hip: token by token; outer_memory_chunked.hip: chunks of 64
// tokens on the matrix cores) share: the call's arguments.
#pragma once
#include "mixers_common.h"

namespace aphro {

struct OuterMemory {
  float* out;
  const void *q, *k, *v, *gate_i, *gate_f;
  int64_t q_stride, k_stride, v_stride, gate_stride;
  float *state_s, *state_n, *state_m;
  const int32_t* slot_of_seq;
  int num_slots;
  const int32_t *q_start, *q_len, *ctx_len;
  int num_seqs;
  int64_t num_tokens;
  int heads, dim, vdim, mode;
  const float* decay;
  float q_scale, gate_cap;
  int qk_heads;
  const float *a_log, *dt_bias, *skip;
  int max_q_len, dtype;
  hipStream_t stream;
};

int outer_memory_check(const OuterMemory& p);
// The token-by-token form over the segments shorter than ``below`` tokens; ``wide``: the work split of prompt portions.
int outer_memory_scan_launch(const OuterMemory& p, int below, bool wide);

}  // namespace aphro
