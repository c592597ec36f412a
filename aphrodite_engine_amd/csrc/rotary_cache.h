// Host interface of the rotation with cache write (paged_attention.hip, rotary_cache_kernel).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace aphro {

struct RotaryCacheCall {
  const int64_t* positions;
  void* query;              // rows q_stride, k_stride and v_stride elements apart, turned in place
  void* key;
  void* value;
  const void* cos_sin;
  void* key_cache;
  void* value_cache;
  const int64_t* slot_mapping;
  int64_t num_tokens;
  int num_heads, num_kv_heads, head_size, block_size;
  int64_t q_stride, k_stride, v_stride;
  int dtype, kv_dtype;
  float k_scale, v_scale;
  const float* slabs;       // not null: the rows are not there yet, but the sum over nslab slabs, slab_stride floats apart, of rows of
  int nslab;                // (num_heads + 2 num_kv_heads) head_size floats; they are written as well
  int64_t slab_stride;
};
int rotary_cache_launch(const RotaryCacheCall& call, hipStream_t st);

}  // namespace aphro
