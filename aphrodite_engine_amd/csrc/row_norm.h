// What the RMS norms of rows share: the sum over a workgroup and its size.
#pragma once
#include "common.h"

namespace aphro {

__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int nw = blockDim.x >> 6;
  if (nw == 1) return v;
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
  for (int w = 0; w < nw; ++w) t += red[w];
  __syncthreads();
  return t;
}

static inline int norm_threads(int hidden) {
  // same thread -> element mapping as add_rms_norm_pack_kernel (fused_decode.hip): the
  // sum-of-squares reduction order, hence every output bit, is shared by the two paths
  int nv = hidden / 8;
  int t = nv <= 1024 ? nv : (nv + 1) / 2;
  t = (t + 63) / 64 * 64;
  return t < 64 ? 64 : (t > 1024 ? 1024 : t);
}

}  // namespace aphro
