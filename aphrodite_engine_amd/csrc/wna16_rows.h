// Host interface of wna16_gemm_rows.hip: int4 GEMM for 65 rows and more, tile heights that fit the batch.
#pragma once
#include <hip/hip_runtime.h>

#include "wna16_strip.h"

namespace aphro {

struct Wna16RowsParams {
  const uint16_t* a;      // f16 [M, lda]
  const uint32_t* qw;     // [K/8, N] exllama order, or the strip-major copy
  const uint32_t* qz;     // [G, N/8]
  const uint16_t* sc;     // [G, N]
  uint16_t* c;            // [M, N], [M, N / 2] with SiluAndMul
  float* partial;         // slabs when ksplit > 1
  int row_slabs;          // K slices stay in partial, [ksplit][M rounded up to tiles][N], for a launch behind this one (with a norm: that one)
  int M, N, K, lda;
  int group_size, zero_offset, ksplit, silu;
  int bf16;               // scales and results are bf16 (else f16)
  // RMS norm behind summed K slices (ksplit > 1): residual' = residual + product, c = norm(residual') * norm_weight
  uint16_t* residual;
  const uint16_t* norm_weight;      // (null: none)
  float norm_eps;
  int tiles_m, tiles_n;   // (filled by the launch, like the next)
  uint32_t inv_group;     // ceil(2^32 / group_size): the group of every k of the matrix by a multiplication
  Wna16StripGeom strip;
};

// 32-row blocks of a workgroup's tile (0: the kernel does not take the call, or needs longer than other_ns >= 0) and K slices, whose
// slabs, ksplit x M rounded up to tiles x N floats, fit slab_bytes
struct Wna16RowsPlan { int mb, ksplit; bool exact; };
Wna16RowsPlan wna16_rows_plan(int64_t M, int64_t N, int64_t K, int64_t group_size, int64_t slab_bytes, int64_t other_ns);
// the same of the form that multiplies exact integers and scales fp32 sums: 65 to 128 rows, float16
Wna16RowsPlan wna16_rows_plan_exact(int64_t M, int64_t N, int64_t K, int64_t group_size, int64_t slab_bytes);
// bytes of Wna16RowsParams::partial
size_t wna16_rows_slab_bytes(const Wna16RowsPlan& plan, int64_t M, int64_t N);
int wna16_rows_launch(const Wna16RowsParams& p, const Wna16RowsPlan& plan, hipStream_t st);

}  // namespace aphro
