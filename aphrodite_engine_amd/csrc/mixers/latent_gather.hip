// The latents that the leading segments of a batch see, one after the other in rows of their own: what a prompt portion multiplies with
// W_uk and W_uv to attend over keys and values per head instead of in the latent.  Segment s has its q_len + ctx_len rows from a multiple of
// 16 on; tables[s] numbers its blocks of 16 rows, so that the rows serve as a paged cache of their own.  A wave copies a row, 16 bytes a lane:
// bound by the rows' bytes (3000 rows of 1 KiB: 5 us, of which the launch is most).
#include "mixers_common.h"

namespace aphro {

struct LatentGatherParams {
  uint16_t* rows;
  int32_t* tables;
  const uint16_t* cache;
  const int32_t* block_tables;
  const int32_t* q_len;
  const int32_t* ctx_len;
  int64_t num_blocks, total;
  int max_blocks, block_size, dim, num_seqs, out_blocks;
};

__global__ __launch_bounds__(256) void latent_gather_kernel(LatentGatherParams p) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= p.total) return;
  // segment of the row: their padded lengths summed up, 64 segments a step
  int64_t at = row;
  int seq = -1;
  for (int base = 0; base < p.num_seqs && seq < 0; base += 64) {
    const int s = base + lane;
    const int n = s < p.num_seqs ? (p.q_len[s] + p.ctx_len[s] + 15) & ~15 : 0;
    int64_t sum = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t up = __shfl_up(sum, d, 64);
      if (lane >= d) sum += up;
    }
    const unsigned long long past = __builtin_amdgcn_ballot_w64(sum > at);
    if (past) {
      const int k = __builtin_ctzll(past);
      seq = base + k;
      at -= __shfl(sum, k, 64) - __shfl(n, k, 64);
    } else {
      at -= __shfl(sum, 63, 64);
    }
  }
  if (seq < 0) return;
  if ((at & 15) == 0 && lane == 0 && (at >> 4) < p.out_blocks) p.tables[(int64_t)seq * p.out_blocks + (at >> 4)] = (int32_t)(row >> 4);
  const int last = p.q_len[seq] + p.ctx_len[seq] - 1;
  const int key = (int)(at < last ? at : last);              // (the padding repeats the last row)
  const int32_t* bt = p.block_tables + (int64_t)seq * p.max_blocks;
  int64_t blk = bt[key / p.block_size];
  if (blk < 0 || blk >= p.num_blocks) blk = 0;               // never read outside the pool
  const uint16_t* src = p.cache + (blk * p.block_size + key % p.block_size) * p.dim;
  uint16_t* dst = p.rows + row * p.dim;
  for (int c = 8 * lane; c < p.dim; c += 512) *reinterpret_cast<u16x8*>(dst + c) = *reinterpret_cast<const u16x8*>(src + c);
}

}  // namespace aphro

using namespace aphro;

extern "C" int aphro_latent_gather(void* rows, int64_t total_rows, int32_t* tables, int out_blocks, const void* cache,
                                   const int32_t* block_tables, int max_blocks, int64_t num_blocks, int block_size, const int32_t* q_len,
                                   const int32_t* ctx_len, int num_seqs, int dim, int dtype, void* stream) {
  if (total_rows == 0) return APHRO_OK;
  APHRO_CHECK(dtype == APHRO_BF16, "latent_gather: bf16 rows");
  APHRO_CHECK(rows && tables && cache && block_tables && q_len && ctx_len, "latent_gather: null argument");
  APHRO_CHECK(dim > 0 && dim % 8 == 0 && (((uintptr_t)rows | (uintptr_t)cache) & 15) == 0, "latent_gather: rows of 16-byte pieces");
  APHRO_CHECK(total_rows % 16 == 0 && total_rows < (1ll << 31) && out_blocks > 0 && max_blocks > 0 && num_blocks > 0 && block_size > 0 && num_seqs > 0,
              "latent_gather: bad geometry");
  LatentGatherParams p;
  p.rows = (uint16_t*)rows; p.tables = tables; p.cache = (const uint16_t*)cache; p.block_tables = block_tables;
  p.q_len = q_len; p.ctx_len = ctx_len; p.num_blocks = num_blocks; p.total = total_rows; p.max_blocks = max_blocks;
  p.block_size = block_size; p.dim = dim; p.num_seqs = num_seqs; p.out_blocks = out_blocks;
  hipLaunchKernelGGL(latent_gather_kernel, dim3((unsigned)((total_rows + 3) / 4)), dim3(256), 0, (hipStream_t)stream, p);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}
