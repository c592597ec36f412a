// Helpers of the recurrences that run in chunks of 64 tokens (outer_memory_chunked.hip, delta_rule_chunked.hip): which chunk a
// workgroup owns, cumulative log decays, 16-byte loads, fp32 matrix-core products.
#pragma once
#include "mixers_common.h"

namespace aphro {

constexpr int CHUNK = 64;

// fp32 product on the matrix cores: D[i][j] += sum over four k of A[i][k] B[k][j].  Lane l gives A[l % 16][k] and B[k][l % 16] for k =
// l / 16 and holds D[4 (l / 16) + r][l % 16].  Which four of the k a call covers is the caller's choice as long as A and B agree:
// here lane group g = l / 16 brings four (or eight) NEIGHBOURING k per load and one of them per call.
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// A matrix of DP columns in the fragments that fp32 and 16-bit products read: 1 KiB each, a lane's four numbers next to each other.  Lane (li, lg) =
// (l % 16, l / 16) of fragment (i, 2 j + u) has row 16 i + li, columns 32 j + 8 lg + 4 u + (0..3).  As rows, a load of 16 bytes a lane would meet another
// cache line in every lane of four.  Here: where the lane's columns 16 j + 4 lg + (0..3) of row 16 i + li begin, as a 16 x 16 product leaves them.
template <int DP>
__device__ __forceinline__ int frag8(int i, int j, int li, int lg) { return (i * (DP / 16) + (j & ~1) + (lg & 1)) * 256 + (((j & 1) * 2 + (lg >> 1)) * 16 + li) * 4; }

// A barrier for what lies in LDS only: __syncthreads() also waits for the loads from memory that are still on their way.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Inclusive prefix sum over the wave: within sixteens, then the sixteens ahead (lane choices inside the instruction; by way of LDS the six steps took
// 600 cycles of a chunk).
template <int CTRL, int ROWS>
__device__ __forceinline__ int from_lane(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false); }
__device__ __forceinline__ int wave_incl_sum(int v) {
  v += from_lane<0x111, 0xf>(v);       // row_shr 1, 2, 4, 8
  v += from_lane<0x112, 0xf>(v);
  v += from_lane<0x114, 0xf>(v);
  v += from_lane<0x118, 0xf>(v);
  v += from_lane<0x142, 0xa>(v);       // row_bcast 15 to rows 1 and 3, 31 to rows 2 and 3
  v += from_lane<0x143, 0xc>(v);
  return v;
}

// (In what follows a unit is a chunk, or a group of chunks of one segment.)
__device__ __forceinline__ int chunks_of(int n, int min_len, int unit = CHUNK) { return n >= min_len ? (n + unit - 1) / unit : 0; }

// Chunk ``id`` of the batch's segments of at least min_len tokens, counted in order: segment s, chunk c of it, and what the segment is; false: there are
// fewer.  Every wave of a workgroup works it out for itself (64 segments a step); what the segment is comes with the lengths, not behind them -- at the
// start of a launch a load takes 1 700 cycles.
struct ChunkPlace {
  int s, c, len, start, slot;
};
template <typename P>
__device__ __forceinline__ bool locate_chunk(int id, const P& p, int min_len, ChunkPlace& at, int unit = CHUNK) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int s0 = 0; s0 < p.num_seqs; s0 += 64) {
    const int seg = min(s0 + lane, p.num_seqs - 1), len = p.q_len[seg], start = p.q_start[seg], slot = p.slot_of_seq[seg];
    const int cnt = s0 + lane < p.num_seqs ? chunks_of(len, min_len, unit) : 0;
    const int incl = wave_incl_sum(cnt) + before;
    const uint64_t past = __ballot(incl > id);
    if (past) {
      const int l = __ffsll((unsigned long long)past) - 1;
      at.s = s0 + l;
      at.c = id - (__builtin_amdgcn_readlane(incl, l) - __builtin_amdgcn_readlane(cnt, l));
      at.len = __builtin_amdgcn_readlane(len, l), at.start = __builtin_amdgcn_readlane(start, l), at.slot = __builtin_amdgcn_readlane(slot, l);
      return true;
    }
    before = __builtin_amdgcn_readlane(incl, 63);
  }
  return false;
}

// Number of chunks ahead of segment s.
__device__ __forceinline__ int chunks_before(int s, const int32_t* __restrict__ q_len, int min_len, int unit = CHUNK) {
  const int lane = threadIdx.x & 63;
  int sum = 0;
  for (int s0 = 0; s0 < s; s0 += 64) sum += __builtin_amdgcn_readlane(wave_incl_sum(s0 + lane < s ? chunks_of(q_len[s0 + lane], min_len, unit) : 0), 63);
  return __builtin_amdgcn_readfirstlane(sum);
}

// The most chunks that num_tokens rows in num_seqs segments can hold.
inline int64_t max_chunks(int64_t num_tokens, int num_seqs, int min_len, int unit = CHUNK) {
  const int64_t longs = num_tokens / min_len;
  return num_tokens / unit + (longs < num_seqs ? longs : num_seqs);
}

// A call's chunks run in spans of as many as the workspace holds, the state between them in the state tensors (fp32, as the chunks carry it: the
// span's length does not show in the results).  Chunks [begin, end) of segment s in the span from chunk id ``chunk0`` on; ``first``: where
// the segment's chunk 0 would lie in the span's arrays.
constexpr int64_t SPAN_BYTES = 256 << 20;       // 38 chunks of 32 heads of the delta rule's 128 x 128, the widest: enough for the chip.  16384 tokens in spans
// against all at once: delta rule 16 / 32 heads 1712 / 2687 -> 1748 / 2682 us, state space of 64 heads 1227 -> 1310 us
__device__ __forceinline__ bool span_of(int s, int nc, const int32_t* __restrict__ q_len, int min_len, int chunk0, int span, int& begin, int& end, int64_t& first, int unit = CHUNK) {
  const int64_t rel = (int64_t)chunks_before(s, q_len, min_len, unit) - chunk0;
  first = rel;
  begin = rel < 0 ? (int)-rel : 0;
  end = rel + nc > span ? (int)(span - rel) : nc;
  return begin < end;
}

// The most of ``chunks`` chunks whose parts, floats(n) floats of n chunks, fit ``bytes``.
template <typename F>
inline int64_t span_chunks(int64_t chunks, int64_t bytes, F floats) {
  const int64_t fixed = floats(0), four = floats(4) - fixed;
  int64_t n = (bytes / 4 - fixed) / four * 4 + 4;
  if (n > chunks) n = chunks;
  while (n > 0 && floats(n) * 4 > bytes) --n;
  return n;
}
template <typename F>
inline int64_t span_workspace(int64_t chunks, F floats) {
  int64_t n = span_chunks(chunks, floats(0) * 4 + SPAN_BYTES, floats);
  if (n < 1) n = chunks < 1 ? chunks : 1;
  return floats(n) * 4;
}

// Inclusive prefix sum over the wave, in 64 bits: differences of two prefixes keep a small decay exact behind a large one.
template <int CTRL, int ROWS>
__device__ __forceinline__ double from_lane(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)from_lane<CTRL, ROWS>((int)(uint32_t)b), hi = (uint32_t)from_lane<CTRL, ROWS>((int)(uint32_t)(b >> 32));
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double wave_incl_sum(double v) {
  v += from_lane<0x111, 0xf>(v);
  v += from_lane<0x112, 0xf>(v);
  v += from_lane<0x114, 0xf>(v);
  v += from_lane<0x118, 0xf>(v);
  v += from_lane<0x142, 0xa>(v);
  v += from_lane<0x143, 0xc>(v);
  return v;
}
__device__ __forceinline__ double of_lane(double v, int l) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l) << 32 | (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l));
}

// 2^t for a difference of two prefixes.  Rounding t to fp32 costs |t| 2^-24 of a factor of size 2^t: half an ulp of one at the most.
__device__ __forceinline__ float exp2_d(double t) { return __builtin_amdgcn_exp2f((float)t); }

// A log decay as it enters a prefix: in units of ln 2, and finite (2^-1e5 is zero however it is split).
__device__ __forceinline__ double log2_decay(float la) { return 1.4426950408889634 * (double)(la < -1e5f ? -1e5f : la); }

// Eight neighbouring numbers of a row, as fp32; zeros from ``limit`` on.  VEC: the address is a multiple of 16 bytes and the row's
// length a multiple of eight.
template <typename T, bool VEC>
__device__ __forceinline__ void load8(const typename T::storage* __restrict__ row, int at, int limit, float (&x)[8]) {
  if constexpr (VEC) {
    if (at < limit) {
      if constexpr (sizeof(typename T::storage) == 2) {
        const u16x8 w = *reinterpret_cast<const u16x8*>(row + at);
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = T::to_f32(w[i]);
      } else {
        const f32x4 a = *reinterpret_cast<const f32x4*>(row + at), b = *reinterpret_cast<const f32x4*>(row + at + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = a[i], x[4 + i] = b[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = 0.f;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = at + i < limit ? T::to_f32(row[at + i]) : 0.f;
  }
}

// The same as they lie in memory: bf16 bits.
template <bool VEC>
__device__ __forceinline__ u16x8 load8_bits(const uint16_t* __restrict__ row, int at, int limit) {
  u16x8 w = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  if constexpr (VEC) {
    if (at < limit) w = *reinterpret_cast<const u16x8*>(row + at);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (at + i < limit) w[i] = row[at + i];
  }
  return w;
}

// An fp32 number as the sum of three bf16 ones, exactly (8 + 8 + 8 bits of its 24; below about 2^-110 the last bits fall out of bf16's range): a product with a bf16 number is then three products on the
// 16-bit matrix cores, each exact, for a quarter of the time of the fp32 ones.  What is not finite stays in the first part.
__device__ __forceinline__ void split3(float x, uint16_t (&p)[3]) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const bool fin = (u & 0x7f800000u) != 0x7f800000u;
  const float h = __builtin_bit_cast(float, u & 0xffff0000u), r = fin ? x - h : 0.f;
  const uint32_t ur = __builtin_bit_cast(uint32_t, r);
  const float l = r - __builtin_bit_cast(float, ur & 0xffff0000u);
  p[0] = (uint16_t)((u >> 16) | (x != x ? 0x40u : 0u));
  p[1] = (uint16_t)(ur >> 16);
  p[2] = (uint16_t)(__builtin_bit_cast(uint32_t, l) >> 16);
}
__device__ __forceinline__ f32x4 mfma16(u16x8 a, u16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

inline bool rows_of_16_bytes(const void* p, int64_t stride, int head, int elem) {
  return ((uintptr_t)p & 15) == 0 && (stride * elem) % 16 == 0 && head % 8 == 0;
}

__device__ __forceinline__ bool finite_f(float x) { return fabsf(x) <= 3.402823466e38f; }

}  // namespace aphro
