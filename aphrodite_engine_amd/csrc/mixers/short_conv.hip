// Short causal convolution over time on every channel of a projection's output, for a batch of segments:
//   y_t[c] = sum_j w[c, j] * u_(t - taps + 1 + j)[c]  (+ b[c]),   zeros before the sequence's start.
// The taps - 1 inputs that precede a segment come from the request's state slot, which afterwards holds the last taps - 1
// inputs of the sequence.  A segment that starts a sequence never reads its slot, and no input older than the sequence's
// start is read from it either, so a slot taken over from another request needs no clearing.
//
// The channels are [q | k | v]: the q part goes to a dense output, the k and v parts straight into the token-major paged
// cache at the rows' slots (what attention reads is the convolved key and value).  Products and sums are fp32, one rounding
// to the storage type.  act 1: silu on the convolution's result (fp32, before the rounding).
#include "mixers_common.h"

namespace aphro {

constexpr int SC_MAX_TAPS = 16;

template <typename T>
__global__ void short_conv_kernel(typename T::storage* __restrict__ q_out, int64_t q_out_stride,
                                  typename T::storage* __restrict__ k_cache, typename T::storage* __restrict__ v_cache,
                                  const int64_t* __restrict__ cache_slots, int64_t num_cache_slots,
                                  const typename T::storage* __restrict__ u, int64_t u_stride,
                                  const typename T::storage* __restrict__ w, const typename T::storage* __restrict__ bias,
                                  const typename T::storage* __restrict__ state,
                                  const int32_t* __restrict__ state_slots, const int32_t* __restrict__ q_start,
                                  const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ seq_of_token, int cq, int ck,
                                  int cv, int taps, int act) {
  const int64_t t = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  const int C = cq + ck + cv;
  if (c >= C) return;
  const int s = seq_of_token[t];
  const int r = (int)t - q_start[s], ctx = ctx_len[s];
  const typename T::storage* st = state ? state + ((int64_t)state_slots[s] * (taps - 1)) * C + c : nullptr;
  float acc = bias ? T::to_f32(bias[c]) : 0.f;
  for (int j = 0; j < taps; ++j) {
    const int i = r - taps + 1 + j;            // row of the segment, negative: before it
    float x = 0.f;
    if (i >= 0) x = T::to_f32(u[(t - r + i) * u_stride + c]);
    else if (ctx + i >= 0) x = T::to_f32(st[(int64_t)(taps - 1 + i) * C]);
    acc += T::to_f32(w[(int64_t)c * taps + j]) * x;
  }
  if (act) acc = silu_f(acc);
  const typename T::storage y = T::from_f32(acc);
  if (c < cq) {
    q_out[t * q_out_stride + c] = y;
  } else {
    const int64_t slot = cache_slots[t];
    if (slot < 0 || slot >= num_cache_slots) return;
    if (c < cq + ck) k_cache[slot * ck + (c - cq)] = y;
    else v_cache[slot * cv + (c - cq - ck)] = y;
  }
}

template <typename T>
__device__ __forceinline__ void sc_store8(typename T::storage* p, const float* v) {
  if constexpr (sizeof(typename T::storage) == 2) {
    u16x8 r;
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = T::from_f32(v[j]);
    *reinterpret_cast<u16x8*>(p) = r;
  } else {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4*>(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
  }
}

// The same convolution for channel counts that are multiples of 8 and 16-byte-aligned rows: a thread owns 8 channels of TOK
// consecutive rows, reads the TOK + TAPS - 1 input rows they need once (16 bytes each) and its 8 x TAPS weights once.
// Bound by the rows' way in and out; what it takes beside is a chain of loads, so the rows and weights (which need no segment) go out
// first, then what the rows of the tile are (uniform over the workgroup), all at once, and the rows wait in the registers as they lay in
// memory.  A tile whose taps lie in one segment turns every number to fp32 once.  With the segments looked up row by row between the rows'
// stores and 4 rows a thread, 4 taps with silu, us before / here (the states' launch, 5, included): 6144 channels, 2000 rows beside 24 single
// ones 30.3 / 22.2, 4096 rows 40.8 / 29.3, 32 single rows 15.3 / 9.4; 12288 channels, 2560 rows 47.0 / 33.8 (bf16 by the converter).
template <typename T, int TAPS, int TOK>
__global__ __launch_bounds__(256) void short_conv_vec8_kernel(
    typename T::storage* __restrict__ q_out, int64_t q_out_stride, typename T::storage* __restrict__ k_cache,
    typename T::storage* __restrict__ v_cache, const int64_t* __restrict__ cache_slots, int64_t num_cache_slots,
    const typename T::storage* __restrict__ u, int64_t u_stride, const typename T::storage* __restrict__ w,
    const typename T::storage* __restrict__ bias,
    const typename T::storage* __restrict__ state, const int32_t* __restrict__ state_slots, const int32_t* __restrict__ q_start,
    const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ seq_of_token, int64_t num_tokens, int cq, int ck, int cv,
    int act) {
  const int C = cq + ck + cv, c_raw = (blockIdx.y * blockDim.x + threadIdx.x) * 8;
  const bool work = c_raw < C;
  const int c0 = work ? c_raw : 0;
  const int64_t t0 = (int64_t)blockIdx.x * TOK;
  Chunk8<T> rows[TOK + TAPS - 1], wr[TAPS], br;
#pragma unroll
  for (int x = 0; x < TOK + TAPS - 1; ++x) {
    const int64_t gr = t0 - (TAPS - 1) + x;                  // a row outside the batch is never used: any row in its place
    rows[x].load(u + (gr < 0 ? 0 : gr < num_tokens ? gr : num_tokens - 1) * u_stride + c0);
  }
#pragma unroll
  for (int x = 0; x < TAPS; ++x) wr[x].load(w + (int64_t)c0 * TAPS + 8 * x);
  br.clear();
  if (bias) br.load(bias + c0);
  int seq[TOK], back0[TOK], ctx[TOK];
  int64_t cslot[TOK];
#pragma unroll
  for (int k = 0; k < TOK; ++k) {
    const int64_t t = t0 + k < num_tokens ? t0 + k : num_tokens - 1;
    seq[k] = seq_of_token[t];
    cslot[k] = ck + cv > 0 ? cache_slots[t] : 0;
  }
#pragma unroll
  for (int k = 0; k < TOK; ++k) {
    const int64_t t = t0 + k < num_tokens ? t0 + k : num_tokens - 1;
    back0[k] = (int)t - q_start[seq[k]];                     // rows of the segment ahead of this one
    ctx[k] = ctx_len[seq[k]];
  }
  if (!work) return;
  float wv[TAPS][8], bv[8];                    // wv[j][i] = w[c0 + i, j]
  {
    float flat[8 * TAPS];
#pragma unroll
    for (int x = 0; x < TAPS; ++x) wr[x].floats(flat + 8 * x);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < TAPS; ++j) wv[j][i] = flat[i * TAPS + j];
  }
  br.floats(bv);
  auto finish = [&](int k, float (&acc)[8]) {
    if (act) {
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = silu_f(acc[i]);
    }
    if (c0 < cq) {
      sc_store8<T>(q_out + (t0 + k) * q_out_stride + c0, acc);
    } else {
      const int64_t slot = cslot[k];
      if (slot < 0 || slot >= num_cache_slots) return;
      if (c0 < cq + ck) sc_store8<T>(k_cache + slot * ck + (c0 - cq), acc);
      else sc_store8<T>(v_cache + slot * cv + (c0 - cq - ck), acc);
    }
  };
  if (t0 + TOK <= num_tokens && seq[0] == seq[TOK - 1] && back0[0] >= TAPS - 1) {      // every tap of the tile lies in one segment
    float x[TOK + TAPS - 1][8];
#pragma unroll
    for (int r = 0; r < TOK + TAPS - 1; ++r) rows[r].floats(x[r]);
#pragma unroll
    for (int k = 0; k < TOK; ++k) {
      float acc[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = bv[i];
#pragma unroll
      for (int j = 0; j < TAPS; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += wv[j][i] * x[k + j][i];
      finish(k, acc);
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < TOK; ++k) {
    if (t0 + k >= num_tokens) break;
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = bv[i];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
      const int back = back0[k] - TAPS + 1 + j;              // row of the segment, negative: before it
      Chunk8<T> win = rows[k + j];
      if (back < 0) {
        win.clear();
        if (ctx[k] + back >= 0) win.load(state + ((int64_t)state_slots[seq[k]] * (TAPS - 1) + (TAPS - 1 + back)) * C + c0);
      }
      float x[8];
      win.floats(x);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] += wv[j][i] * x[i];
    }
    finish(k, acc);
  }
}

// After the convolution: the slot takes the last taps - 1 inputs of the sequence (from the segment, or -- for a segment
// shorter than that -- from what the slot held, moved up).  One thread owns a channel of a segment and reads all it needs
// before it writes.
template <typename T>
__global__ void short_conv_state_kernel(typename T::storage* __restrict__ state, const typename T::storage* __restrict__ u,
                                        int64_t u_stride, const int32_t* __restrict__ state_slots,
                                        const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len,
                                        const int32_t* __restrict__ ctx_len, int C, int taps) {
  const int s = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int n = q_len[s], ctx = ctx_len[s], keep = taps - 1;
  typename T::storage* st = state + ((int64_t)state_slots[s] * keep) * C + c;
  typename T::storage val[SC_MAX_TAPS];
  for (int m = 0; m < keep; ++m) {
    const int p = ctx + n - keep + m;          // position in the sequence
    typename T::storage x = T::from_f32(0.f);
    if (p >= ctx) x = u[((int64_t)q_start[s] + (p - ctx)) * u_stride + c];
    else if (p >= 0) x = st[(int64_t)(p - ctx + keep) * C];
    val[m] = x;
  }
  for (int m = 0; m < keep; ++m) st[(int64_t)m * C] = val[m];
}

}  // namespace aphro

using namespace aphro;

extern "C" int aphro_short_conv_state(void* state, const void* u, int64_t u_stride, const int32_t* state_slots, const int32_t* q_start,
                                      const int32_t* q_len, const int32_t* ctx_len, int num_seqs, int channels, int taps, int dtype,
                                      void* stream) {
  APHRO_CHECK(state && u && state_slots && q_start && q_len && ctx_len && num_seqs > 0 && channels > 0 && (channels + 255) / 256 <= 65535 &&
                  u_stride >= channels && taps >= 2 && taps <= SC_MAX_TAPS, "short_conv_state: bad arguments (%d taps)", taps);
  MIX_DISPATCH_DTYPE(dtype, {
    typedef typename T::storage S;
    hipLaunchKernelGGL((short_conv_state_kernel<T>), dim3((unsigned)num_seqs, (unsigned)((channels + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, (S*)state, (const S*)u, u_stride, state_slots, q_start, q_len, ctx_len, channels, taps);
  });
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

extern "C" int aphro_short_conv(void* q_out, int64_t q_out_stride, void* k_cache, void* v_cache, const int64_t* cache_slots,
                                int64_t num_cache_slots, const void* u, int64_t u_stride, const void* w, const void* bias,
                                void* state,
                                const int32_t* state_slots, const int32_t* q_start, const int32_t* q_len,
                                const int32_t* ctx_len, const int32_t* seq_of_token, int64_t num_tokens, int num_seqs, int cq,
                                int ck, int cv, int taps, int act, int dtype, void* stream) {
  if (num_tokens == 0) return APHRO_OK;
  const int C = cq + ck + cv;
  APHRO_CHECK(u && w && q_start && q_len && ctx_len && seq_of_token && num_seqs > 0 && cq >= 0 && ck >= 0 && cv >= 0 && C > 0,
              "short_conv: bad arguments");
  APHRO_CHECK(taps >= 1 && taps <= SC_MAX_TAPS, "short_conv: %d taps (1 .. %d)", taps, SC_MAX_TAPS);
  APHRO_CHECK(act == 0 || act == 1, "short_conv: activation %d (0 none, 1 silu)", act);
  APHRO_CHECK(taps == 1 || (state && state_slots), "short_conv: more than one tap needs the state slots");
  APHRO_CHECK(u_stride >= C && (cq == 0 || (q_out && q_out_stride >= cq)), "short_conv: row strides smaller than the rows");
  APHRO_CHECK(ck + cv == 0 || (k_cache && v_cache && cache_slots && num_cache_slots > 0 && ck > 0 && cv > 0),
              "short_conv: key / value channels need the cache and the rows' slots");
  APHRO_CHECK(num_tokens <= 0x7fffffff && (C + 255) / 256 <= 65535, "short_conv: too large");
  const auto al16 = [](const void* ptr) { return ((uintptr_t)ptr & 15) == 0; };
  const bool vec = taps >= 2 && taps <= 4 && (cq & 7) == 0 && (ck & 7) == 0 && (cv & 7) == 0 && (u_stride & 7) == 0 &&
                   (q_out_stride & 7) == 0 && al16(u) && al16(w) && al16(bias) && al16(q_out) && al16(k_cache) && al16(v_cache) && al16(state);
  // rows a thread: 4 where that leaves four workgroups for every CU, else 2 (48 rows of 6144 channels 7.7 us, with 4 10.6).  With 8 the chip is
  // filled once and loads, sums and stores take turns: 2024 rows of 6144 24.8 us, with 4 22.2; 4096 rows 30.0 / 29.3
  const int threads = C / 8 >= 256 ? 256 : (C / 8 + 63) / 64 * 64;
  const unsigned parts = (unsigned)((C / 8 + threads - 1) / threads);
  const bool tall = (num_tokens + 3) / 4 * parts >= 4 * device_cu_count();
#define SC_VEC_TOK(TAPS, TOK)                                                                                                  \
  hipLaunchKernelGGL((short_conv_vec8_kernel<T, TAPS, TOK>), dim3((unsigned)((num_tokens + TOK - 1) / TOK), parts), dim3(threads), 0, (hipStream_t)stream,  \
                     (S*)q_out, q_out_stride, (S*)k_cache,                                                                     \
                     (S*)v_cache, cache_slots, num_cache_slots, (const S*)u, u_stride, (const S*)w, (const S*)bias, (const S*)state, state_slots, \
                     q_start, ctx_len, seq_of_token, num_tokens, cq, ck, cv, act)
#define SC_VEC(TAPS)                 \
  do {                               \
    if (tall) SC_VEC_TOK(TAPS, 4);   \
    else SC_VEC_TOK(TAPS, 2);        \
  } while (0)
  MIX_DISPATCH_DTYPE(dtype, {
    typedef typename T::storage S;
    if (vec && taps == 2) SC_VEC(2);
    else if (vec && taps == 3) SC_VEC(3);
    else if (vec && taps == 4) SC_VEC(4);
    else
    hipLaunchKernelGGL((short_conv_kernel<T>), dim3((unsigned)num_tokens, (unsigned)((C + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, (S*)q_out, q_out_stride, (S*)k_cache, (S*)v_cache, cache_slots, num_cache_slots,
                       (const S*)u, u_stride, (const S*)w, (const S*)bias, (const S*)state, state_slots, q_start, ctx_len, seq_of_token, cq, ck,
                       cv, taps, act);
  });
#undef SC_VEC
#undef SC_VEC_TOK
  APHRO_LAUNCH_CHECK();
  if (taps == 1) return APHRO_OK;
  return aphro_short_conv_state(state, u, u_stride, state_slots, q_start, q_len, ctx_len, num_seqs, C, taps, dtype, stream);
}
