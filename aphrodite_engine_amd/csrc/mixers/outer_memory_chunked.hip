// Gated outer-product memories (outer_memory.hip has the recurrence) over prompt portions, in chunks of 64 tokens on the matrix
// cores.  With G_i the sum of log a over a chunk's tokens up to i and S the state ahead of the chunk:
//     o_i = e^{G_i} S^T q_i + sum_{j <= i} e^{G_i - G_j} b_j (q_i . k_j) v_j,      S' = e^{G_63} S + sum_j e^{G_63 - G_j} b_j k_j v_j^T
// so three launches do what a scan does token by token:
//   1. om_chunk_update: every chunk's own sum U (d x 64 value columns a workgroup) and its decay -- all chunks at once
//   2. om_chunk_carry:  S through the chunks, elementwise; U is replaced by the state ahead of its chunk
//   3. om_chunk_out:    o of every chunk -- all chunks at once
// and mLSTM's running maximum (a recurrence of its own, one number per head and token) is worked out ahead of them by om_gates.
//
// Everything is fp32, products on v_mfma_f32_16x16x4_f32 (what enters the recurrence is fp32 and stays so); G is summed in 64 bits, so that a small decay keeps its digits behind a large one.
// Only the differences G_i - G_j <= 0 are exponentiated: nothing overflows however strong the decay.
//
// What bounds it: the fp32 products (the matrix pipe is busy half of the time in launches 1 and 3) and the states between the chunks
// (written once, read and written once, read once: dim x vdim x 4 bytes a chunk and head).  A scan is bound by the latency of its
// token chain.  One portion of 4096 tokens, scan -> chunks: decay 8 x 64 x 128 1106 -> 60 us, mLSTM 4 x 128 x 256 2170 -> 113 us, state
// space 64 x 128 x 64 1476 -> 274 us (128 heads: 1482 -> 575 us).  With mLSTM's and the state space's bf16 inputs on the 16-bit units (the *16
// kernels): mLSTM 4096 tokens 112 -> 95 us, state space 2000 tokens 146 -> 111, three portions of 300, 128 heads 171 -> 137; error against 64
// bits 4.8e-7 -> 2.5e-7 and 1.05e-7 -> 0.94e-7.
// Outputs lie as the products leave them: scores as K Q^T and results as V^T P^T, so that a score's registers are the next product's
// operand and a lane holds four neighbouring value columns of one token.  Row pitches are 4 floats over a multiple of 32: the
// eight lanes that a 16-byte LDS access serves at a time fall on all 32 banks.
#include "outer_memory.h"
#include "chunked_scan.h"

namespace aphro {

constexpr int OMC_COLS = 64;                // value columns of a workgroup
constexpr int OMC_PITCH = CHUNK + 4;

struct OMChunk {
  OuterMemory p;
  int min_len;            // segments shorter than this are the scan's
  int chunk0, span;       // the chunks of these launches (below: [chunks] of one span)
  int vpad;               // vdim rounded up to 16
  float* u;               // [chunks, heads, vpad, DP] U, then the state ahead of the chunk
  float* un;              // mLSTM: [chunks, heads, DP], the same of the normaliser
  float* total;           // [chunks, heads] decay over the chunk
  float *la, *gb, *em;    // mLSTM: [heads, tokens] log decay, write strength, e^{-m}
};

// ---- mLSTM gates ---------------------------------------------------------------------------------------------------------------
// m_t = max(f_t + m_{t-1}, i_t) composes: (F, I) then (F', I') is (F + F', max(I + F', I')).  A thread folds four neighbouring tokens, a
// wave its threads, the workgroup its waves; then every token takes log a_t = f_t + m_{t-1} - m_t from the SAME rounded m that its
// neighbours use, so the state's scale stays consistent whatever the order of the folds.
constexpr int OMG_TOKENS = 4096;
template <typename T>
__global__ __launch_bounds__(1024) void om_gates_kernel(OMChunk a) {
  typedef typename T::storage ST;
  __shared__ float ms[OMG_TOKENS + 1], wf[16], wi[16];
  const OuterMemory& p = a.p;
  const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = p.q_len[s], slot = p.slot_of_seq[s];
  if (n < a.min_len || slot < 0 || slot >= p.num_slots) return;
  const int64_t t0 = p.q_start[s];
  const int ncopy = (p.vdim + 15) >> 4;
  float* mptr = p.state_m + ((int64_t)slot * p.heads + h) * ncopy;
  float m0 = p.ctx_len[s] == 0 ? 0.f : mptr[0];
  const ST* gi = (const ST*)p.gate_i + t0 * p.gate_stride + h;
  const ST* gf = (const ST*)p.gate_f + t0 * p.gate_stride + h;
  const int64_t row = (int64_t)h * p.num_tokens + t0;
  for (int base = 0; base < n; base += OMG_TOKENS) {
    const int cnt = min(OMG_TOKENS, n - base);
    float f[4], ig[4], F = 0.f, I = -INFINITY;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = 4 * tid + u;
      f[u] = 0.f, ig[u] = -INFINITY;                                     // (a token that is not there: m passes)
      if (t < cnt) {
        ig[u] = p.gate_cap * tanhf(T::to_f32(gi[(int64_t)(base + t) * p.gate_stride]) / p.gate_cap);
        f[u] = log_sigmoid_f(p.gate_cap * tanhf(T::to_f32(gf[(int64_t)(base + t) * p.gate_stride]) / p.gate_cap));
      }
      F += f[u];
      I = fmaxf(I + f[u], ig[u]);
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float F2 = __shfl_up(F, o, 64), I2 = __shfl_up(I, o, 64);
      if (lane >= o) {
        I = fmaxf(I2 + F, I);
        F += F2;
      }
    }
    if (lane == 63) wf[wave] = F, wi[wave] = I;
    float ef = __shfl_up(F, 1, 64), ei = __shfl_up(I, 1, 64);            // what lies ahead of the thread in its wave
    if (lane == 0) ef = 0.f, ei = -INFINITY;
    __syncthreads();
    float m = m0;
    for (int w = 0; w < wave; ++w) m = fmaxf(m + wf[w], wi[w]);
    m = fmaxf(m + ef, ei);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      m = fmaxf(f[u] + m, ig[u]);
      if (4 * tid + u < cnt) ms[4 * tid + u + 1] = m;
    }
    if (tid == 0) ms[0] = m0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = 4 * tid + u;
      if (t < cnt) {
        const float mt = ms[t + 1];
        a.la[row + base + t] = f[u] + ms[t] - mt;
        a.gb[row + base + t] = expf(ig[u] - mt);
        a.em[row + base + t] = expf(-mt);
      }
    }
    m0 = ms[cnt];
    __syncthreads();
  }
  for (int c = tid; c < ncopy; c += 1024) mptr[c] = m0;
}

// ---- the chunk's gates ------------------------------------------------------------------------------------------------------------
// Log decay (base 2) and write strength of the wave's lane's token; lanes past the chunk's end neither decay nor write.
template <typename T, int MODE>
__device__ __forceinline__ void chunk_gate(const OMChunk& a, int h, int64_t row0, int lane, int cnt, double& la, float& b) {
  const OuterMemory& p = a.p;
  la = 0.0, b = 0.f;
  if (lane >= cnt) return;
  if constexpr (MODE == 0) {
    const float d = fabsf(p.decay[h]);                                  // (a negative decay: its sign is put back per pair)
    la = d == 1.f ? 0.0 : fmax(log2((double)d), -1e5);
    if (d != d) la = d;
    b = 1.f;
  } else if constexpr (MODE == 1) {
    la = log2_decay(a.la[(int64_t)h * p.num_tokens + row0 + lane]);
    b = a.gb[(int64_t)h * p.num_tokens + row0 + lane];
  } else {
    const float dt = softplus_f(T::to_f32(((const typename T::storage*)p.gate_i)[(row0 + lane) * p.gate_stride + h]) + p.dt_bias[h]);
    la = log2_decay(-expf(p.a_log[h]) * dt);
    b = dt;
  }
}

template <int MODE>
__device__ __forceinline__ float act_k(float x) { return MODE == 0 ? silu_f(x) : x; }

// ---- 1. every chunk's own sum ------------------------------------------------------------------------------------------------------
template <typename T, int MODE, int DP, bool VEC>
__global__ __launch_bounds__(256) void om_chunk_update_kernel(OMChunk a) {
  typedef typename T::storage ST;
  __shared__ __attribute__((aligned(16))) float kt[DP * OMC_PITCH];
  __shared__ __attribute__((aligned(16))) float vt[OMC_COLS * OMC_PITCH];
  const OuterMemory& p = a.p;
  int s, c;
  if (!locate_chunk(a.chunk0 + blockIdx.x, p.q_len, p.num_seqs, a.min_len, s, c)) return;
  const int slot = p.slot_of_seq[s];
  if (slot < 0 || slot >= p.num_slots) return;
  const int h = blockIdx.y, c0 = blockIdx.z * OMC_COLS, hk = MODE == 2 ? h / (p.heads / p.qk_heads) : h;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cnt = min(CHUNK, p.q_len[s] - c * CHUNK);
  const int64_t row0 = (int64_t)p.q_start[s] + c * CHUNK;
  // lane = token; the four waves divide the key numbers and the value columns.  Every load is on its way before the first is used.
  const int64_t row = row0 + min(lane, cnt - 1);
  const ST* kr = (const ST*)p.k + row * p.k_stride + (int64_t)hk * p.dim;
  const ST* vr = (const ST*)p.v + row * p.v_stride + (int64_t)h * p.vdim + c0;
  float kx[DP / 32][8], vx[OMC_COLS / 32][8];
#pragma unroll
  for (int it = 0; it < DP / 32; ++it) load8<T, VEC>(kr, wave * (DP / 4) + it * 8, p.dim, kx[it]);
#pragma unroll
  for (int it = 0; it < OMC_COLS / 32; ++it) load8<T, VEC>(vr, wave * (OMC_COLS / 4) + it * 8, p.vdim - c0, vx[it]);
  double la;
  float b;
  chunk_gate<T, MODE>(a, h, row0, lane, cnt, la, b);
  const double g = wave_incl_sum(la, lane), gend = __shfl(g, 63, 64);
  float w = exp2_d(gend - g) * b, all = exp2_d(gend);
  if (MODE == 0 && p.decay[h] < 0.f) {
    if ((cnt - 1 - lane) & 1) w = -w;
    if (cnt & 1) all = -all;
  }
  if (blockIdx.z == 0 && tid == 0) a.total[(int64_t)blockIdx.x * p.heads + h] = all;
#pragma unroll
  for (int it = 0; it < DP / 32; ++it)
#pragma unroll
    for (int i = 0; i < 8; ++i) kt[(wave * (DP / 4) + it * 8 + i) * OMC_PITCH + lane] = lane < cnt ? act_k<MODE>(kx[it][i]) * w : 0.f;
#pragma unroll
  for (int it = 0; it < OMC_COLS / 32; ++it)
#pragma unroll
    for (int i = 0; i < 8; ++i) vt[(wave * (OMC_COLS / 4) + it * 8 + i) * OMC_PITCH + lane] = lane < cnt ? act_k<MODE>(vx[it][i]) : 0.f;
  __syncthreads();
  const int li = lane & 15, lg = lane >> 4;
  const int nct = min(OMC_COLS / 16, (p.vdim - c0 + 15) >> 4);
  constexpr int DT = DP / 64;                              // 16-row tiles of a wave
  f32x4 acc[DT][OMC_COLS / 16] = {};
#pragma unroll
  for (int kk = 0; kk < CHUNK / 16; ++kk) {
    f32x4 av[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      av[dt] = *reinterpret_cast<const f32x4*>(&kt[((wave * DT + dt) * 16 + li) * OMC_PITCH + 16 * kk + 4 * lg]);
#pragma unroll
    for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
      if (ct >= nct) break;
      const f32x4 bv = *reinterpret_cast<const f32x4*>(&vt[(ct * 16 + li) * OMC_PITCH + 16 * kk + 4 * lg]);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[dt][ct] = mfma4(av[dt][m], bv[m], acc[dt][ct]);
    }
  }
  float* u = a.u + (((int64_t)blockIdx.x * p.heads + h) * a.vpad + c0) * DP;
#pragma unroll
  for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
    if (ct >= nct) break;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      *reinterpret_cast<f32x4*>(&u[(ct * 16 + li) * DP + (wave * DT + dt) * 16 + 4 * lg]) = acc[dt][ct];
  }
  if (MODE == 1 && blockIdx.z == 0 && tid < DP) {
    float sum = 0.f;
    for (int t = 0; t < CHUNK; t += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(&kt[tid * OMC_PITCH + t]);
      sum += (x[0] + x[1]) + (x[2] + x[3]);
    }
    a.un[((int64_t)blockIdx.x * p.heads + h) * DP + tid] = sum;
  }
}

// The same where keys and values enter as the bf16 numbers they are (mLSTM, state space): U = sum_j k_j (w_j v_j)^T with the second factor in
// three bf16 parts.  Keys that are not finite would meet a part that is zero: such a chunk multiplies in fp32, from the same LDS.
template <int MODE, int DP, bool VEC>
__global__ __launch_bounds__(256) void om_chunk_update16_kernel(OMChunk a) {
  constexpr int PITCH = CHUNK + 8;
  __shared__ __attribute__((aligned(16))) uint16_t kt[DP * PITCH];
  __shared__ __attribute__((aligned(16))) uint16_t vt[3][OMC_COLS * PITCH];
  __shared__ float ws[CHUNK];
  const OuterMemory& p = a.p;
  int s, c;
  if (!locate_chunk(a.chunk0 + blockIdx.x, p.q_len, p.num_seqs, a.min_len, s, c)) return;
  const int slot = p.slot_of_seq[s];
  if (slot < 0 || slot >= p.num_slots) return;
  const int h = blockIdx.y, c0 = blockIdx.z * OMC_COLS, hk = MODE == 2 ? h / (p.heads / p.qk_heads) : h;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cnt = min(CHUNK, p.q_len[s] - c * CHUNK);
  const int64_t row0 = (int64_t)p.q_start[s] + c * CHUNK;
  const int64_t row = row0 + min(lane, cnt - 1);
  const uint16_t* kr = (const uint16_t*)p.k + row * p.k_stride + (int64_t)hk * p.dim;
  const uint16_t* vr = (const uint16_t*)p.v + row * p.v_stride + (int64_t)h * p.vdim + c0;
  u16x8 kx[DP / 32], vx[OMC_COLS / 32];
#pragma unroll
  for (int it = 0; it < DP / 32; ++it) kx[it] = load8_bits<VEC>(kr, wave * (DP / 4) + it * 8, p.dim);
#pragma unroll
  for (int it = 0; it < OMC_COLS / 32; ++it) vx[it] = load8_bits<VEC>(vr, wave * (OMC_COLS / 4) + it * 8, p.vdim - c0);
  double la;
  float b;
  chunk_gate<BFloat, MODE>(a, h, row0, lane, cnt, la, b);
  const double g = wave_incl_sum(la, lane), gend = __shfl(g, 63, 64);
  const float w = exp2_d(gend - g) * b, all = exp2_d(gend);
  if (blockIdx.z == 0 && tid == 0) a.total[(int64_t)blockIdx.x * p.heads + h] = all;
  if (tid < CHUNK) ws[tid] = lane < cnt ? w : 0.f;
  bool odd = false;                                                      // a key that is not finite
#pragma unroll
  for (int it = 0; it < DP / 32; ++it)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint16_t x = lane < cnt ? kx[it][i] : (uint16_t)0;
      odd |= (x & 0x7f80u) == 0x7f80u;
      kt[(wave * (DP / 4) + it * 8 + i) * PITCH + lane] = x;
    }
#pragma unroll
  for (int it = 0; it < OMC_COLS / 32; ++it)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      uint16_t part[3];
      split3(lane < cnt ? BFloat::to_f32(vx[it][i]) * w : 0.f, part);
#pragma unroll
      for (int n = 0; n < 3; ++n) vt[n][(wave * (OMC_COLS / 4) + it * 8 + i) * PITCH + lane] = part[n];
    }
  odd = __syncthreads_or(odd);
  const int li = lane & 15, lg = lane >> 4;
  const int nct = min(OMC_COLS / 16, (p.vdim - c0 + 15) >> 4);
  constexpr int DT = DP / 64;                              // 16-row tiles of a wave
  f32x4 acc[DT][OMC_COLS / 16] = {};
#pragma unroll
  for (int kk = 0; kk < CHUNK / 32; ++kk) {
    u16x8 av[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) av[dt] = *reinterpret_cast<const u16x8*>(&kt[((wave * DT + dt) * 16 + li) * PITCH + 32 * kk + 8 * lg]);
#pragma unroll
    for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
      if (ct >= nct) break;
      u16x8 bv[3];
#pragma unroll
      for (int n = 0; n < 3; ++n) bv[n] = *reinterpret_cast<const u16x8*>(&vt[n][(ct * 16 + li) * PITCH + 32 * kk + 8 * lg]);
      if (!odd) {
#pragma unroll
        for (int n = 2; n >= 0; --n)
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) acc[dt][ct] = mfma16(av[dt], bv[n], acc[dt][ct]);
      } else {
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          const float x = (BFloat::to_f32(bv[2][m]) + BFloat::to_f32(bv[1][m])) + BFloat::to_f32(bv[0][m]);
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) acc[dt][ct] = mfma4(BFloat::to_f32(av[dt][m]), x, acc[dt][ct]);
        }
      }
    }
  }
  float* u = a.u + (((int64_t)blockIdx.x * p.heads + h) * a.vpad + c0) * DP;
#pragma unroll
  for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
    if (ct >= nct) break;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      *reinterpret_cast<f32x4*>(&u[(ct * 16 + li) * DP + (wave * DT + dt) * 16 + 4 * lg]) = acc[dt][ct];
  }
  if (MODE == 1 && blockIdx.z == 0 && tid < DP) {
    float sum = 0.f;
    for (int t = 0; t < CHUNK; t += 8) {
      const u16x8 x = *reinterpret_cast<const u16x8*>(&kt[tid * PITCH + t]);
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += BFloat::to_f32(x[i]) * ws[t + i];
    }
    a.un[((int64_t)blockIdx.x * p.heads + h) * DP + tid] = sum;
  }
}

// ---- 2. the state through the chunks -------------------------------------------------------------------------------------------------
// A thread carries four neighbouring key rows of one value column (mLSTM: behind them, one number of the normaliser); U of eight to
// sixteen chunks is in flight ahead of the chain.
template <int MODE, int DP>
__global__ __launch_bounds__(64) void om_chunk_carry_kernel(OMChunk a) {
  const OuterMemory& p = a.p;
  const int s = blockIdx.z, h = blockIdx.y;
  const int n = p.q_len[s], slot = p.slot_of_seq[s];
  if (n < a.min_len || slot < 0 || slot >= p.num_slots) return;
  int begin, nc;
  int64_t first;
  if (!span_of(s, (n + CHUNK - 1) / CHUNK, p.q_len, a.min_len, a.chunk0, a.span, begin, nc, first)) return;
  const bool fresh = begin == 0 && p.ctx_len[s] == 0;
  first += begin, nc -= begin;                             // (chunks are numbered from the span's first from here on)
  const int x = blockIdx.x * 64 + threadIdx.x, quads = a.vpad * (DP / 4);
  const float* tot = a.total + first * p.heads + h;
  if (MODE == 1 && x >= quads && x < quads + DP) {
    const int d = x - quads, ncopy = (p.vdim + 15) >> 4;
    float* nbase = p.state_n + ((int64_t)slot * p.heads + h) * ncopy * p.dim;
    float S = !fresh && d < p.dim ? nbase[d] : 0.f;
    float* un = a.un + (first * p.heads + h) * DP + d;
    for (int c = 0; c < nc; ++c) {
      const float u = un[(int64_t)c * p.heads * DP];
      un[(int64_t)c * p.heads * DP] = S;
      S = tot[(int64_t)c * p.heads] * S + u;
    }
    if (d < p.dim)
      for (int cp = 0; cp < ncopy; ++cp) nbase[(int64_t)cp * p.dim + d] = S;
    return;
  }
  if (x >= quads) return;
  const int e = x / (DP / 4), d = (x % (DP / 4)) * 4;
  float* sb = p.state_s + ((int64_t)slot * p.heads + h) * p.dim * (int64_t)p.vdim + e;
  f32x4 S = {};
  if (!fresh && e < p.vdim)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (d + i < p.dim) S[i] = sb[(int64_t)(d + i) * p.vdim];
  float* u = a.u + (first * p.heads + h) * a.vpad * (int64_t)DP + (int64_t)e * DP + d;
  const int64_t step = (int64_t)p.heads * a.vpad * DP;
  constexpr int AHEAD = 8;
  f32x4 w[2][AHEAD];
  float t[2][AHEAD];
  auto fetch = [&](int c0, f32x4 (&x)[AHEAD], float (&y)[AHEAD]) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (c0 + i < nc) {
        x[i] = *reinterpret_cast<const f32x4*>(u + (c0 + i) * step);
        y[i] = tot[(int64_t)(c0 + i) * p.heads];
      }
  };
  auto carry = [&](int c0, const f32x4 (&x)[AHEAD], const float (&y)[AHEAD]) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (c0 + i < nc) {
        *reinterpret_cast<f32x4*>(u + (c0 + i) * step) = S;
#pragma unroll
        for (int r = 0; r < 4; ++r) S[r] = y[i] * S[r] + x[i][r];
      }
  };
  fetch(0, w[0], t[0]);
  for (int c0 = 0; c0 < nc; c0 += 2 * AHEAD) {
    fetch(c0 + AHEAD, w[1], t[1]);
    carry(c0, w[0], t[0]);
    fetch(c0 + 2 * AHEAD, w[0], t[0]);
    carry(c0 + AHEAD, w[1], t[1]);
  }
  if (e < p.vdim)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (d + i < p.dim) sb[(int64_t)(d + i) * p.vdim] = S[i];
}

// ---- 3. every chunk's outputs ---------------------------------------------------------------------------------------------------------
template <typename T, int MODE, int DP, bool VEC>
__global__ __launch_bounds__(256) void om_chunk_out_kernel(OMChunk a) {
  typedef typename T::storage ST;
  constexpr int KP = DP + 4;
  __shared__ __attribute__((aligned(16))) float ks[CHUNK * KP];          // afterwards, for numbers that are not finite: the scores
  __shared__ __attribute__((aligned(16))) float vt[OMC_COLS * OMC_PITCH];
  __shared__ double gs[CHUNK];
  __shared__ float bs[CHUNK];
  const OuterMemory& p = a.p;
  int s, c;
  if (!locate_chunk(a.chunk0 + blockIdx.x, p.q_len, p.num_seqs, a.min_len, s, c)) return;
  const int slot = p.slot_of_seq[s];
  if (slot < 0 || slot >= p.num_slots) return;
  const int h = blockIdx.y, c0 = blockIdx.z * OMC_COLS, hk = MODE == 2 ? h / (p.heads / p.qk_heads) : h;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int cnt = min(CHUNK, p.q_len[s] - c * CHUNK);
  const int64_t row0 = (int64_t)p.q_start[s] + c * CHUNK;
  const int64_t row = row0 + min(lane, cnt - 1);
  const ST* kr = (const ST*)p.k + row * p.k_stride + (int64_t)hk * p.dim;
  const ST* vr = (const ST*)p.v + row * p.v_stride + (int64_t)h * p.vdim + c0;
  // the workgroup's keys and values are on their way while the waves multiply with the state; lane = token here
  float kx[DP / 32][8], vx[OMC_COLS / 32][8];
#pragma unroll
  for (int it = 0; it < DP / 32; ++it) load8<T, VEC>(kr, wave * (DP / 4) + it * 8, p.dim, kx[it]);
#pragma unroll
  for (int it = 0; it < OMC_COLS / 32; ++it) load8<T, VEC>(vr, wave * (OMC_COLS / 4) + it * 8, p.vdim - c0, vx[it]);
  // a wave's sixteen queries: lane li's query, eight neighbouring numbers a step.  Later queries see more tokens: the tiles go round the
  // waves from workgroup to workgroup, so that no SIMD has all the long ones.
  const int qt = (wave + blockIdx.x + blockIdx.y) & 3, qi = qt * 16 + li;
  float q[DP / 32][8];
  {
    const ST* qr = (const ST*)p.q + (row0 + min(qi, cnt - 1)) * p.q_stride + (int64_t)hk * p.dim;
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk) {
      load8<T, VEC>(qr, 32 * kk + 8 * lg, p.dim, q[kk]);
#pragma unroll
      for (int i = 0; i < 8; ++i) q[kk][i] = MODE == 0 ? silu_f(q[kk][i]) : MODE == 1 ? q[kk][i] * p.q_scale : q[kk][i];
    }
  }
  const int nct = min(OMC_COLS / 16, (p.vdim - c0 + 15) >> 4);
  // what the state ahead of the chunk gives
  const float* st = a.u + (((int64_t)blockIdx.x * p.heads + h) * a.vpad + c0) * DP;
  f32x4 acc[OMC_COLS / 16] = {};
#pragma unroll
  for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
    if (ct >= nct) break;
    const float* sr = st + (ct * 16 + li) * DP + 8 * lg;
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk) {
      const f32x4 s0 = *reinterpret_cast<const f32x4*>(sr + 32 * kk), s1 = *reinterpret_cast<const f32x4*>(sr + 32 * kk + 4);
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[ct] = mfma4(s0[m], q[kk][m], acc[ct]);
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[ct] = mfma4(s1[m], q[kk][4 + m], acc[ct]);
    }
  }
  bool odd = false;                                                      // a value that is not finite
#pragma unroll
  for (int it = 0; it < DP / 32; ++it) {
    const int d = wave * (DP / 4) + it * 8;
    f32x4 lo, hi;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      lo[i] = lane < cnt ? act_k<MODE>(kx[it][i]) : 0.f;
      hi[i] = lane < cnt ? act_k<MODE>(kx[it][4 + i]) : 0.f;
    }
    *reinterpret_cast<f32x4*>(&ks[lane * KP + d]) = lo;
    *reinterpret_cast<f32x4*>(&ks[lane * KP + d + 4]) = hi;
  }
#pragma unroll
  for (int it = 0; it < OMC_COLS / 32; ++it) {
    const int e = wave * (OMC_COLS / 4) + it * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float val = lane < cnt ? act_k<MODE>(vx[it][i]) : 0.f;
      odd |= !finite_f(val);
      vt[(e + i) * OMC_PITCH + lane] = val;
    }
  }
  if (wave == 0) {
    double la;
    float b;
    chunk_gate<T, MODE>(a, h, row0, lane, cnt, la, b);
    gs[lane] = wave_incl_sum(la, lane);
    bs[lane] = b;
  }
  odd = __syncthreads_or(odd);
  const bool neg = MODE == 0 && p.decay[h] < 0.f;
  const double gq = gs[qi];
  const float eq = (neg && !(qi & 1) ? -1.f : 1.f) * exp2_d(gq);           // the state has decayed qi + 1 times
#pragma unroll
  for (int ct = 0; ct < OMC_COLS / 16; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[ct][r] *= eq;
  float nq = 0.f;                                                       // mLSTM: the lane's part of n . q
  if constexpr (MODE == 1) {
    const float* nb = a.un + ((int64_t)blockIdx.x * p.heads + h) * DP + 8 * lg;
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk)
#pragma unroll
      for (int i = 0; i < 8; ++i) nq += q[kk][i] * nb[32 * kk + i];
    nq *= eq;
  }
  // the chunk's own tokens up to the query's
  f32x4 pr[CHUNK / 16];
#pragma unroll
  for (int jt = 0; jt < CHUNK / 16; ++jt) {
    if (jt > qt) break;
    f32x4 sc = {};
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk) {
      const float* kp = &ks[(jt * 16 + li) * KP + 32 * kk + 8 * lg];
      const f32x4 k0 = *reinterpret_cast<const f32x4*>(kp), k1 = *reinterpret_cast<const f32x4*>(kp + 4);
#pragma unroll
      for (int m = 0; m < 4; ++m) sc = mfma4(k0[m], q[kk][m], sc);
#pragma unroll
      for (int m = 0; m < 4; ++m) sc = mfma4(k1[m], q[kk][4 + m], sc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = jt * 16 + 4 * lg + r;
      float w = 0.f;
      if (j <= qi) w = sc[r] * (exp2_d(gq - gs[j]) * bs[j]);
      pr[jt][r] = neg && ((qi - j) & 1) ? -w : w;
      if (MODE == 1) nq += w;
    }
    if (!odd) {
#pragma unroll
      for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
        if (ct >= nct) break;
        const f32x4 vv = *reinterpret_cast<const f32x4*>(&vt[(ct * 16 + li) * OMC_PITCH + jt * 16 + 4 * lg]);
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[ct] = mfma4(vv[m], pr[jt][m], acc[ct]);
      }
    }
  }
  if (odd) {
    // zero times a value that is not finite is not zero: a token behind the query must not be multiplied at all
    __syncthreads();                                                     // every wave is through with the keys
    float* ps = ks;                                                      // [64 queries][64 + 1]
#pragma unroll
    for (int jt = 0; jt < CHUNK / 16; ++jt)
      if (jt <= qt)
#pragma unroll
        for (int r = 0; r < 4; ++r) ps[qi * (CHUNK + 1) + jt * 16 + 4 * lg + r] = pr[jt][r];
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < OMC_COLS / 16; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float sum = 0.f;
        for (int j = 0; j <= qi; ++j) sum += ps[qi * (CHUNK + 1) + j] * vt[(ct * 16 + 4 * lg + r) * OMC_PITCH + j];
        acc[ct][r] += sum;
      }
  }
  float inv = 1.f;
  if constexpr (MODE == 1) {
    nq += __shfl_xor(nq, 16, 64);
    nq += __shfl_xor(nq, 32, 64);
    const float em = a.em[(int64_t)h * p.num_tokens + row0 + min(qi, cnt - 1)];
    inv = fmaxf(fabsf(nq), em) + 1e-6f;
  }
  if (qi >= cnt) return;
  const float skip = MODE == 2 ? p.skip[h] : 0.f;
  float* o = p.out + (row0 + qi) * ((int64_t)p.heads * p.vdim) + (int64_t)h * p.vdim + c0;
#pragma unroll
  for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
    if (ct >= nct) break;
    const int e = ct * 16 + 4 * lg;
    f32x4 x = acc[ct];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (MODE == 1) x[r] = x[r] / inv;
      if (MODE == 2) x[r] += skip * vt[(e + r) * OMC_PITCH + qi];
    }
    if ((p.vdim & 3) == 0) {
      if (c0 + e < p.vdim) *reinterpret_cast<f32x4*>(o + e) = x;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (c0 + e + r < p.vdim) o[e + r] = x[r];
    }
  }
}

// The same where keys, queries and values enter as the bf16 numbers they are (mLSTM, state space): scores are bf16 products as they stand, the
// weights that meet the values go in three bf16 parts; only the state's product stays on the fp32 units.
template <int MODE, int DP, bool VEC>
__global__ __launch_bounds__(256, MODE == 2 ? 4 : 3) void om_chunk_out16_kernel(OMChunk a) {
  constexpr int KP = DP + 8, VP = CHUNK + 8, SCORES = CHUNK * (CHUNK + 1) * 4, KEYS = CHUNK * KP * 2;
  __shared__ __attribute__((aligned(16))) unsigned char room[KEYS > SCORES ? KEYS : SCORES];      // keys; for values that are not finite, then: the scores
  __shared__ __attribute__((aligned(16))) uint16_t vt[OMC_COLS * VP];
  __shared__ double gs[CHUNK];
  __shared__ float bs[CHUNK];
  uint16_t* ks = reinterpret_cast<uint16_t*>(room);
  const OuterMemory& p = a.p;
  int s, c;
  if (!locate_chunk(a.chunk0 + blockIdx.x, p.q_len, p.num_seqs, a.min_len, s, c)) return;
  const int slot = p.slot_of_seq[s];
  if (slot < 0 || slot >= p.num_slots) return;
  const int h = blockIdx.y, c0 = blockIdx.z * OMC_COLS, hk = MODE == 2 ? h / (p.heads / p.qk_heads) : h;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int cnt = min(CHUNK, p.q_len[s] - c * CHUNK);
  const int64_t row0 = (int64_t)p.q_start[s] + c * CHUNK;
  const int64_t row = row0 + min(lane, cnt - 1);
  const uint16_t* kr = (const uint16_t*)p.k + row * p.k_stride + (int64_t)hk * p.dim;
  const uint16_t* vr = (const uint16_t*)p.v + row * p.v_stride + (int64_t)h * p.vdim + c0;
  u16x8 kx[DP / 32], vx[OMC_COLS / 32];
#pragma unroll
  for (int it = 0; it < DP / 32; ++it) kx[it] = load8_bits<VEC>(kr, wave * (DP / 4) + it * 8, p.dim);
#pragma unroll
  for (int it = 0; it < OMC_COLS / 32; ++it) vx[it] = load8_bits<VEC>(vr, wave * (OMC_COLS / 4) + it * 8, p.vdim - c0);
  const int qt = (wave + blockIdx.x + blockIdx.y) & 3, qi = qt * 16 + li;      // (which queries a wave has: as above)
  u16x8 q[DP / 32];
  {
    const uint16_t* qr = (const uint16_t*)p.q + (row0 + min(qi, cnt - 1)) * p.q_stride + (int64_t)hk * p.dim;
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk) q[kk] = load8_bits<VEC>(qr, 32 * kk + 8 * lg, p.dim);
  }
  const int nct = min(OMC_COLS / 16, (p.vdim - c0 + 15) >> 4);
  const float* st = a.u + (((int64_t)blockIdx.x * p.heads + h) * a.vpad + c0) * DP;
  f32x4 acc[OMC_COLS / 16] = {};
#pragma unroll
  for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
    if (ct >= nct) break;
    const float* sr = st + (ct * 16 + li) * DP + 8 * lg;
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk) {
      const f32x4 s0 = *reinterpret_cast<const f32x4*>(sr + 32 * kk), s1 = *reinterpret_cast<const f32x4*>(sr + 32 * kk + 4);
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[ct] = mfma4(s0[m], BFloat::to_f32(q[kk][m]), acc[ct]);
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[ct] = mfma4(s1[m], BFloat::to_f32(q[kk][4 + m]), acc[ct]);
    }
  }
  bool odd = false;                                                      // a value that is not finite
#pragma unroll
  for (int it = 0; it < DP / 32; ++it)
    *reinterpret_cast<u16x8*>(&ks[lane * KP + wave * (DP / 4) + it * 8]) = lane < cnt ? kx[it] : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int it = 0; it < OMC_COLS / 32; ++it)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint16_t x = lane < cnt ? vx[it][i] : (uint16_t)0;
      odd |= (x & 0x7f80u) == 0x7f80u;
      vt[(wave * (OMC_COLS / 4) + it * 8 + i) * VP + lane] = x;
    }
  if (wave == 0) {
    double la;
    float b;
    chunk_gate<BFloat, MODE>(a, h, row0, lane, cnt, la, b);
    gs[lane] = wave_incl_sum(la, lane);
    bs[lane] = b;
  }
  odd = __syncthreads_or(odd);
  const double gq = gs[qi];
  const float scale = MODE == 1 ? p.q_scale : 1.f, eq = exp2_d(gq) * scale;
#pragma unroll
  for (int ct = 0; ct < OMC_COLS / 16; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[ct][r] *= eq;
  float nq = 0.f;                                                       // mLSTM: the lane's part of n . q
  if constexpr (MODE == 1) {
    const float* nb = a.un + ((int64_t)blockIdx.x * p.heads + h) * DP + 8 * lg;
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk)
#pragma unroll
      for (int i = 0; i < 8; ++i) nq += BFloat::to_f32(q[kk][i]) * nb[32 * kk + i];
    nq *= eq;
  }
  // the chunk's own tokens up to the query's, 32 a step: lane group lg has tokens 4 lg .. 4 lg + 3 of either half
  f32x4 pr[CHUNK / 16];
#pragma unroll
  for (int jp = 0; jp < CHUNK / 32; ++jp) {
    if (2 * jp > qt) break;
    u16x8 part[3];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int jt = 2 * jp + half;
      f32x4 sc = {};
      if (jt <= qt) {
#pragma unroll
        for (int kk = 0; kk < DP / 32; ++kk) sc = mfma16(*reinterpret_cast<const u16x8*>(&ks[(jt * 16 + li) * KP + 32 * kk + 8 * lg]), q[kk], sc);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = jt * 16 + 4 * lg + r;
        float w = 0.f;
        if (j <= qi) w = sc[r] * scale * (exp2_d(gq - gs[j]) * bs[j]);
        pr[jt][r] = w;
        if (MODE == 1) nq += w;
        uint16_t x[3];
        split3(w, x);
#pragma unroll
        for (int n = 0; n < 3; ++n) part[n][4 * half + r] = x[n];
      }
    }
    if (!odd) {
#pragma unroll
      for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
        if (ct >= nct) break;
        const uint16_t* vp = &vt[(ct * 16 + li) * VP + 32 * jp + 4 * lg];
        const u32x2 lo = *reinterpret_cast<const u32x2*>(vp), hi = *reinterpret_cast<const u32x2*>(vp + 16);
        const u16x8 vv = __builtin_bit_cast(u16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
#pragma unroll
        for (int n = 2; n >= 0; --n) acc[ct] = mfma16(vv, part[n], acc[ct]);
      }
    }
  }
  if (odd) {
    // zero times a value that is not finite is not zero: a token behind the query must not be multiplied at all
    __syncthreads();                                                     // every wave is through with the keys
    float* ps = reinterpret_cast<float*>(room);                          // [64 queries][64 + 1]
#pragma unroll
    for (int jt = 0; jt < CHUNK / 16; ++jt)
      if (jt <= qt)
#pragma unroll
        for (int r = 0; r < 4; ++r) ps[qi * (CHUNK + 1) + jt * 16 + 4 * lg + r] = pr[jt][r];
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < OMC_COLS / 16; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float sum = 0.f;
        for (int j = 0; j <= qi; ++j) sum += ps[qi * (CHUNK + 1) + j] * BFloat::to_f32(vt[(ct * 16 + 4 * lg + r) * VP + j]);
        acc[ct][r] += sum;
      }
  }
  float inv = 1.f;
  if constexpr (MODE == 1) {
    nq += __shfl_xor(nq, 16, 64);
    nq += __shfl_xor(nq, 32, 64);
    const float em = a.em[(int64_t)h * p.num_tokens + row0 + min(qi, cnt - 1)];
    inv = fmaxf(fabsf(nq), em) + 1e-6f;
  }
  if (qi >= cnt) return;
  const float skip = MODE == 2 ? p.skip[h] : 0.f;
  float* o = p.out + (row0 + qi) * ((int64_t)p.heads * p.vdim) + (int64_t)h * p.vdim + c0;
#pragma unroll
  for (int ct = 0; ct < OMC_COLS / 16; ++ct) {
    if (ct >= nct) break;
    const int e = ct * 16 + 4 * lg;
    f32x4 x = acc[ct];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (MODE == 1) x[r] = x[r] / inv;
      if (MODE == 2) x[r] += skip * BFloat::to_f32(vt[(e + r) * VP + qi]);
    }
    if ((p.vdim & 3) == 0) {
      if (c0 + e < p.vdim) *reinterpret_cast<f32x4*>(o + e) = x;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (c0 + e + r < p.vdim) o[e + r] = x[r];
    }
  }
}

// Sizes of the workspace's parts for so many chunks, in floats: U, the normaliser's, decays, gates (of all tokens).
static void om_chunk_parts(const OuterMemory& p, int64_t chunks, int64_t (&n)[4]) {
  const int64_t dp = p.dim <= 64 ? 64 : 128, vpad = (p.vdim + 15) / 16 * 16;
  n[0] = chunks * p.heads * vpad * dp;
  n[1] = p.mode == 1 ? chunks * p.heads * dp : 0;
  n[2] = (chunks * p.heads + 3) / 4 * 4;
  n[3] = p.mode == 1 ? 3 * p.heads * p.num_tokens : 0;
}
static int64_t om_chunk_floats(const OuterMemory& p, int64_t chunks) {
  int64_t n[4];
  om_chunk_parts(p, chunks, n);
  return n[0] + n[1] + n[2] + n[3];
}

template <typename T, int MODE, int DP, bool VEC>
static void om_chunk_launch(OMChunk a, int64_t chunks) {
  const OuterMemory& p = a.p;
  const dim3 grid((unsigned)a.span, (unsigned)p.heads, (unsigned)((p.vdim + OMC_COLS - 1) / OMC_COLS));
  const unsigned items = (unsigned)a.vpad * (DP / 4) + (MODE == 1 ? DP : 0);
  if (MODE == 1) hipLaunchKernelGGL((om_gates_kernel<T>), dim3((unsigned)p.num_seqs, (unsigned)p.heads), dim3(1024), 0, p.stream, a);
  for (; a.chunk0 < chunks; a.chunk0 += a.span) {
    constexpr bool B16 = sizeof(typename T::storage) == 2 && MODE != 0;
    if constexpr (B16) hipLaunchKernelGGL((om_chunk_update16_kernel<MODE, DP, VEC>), grid, dim3(256), 0, p.stream, a);
    else hipLaunchKernelGGL((om_chunk_update_kernel<T, MODE, DP, VEC>), grid, dim3(256), 0, p.stream, a);
    hipLaunchKernelGGL((om_chunk_carry_kernel<MODE, DP>), dim3((items + 63) / 64, (unsigned)p.heads, (unsigned)p.num_seqs), dim3(64), 0, p.stream, a);
    if constexpr (B16) hipLaunchKernelGGL((om_chunk_out16_kernel<MODE, DP, VEC>), grid, dim3(256), 0, p.stream, a);
    else hipLaunchKernelGGL((om_chunk_out_kernel<T, MODE, DP, VEC>), grid, dim3(256), 0, p.stream, a);
  }
}

}  // namespace aphro

using namespace aphro;

extern "C" int64_t aphro_outer_memory_chunked_workspace(int num_seqs, int64_t num_tokens, int heads, int dim, int vdim, int mode, int min_len) {
  if (num_seqs <= 0 || num_tokens <= 0 || heads <= 0 || dim <= 0 || dim > 128 || vdim <= 0 || mode < 0 || mode > 2 || min_len <= 0) return 0;
  OuterMemory p = {};
  p.num_seqs = num_seqs, p.num_tokens = num_tokens, p.heads = heads, p.dim = dim, p.vdim = vdim, p.mode = mode;
  return span_workspace(max_chunks(num_tokens, num_seqs, num_seqs == 1 ? 1 : min_len), [&](int64_t n) { return om_chunk_floats(p, n); });
}

extern "C" int aphro_outer_memory_chunked(float* out, const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                                          const void* v, int64_t v_stride, const void* gate_i, const void* gate_f,
                                          int64_t gate_stride, float* state_s, float* state_n, float* state_m,
                                          const int32_t* slot_of_seq, int num_slots, const int32_t* q_start, const int32_t* q_len,
                                          const int32_t* ctx_len, int num_seqs, int64_t num_tokens, int heads, int dim, int vdim,
                                          int mode, const float* decay, float q_scale, float gate_cap, int qk_heads,
                                          const float* a_log, const float* dt_bias, const float* skip, int min_len, float* workspace,
                                          int64_t workspace_bytes, int dtype, void* stream) {
  if (num_tokens == 0 || num_seqs == 0) return APHRO_OK;
  OMChunk a = {};
  a.p = {out, q, k, v, gate_i, gate_f, q_stride, k_stride, v_stride, gate_stride, state_s, state_n, state_m, slot_of_seq,
         num_slots, q_start, q_len, ctx_len, num_seqs, num_tokens, heads, dim, vdim, mode, decay, q_scale, gate_cap, qk_heads,
         a_log, dt_bias, skip, min_len, dtype, (hipStream_t)stream};
  const OuterMemory& p = a.p;
  const int rc = outer_memory_check(p);
  if (rc != APHRO_OK) return rc;
  APHRO_CHECK(dim <= 128 && min_len > 0 && num_seqs <= 65535, "outer_memory_chunked: dim %d (<= 128), %d segments (<= 65535) from %d tokens on", dim, num_seqs, min_len);
  if (num_seqs == 1) min_len = 1;
  const int64_t chunks = max_chunks(num_tokens, num_seqs, min_len);
  APHRO_CHECK(chunks <= 0x3fffffff, "outer_memory_chunked: too many tokens");
  const int64_t span = span_chunks(chunks, workspace_bytes, [&](int64_t m) { return om_chunk_floats(p, m); });
  APHRO_CHECK(((uintptr_t)out & 15) == 0 && (chunks == 0 || (workspace && ((uintptr_t)workspace & 15) == 0 && span > 0)),
              "outer_memory_chunked: a workspace of %lld bytes at least, 16-byte aligned, is needed", (long long)om_chunk_floats(p, 1) * 4);
  int64_t n[4];
  om_chunk_parts(p, span, n);
  a.chunk0 = 0, a.span = (int)span;
  a.min_len = min_len;
  a.vpad = (vdim + 15) / 16 * 16;
  a.u = workspace;
  a.un = a.u + n[0];
  a.total = a.un + n[1];
  a.la = a.total + n[2];
  a.gb = a.la + (int64_t)heads * num_tokens;
  a.em = a.gb + (int64_t)heads * num_tokens;
  if (num_seqs > 1) {                                       // (a single segment: chunks, whatever its length)
    const int rs = outer_memory_scan_launch(p, min_len, min_len > 32);
    if (rs != APHRO_OK || chunks == 0) return rs;
  }
  const int elem = dtype == APHRO_BF16 ? 2 : 4;
  const bool vec = rows_of_16_bytes(q, q_stride, dim, elem) && rows_of_16_bytes(k, k_stride, dim, elem) && rows_of_16_bytes(v, v_stride, vdim, elem);
#define OMC_LAUNCH(MODE)                                                                  \
  do {                                                                                    \
    if (dim <= 64) {                                                                      \
      if (vec) om_chunk_launch<T, MODE, 64, true>(a, chunks);                   \
      else om_chunk_launch<T, MODE, 64, false>(a, chunks);                      \
    } else {                                                                              \
      if (vec) om_chunk_launch<T, MODE, 128, true>(a, chunks);                  \
      else om_chunk_launch<T, MODE, 128, false>(a, chunks);                     \
    }                                                                                     \
  } while (0)
  MIX_DISPATCH_DTYPE(dtype, {
    if (mode == 0) OMC_LAUNCH(0);
    else if (mode == 1) OMC_LAUNCH(1);
    else OMC_LAUNCH(2);
  });
#undef OMC_LAUNCH
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}
