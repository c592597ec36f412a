// Gated outer-product memories: per (request slot, head) a matrix state S [dim, vdim] with
//     S <- a_t S + b_t k_t v_t^T,     o_t = S^T q_t   [ / normaliser ]
// scanned token by token over each segment of the batch -- prompt portions and single decoded tokens alike -- from the
// state an earlier step left in the slot (or from zero for a sequence's first tokens), and written back in place.
//   mode 0, decay linear attention: q, k, v through silu, a_t = a fixed per-head decay, b_t = 1.
//   mode 1, mLSTM: exponential input gate and sigmoid forget gate in log space under a running maximum m (which starts at
//   ZERO), a normaliser vector n that follows the same recurrence with k alone, and the guarded division of the output.
//   mode 2, selective state space (Mamba-2): dt_t = softplus(raw + dt_bias), a_t = exp(-exp(A_log) dt_t), b_t = dt_t per head;
//   keys and queries (that literature's B and C) are shared by groups of neighbouring heads; o_t gains D v_t.
// State, gates, decays and the accumulation are fp32 whatever the activations' storage.
//
// Work split: a workgroup of 256 threads owns 64 (or, for prompt portions, 16) value columns of one (segment, head): thread
// = (column c, slice sl) with the key dimension cut into 4 (or 16) slices of DPT rows held in registers; q / k / v of 16 tokens at a time are staged in LDS with
// their activations applied (the next 16 tokens' raw values are already in flight in registers), the per-token partial dot products are folded over the slices with DPP moves.  The
// mLSTM gate recurrence of a 16-token stage runs in wave 0 (lane = token for the transcendental parts, a 16-step max-plus
// loop for m) before the stage is released to all waves.
#include "outer_memory.h"

namespace aphro {

constexpr int OMS_CH = 16, OMR_CH = 8;          // tokens of a stage

template <typename T, int MODE, int DPT>
__global__ __launch_bounds__(256) void outer_memory_scan_kernel(
    float* __restrict__ out, const typename T::storage* __restrict__ q, int64_t q_stride,
    const typename T::storage* __restrict__ k, int64_t k_stride, const typename T::storage* __restrict__ v, int64_t v_stride,
    const typename T::storage* __restrict__ gate_i, const typename T::storage* __restrict__ gate_f, int64_t gate_stride,
    float* __restrict__ state_s, float* __restrict__ state_n, float* __restrict__ state_m,
    const int32_t* __restrict__ slot_of_seq, int num_slots, const int32_t* __restrict__ q_start,
    const int32_t* __restrict__ q_len, const int32_t* __restrict__ ctx_len, int below, int heads, int dim, int vdim,
    const float* __restrict__ decay, float q_scale, float gate_cap, int qk_heads, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, const float* __restrict__ skip) {
  constexpr int SLOG = 4, NS = 1 << SLOG;     // slices of the key dimension = lanes that share a column
  constexpr int TW = 256 >> SLOG;      // value columns per workgroup
  constexpr int DP = NS * DPT;
  __shared__ __attribute__((aligned(16))) float qs[OMS_CH][DP];
  __shared__ __attribute__((aligned(16))) float ks[OMS_CH][DP];
  __shared__ float vs[OMS_CH][TW];
  __shared__ float a_s[OMS_CH], b_s[OMS_CH], em_s[OMS_CH];
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * TW;
  const int ncopy = (vdim + 15) >> 4, copy0 = c0 >> 4;          // n and m are kept once per 16 value columns
  const int tid = threadIdx.x, c = tid >> SLOG, sl = tid & (NS - 1), col = c0 + c;
  const int hq = MODE == 2 ? h / (heads / qk_heads) : h;    // head of q and k
  const int n = q_len[s];
  const int slot = slot_of_seq[s];
  if (n <= 0 || n >= below || slot < 0 || slot >= num_slots) return;
  const int64_t t0 = q_start[s];
  const bool fresh = ctx_len[s] == 0;
  float S[DPT], nv[DPT];
  float m = 0.f;                                            // wave 0 only (uniform)
  float* sbase = state_s + ((int64_t)slot * heads + h) * dim * (int64_t)vdim;
  float* nbase = MODE == 1 ? state_n + (((int64_t)slot * heads + h) * ncopy + copy0) * dim : nullptr;
  float* mptr = MODE == 1 ? state_m + ((int64_t)slot * heads + h) * ncopy + copy0 : nullptr;
#pragma unroll
  for (int i = 0; i < DPT; ++i) {
    const int r = sl * DPT + i;
    S[i] = (!fresh && r < dim && col < vdim) ? sbase[(int64_t)r * vdim + col] : 0.f;
    nv[i] = (MODE == 1 && !fresh && r < dim) ? nbase[r] : 0.f;
  }
  if (MODE == 1 && !fresh) m = *mptr;
  const float dec = MODE == 0 ? decay[h] : 0.f;
  const float neg_rate = MODE == 2 ? -expf(a_log[h]) : 0.f, dtb = MODE == 2 ? dt_bias[h] : 0.f, skip_h = MODE == 2 ? skip[h] : 0.f;

  // raw q / k / v (and gates) of the next stage travel in registers while the current stage is scanned
  constexpr int NQ = (OMS_CH * DP + 255) / 256, NV = (OMS_CH * TW + 255) / 256;
  float rq[NQ], rk[NQ], rv[NV], rgi = 0.f, rgf = 0.f;
  auto fetch = [&](int base) {
    const int cnt = min(OMS_CH, n - base);
#pragma unroll
    for (int it = 0; it < NQ; ++it) {
      const int idx = tid + 256 * it, tt = idx / DP, r = idx % DP;
      rq[it] = rk[it] = 0.f;
      if (tt < cnt && r < dim) {
        rq[it] = T::to_f32(q[(t0 + base + tt) * q_stride + hq * dim + r]);
        rk[it] = T::to_f32(k[(t0 + base + tt) * k_stride + hq * dim + r]);
      }
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = tid + 256 * it, tt = idx / TW, cc = idx % TW;
      rv[it] = (tt < cnt && c0 + cc < vdim) ? T::to_f32(v[(t0 + base + tt) * v_stride + h * vdim + c0 + cc]) : 0.f;
    }
    if (MODE == 1 && tid < cnt) {
      rgi = T::to_f32(gate_i[(t0 + base + tid) * gate_stride + h]);
      rgf = T::to_f32(gate_f[(t0 + base + tid) * gate_stride + h]);
    }
    if (MODE == 2 && tid < cnt) rgi = T::to_f32(gate_i[(t0 + base + tid) * gate_stride + h]);
  };
  fetch(0);
  for (int base = 0; base < n; base += OMS_CH) {
    const int cnt = min(OMS_CH, n - base);
    __syncthreads();                                        // the previous stage is consumed
#pragma unroll
    for (int it = 0; it < NQ; ++it) {
      const int idx = tid + 256 * it, tt = idx / DP, r = idx % DP;
      if (tt < OMS_CH) {
        qs[tt][r] = MODE == 0 ? silu_f(rq[it]) : MODE == 1 ? rq[it] * q_scale : rq[it];
        ks[tt][r] = MODE == 0 ? silu_f(rk[it]) : rk[it];
      }
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = tid + 256 * it;
      if (idx < OMS_CH * TW) vs[idx / TW][idx % TW] = MODE == 0 ? silu_f(rv[it]) : rv[it];
    }
    if (MODE == 2 && tid < cnt) {
      const float dt = softplus_f(rgi + dtb);
      a_s[tid] = expf(neg_rate * dt);
      b_s[tid] = dt;
    }
    if (MODE == 1 && tid < 64) {
      float gi = 0.f, gf = 0.f;
      if (tid < cnt) {
        gi = gate_cap * tanhf(rgi / gate_cap);
        gf = log_sigmoid_f(gate_cap * tanhf(rgf / gate_cap));
      }
      float m_prev_mine = 0.f, m_mine = 0.f;
      for (int tt = 0; tt < cnt; ++tt) {
        const float f = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gf), tt));
        const float ig = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gi), tt));
        const float m_new = fmaxf(f + m, ig);
        if (tid == tt) {
          m_prev_mine = m;
          m_mine = m_new;
        }
        m = m_new;
      }
      if (tid < cnt) {
        a_s[tid] = expf(gf + m_prev_mine - m_mine);
        b_s[tid] = expf(gi - m_mine);
        em_s[tid] = expf(-m_mine);
      }
    }
    __syncthreads();
    if (base + OMS_CH < n) fetch(base + OMS_CH);
#pragma unroll 4
    for (int tt = 0; tt < cnt; ++tt) {
      const float a = MODE != 0 ? a_s[tt] : dec;
      const float b = MODE != 0 ? b_s[tt] : 1.0f;
      const float vv = vs[tt][c] * b;
      float part[4] = {0.f, 0.f, 0.f, 0.f}, npart[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i4 = 0; i4 < DPT; i4 += 4) {
        const f32x4 kk = *reinterpret_cast<const f32x4*>(&ks[tt][sl * DPT + i4]);
        const f32x4 qq = *reinterpret_cast<const f32x4*>(&qs[tt][sl * DPT + i4]);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          S[i4 + u] = a * S[i4 + u] + kk[u] * vv;
          part[u] += S[i4 + u] * qq[u];
          if (MODE == 1) {
            nv[i4 + u] = a * nv[i4 + u] + b * kk[u];
            npart[u] += nv[i4 + u] * qq[u];
          }
        }
      }
      float po = (part[0] + part[1]) + (part[2] + part[3]);
      po = group_sum<SLOG>(po);
      if (MODE == 1) {
        float pn = (npart[0] + npart[1]) + (npart[2] + npart[3]);
        pn = group_sum<SLOG>(pn);
        po = po / (fmaxf(fabsf(pn), em_s[tt]) + 1e-6f);
      }
      if (MODE == 2) po += skip_h * vs[tt][c];
      if (sl == 0 && col < vdim) out[(t0 + base + tt) * ((int64_t)heads * vdim) + h * vdim + col] = po;
    }
  }
#pragma unroll
  for (int i = 0; i < DPT; ++i) {
    const int r = sl * DPT + i;
    if (r < dim && col < vdim) sbase[(int64_t)r * vdim + col] = S[i];
    if (MODE == 1 && c == 0 && r < dim)
      for (int cp = 0; cp < TW / 16 && copy0 + cp < ncopy; ++cp) nbase[(int64_t)cp * dim + r] = nv[i];
  }
  if (MODE == 1 && tid == 0)
    for (int cp = 0; cp < TW / 16 && copy0 + cp < ncopy; ++cp) mptr[cp] = m;
}

// The same for short segments -- decoded tokens, one per request -- where the state's way through memory and back is the work: a thread
// owns 4 neighbouring columns of NI rows, so the state comes in 16-byte pieces, 256 contiguous bytes a row and workgroup, all of them
// in flight together with the first tokens' numbers; a token's partial sums meet in LDS once a stage, not once a token.
// The split above with 4 lanes a column (4-byte pieces, 64 contiguous bytes, 160 to 210 registers: 2 or 3 waves a SIMD) took, in us against
// here: single tokens of 32 sequences, decay 16 heads of 64 x 128 10.7 / 7.8, mLSTM 8 of 128 x 256 39.8 / 15.5 (4.3 TB/s), state space 128 of
// 128 x 64 79.8 / 46.3 (5.8 TB/s); of one, 6.4 / 4.4 and 9.5 / 5.9; four segments of 8 tokens, mLSTM 22.4 / 11.3; three of 31, decay 17.3 / 14.0.
template <typename T, int MODE, int NI>
__global__ __launch_bounds__(256, NI <= 8 ? 4 : 2) void outer_memory_rows_kernel(
    float* __restrict__ out, const typename T::storage* __restrict__ q, int64_t q_stride,
    const typename T::storage* __restrict__ k, int64_t k_stride, const typename T::storage* __restrict__ v, int64_t v_stride,
    const typename T::storage* __restrict__ gate_i, const typename T::storage* __restrict__ gate_f, int64_t gate_stride,
    float* __restrict__ state_s, float* __restrict__ state_n, float* __restrict__ state_m,
    const int32_t* __restrict__ slot_of_seq, int num_slots, const int32_t* __restrict__ q_start,
    const int32_t* __restrict__ q_len, const int32_t* __restrict__ ctx_len, int below, int heads, int dim, int vdim,
    const float* __restrict__ decay, float q_scale, float gate_cap, int qk_heads, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, const float* __restrict__ skip) {
  constexpr int TW = 64;               // value columns per workgroup
  constexpr int DP = 16 * NI;          // rows of the state, padded
  __shared__ __attribute__((aligned(16))) float qs[OMR_CH][DP];
  __shared__ __attribute__((aligned(16))) float ks[OMR_CH][DP];
  __shared__ __attribute__((aligned(16))) float vs[OMR_CH][TW];
  __shared__ float a_s[OMR_CH], b_s[OMR_CH], em_s[OMR_CH];
  __shared__ __attribute__((aligned(16))) float po_s[OMR_CH][4][TW];      // [token][wave]: S^T q of the wave's rows
  __shared__ float pn_s[OMR_CH][4];
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * TW;
  const int ncopy = (vdim + 15) >> 4, copy0 = c0 >> 4;          // n and m are kept once per 16 value columns
  const int tid = threadIdx.x, wave = tid >> 6, cg = tid & 15, rr = tid >> 4, col = c0 + 4 * cg;
  const int hq = MODE == 2 ? h / (heads / qk_heads) : h;    // head of q and k
  const int n = q_len[s];
  const int slot = slot_of_seq[s];
  if (n <= 0 || n >= below || slot < 0 || slot >= num_slots) return;
  const int64_t t0 = q_start[s];
  const bool fresh = ctx_len[s] == 0;
  f32x4 S[NI];
  float nr = 0.f;                                           // the normaliser's row tid
  float m = 0.f;                                            // wave 0 only (uniform)
  float* sbase = state_s + ((int64_t)slot * heads + h) * dim * (int64_t)vdim;
  float* nbase = MODE == 1 ? state_n + (((int64_t)slot * heads + h) * ncopy + copy0) * dim : nullptr;
  float* mptr = MODE == 1 ? state_m + ((int64_t)slot * heads + h) * ncopy + copy0 : nullptr;
  const bool in = col < vdim;                               // (vdim is a multiple of 4)
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = rr * NI + i;
    S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!fresh && in && r < dim) S[i] = *reinterpret_cast<const f32x4*>(sbase + (int64_t)r * vdim + col);
  }
  if (MODE == 1 && !fresh && tid < dim) nr = nbase[tid];
  if (MODE == 1 && !fresh) m = *mptr;
  const float dec = MODE == 0 ? decay[h] : 0.f;
  const float neg_rate = MODE == 2 ? -expf(a_log[h]) : 0.f, dtb = MODE == 2 ? dt_bias[h] : 0.f, skip_h = MODE == 2 ? skip[h] : 0.f;

  // raw q / k / v (and gates) of the next stage travel in registers while the current stage is scanned
  constexpr int NQ = (OMR_CH * DP + 255) / 256, NV = (OMR_CH * TW + 255) / 256;
  float rq[NQ], rk[NQ], rv[NV], rgi = 0.f, rgf = 0.f;
  auto fetch = [&](int base) {
    const int cnt = min(OMR_CH, n - base);
#pragma unroll
    for (int it = 0; it < NQ; ++it) {
      const int idx = tid + 256 * it, tt = idx / DP, r = idx % DP;
      rq[it] = rk[it] = 0.f;
      if (tt < cnt && r < dim) {
        rq[it] = T::to_f32(q[(t0 + base + tt) * q_stride + hq * dim + r]);
        rk[it] = T::to_f32(k[(t0 + base + tt) * k_stride + hq * dim + r]);
      }
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = tid + 256 * it, tt = idx / TW, cc = idx % TW;
      rv[it] = (tt < cnt && c0 + cc < vdim) ? T::to_f32(v[(t0 + base + tt) * v_stride + h * vdim + c0 + cc]) : 0.f;
    }
    if (MODE == 1 && tid < cnt) {
      rgi = T::to_f32(gate_i[(t0 + base + tid) * gate_stride + h]);
      rgf = T::to_f32(gate_f[(t0 + base + tid) * gate_stride + h]);
    }
    if (MODE == 2 && tid < cnt) rgi = T::to_f32(gate_i[(t0 + base + tid) * gate_stride + h]);
  };
  fetch(0);
  for (int base = 0; base < n; base += OMR_CH) {
    const int cnt = min(OMR_CH, n - base);
    __syncthreads();                                        // the previous stage is consumed
#pragma unroll
    for (int it = 0; it < NQ; ++it) {
      const int idx = tid + 256 * it, tt = idx / DP, r = idx % DP;
      if (tt < OMR_CH) {
        qs[tt][r] = MODE == 0 ? silu_f(rq[it]) : MODE == 1 ? rq[it] * q_scale : rq[it];
        ks[tt][r] = MODE == 0 ? silu_f(rk[it]) : rk[it];
      }
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = tid + 256 * it;
      if (idx < OMR_CH * TW) vs[idx / TW][idx % TW] = MODE == 0 ? silu_f(rv[it]) : rv[it];
    }
    if (MODE == 2 && tid < cnt) {
      const float dt = softplus_f(rgi + dtb);
      a_s[tid] = expf(neg_rate * dt);
      b_s[tid] = dt;
    }
    if (MODE == 1 && tid < 64) {
      float gi = 0.f, gf = 0.f;
      if (tid < cnt) {
        gi = gate_cap * tanhf(rgi / gate_cap);
        gf = log_sigmoid_f(gate_cap * tanhf(rgf / gate_cap));
      }
      float m_prev_mine = 0.f, m_mine = 0.f;
      for (int tt = 0; tt < cnt; ++tt) {
        const float f = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gf), tt));
        const float ig = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gi), tt));
        const float m_new = fmaxf(f + m, ig);
        if (tid == tt) {
          m_prev_mine = m;
          m_mine = m_new;
        }
        m = m_new;
      }
      if (tid < cnt) {
        a_s[tid] = expf(gf + m_prev_mine - m_mine);
        b_s[tid] = expf(gi - m_mine);
        em_s[tid] = expf(-m_mine);
      }
    }
    __syncthreads();
    if (base + OMR_CH < n) fetch(base + OMR_CH);
    for (int tt = 0; tt < cnt; ++tt) {
      const float a = MODE != 0 ? a_s[tt] : dec;
      const float b = MODE != 0 ? b_s[tt] : 1.0f;
      const f32x4 v4 = *reinterpret_cast<const f32x4*>(&vs[tt][4 * cg]);
      float part[4] = {0.f, 0.f, 0.f, 0.f}, x[NI];
      lds_row<NI>(&ks[tt][rr * NI], x);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int u = 0; u < 4; ++u) S[i][u] = a * S[i][u] + x[i] * (v4[u] * b);
      lds_row<NI>(&qs[tt][rr * NI], x);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int u = 0; u < 4; ++u) part[u] += S[i][u] * x[i];
      po_s[tt][wave][4 * cg + scatter_index4(tid)] = scatter_sum4(part);
      if (MODE == 1) {
        float pn = 0.f;
        if (tid < DP) {
          nr = a * nr + b * ks[tt][tid];
          pn = nr * qs[tt][tid];
        }
        pn = wave_sum(pn);
        if ((tid & 63) == 0) pn_s[tt][wave] = pn;
      }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int tt = (tid + 256 * it) / TW, c = tid % TW;
      if (tt >= cnt || c0 + c >= vdim) continue;
      float po = (po_s[tt][0][c] + po_s[tt][1][c]) + (po_s[tt][2][c] + po_s[tt][3][c]);
      if (MODE == 1) {
        const float pn = (pn_s[tt][0] + pn_s[tt][1]) + (pn_s[tt][2] + pn_s[tt][3]);
        po = po / (fmaxf(fabsf(pn), em_s[tt]) + 1e-6f);
      }
      if (MODE == 2) po += skip_h * vs[tt][c];
      out[(t0 + base + tt) * ((int64_t)heads * vdim) + h * vdim + c0 + c] = po;
    }
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = rr * NI + i;
    if (in && r < dim) *reinterpret_cast<f32x4*>(sbase + (int64_t)r * vdim + col) = S[i];
  }
  if (MODE == 1 && tid < dim)
    for (int cp = 0; cp < TW / 16 && copy0 + cp < ncopy; ++cp) nbase[(int64_t)cp * dim + tid] = nr;
  if (MODE == 1 && tid == 0)
    for (int cp = 0; cp < TW / 16 && copy0 + cp < ncopy; ++cp) mptr[cp] = m;
}

int outer_memory_check(const OuterMemory& p) {
  APHRO_CHECK(p.out && p.q && p.k && p.v && p.state_s && p.slot_of_seq && p.q_start && p.q_len && p.ctx_len, "outer_memory_scan: null argument");
  APHRO_CHECK(p.mode >= 0 && p.mode <= 2, "outer_memory_scan: mode %d", p.mode);
  APHRO_CHECK(p.qk_heads > 0 && p.heads % p.qk_heads == 0 && (p.mode == 2 || p.qk_heads == p.heads), "outer_memory_scan: %d heads over %d query/key heads", p.heads, p.qk_heads);
  APHRO_CHECK(p.mode == 0 ? p.decay != nullptr : p.mode == 2 ? (p.gate_i && p.a_log && p.dt_bias && p.skip && p.gate_stride >= p.heads) : (p.gate_i && p.gate_f && p.state_n && p.state_m && p.gate_cap > 0.f && p.gate_stride >= p.heads),
              "outer_memory_scan: mode %d lacks its gate arguments", p.mode);
  APHRO_CHECK(p.heads > 0 && p.heads <= 65535 && p.dim > 0 && p.dim <= 256 && p.vdim > 0 && p.vdim <= 64 * 65535 && p.num_slots > 0 && p.num_seqs > 0,
              "outer_memory_scan: heads %d dim %d (<= 256) vdim %d", p.heads, p.dim, p.vdim);
  APHRO_CHECK(p.q_stride >= (int64_t)p.qk_heads * p.dim && p.k_stride >= (int64_t)p.qk_heads * p.dim && p.v_stride >= (int64_t)p.heads * p.vdim,
              "outer_memory_scan: row strides smaller than the rows");
  return APHRO_OK;
}

// Prompt portions, and value heads of no multiple of 4: 16 lanes per value column (16 columns per workgroup), so that a long sequential
// scan spreads over many waves with little work per token and lane.  Short segments: outer_memory_rows_kernel.
int outer_memory_scan_launch(const OuterMemory& p, int below, bool wide) {
  wide = wide || p.vdim % 4 != 0 || ((uintptr_t)p.state_s & 15) != 0;
  const int tw = wide ? 16 : 64;
  const dim3 grid((unsigned)p.num_seqs, (unsigned)p.heads, (unsigned)((p.vdim + tw - 1) / tw));
#define OMS_LAUNCH(KERNEL, ...)                                                                                             \
  hipLaunchKernelGGL((KERNEL<T, __VA_ARGS__>), grid, dim3(256), 0, p.stream, p.out, (const S*)p.q,                               \
                     p.q_stride, (const S*)p.k, p.k_stride, (const S*)p.v, p.v_stride, (const S*)p.gate_i, (const S*)p.gate_f, p.gate_stride, \
                     p.state_s, p.state_n, p.state_m, p.slot_of_seq, p.num_slots, p.q_start, p.q_len, p.ctx_len, below, p.heads, p.dim, p.vdim, \
                     p.decay, p.q_scale, p.gate_cap, p.qk_heads, p.a_log, p.dt_bias, p.skip)
#define OMS_BY_DIM(MODE)                                                       \
  do {                                                                         \
    if (wide) {                                                                \
      if (p.dim <= 64) OMS_LAUNCH(outer_memory_scan_kernel, MODE, 4);          \
      else if (p.dim <= 128) OMS_LAUNCH(outer_memory_scan_kernel, MODE, 8);    \
      else OMS_LAUNCH(outer_memory_scan_kernel, MODE, 16);                     \
    } else if (p.dim <= 32) OMS_LAUNCH(outer_memory_rows_kernel, MODE, 2);     \
    else if (p.dim <= 64) OMS_LAUNCH(outer_memory_rows_kernel, MODE, 4);       \
    else if (p.dim <= 96) OMS_LAUNCH(outer_memory_rows_kernel, MODE, 6);       \
    else if (p.dim <= 128) OMS_LAUNCH(outer_memory_rows_kernel, MODE, 8);      \
    else OMS_LAUNCH(outer_memory_rows_kernel, MODE, 16);                       \
  } while (0)
  MIX_DISPATCH_DTYPE(p.dtype, {
    typedef typename T::storage S;
    if (p.mode == 0) OMS_BY_DIM(0);
    else if (p.mode == 1) OMS_BY_DIM(1);
    else OMS_BY_DIM(2);
  });
#undef OMS_BY_DIM
#undef OMS_LAUNCH
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

}  // namespace aphro

using namespace aphro;

extern "C" int aphro_outer_memory_scan(float* out, const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                                       const void* v, int64_t v_stride, const void* gate_i, const void* gate_f,
                                       int64_t gate_stride, float* state_s, float* state_n, float* state_m,
                                       const int32_t* slot_of_seq, int num_slots, const int32_t* q_start, const int32_t* q_len,
                                       const int32_t* ctx_len, int num_seqs, int64_t num_tokens, int heads, int dim, int vdim,
                                       int mode, const float* decay, float q_scale, float gate_cap, int qk_heads,
                                       const float* a_log, const float* dt_bias, const float* skip, int max_q_len, int dtype,
                                       void* stream) {
  if (num_tokens == 0 || num_seqs == 0) return APHRO_OK;
  const OuterMemory p = {out, q, k, v, gate_i, gate_f, q_stride, k_stride, v_stride, gate_stride, state_s, state_n, state_m, slot_of_seq,
                         num_slots, q_start, q_len, ctx_len, num_seqs, num_tokens, heads, dim, vdim, mode, decay, q_scale, gate_cap, qk_heads,
                         a_log, dt_bias, skip, max_q_len, dtype, (hipStream_t)stream};
  const int rc = outer_memory_check(p);
  return rc != APHRO_OK ? rc : outer_memory_scan_launch(p, 0x7fffffff, max_q_len >= 32);
}
