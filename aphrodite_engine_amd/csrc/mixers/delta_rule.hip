// Gated delta rule: per (request slot, head) a matrix state S [dim, vdim] that forgets, corrects what it holds under the key
// towards the new value, and is read AFTER the write:
//     S <- g_t S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
// (CHANNEL form: g_t is a vector over the key dimension, one decay per row of S: g_t[r] = exp(-exp(A_log) softplus(a_t[r] + dt_bias[r])))
// with k and q made unit vectors per head (x / sqrt(sum x^2 + norm_eps); q times q_scale), beta_t = sigmoid(b_t) and
// g_t = exp(-exp(A_log) * softplus(a_t + dt_bias)) per head.  State, the unit norms, beta, g and every sum are fp32 whatever
// the activations' storage.  Query / key head of value head h: h / (heads / kv_heads).
//
// With r_k = S_old^T k and r_q = S_old^T q (ONE pass over the state, two dot products per column):
//     u = beta (v - g r_k),   S_new = g S_old + k u^T,   o = g r_q + (k . q) u
// so a token costs one read pass and one update pass over the registers that hold the state.  In the CHANNEL form the read pass
// decays the rows as it goes (S <- g S, r_k = S^T k, r_q = S^T q) and the update adds k u^T: the same number of operations.
//
// Work split (that of the gated outer-product memories): a workgroup of 256 threads owns 16 value
// columns of one (segment, head); thread = (column, slice of the key dimension); 16 tokens at a time are staged in LDS, sixteen
// lanes per token, which also make the token's unit norms, k . q, beta and g; the next 16 tokens' raw values are in flight in
// registers meanwhile.  The per-token partial dot products are folded over the slices with DPP moves.
//
// gated_head_rms_norm: out = o / rms(o over the head's vdim) * weight[vdim] * act(gate), one wave per (token, head).
#include "delta_rule.h"

namespace aphro {

constexpr int GDR_CH = 16;

template <typename T, int DPT, bool CHANNEL>
__global__ __launch_bounds__(256) void gated_delta_scan_kernel(
    float* __restrict__ out, const typename T::storage* __restrict__ q, int64_t q_stride,
    const typename T::storage* __restrict__ k, int64_t k_stride, const typename T::storage* __restrict__ v, int64_t v_stride,
    const typename T::storage* __restrict__ b, int64_t b_stride, const typename T::storage* __restrict__ a, int64_t a_stride,
    const float* __restrict__ a_log, const float* __restrict__ dt_bias, float* __restrict__ state,
    const int32_t* __restrict__ slot_of_seq, int num_slots, const int32_t* __restrict__ q_start,
    const int32_t* __restrict__ q_len, const int32_t* __restrict__ ctx_len, int below, int heads, int kv_heads, int dim, int vdim,
    float q_scale, float norm_eps) {
  constexpr int SLOG = 4, NS = 1 << SLOG;     // slices of the key dimension = lanes that share a column
  constexpr int TW = 256 >> SLOG;      // value columns per workgroup
  constexpr int DP = NS * DPT;         // key dimension, padded
  constexpr int NQ = (DP + 15) / 16;   // numbers of q (and of k) a staging lane holds: sixteen lanes per token
  constexpr int NV = (GDR_CH * TW + 255) / 256;
  __shared__ __attribute__((aligned(16))) float qs[GDR_CH][DP];
  __shared__ __attribute__((aligned(16))) float ks[GDR_CH][DP];
  __shared__ __attribute__((aligned(16))) float gs[CHANNEL ? GDR_CH : 1][CHANNEL ? DP : 1];
  __shared__ float vs[GDR_CH][TW];
  __shared__ float g_s[GDR_CH], b_s[GDR_CH], kq_s[GDR_CH];
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * TW;
  const int hk = h / (heads / kv_heads);
  const int tid = threadIdx.x, c = tid >> SLOG, sl = tid & (NS - 1), col = c0 + c;
  const int n = q_len[s];
  const int slot = slot_of_seq[s];
  if (n <= 0 || n >= below || slot < 0 || slot >= num_slots) return;
  const int64_t t0 = q_start[s];
  const bool fresh = ctx_len[s] == 0;
  float S[DPT];
  float* sbase = state + ((int64_t)slot * heads + h) * dim * (int64_t)vdim;
#pragma unroll
  for (int i = 0; i < DPT; ++i) {
    const int r = sl * DPT + i;
    S[i] = (!fresh && r < dim && col < vdim) ? sbase[(int64_t)r * vdim + col] : 0.f;
  }
  const float neg_rate = -expf(a_log[h]), dtb = CHANNEL ? 0.f : dt_bias[h];
  const int stok = tid >> 4, sln = tid & 15;               // staging: token of the stage, lane within the token

  float rq[NQ], rk[NQ], rv[NV], rb = 0.f, ra = 0.f;
  float rg[CHANNEL ? NQ : 1], dtc[CHANNEL ? NQ : 1];       // per-channel decay: raw values of the next stage, the lane's dt_bias
  if constexpr (CHANNEL) {
#pragma unroll
    for (int it = 0; it < NQ; ++it) {
      const int r = sln + 16 * it;
      dtc[it] = r < dim ? dt_bias[h * dim + r] : 0.f;
    }
  }
  auto fetch = [&](int base) {
    const int cnt = min(GDR_CH, n - base);
#pragma unroll
    for (int it = 0; it < NQ; ++it) {
      const int r = sln + 16 * it;
      rq[it] = rk[it] = 0.f;
      if (stok < cnt && r < dim) {
        rq[it] = T::to_f32(q[(t0 + base + stok) * q_stride + hk * dim + r]);
        rk[it] = T::to_f32(k[(t0 + base + stok) * k_stride + hk * dim + r]);
        if constexpr (CHANNEL) rg[it] = T::to_f32(a[(t0 + base + stok) * a_stride + (int64_t)h * dim + r]);
      } else if constexpr (CHANNEL) {
        rg[it] = 0.f;
      }
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = tid + 256 * it, tt = idx / TW, cc = idx % TW;
      rv[it] = (tt < cnt && c0 + cc < vdim) ? T::to_f32(v[(t0 + base + tt) * v_stride + h * vdim + c0 + cc]) : 0.f;
    }
    if (sln == 0 && stok < cnt) {
      rb = T::to_f32(b[(t0 + base + stok) * b_stride + h]);
      if constexpr (!CHANNEL) ra = T::to_f32(a[(t0 + base + stok) * a_stride + h]);
    }
  };
  fetch(0);
  for (int base = 0; base < n; base += GDR_CH) {
    const int cnt = min(GDR_CH, n - base);
    __syncthreads();                                        // the previous stage is consumed
    {
      float sq = 0.f, sk = 0.f;
#pragma unroll
      for (int it = 0; it < NQ; ++it) {
        sq += rq[it] * rq[it];
        sk += rk[it] * rk[it];
      }
      sq = group_sum<4>(sq);
      sk = group_sum<4>(sk);
      const float fq = q_scale / sqrtf(sq + norm_eps), fk = 1.0f / sqrtf(sk + norm_eps);
      float kq = 0.f;
#pragma unroll
      for (int it = 0; it < NQ; ++it) {
        const int r = sln + 16 * it;
        const float qv = rq[it] * fq, kv = rk[it] * fk;
        kq += qv * kv;
        if (r < DP) {
          qs[stok][r] = qv;
          ks[stok][r] = kv;
          if constexpr (CHANNEL) gs[stok][r] = expf(neg_rate * softplus_f(rg[it] + dtc[it]));
        }
      }
      kq = group_sum<4>(kq);
      if (sln == 0) {
        kq_s[stok] = kq;
        b_s[stok] = sigmoid_f(rb);
        if constexpr (!CHANNEL) g_s[stok] = expf(neg_rate * softplus_f(ra + dtb));
      }
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = tid + 256 * it;
      if (idx < GDR_CH * TW) vs[idx / TW][idx % TW] = rv[it];
    }
    __syncthreads();
    if (base + GDR_CH < n) fetch(base + GDR_CH);
#pragma unroll 2
    for (int tt = 0; tt < cnt; ++tt) {
      const float g = CHANNEL ? 1.f : g_s[tt], beta = b_s[tt], kq = kq_s[tt];
      float pk[4] = {0.f, 0.f, 0.f, 0.f}, pq[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i4 = 0; i4 < DPT; i4 += 4) {
        const f32x4 kk = *reinterpret_cast<const f32x4*>(&ks[tt][sl * DPT + i4]);
        const f32x4 qq = *reinterpret_cast<const f32x4*>(&qs[tt][sl * DPT + i4]);
        if constexpr (CHANNEL) {
          const f32x4 gg = *reinterpret_cast<const f32x4*>(&gs[tt][sl * DPT + i4]);
#pragma unroll
          for (int e = 0; e < 4; ++e) S[i4 + e] *= gg[e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pk[e] += S[i4 + e] * kk[e];
          pq[e] += S[i4 + e] * qq[e];
        }
      }
      const float rk_ = group_sum<SLOG>((pk[0] + pk[1]) + (pk[2] + pk[3]));
      const float rq_ = group_sum<SLOG>((pq[0] + pq[1]) + (pq[2] + pq[3]));
      const float u = beta * (vs[tt][c] - g * rk_);
#pragma unroll
      for (int i4 = 0; i4 < DPT; i4 += 4) {
        const f32x4 kk = *reinterpret_cast<const f32x4*>(&ks[tt][sl * DPT + i4]);
#pragma unroll
        for (int e = 0; e < 4; ++e) S[i4 + e] = (CHANNEL ? S[i4 + e] : g * S[i4 + e]) + kk[e] * u;
      }
      if (sl == 0 && col < vdim) out[(t0 + base + tt) * ((int64_t)heads * vdim) + h * vdim + col] = g * rq_ + kq * u;
    }
  }
#pragma unroll
  for (int i = 0; i < DPT; ++i) {
    const int r = sl * DPT + i;
    if (r < dim && col < vdim) sbase[(int64_t)r * vdim + col] = S[i];
  }
}

// The same for short segments -- decoded tokens, one per request -- where the state's way through memory and back is the work: a thread
// owns 4 neighbouring columns of NI rows, so the state comes in 16-byte pieces, 256 contiguous bytes a row and workgroup, all of them
// in flight together with the first tokens' numbers; a token's two dot products meet in LDS behind one barrier.
// The split above with 4 lanes a column (4-byte pieces, 64 contiguous bytes, up to 170 registers) took, in us against
// here: single tokens of 32 sequences, 32 heads of 128 x 128, a decay per channel 49.6 / 32.6 (4.1 TB/s), per head 49.8 / 28.0; of 24, 16 heads
// 22.4 / 12.6; of one 10.3 / 6.9; three of 8 tokens 15.3 / 11.9, four of 31 31.1 / 32.2.
template <typename T, int NI, bool CHANNEL>
__global__ __launch_bounds__(256, NI <= 8 ? 4 : 2) void gated_delta_rows_kernel(
    float* __restrict__ out, const typename T::storage* __restrict__ q, int64_t q_stride,
    const typename T::storage* __restrict__ k, int64_t k_stride, const typename T::storage* __restrict__ v, int64_t v_stride,
    const typename T::storage* __restrict__ b, int64_t b_stride, const typename T::storage* __restrict__ a, int64_t a_stride,
    const float* __restrict__ a_log, const float* __restrict__ dt_bias, float* __restrict__ state,
    const int32_t* __restrict__ slot_of_seq, int num_slots, const int32_t* __restrict__ q_start,
    const int32_t* __restrict__ q_len, const int32_t* __restrict__ ctx_len, int below, int heads, int kv_heads, int dim, int vdim,
    float q_scale, float norm_eps) {
  constexpr int CH = 8, LPT = 32;      // tokens of a stage, staging lanes a token
  constexpr int TW = 64;               // value columns per workgroup
  constexpr int DP = 16 * NI;          // key dimension, padded
  constexpr int NQ = DP / LPT;         // numbers of q (and of k) a staging lane holds
  constexpr int NV = CH * TW / 256;
  __shared__ __attribute__((aligned(16))) float qs[CH][DP];
  __shared__ __attribute__((aligned(16))) float ks[CH][DP];
  __shared__ __attribute__((aligned(16))) float gs[CHANNEL ? CH : 1][CHANNEL ? DP : 1];
  __shared__ __attribute__((aligned(16))) float vs[CH][TW];
  __shared__ __attribute__((aligned(16))) float dots[2][4][2][TW];      // [token's parity][wave][S^T k, S^T q]
  __shared__ float g_s[CH], b_s[CH], kq_s[CH];
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * TW;
  const int hk = h / (heads / kv_heads);
  const int tid = threadIdx.x, wave = tid >> 6, cg = tid & 15, rr = tid >> 4, col = c0 + 4 * cg;
  const int n = q_len[s];
  const int slot = slot_of_seq[s];
  if (n <= 0 || n >= below || slot < 0 || slot >= num_slots) return;
  const int64_t t0 = q_start[s];
  const bool fresh = ctx_len[s] == 0, in = col < vdim;       // (vdim is a multiple of 4)
  f32x4 S[NI];
  float* sbase = state + ((int64_t)slot * heads + h) * dim * (int64_t)vdim;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = rr * NI + i;
    S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!fresh && in && r < dim) S[i] = *reinterpret_cast<const f32x4*>(sbase + (int64_t)r * vdim + col);
  }
  const float neg_rate = -expf(a_log[h]), dtb = CHANNEL ? 0.f : dt_bias[h];
  const int stok = tid / LPT, sln = tid % LPT;               // staging: token of the stage, lane within the token
  float rq[NQ], rk[NQ], rv[NV], rb = 0.f, ra = 0.f;
  float rg[CHANNEL ? NQ : 1], dtc[CHANNEL ? NQ : 1];
  if constexpr (CHANNEL) {
#pragma unroll
    for (int it = 0; it < NQ; ++it) {
      const int r = sln + LPT * it;
      dtc[it] = r < dim ? dt_bias[h * dim + r] : 0.f;
    }
  }
  auto fetch = [&](int base) {
    const int cnt = min(CH, n - base);
#pragma unroll
    for (int it = 0; it < NQ; ++it) {
      const int r = sln + LPT * it;
      rq[it] = rk[it] = 0.f;
      if (stok < cnt && r < dim) {
        rq[it] = T::to_f32(q[(t0 + base + stok) * q_stride + hk * dim + r]);
        rk[it] = T::to_f32(k[(t0 + base + stok) * k_stride + hk * dim + r]);
        if constexpr (CHANNEL) rg[it] = T::to_f32(a[(t0 + base + stok) * a_stride + (int64_t)h * dim + r]);
      } else if constexpr (CHANNEL) {
        rg[it] = 0.f;
      }
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = tid + 256 * it, tt = idx / TW, cc = idx % TW;
      rv[it] = (tt < cnt && c0 + cc < vdim) ? T::to_f32(v[(t0 + base + tt) * v_stride + h * vdim + c0 + cc]) : 0.f;
    }
    if (sln == 0 && stok < cnt) {
      rb = T::to_f32(b[(t0 + base + stok) * b_stride + h]);
      if constexpr (!CHANNEL) ra = T::to_f32(a[(t0 + base + stok) * a_stride + h]);
    }
  };
  fetch(0);
  for (int base = 0; base < n; base += CH) {
    const int cnt = min(CH, n - base);
    __syncthreads();                                        // the previous stage is consumed
    {
      float sq = 0.f, sk = 0.f;
#pragma unroll
      for (int it = 0; it < NQ; ++it) {
        sq += rq[it] * rq[it];
        sk += rk[it] * rk[it];
      }
      sq = group_sum<5>(sq);
      sk = group_sum<5>(sk);
      const float fq = q_scale / sqrtf(sq + norm_eps), fk = 1.0f / sqrtf(sk + norm_eps);
      float kq = 0.f;
#pragma unroll
      for (int it = 0; it < NQ; ++it) {
        const int r = sln + LPT * it;
        const float qv = rq[it] * fq, kv = rk[it] * fk;
        kq += qv * kv;
        qs[stok][r] = qv;
        ks[stok][r] = kv;
        if constexpr (CHANNEL) gs[stok][r] = expf(neg_rate * softplus_f(rg[it] + dtc[it]));
      }
      kq = group_sum<5>(kq);
      if (sln == 0) {
        kq_s[stok] = kq;
        b_s[stok] = sigmoid_f(rb);
        if constexpr (!CHANNEL) g_s[stok] = expf(neg_rate * softplus_f(ra + dtb));
      }
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = tid + 256 * it;
      vs[idx / TW][idx % TW] = rv[it];
    }
    __syncthreads();
    if (base + CH < n) fetch(base + CH);
    for (int tt = 0; tt < cnt; ++tt) {
      const float g = CHANNEL ? 1.f : g_s[tt], beta = b_s[tt], kq = kq_s[tt];
      float pk[4] = {0.f, 0.f, 0.f, 0.f}, pq[4] = {0.f, 0.f, 0.f, 0.f};
      float kk[NI], qq[NI];
      lds_row<NI>(&ks[tt][rr * NI], kk);
      lds_row<NI>(&qs[tt][rr * NI], qq);
      if constexpr (CHANNEL) {
        float gg[NI];
        lds_row<NI>(&gs[tt][rr * NI], gg);
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) S[i][e] *= gg[i];
      }
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pk[e] += S[i][e] * kk[i];
          pq[e] += S[i][e] * qq[i];
        }
      float (*d)[2][TW] = dots[tt & 1];                      // the other one may still be read; this one was, before the last barrier
      d[wave][0][4 * cg + scatter_index4(tid)] = scatter_sum4(pk);
      d[wave][1][4 * cg + scatter_index4(tid)] = scatter_sum4(pq);
      __syncthreads();
      f32x4 dk[4], dq[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        dk[w] = *reinterpret_cast<const f32x4*>(&d[w][0][4 * cg]);
        dq[w] = *reinterpret_cast<const f32x4*>(&d[w][1][4 * cg]);
      }
      const f32x4 v4 = *reinterpret_cast<const f32x4*>(&vs[tt][4 * cg]);
      float u[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) u[e] = beta * (v4[e] - g * ((dk[0][e] + dk[1][e]) + (dk[2][e] + dk[3][e])));
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[i][e] = (CHANNEL ? S[i][e] : g * S[i][e]) + kk[i] * u[e];
      if (rr == 0 && in) {
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = g * ((dq[0][e] + dq[1][e]) + (dq[2][e] + dq[3][e])) + kq * u[e];
        *reinterpret_cast<f32x4*>(out + (t0 + base + tt) * ((int64_t)heads * vdim) + h * vdim + col) = o;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = rr * NI + i;
    if (in && r < dim) *reinterpret_cast<f32x4*>(sbase + (int64_t)r * vdim + col) = S[i];
  }
}

// act: 0 sigmoid(gate), 1 silu(gate); gate NULL: none.  weight [vdim] is shared by the heads (NULL: ones).
template <typename T>
__global__ __launch_bounds__(256) void gated_head_rms_norm_kernel(typename T::storage* __restrict__ out, int64_t out_stride,
                                                                  const float* __restrict__ x, const typename T::storage* __restrict__ weight,
                                                                  const typename T::storage* __restrict__ gate, int64_t gate_stride,
                                                                  int64_t num_tokens, int heads, int vdim, float eps, int act) {
  const int lane = threadIdx.x & 63;
  const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= num_tokens * heads) return;
  const int64_t t = unit / heads;
  const int h = (int)(unit - t * heads);
  const float* xr = x + (t * heads + h) * (int64_t)vdim;
  float ss = 0.f;
  for (int i = lane; i < vdim; i += 64) ss += xr[i] * xr[i];
  const float rstd = 1.0f / sqrtf(wave_sum(ss) / (float)vdim + eps);
  for (int i = lane; i < vdim; i += 64) {
    float val = xr[i] * rstd;
    if (weight) val *= T::to_f32(weight[i]);
    if (gate) {
      const float gv = T::to_f32(gate[t * gate_stride + (int64_t)h * vdim + i]);
      val *= act == 1 ? silu_f(gv) : sigmoid_f(gv);
    }
    out[t * out_stride + (int64_t)h * vdim + i] = T::from_f32(val);
  }
}

int gated_delta_check(const GatedDelta& p) {
  APHRO_CHECK(p.out && p.q && p.k && p.v && p.b && p.a && p.a_log && p.dt_bias && p.state && p.slot_of_seq && p.q_start && p.q_len && p.ctx_len,
              "gated_delta_scan: null argument");
  APHRO_CHECK(p.heads > 0 && p.heads <= 65535 && p.kv_heads > 0 && p.heads % p.kv_heads == 0 && p.dim > 0 && p.dim <= 256 && p.vdim > 0 &&
                  p.vdim <= 16 * 65535 && p.num_slots > 0,
              "gated_delta_scan: heads %d over %d key heads, dim %d (<= 256), vdim %d", p.heads, p.kv_heads, p.dim, p.vdim);
  APHRO_CHECK(p.q_stride >= (int64_t)p.kv_heads * p.dim && p.k_stride >= (int64_t)p.kv_heads * p.dim && p.v_stride >= (int64_t)p.heads * p.vdim &&
                  p.b_stride >= p.heads && p.a_stride >= (p.channel_decay ? (int64_t)p.heads * p.dim : (int64_t)p.heads), "gated_delta_scan: row strides smaller than the rows");
  return APHRO_OK;
}

// Prompt portions, and value heads of no multiple of 4, on 16 lanes per value column; short segments on gated_delta_rows_kernel.
int gated_delta_scan_launch(const GatedDelta& p, int below, bool wide) {
  wide = wide || p.vdim % 4 != 0 || (((uintptr_t)p.state | (uintptr_t)p.out) & 15) != 0;
  const int tw = wide ? 16 : 64;
  const dim3 grid((unsigned)p.num_seqs, (unsigned)p.heads, (unsigned)((p.vdim + tw - 1) / tw));
#define GDR_LAUNCH1(KERNEL, N, CHANNEL)                                                                                                \
  hipLaunchKernelGGL((KERNEL<T, N, CHANNEL>), grid, dim3(256), 0, p.stream, p.out, (const S*)p.q, p.q_stride,                          \
                     (const S*)p.k, p.k_stride, (const S*)p.v, p.v_stride, (const S*)p.b, p.b_stride, (const S*)p.a, p.a_stride, p.a_log, p.dt_bias, \
                     p.state, p.slot_of_seq, p.num_slots, p.q_start, p.q_len, p.ctx_len, below, p.heads, p.kv_heads, p.dim, p.vdim, p.q_scale, p.norm_eps)
#define GDR_LAUNCH(KERNEL, N)                             \
  do {                                                    \
    if (p.channel_decay) GDR_LAUNCH1(KERNEL, N, true);    \
    else GDR_LAUNCH1(KERNEL, N, false);                   \
  } while (0)
  MIX_DISPATCH_DTYPE(p.dtype, {
    typedef typename T::storage S;
    if (wide) {
      if (p.dim <= 64) GDR_LAUNCH(gated_delta_scan_kernel, 4);
      else if (p.dim <= 128) GDR_LAUNCH(gated_delta_scan_kernel, 8);
      else GDR_LAUNCH(gated_delta_scan_kernel, 16);
    } else if (p.dim <= 32) GDR_LAUNCH(gated_delta_rows_kernel, 2);
    else if (p.dim <= 64) GDR_LAUNCH(gated_delta_rows_kernel, 4);
    else if (p.dim <= 128) GDR_LAUNCH(gated_delta_rows_kernel, 8);
    else GDR_LAUNCH(gated_delta_rows_kernel, 16);
  });
#undef GDR_LAUNCH
#undef GDR_LAUNCH1
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

}  // namespace aphro

using namespace aphro;

extern "C" int aphro_gated_delta_scan(float* out, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                                      int64_t v_stride, const void* b, int64_t b_stride, const void* a, int64_t a_stride,
                                      const float* a_log, const float* dt_bias, float* state, const int32_t* slot_of_seq,
                                      int num_slots, const int32_t* q_start, const int32_t* q_len, const int32_t* ctx_len,
                                      int num_seqs, int64_t num_tokens, int heads, int kv_heads, int dim, int vdim, int channel_decay,
                                      float q_scale, float norm_eps, int max_q_len, int dtype, void* stream) {
  if (num_tokens == 0 || num_seqs == 0) return APHRO_OK;
  const GatedDelta p = {out, q, k, v, b, a, q_stride, k_stride, v_stride, b_stride, a_stride, a_log, dt_bias, state, slot_of_seq, num_slots,
                        q_start, q_len, ctx_len, num_seqs, num_tokens, heads, kv_heads, dim, vdim, channel_decay, q_scale, norm_eps, dtype,
                        (hipStream_t)stream};
  const int rc = gated_delta_check(p);
  return rc != APHRO_OK ? rc : gated_delta_scan_launch(p, 0x7fffffff, max_q_len >= 32);
}

extern "C" int aphro_gated_head_rms_norm(void* out, int64_t out_stride, const float* x, const void* weight, const void* gate,
                                         int64_t gate_stride, int64_t num_tokens, int heads, int vdim, float eps, int act, int dtype,
                                         void* stream) {
  if (num_tokens == 0) return APHRO_OK;
  APHRO_CHECK(out && x && heads > 0 && vdim > 0 && out_stride >= (int64_t)heads * vdim && (!gate || gate_stride >= (int64_t)heads * vdim) &&
                  (act == 0 || act == 1), "gated_head_rms_norm: bad arguments (%d heads of %d)", heads, vdim);
  if (group_rms_norm_launch(out, out_stride, x, weight, true, gate, gate_stride, num_tokens, heads * vdim, vdim, eps, 1.0f, act, dtype, (hipStream_t)stream)) {
    APHRO_LAUNCH_CHECK();
    return APHRO_OK;
  }
  const int64_t units = num_tokens * heads;
  APHRO_CHECK((units + 3) / 4 <= 0x7fffffff, "gated_head_rms_norm: too many rows");
  MIX_DISPATCH_DTYPE(dtype, {
    typedef typename T::storage S;
    hipLaunchKernelGGL((gated_head_rms_norm_kernel<T>), dim3((unsigned)((units + 3) / 4)), dim3(256), 0, (hipStream_t)stream, (S*)out,
                       out_stride, x, (const S*)weight, (const S*)gate, gate_stride, num_tokens, heads, vdim, eps, act);
  });
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}
