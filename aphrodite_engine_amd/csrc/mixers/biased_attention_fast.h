// bf16 fast paths of the distance-biased attention (same semantics as biased_attention.hip, which stays the fp32 path and
// the path of sizes these do not tile).  EXT (the form DBA_MASKED) adds, at run time: a sliding window or chunks (both give every row an oldest key;
// key tiles older than that are not visited), a tanh soft cap on the scores, a per-head sink in the denominator and an
// elementwise gate.  DBA_GATED is the plain form with the elementwise gate (and none of
// the branches of the masked loop).  Every form is a translation unit of its own.
//
//  * dba_prefill_kernel<DK, DV>: segments of >= DBA_MFMA_MIN_LEN rows.  A workgroup of four waves owns 64 consecutive
//    query rows of one (segment, head), 16 rows per wave, and walks the visible keys 64 at a time: the K rows and V rows of
//    the tile come from the paged cache with 16-byte loads into LDS (K chunk-swizzled, V transposed), together with the 127
//    bias values the tile can need (the table is indexed by distance, and a 64 x 64 tile spans 127 distances); the next
//    tile's cache rows are fetched into registers while the current tile's products run.
//    S^T = K Q^T on v_mfma_f32_16x16x32_bf16, so that the probabilities come out in the B-operand layout of O^T = V^T P^T
//    (keys of the two 16-key halves interleaved per lane group, V fragments read in the same order); temperature, bias,
//    mask and the online softmax are fp32 on the accumulator registers.
//  * dba_prefill32_kernel: the same for rows of 128 values, see there.
//  * dba_decode_kernel<QH, CHL>: the other rows (single decoded tokens, short portions), one workgroup per (row, kv head)
//    serving QH query heads of that kv head from one pass over the keys.  A key row is read by 2^CHL lanes x 16 bytes,
//    64 / 2^CHL keys per load instruction (fully coalesced); the partial dot products fold over the lanes of a key with
//    DPP shuffles; scores and probabilities stay in that layout (4 keys x QH per lane and step), which is also the layout
//    the V pass wants, so nothing is redistributed; K and V of a step are fetched together.  Four waves take the steps
//    round-robin and merge their (max, sum, acc) in LDS; long key ranges are also split over workgroups (grid z), whose
//    partial results dba_merge_kernel combines.
//  * dba_decode128_kernel<QH>: the same for rows of 128 values in blocks of whole 16-key tiles, see there.
#pragma once
#include "biased_attention.h"

namespace aphro {

// row of key `key` in the token-major cache ([block, offset] -> block * block_size + offset), following the block table
__device__ __forceinline__ int dba_slot(const DBAParams& p, const int32_t* bt, int key) {
  int blk, off;
  if (p.bs_shift >= 0) {
    blk = bt[key >> p.bs_shift];
    off = key & (p.block_size - 1);
  } else {
    blk = bt[key / p.block_size];
    off = key % p.block_size;
  }
  if (blk < 0 || blk >= p.num_blocks) blk = 0;             // never read outside the pool
  return blk * p.block_size + off;
}

__device__ __forceinline__ float dba_temp(const DBAParams& p, int pos) {
  return p.temp_coef != 0.f ? 1.0f + p.temp_coef * logf((float)((pos + 1) / p.temp_every + 1)) : 1.0f;
}

// Segment of a rank among items that the segments have `count(q_len)` of, one segment's after the other's (-1: there are fewer); rank
// becomes the item's number in its segment, mine the segment's items.  One wave, 64 segments a step.
template <typename F>
__device__ __forceinline__ int dba_segment(const DBAParams& p, int& rank, int& mine, F count) {
  const int lane = threadIdx.x & 63;
  for (int base = 0; base < p.num_seqs; base += 64) {
    const int n = base + lane < p.num_seqs ? count(p.q_len[base + lane]) : 0;
    int sum = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(sum, d, 64);
      if (lane >= d) sum += up;
    }
    const unsigned long long past = __builtin_amdgcn_ballot_w64(sum > rank);
    if (past) {
      const int at = __builtin_ctzll(past);
      mine = __builtin_amdgcn_readlane(n, at);
      rank -= __builtin_amdgcn_readlane(sum, at) - mine;
      return base + at;
    }
    rank -= __builtin_amdgcn_readlane(sum, 63);
  }
  return -1;
}

// Row and segment of the decode kernel's workgroup number `x` (-1: none).  Beside prompt portions only the rows of short segments are
// numbered: 2000 portion rows would otherwise start and end thousands of workgroups, and the key ranges be split for their number.
__device__ __forceinline__ int dba_short_row(const DBAParams& p, int x, int& seq) {
  if (!p.mixed) {
    seq = p.seq_of_token[x];
    return p.q_len[seq] >= p.min_len ? -1 : x;
  }
  int mine;
  seq = dba_segment(p, x, mine, [&](int len) { return len < p.min_len ? len : 0; });
  return seq < 0 ? -1 : p.q_start[seq] + x;
}

// Oldest key the row at `pos` sees: its window's first key, its chunk's first key, or key 0.
__device__ __forceinline__ int dba_first_key(const DBAParams& p, int pos) {
  int lo = 0;
  if (p.window > 0) lo = max(lo, pos - p.window + 1);
  if (p.chunk > 0) lo = max(lo, pos / p.chunk * p.chunk);
  return lo;
}

// cap * tanh(x / cap) of a score in units of ln 2 (tanh z = 1 - 2 / (e^2z + 1); a large z ends at exactly 1)
__device__ __forceinline__ float dba_cap2(const DBAParams& p, float x) {
  const float e = __builtin_amdgcn_exp2f(x * p.cap_in);
  return p.cap_out - 2.f * p.cap_out * __builtin_amdgcn_rcpf(e + 1.f);
}

// a decoded row's column: o = sum of e^(s - M) v, L = sum of e^(s - M); sink, gate, scale and store
template <int FORM>
__device__ __forceinline__ void dba_finish(const DBAParams& p, int t, int head, int col, float M, float L, float o) {
  constexpr bool EXT = FORM == DBA_MASKED;
  float sig = p.out_scale;
  if (p.gate) {
    const int at = FORM != DBA_PLAIN && p.gate_cols ? head * p.vdim + col : head;
    sig *= sigmoid_f(BFloat::to_f32(p.gate[(int64_t)t * p.gate_stride + at]));
  }
  if (EXT && p.sink) {
    const float sk = p.sink[head], M2 = fmaxf(M, sk), a = expf(M - M2);
    o *= a;
    L = L * a + expf(sk - M2);
  }
  p.out[(int64_t)t * p.out_stride + head * p.vdim + col] = BFloat::from_f32(o * sig / L);
}

constexpr int PF_BM = 64, PF_BN = 64, PF_VT = PF_BN + 4;

// One thread's share of a key tile on its way from the cache to LDS: K chunks (one key, 16 bytes) and V chunk pairs (two
// neighbouring keys, so that the transposed LDS stores are whole dwords).
template <int DK, int DV>
struct PFStage {
  static constexpr int NCHK = DK / 8, NCHV = DV / 8;
  static constexpr int KI = (PF_BN * NCHK + 255) / 256, VI = (PF_BN / 2 * NCHV + 255) / 256;
  u16x8 k[KI], v0[VI], v1[VI];
};

template <int DK, int DV>
__device__ __forceinline__ void pf_load(PFStage<DK, DV>& st, const DBAParams& p, const int32_t* bt, int kvh, int t0, int nk) {
  constexpr int NCHK = DK / 8, NCHV = DV / 8;
  const int64_t krow = (int64_t)p.kv_heads * DK, vrow = (int64_t)p.kv_heads * DV;
#pragma unroll
  for (int it = 0; it < PFStage<DK, DV>::KI; ++it) {
    const int i = threadIdx.x + 256 * it;
    if (i < PF_BN * NCHK) {
      const int tok = i / NCHK, ch = i % NCHK;
      const int key = min(t0 + tok, nk - 1);
      st.k[it] = *reinterpret_cast<const u16x8*>(p.k_cache + (int64_t)dba_slot(p, bt, key) * krow + kvh * DK + 8 * ch);
    }
  }
#pragma unroll
  for (int it = 0; it < PFStage<DK, DV>::VI; ++it) {
    const int i = threadIdx.x + 256 * it;
    if (i < PF_BN / 2 * NCHV) {
      const int tp = i / NCHV, ch = i % NCHV;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int key = min(t0 + 2 * tp + half, nk - 1);
        u16x8 vv = *reinterpret_cast<const u16x8*>(p.v_cache + (int64_t)dba_slot(p, bt, key) * vrow + kvh * DV + 8 * ch);
        if (t0 + 2 * tp + half >= nk) vv = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
        if (half == 0) st.v0[it] = vv;
        else st.v1[it] = vv;
      }
    }
  }
}

template <int DK, int DV>
__device__ __forceinline__ void pf_store(const PFStage<DK, DV>& st, uint16_t* k_lds, uint16_t* vt_lds) {
  constexpr int NCHK = DK / 8, NCHV = DV / 8;
  constexpr int SWZ = (NCHK & -NCHK) - 1;
#pragma unroll
  for (int it = 0; it < PFStage<DK, DV>::KI; ++it) {
    const int i = threadIdx.x + 256 * it;
    if (i < PF_BN * NCHK) {
      const int tok = i / NCHK, ch = i % NCHK;
      *reinterpret_cast<u16x8*>(&k_lds[tok * DK + 8 * (ch ^ (tok & SWZ))]) = st.k[it];
    }
  }
#pragma unroll
  for (int it = 0; it < PFStage<DK, DV>::VI; ++it) {
    const int i = threadIdx.x + 256 * it;
    if (i < PF_BN / 2 * NCHV) {
      const int tp = i / NCHV, ch = i % NCHV;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        *reinterpret_cast<uint32_t*>(&vt_lds[(8 * ch + j) * PF_VT + 2 * tp]) = (uint32_t)st.v0[it][j] | ((uint32_t)st.v1[it][j] << 16);
    }
  }
}

// QT query heads of one kv head share a workgroup: the K and V fragments read from LDS feed QT products each, and the
// tile's trip from the cache to LDS is paid once for them.
template <int DK, int DV, int QT, int FORM>
__global__ __launch_bounds__(256) void dba_prefill_kernel(DBAParams p) {
  constexpr bool EXT = FORM == DBA_MASKED;
  constexpr int NCHK = DK / 8, NKS = DK / 32, NDT = DV / 16, NH = PF_BN / 16, NPK = PF_BN / 32;
  constexpr int SWZ = (NCHK & -NCHK) - 1;
  constexpr int NWIN = PF_BM + PF_BN - 1;
  __shared__ __attribute__((aligned(16))) uint16_t k_lds[PF_BN * DK];
  __shared__ __attribute__((aligned(16))) uint16_t vt_lds[DV * PF_VT];
  __shared__ float bias_win[QT][NWIN + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const int seq = blockIdx.y;
  const int len = p.q_len[seq];
  if (len < p.min_len) return;
  const int ntiles = (len + PF_BM - 1) / PF_BM;
  // Workgroups go to the 8 XCDs round-robin by their linear index, and each XCD has its own L2: the (tile, head unit) pairs
  // are numbered so that every query head of one kv head -- the workgroups that read the same keys and values -- lands on
  // the same XCD (or the same few, when there are fewer kv heads than XCDs).  Within an XCD: longest key ranges first.
  int unit, rank;                                           // head unit: QT consecutive query heads
  {
    constexpr int NX = 8;
    const int G = p.kv_heads, QU = p.heads / p.kv_heads / QT, x = blockIdx.x % NX, j = blockIdx.x / NX;
    if (G % NX == 0) {
      const int ux = (G / NX) * QU, ul = j % ux;            // units served by this XCD, this workgroup's among them
      rank = j / ux;
      unit = ((ul / QU) * NX + x) * QU + ul % QU;
    } else if (NX % G == 0) {
      const int share = NX / G, pair = j * share + x / G;   // XCDs per kv head; (tile, unit) pair of that kv head
      rank = pair / QU;
      unit = (x % G) * QU + pair % QU;
    } else {
      rank = blockIdx.x / (p.heads / QT);
      unit = blockIdx.x % (p.heads / QT);
    }
  }
  const int tile = ntiles - 1 - rank;
  if (tile < 0 || rank >= p.max_tiles) return;
  const int head0 = unit * QT;
  const int ctx = p.ctx_len[seq], s0 = p.q_start[seq];
  const int kvh = head0 / (p.heads / p.kv_heads);
  const int q0 = tile * PF_BM;
  const int qrow = q0 + 16 * wave + c;
  const bool qvalid = qrow < len;
  const int qpos = ctx + qrow;
  constexpr float LOG2E = 1.4426950408889634f;
  const float qs = p.scale * dba_temp(p, qpos) * LOG2E;     // scores in units of ln 2: the exponentials are exp2
  u32x4 qf[QT][NKS];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const uint16_t* qp = p.q + (int64_t)(s0 + min(qrow, len - 1)) * p.q_stride + (head0 + t) * DK;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qf[t][ks] = *reinterpret_cast<const u32x4*>(qp + 32 * ks + 8 * g);
  }
  f32x4 o[QT][NDT];
  float m_run[QT], l_run[QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    m_run[t] = -1e28f;                                      // above a masked score: a row without a visible key so far adds nothing
    l_run[t] = 0.f;
#pragma unroll
    for (int i = 0; i < NDT; ++i) o[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int32_t* bt = p.block_tables + (int64_t)seq * p.max_blocks;
  const int nk = ctx + min(len, q0 + PF_BM);               // keys the tile's last row sees
  // EXT: the oldest key a row sees grows with the row; the walk starts at the key tile of the workgroup's first row
  const int lo_row = EXT ? dba_first_key(p, qpos) : 0;
  const int lo_wave0 = EXT ? dba_first_key(p, ctx + q0 + 16 * wave) : 0, lo_wave1 = EXT ? dba_first_key(p, ctx + q0 + 16 * wave + 15) : 0;
  const int t_first = EXT ? dba_first_key(p, ctx + q0) & ~(PF_BN - 1) : 0;

  PFStage<DK, DV> st;
  pf_load<DK, DV>(st, p, bt, kvh, t_first, nk);
  for (int t0 = t_first; t0 < nk; t0 += PF_BN) {
    __syncthreads();                                        // the previous tile is consumed
    pf_store<DK, DV>(st, k_lds, vt_lds);
    const int dmin = ctx + q0 - t0 - (PF_BN - 1);           // distance of (first row, last key of the tile)
    if (threadIdx.x < QT * 128) {
      const int t = threadIdx.x >> 7, x = threadIdx.x & 127;
      if (x < NWIN) {
        float b = 0.f;
        if (p.bias_lut) {
          const int dist = dmin + x;
          b = p.bias_lut[(int64_t)(head0 + t) * p.lut_len + (dist < 0 ? 0 : (dist < p.lut_len ? dist : p.lut_len - 1))] * LOG2E;
        }
        bias_win[t][x] = b;
      }
    }
    __syncthreads();
    if (t0 + PF_BN < nk) pf_load<DK, DV>(st, p, bt, kvh, t0 + PF_BN, nk);      // in flight during this tile's products
    if (t0 > ctx + q0 + 16 * wave + 15) continue;           // every key of the tile is ahead of the wave's rows
    if (EXT && t0 + PF_BN <= lo_wave0) continue;            // ... or behind what any of them sees
    const bool below = EXT && t0 < lo_wave1;                // some key of the tile is older than what some row of the wave sees
    f32x4 s[QT][NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
#pragma unroll
      for (int t = 0; t < QT; ++t) s[t][h] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int tok = 16 * h + c;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const int ch = (4 * ks + g) ^ (tok & SWZ);
        const u32x4 kf = *reinterpret_cast<const u32x4*>(&k_lds[tok * DK + 8 * ch]);
#pragma unroll
        for (int t = 0; t < QT; ++t)
          s[t][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kf), __builtin_bit_cast(bf16x8, qf[t][ks]),
                                                            s[t][h], 0, 0, 0);
      }
    }
    const bool diag = t0 + PF_BN - 1 > ctx + q0 + 16 * wave; // some key of the tile is ahead of some row of the wave
    u32x4 pf[QT][NPK];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      float pv[NH][4];
      float mx = -1e30f;
      const float* bw = &bias_win[t][qpos - t0 - dmin - 4 * g];    // bias of (this row, key t0 + 4 g); keys count downwards
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float xv = s[t][h][r] * qs;
          if (EXT && p.softcap > 0.f) xv = dba_cap2(p, xv);
          xv += bw[-(16 * h + r)];
          if (diag) xv = t0 + 16 * h + 4 * g + r <= qpos ? xv : -1e30f;
          if (below) xv = t0 + 16 * h + 4 * g + r >= lo_row ? xv : -1e30f;
          pv[h][r] = xv;
          mx = fmaxf(mx, xv);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m_run[t], mx);              // finite for every row that is kept: key 0 is visible
      const float alpha = __builtin_amdgcn_exp2f(m_run[t] - m_new);
      m_run[t] = m_new;
      float lsum = 0.f;
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float e = __builtin_amdgcn_exp2f(pv[h][r] - m_new);    // a masked score is 1e30 below: exactly 0
          pv[h][r] = e;
          lsum += e;
        }
      l_run[t] = l_run[t] * alpha + lsum;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) o[t][dt] *= alpha;
#pragma unroll
      for (int pk = 0; pk < NPK; ++pk)
        pf[t][pk] = u32x4{pack2_16<true>(pv[2 * pk][0], pv[2 * pk][1]), pack2_16<true>(pv[2 * pk][2], pv[2 * pk][3]),
                          pack2_16<true>(pv[2 * pk + 1][0], pv[2 * pk + 1][1]), pack2_16<true>(pv[2 * pk + 1][2], pv[2 * pk + 1][3])};
    }
#pragma unroll
    for (int pk = 0; pk < NPK; ++pk) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        const uint16_t* vr = &vt_lds[(16 * dt + c) * PF_VT + 32 * pk + 4 * g];
        const u32x2 lo = *reinterpret_cast<const u32x2*>(vr);
        const u32x2 hi = *reinterpret_cast<const u32x2*>(vr + 16);
        const u32x4 vf = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int t = 0; t < QT; ++t)
          o[t][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vf), __builtin_bit_cast(bf16x8, pf[t][pk]),
                                                             o[t][dt], 0, 0, 0);
      }
    }
  }
  if (!qvalid) return;                                      // (after the last shuffle-free point: the sums below are per lane group)
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    float l = l_run[t];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    float f = (l > 0.f ? 1.f / l : 0.f) * p.out_scale;
    if (EXT && p.sink) {                                    // one more term of the denominator, without a value
      const float s2 = p.sink[head0 + t] * LOG2E, M = fmaxf(m_run[t], s2), a = __builtin_amdgcn_exp2f(m_run[t] - M);
      f = a / (l * a + __builtin_amdgcn_exp2f(s2 - M)) * p.out_scale;
    }
    if (p.gate && !(FORM != DBA_PLAIN && p.gate_cols)) f *= sigmoid_f(BFloat::to_f32(p.gate[(int64_t)(s0 + qrow) * p.gate_stride + head0 + t]));
    uint16_t* op = p.out + (int64_t)(s0 + qrow) * p.out_stride + (head0 + t) * DV;
    if constexpr (FORM != DBA_PLAIN) {
      const uint16_t* gp = p.gate && p.gate_cols ? p.gate + (int64_t)(s0 + qrow) * p.gate_stride + (head0 + t) * DV : nullptr;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = o[t][dt][r] * f;
        const int c0 = 16 * dt + 4 * g;
        if (p.vec4) {                                       // rows of out and gate are 8-byte aligned
          if (gp) {
            const u16x4 gv = *reinterpret_cast<const u16x4*>(gp + c0);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] *= sigmoid_f(BFloat::to_f32(gv[r]));
          }
          *reinterpret_cast<u16x4*>(op + c0) = u16x4{BFloat::from_f32(v[0]), BFloat::from_f32(v[1]), BFloat::from_f32(v[2]), BFloat::from_f32(v[3])};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) op[c0 + r] = BFloat::from_f32(gp ? v[r] * sigmoid_f(BFloat::to_f32(gp[c0 + r])) : v[r]);
        }
      }
      continue;
    }
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
#pragma unroll
      for (int r = 0; r < 4; ++r) op[16 * dt + 4 * g + r] = BFloat::from_f32(o[t][dt][r] * f);
    }
  }
}

template <int QH, int CHL, int FORM>
__global__ __launch_bounds__(256) void dba_decode_kernel(DBAParams p) {
  constexpr bool EXT = FORM == DBA_MASKED;
  constexpr int CH = 1 << CHL;       // lanes per key row (16 bytes each)
  constexpr int KP = 64 / CH;        // keys per load instruction
  constexpr int NI = 4;              // load instructions per step of the online softmax (few: registers buy occupancy)
  constexpr int KT = NI * KP;        // keys per step
  __shared__ float merge[4][QH][2 + 8 * CH];
  // grid y: the kv heads, each with the groups of QH query heads that cover its own (the last group may be partly empty:
  // its surplus lanes repeat the kv head's last query head and write nothing)
  const int per_kv = p.heads / p.kv_heads, groups = (per_kv + QH - 1) / QH;
  const int kvh = blockIdx.y / groups, sub0 = (blockIdx.y % groups) * QH, hbase = kvh * per_kv;
  int seq;
  const int t = dba_short_row(p, blockIdx.x, seq);
  if (t < 0) return;                                       // the prompt kernel's share
  const int pos = p.ctx_len[seq] + (t - p.q_start[seq]);
  const int k0 = EXT ? dba_first_key(p, pos) : 0;          // oldest visible key
  const int nkeys = pos + 1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ck = lane & (CH - 1), kg = lane >> CHL;
  const bool kin = 8 * ck < p.dim, vin = 8 * ck < p.vdim;
  const float qs = p.scale * dba_temp(p, pos);
  float qv[QH][8];
#pragma unroll
  for (int qh = 0; qh < QH; ++qh) {
    u16x8 raw = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    if (kin) raw = *reinterpret_cast<const u16x8*>(p.q + (int64_t)t * p.q_stride + (hbase + min(sub0 + qh, per_kv - 1)) * p.dim + 8 * ck);
#pragma unroll
    for (int j = 0; j < 8; ++j) qv[qh][j] = BFloat::to_f32(raw[j]);
  }
  const int32_t* bt = p.block_tables + (int64_t)seq * p.max_blocks;
  const int64_t krow = (int64_t)p.kv_heads * p.dim, vrow = (int64_t)p.kv_heads * p.vdim;
  float m[QH], l[QH], acc[QH][8];
#pragma unroll
  for (int qh = 0; qh < QH; ++qh) {
    m[qh] = -INFINITY;
    l[qh] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[qh][j] = 0.f;
  }
  const int ntiles = (nkeys - k0 + KT - 1) / KT;
  const int nsplit = gridDim.z, tps = (ntiles + nsplit - 1) / nsplit;
  const int tile_end = min(ntiles, ((int)blockIdx.z + 1) * tps);
  for (int tile = (int)blockIdx.z * tps + wave; tile < tile_end; tile += 4) {
    float sc[NI][QH];
    u16x8 vv[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int key = k0 + tile * KT + i * KP + kg;
      const bool valid = key < nkeys;
      const int64_t slot = dba_slot(p, bt, valid ? key : k0);
      u16x8 kk = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
      vv[i] = kk;
      if (valid && kin) kk = *reinterpret_cast<const u16x8*>(p.k_cache + slot * krow + kvh * p.dim + 8 * ck);
      if (valid && vin) vv[i] = *reinterpret_cast<const u16x8*>(p.v_cache + slot * vrow + kvh * p.vdim + 8 * ck);
      float kf[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) kf[j] = BFloat::to_f32(kk[j]);
      const int dist = pos - key;
#pragma unroll
      for (int qh = 0; qh < QH; ++qh) {
        float d = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) d += qv[qh][j] * kf[j];
        d = group_sum<CHL>(d);
        float b = 0.f;
        if (p.bias_lut && valid)
          b = p.bias_lut[(int64_t)(hbase + min(sub0 + qh, per_kv - 1)) * p.lut_len + (dist < p.lut_len ? dist : p.lut_len - 1)];
        float x = d * qs;
        if (EXT && p.softcap > 0.f) x = p.softcap * tanhf(x / p.softcap);
        sc[i][qh] = valid ? x + b : -INFINITY;
      }
    }
#pragma unroll
    for (int qh = 0; qh < QH; ++qh) {
      float mx = sc[0][qh];
#pragma unroll
      for (int i = 1; i < NI; ++i) mx = fmaxf(mx, sc[i][qh]);
#pragma unroll
      for (int o = CH; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
      const float m_new = fmaxf(m[qh], mx);                // finite: the tile's first key exists
      const float alpha = (m[qh] == -INFINITY) ? 0.f : __expf(m[qh] - m_new);
      m[qh] = m_new;
      float ls = 0.f;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const float e = (sc[i][qh] == -INFINITY) ? 0.f : __expf(sc[i][qh] - m_new);
        sc[i][qh] = e;
        ls += e;
      }
      l[qh] = l[qh] * alpha + ls;                          // this key group's share; groups are summed at the end
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[qh][j] *= alpha;
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float vf = BFloat::to_f32(vv[i][j]);
#pragma unroll
        for (int qh = 0; qh < QH; ++qh) acc[qh][j] += sc[i][qh] * vf;
      }
    }
  }
  // fold the key groups of the wave, then the four waves
#pragma unroll
  for (int qh = 0; qh < QH; ++qh) {
#pragma unroll
    for (int o = CH; o < 64; o <<= 1) {
      l[qh] += __shfl_xor(l[qh], o, 64);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[qh][j] += __shfl_xor(acc[qh][j], o, 64);
    }
    if (lane == 0) {
      merge[wave][qh][0] = m[qh];
      merge[wave][qh][1] = l[qh];
    }
    if (kg == 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) merge[wave][qh][2 + 8 * ck + j] = acc[qh][j];
    }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < QH * p.vdim; idx += 256) {
    const int qh = idx / p.vdim, col = idx % p.vdim;
    if (sub0 + qh >= per_kv) continue;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, merge[w][qh][0]);
    float L = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = (merge[w][qh][0] == -INFINITY) ? 0.f : __expf(merge[w][qh][0] - M);
      L += merge[w][qh][1] * f;
      o += merge[w][qh][2 + col] * f;
    }
    const int head = hbase + sub0 + qh;
    if (nsplit > 1) {                                       // this split's share; dba_merge_kernel finishes the row
      float* w = p.ws + (((int64_t)t * p.heads + head) * nsplit + blockIdx.z) * (2 + p.vdim);
      if (col == 0) {
        w[0] = M;
        w[1] = L;
      }
      w[2 + col] = o;
      continue;
    }
    dba_finish<FORM>(p, t, head, col, M, L, o);
  }
}

// The same rows where rows are 128 wide (the width of the models) and a cache block holds whole tiles of 16 keys.  A wave takes 16 keys a
// step, aligned in the block, so that a step's block is one scalar lookup and every address a uniform base and a constant of the lane.
// S = K Q^T is four v_mfma_f32_16x16x32_bf16: a lane ends with keys 4 g + r of head `lane % 16` (QH of the 16 columns are heads, the others
// zeros), which makes temperature, cap, bias, mask and softmax of a step those of 4 numbers.  The V pass stays on the vector ALUs in fp32:
// 16 lanes read a V row of key 4 g + i, and the weight of a head is broadcast to them inside their row of 16 lanes by DPP.  K of the next
// step is asked for behind the products, V behind the V pass, so both are on their way during the softmax; nothing branches around a load.
// Bound by memory latency: a wave has few steps.  us with dba_decode_kernel, whose loads wait for one another behind their masks and which
// spends 660 instructions on a step of 16 keys, and here, merge included: 32 rows of up to 1040 keys, 32 heads on 8 with bias 52.9 / 25.4
// (3.4 TB/s), 16 on 4 34.4 / 16.4; one row of 1000 keys 25.0 / 11.5; 128 rows of up to 2000 364 / 146 (4.3 TB/s); two of 16000 121 / 31;
// 24 rows of up to 700, window 31.2 / 18.8, cap and bias 37.7 / 22.9.
template <int H>
__device__ __forceinline__ float row_bcast(float v) { return dpp_f<0x150 + H>(v); }       // lane H of every row of 16
template <int QH, int H>
__device__ __forceinline__ void dec128_scale(float (&acc)[QH][8], float alpha) {
  const float a = row_bcast<H>(alpha);
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[H][j] *= a;
  if constexpr (H + 1 < QH) dec128_scale<QH, H + 1>(acc, alpha);
}
template <int QH, int H>
__device__ __forceinline__ void dec128_add(float (&acc)[QH][8], float prob, const float* vf) {
  const float w = row_bcast<H>(prob);
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[H][j] += w * vf[j];
  if constexpr (H + 1 < QH) dec128_add<QH, H + 1>(acc, prob, vf);
}

template <int QH, int FORM>
__global__ __launch_bounds__(256, 4) void dba_decode128_kernel(DBAParams p) {
  constexpr bool EXT = FORM == DBA_MASKED;
  constexpr int D = 128;
  __shared__ __attribute__((aligned(16))) float part[4][4][QH][D];      // [wave][lane group]: sums of e^(s - m) v
  __shared__ float stat[4][QH][2];                                       // [wave]: m, l
  const int per_kv = p.heads / p.kv_heads, groups = (per_kv + QH - 1) / QH;
  const int kvh = blockIdx.y / groups, sub0 = (blockIdx.y % groups) * QH, hbase = kvh * per_kv;
  int seq;
  const int t = __builtin_amdgcn_readfirstlane(dba_short_row(p, blockIdx.x, seq));
  if (t < 0) return;                                       // the prompt kernel's share
  seq = __builtin_amdgcn_readfirstlane(seq);
  const int pos = p.ctx_len[seq] + (t - p.q_start[seq]);
  const int k0 = EXT ? dba_first_key(p, pos) : 0;          // oldest visible key
  const int nkeys = pos + 1;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l15 = lane & 15, g = lane >> 4;
  const float qs = p.scale * dba_temp(p, pos);
  const int myhead = hbase + min(sub0 + min(l15, QH - 1), per_kv - 1);
  u16x8 qf[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    qf[kk] = *reinterpret_cast<const u16x8*>(p.q + (int64_t)t * p.q_stride + myhead * D + 32 * kk + 8 * g);
    if (l15 >= QH) qf[kk] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  const int32_t* bt = p.block_tables + (int64_t)seq * p.max_blocks;
  const float* lut = p.bias_lut ? p.bias_lut + (int64_t)myhead * p.lut_len : nullptr;
  const int row = p.kv_heads * D;                          // numbers of a cache row
  const int koff = l15 * row + 8 * g, voff = 4 * g * row + 8 * l15;
  const int first = k0 >> 4, ntiles = ((nkeys + 15) >> 4) - first;
  const int nsplit = gridDim.z, tps = (ntiles + nsplit - 1) / nsplit;
  const int tile_end = min(ntiles, ((int)blockIdx.z + 1) * tps);
  int tile = (int)blockIdx.z * tps + wave;
  float m = -INFINITY, l = 0.f, acc[QH][8], b[4] = {0.f, 0.f, 0.f, 0.f};
  u16x8 kf[4], vv[4];
#pragma unroll
  for (int qh = 0; qh < QH; ++qh)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[qh][j] = 0.f;
  // block of a tile (asked for two steps ahead), and numbers ahead of its first cache row of this kv head
  auto block_of = [&](int tl) { return bt[((first + min(tl, tile_end - 1)) << 4) >> p.bs_shift]; };
  auto base_of = [&](int tl, int blk) -> int64_t {
    if (blk < 0 || blk >= p.num_blocks) blk = 0;           // never read outside the pool
    return ((int64_t)blk * p.block_size + (((first + tl) << 4) & (p.block_size - 1))) * row + kvh * D;
  };
  auto load_k = [&](int tl, int64_t base) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) kf[kk] = *reinterpret_cast<const u16x8*>(p.k_cache + base + koff + 32 * kk);
    if (lut) {
      const int dist = pos - ((first + tl) << 4) - 4 * g;
#pragma unroll
      for (int r = 0; r < 4; ++r) b[r] = lut[max(0, min(dist - r, p.lut_len - 1))];
    }
  };
  auto load_v = [&](int64_t base) {
#pragma unroll
    for (int i = 0; i < 4; ++i) vv[i] = *reinterpret_cast<const u16x8*>(p.v_cache + base + voff + i * row);
  };
  if (tile < tile_end) {
    const int64_t base = base_of(tile, block_of(tile));
    load_k(tile, base);
    load_v(base);
    int blk = block_of(tile + 4);
    while (true) {
      const bool more = tile + 4 < tile_end;
      const int64_t next = base_of(tile + 4, blk);
      blk = block_of(tile + 8);
      f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kf[kk]), __builtin_bit_cast(bf16x8, qf[kk]), s, 0, 0, 0);
      const int key0 = (first + tile) << 4;
      float x[4], mx = -INFINITY;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = key0 + 4 * g + r;
        x[r] = s[r] * qs;
        if (EXT && p.softcap > 0.f) x[r] = p.softcap * tanhf(x[r] / p.softcap);
        x[r] = key >= k0 && key < nkeys ? x[r] + b[r] : -INFINITY;       // slots that hold no key may hold anything
        mx = fmaxf(mx, x[r]);
      }
      if (more) load_k(tile + 4, next);
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m, mx);
      if (__builtin_amdgcn_ballot_w64(m_new > m)) {
        const float alpha = m == -INFINITY ? 0.f : __expf(m - m_new);
        m = m_new;
        l *= alpha;
        dec128_scale<QH, 0>(acc, alpha);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[r] = x[r] == -INFINITY ? 0.f : __expf(x[r] - m);
        l += x[r];                                         // this lane group's share; groups are summed at the end
      }
      if (key0 < k0 || key0 + 16 > nkeys) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (key0 + 4 * g + i < k0 || key0 + 4 * g + i >= nkeys) vv[i] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float vf[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) vf[j] = BFloat::to_f32(vv[i][j]);
        dec128_add<QH, 0>(acc, x[i], vf);
      }
      if (!more) break;
      load_v(next);
      tile += 4;
    }
  }
  // the four lane groups of the four waves meet in LDS
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (g == 0 && l15 < QH) {
    stat[wave][l15][0] = m;
    stat[wave][l15][1] = l;
  }
#pragma unroll
  for (int qh = 0; qh < QH; ++qh) {
    *reinterpret_cast<f32x4*>(&part[wave][g][qh][8 * l15]) = f32x4{acc[qh][0], acc[qh][1], acc[qh][2], acc[qh][3]};
    *reinterpret_cast<f32x4*>(&part[wave][g][qh][8 * l15 + 4]) = f32x4{acc[qh][4], acc[qh][5], acc[qh][6], acc[qh][7]};
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < QH * D; idx += 256) {
    const int qh = idx / D, col = idx % D;
    if (sub0 + qh >= per_kv) continue;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, stat[w][qh][0]);
    float L = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = (stat[w][qh][0] == -INFINITY) ? 0.f : __expf(stat[w][qh][0] - M);
      L += stat[w][qh][1] * f;
      o += ((part[w][0][qh][col] + part[w][1][qh][col]) + (part[w][2][qh][col] + part[w][3][qh][col])) * f;
    }
    const int head = hbase + sub0 + qh;
    if (nsplit > 1) {                                       // this split's share; dba_merge_kernel finishes the row
      float* w = p.ws + (((int64_t)t * p.heads + head) * nsplit + blockIdx.z) * (2 + D);
      if (col == 0) {
        w[0] = M;
        w[1] = L;
      }
      w[2 + col] = o;
      continue;
    }
    dba_finish<FORM>(p, t, head, col, M, L, o);
  }
}

// the key ranges' shares of a row, all asked for at once (there are at most DBA_MAX_SPLITS)
template <int FORM>
__global__ void dba_merge_kernel(DBAParams p, int nsplit) {
  const int head = blockIdx.y;
  int seq;
  const int t = dba_short_row(p, blockIdx.x, seq);
  if (t < 0) return;
  const float* w = p.ws + ((int64_t)t * p.heads + head) * nsplit * (2 + p.vdim);
  float mz[DBA_MAX_SPLITS], lz[DBA_MAX_SPLITS], M = -INFINITY, L = 0.f;
#pragma unroll
  for (int z = 0; z < DBA_MAX_SPLITS; ++z) {
    const float* wz = w + min(z, nsplit - 1) * (2 + p.vdim);
    mz[z] = wz[0];
    lz[z] = wz[1];
  }
#pragma unroll
  for (int z = 0; z < DBA_MAX_SPLITS; ++z) M = fmaxf(M, mz[z]);
#pragma unroll
  for (int z = 0; z < DBA_MAX_SPLITS; ++z) {
    mz[z] = z < nsplit && mz[z] != -INFINITY ? __expf(mz[z] - M) : 0.f;       // the share's weight
    if (mz[z] != 0.f) L += lz[z] * mz[z];
  }
  for (int col = threadIdx.x; col < p.vdim; col += blockDim.x) {
    float oz[DBA_MAX_SPLITS], o = 0.f;
#pragma unroll
    for (int z = 0; z < DBA_MAX_SPLITS; ++z) oz[z] = w[min(z, nsplit - 1) * (2 + p.vdim) + 2 + col];
#pragma unroll
    for (int z = 0; z < DBA_MAX_SPLITS; ++z)
      if (mz[z] != 0.f) o += oz[z] * mz[z];
    dba_finish<FORM>(p, t, head, col, M, L, o);
  }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short dba_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* dba_lds_ptr;

constexpr int P32_BN = 64, P32_TILE = P32_BN * 256;          // keys of a tile, bytes of its K (or V) rows
constexpr int p32_rows(int qt) { return 128 / qt; }
constexpr int p32_pitch(int qt) { return p32_rows(qt) + 72; } // floats of a bias window: rows + 64, 32 bytes past a multiple of 128
constexpr size_t p32_lds(int qt) { return 4 * P32_TILE + (size_t)2 * qt * 4 * p32_pitch(qt) * 4; }

// The same attention for rows of 128 (the width of the models), on 32x32x16 products: a workgroup owns 128 / QT consecutive rows of QT
// query heads of one kv head (QT = 4, 2, 1: as many as divide its heads), a wave 32 rows of one head.  Against dba_prefill_kernel a
// fragment read from LDS feeds 32 columns instead of 16, K and V go from the cache to LDS without a stop in registers (V by whole rows,
// its transpose is the transposing LDS read's), the temperature and the bias are one FMA on a score whose four biases are one aligned
// LDS read, the output is rescaled only when some row's maximum moved, and one barrier a tile does.  Two workgroups of one group share a CU.
// Workgroups are numbered over the row tiles that the segments have, not over the longest segment's times their number: decoded rows
// beside a prompt portion cost none.
// Bound by a tile's chain of steps (products, softmax, products: 2 us where a workgroup is alone on its CU, 1.1 where two share it) more than by any unit:
// without its exponentials, its products or its loads it is 5 to 30 % faster each.  us before / after: 16 heads on 4, 4096 rows with bias 327 / 157,
// without 317 / 135; 2000 rows behind 1024 keys, window 1024 84 / 42, with cap and bias 151 / 98; 32 heads on 8, three segments of 900 to 1400 rows
// with gate 147 / 82, eight of 9 rows 35 / 21; 48 rows 20 / 20 (the launch).  Nothing in a step waits for the tile on its way before its products
// are done (block table entries and biases are asked for ahead of it and looked at in the next step, q is waited for where hipcc sees it), lane
// offsets of whole tiles are constants, the halves' maxima meet without LDS: 143 -> 127, 122 -> 103, 91 -> 79, 69 -> 67 for the first, second, fourth
// and fifth of these, 32 heads on 8 of 8192 rows 591 -> 553.  GROUPS = 2: two such groups of waves take a row tile's key tiles in turn, each in
// LDS of its own, and their sums meet at the end: half the chain (the launch says where).  The groups' own barriers, counted in LDS, in place of the
// workgroup's: 3 % slower.  Loads by 64-bit addresses instead of buffer offsets: 160 for 157; loads between the
// products: 170 to 208 (hipcc waits for them in front of the next LDS read).  V in the order [4 keys][16 bytes] of flash_attn.hip, for which four neighbouring
// lanes read four rows: 192 for 164; fragments as hipcc orders them: 164 for 160; tiles begun at another key by every workgroup: no change.
template <int QT, int FORM, int GROUPS>
__global__ __launch_bounds__(256 * GROUPS, 2) void dba_prefill32_kernel(DBAParams p) {
  constexpr bool EXT = FORM == DBA_MASKED;
  constexpr int D = 128, R = p32_rows(QT), BP = p32_pitch(QT), NB = (QT * (R + 63) + 255) / 256;
  constexpr float LOG2E = 1.4426950408889634f;
  extern __shared__ __attribute__((aligned(16))) unsigned char dba_room[];
  const int group = GROUPS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, tid = threadIdx.x & 255;
  unsigned char* const dba_smem = dba_room + group * p32_lds(QT);
  float* bias_lds = reinterpret_cast<float*>(dba_smem + 4 * P32_TILE);      // [2][QT][4 copies][BP]
  const int lane = threadIdx.x & 63, kh = lane >> 5, l31 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);      // of the group's four
  // ---- head unit and rank among the row tiles (numbering over the XCDs: see dba_prefill_kernel) ------------------------------------
  int unit, rank;
  {
    constexpr int NX = 8;
    const int G = p.kv_heads, QU = p.heads / p.kv_heads / QT, x = blockIdx.x % NX, j = blockIdx.x / NX;
    if (G % NX == 0) {
      const int ux = (G / NX) * QU, ul = j % ux;
      rank = j / ux;
      unit = ((ul / QU) * NX + x) * QU + ul % QU;
    } else if (NX % G == 0) {
      const int share = NX / G, pair = j * share + x / G;
      rank = pair / QU;
      unit = (x % G) * QU + pair % QU;
    } else {
      rank = blockIdx.x / (p.heads / QT);
      unit = blockIdx.x % (p.heads / QT);
    }
  }
  // ---- segment and row tile of the rank: the tiles of the segments one after the other ------------------------------------------------
  int ntiles = 0;
  const int seq = dba_segment(p, rank, ntiles, [&](int len) { return len >= p.min_len ? (len + R - 1) / R : 0; });
  if (seq < 0) return;
  // longest key ranges first; where every workgroup is resident at once, the second half shortest first: the two of a CU even out
  int tile = ntiles - 1 - rank;
  if (p.snake && rank >= (ntiles + 1) / 2) tile = rank - (ntiles + 1) / 2;
  const int len = p.q_len[seq], ctx = p.ctx_len[seq], s0 = p.q_start[seq];
  const int t = wave % QT, head = unit * QT + t, kvh = unit * QT / (p.heads / p.kv_heads);
  const int q0 = tile * R, row0 = q0 + 32 * (wave / QT), qrow = row0 + l31, qpos = ctx + qrow;
  const float qs = p.scale * dba_temp(p, qpos) * LOG2E;      // scores in units of ln 2: the exponentials are exp2
  u32x4 qf[8];
  {
    const uint16_t* qp = p.q + (int64_t)(s0 + min(qrow, len - 1)) * p.q_stride + head * D + 8 * kh;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = *reinterpret_cast<const u32x4*>(qp + 16 * ks);
  }
  const int32_t* bt = p.block_tables + (int64_t)seq * p.max_blocks;
  const int nk = ctx + min(len, q0 + R);                     // keys the tile's last row sees
  const int lo_row = EXT ? dba_first_key(p, qpos) : 0;
  const int lo_wave0 = EXT ? dba_first_key(p, ctx + row0) : 0, lo_wave1 = EXT ? dba_first_key(p, ctx + row0 + 31) : 0;
  const int t_first = EXT ? dba_first_key(p, ctx + q0) & ~(P32_BN - 1) : 0;
  // ---- staging: a wave fetches 16 keys of a tile, 4 keys an instruction, lane L -> key L >> 4: a row's 64-byte lines are asked for by
  // neighbouring lanes.  LDS slot L & 15 holds K's piece slot ^ (key & 15), V's piece slot ^ 4 (key & 3): fragment reads and transposing
  // reads find their banks free -------------------------------------------------------------------------------------------------------
  // rows are addressed inside their block (or, in blocks of fewer than 16 keys, inside the whole cache, which then is below 4 GiB)
  const uint32_t row_bytes = (uint32_t)p.kv_heads * D * 2;
  const bool in_block = p.bs_shift >= 4;
  const uint32_t span = (uint32_t)(in_block ? p.block_size : p.num_blocks * p.block_size) * row_bytes - kvh * D * 2;
  const unsigned char* kb = reinterpret_cast<const unsigned char*>(p.k_cache) + kvh * D * 2;
  const unsigned char* vb = reinterpret_cast<const unsigned char*>(p.v_cache) + kvh * D * 2;
  // block of the wave's 16 keys of the tile at t0 where they share one (past the last key: the last key's): the table's entry as it lies, looked at a
  // tile later -- a look at once would wait for the tile on its way, which left ahead of it
  auto entry_of = [&](int t0) { return p.bs_shift < 4 ? 0 : bt[min(t0 + 16 * wave, (nk - 1) & ~15) >> p.bs_shift]; };
  auto block_of = [&](int entry) {
    const int blk = __builtin_amdgcn_readfirstlane(entry);
    return blk < 0 || blk >= p.num_blocks ? 0 : blk;         // never read outside the pool
  };
  // where the wave's 16 keys all exist, lane offsets are the same in every tile
  const int lrow = lane >> 4, vlane = lrow * (int)row_bytes + (((lane & 15) ^ (lrow << 2)) << 4);
  int klane[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) klane[j] = lrow * (int)row_bytes + (((lane & 15) ^ (4 * j + lrow)) << 4);
  auto fetch = [&](int buf, int t0, int blk) {               // a tile's 16 keys of the wave, K and V
    unsigned char* dst = dba_smem + buf * 2 * P32_TILE + wave * 4096;
    const int64_t base = in_block ? (int64_t)blk * p.block_size * row_bytes : 0;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(kb + base), 0, span, 0x00020000),
                                 rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(vb + base), 0, span, 0x00020000);
    if (in_block && t0 + 16 * wave + 16 <= nk) {
      const uint32_t first = (uint32_t)((t0 + 16 * wave) & (p.block_size - 1)) * row_bytes;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (dba_lds_ptr)(dst + j * 1024), 16, klane[j], first + 4 * j * row_bytes, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (dba_lds_ptr)(dst + P32_TILE + j * 1024), 16, vlane, first + 4 * j * row_bytes, 0, 0);
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int key = min(t0 + 16 * wave + 4 * j + lrow, nk - 1);
      const uint32_t at = (uint32_t)(in_block ? key & (p.block_size - 1) : dba_slot(p, bt, key)) * row_bytes;
      const int ko = (int)(at + (((lane & 15) ^ (4 * j + lrow)) << 4)), vo = (int)(at + (((lane & 15) ^ (lrow << 2)) << 4));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (dba_lds_ptr)(dst + j * 1024), 16, ko, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (dba_lds_ptr)(dst + P32_TILE + j * 1024), 16, vo, 0, 0, 0);
    }
  };
  // ---- bias of a tile: entry x of a head's window is the distance (ctx + q0 - t0 + R - 1) - x; a row reads 4 neighbours at a time, and
  // the copy shifted by its own misalignment makes them 16 aligned bytes -----------------------------------------------------------------
  float bias_reg[NB];
  auto bias_load = [&](int t0) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int x = tid + 256 * i, h = x / (R + 63), e = x - h * (R + 63);
      const int dist = ctx + q0 - t0 + R - 1 - e;
      bias_reg[i] = p.bias_lut[(int64_t)(unit * QT + min(h, QT - 1)) * p.lut_len + min(max(dist, 0), p.lut_len - 1)];
    }
  };
  auto bias_store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int x = tid + 256 * i, h = x / (R + 63), e = x - h * (R + 63);
      if (h < QT)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (e >= c) bias_lds[((buf * QT + h) * 4 + c) * BP + e - c] = bias_reg[i] * LOG2E;
    }
  };
  const int bx = R - 1 - (qrow - q0), bias_at = (t * 4 + (bx & 3)) * BP + (bx & ~3) + 4 * kh;
  f32x16 o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float m_run = -1e28f, l_run = 0.f;                         // above a masked score: a row without a visible key so far adds nothing
  const int kaddr = l31 * 256 + ((kh ^ (l31 & 15)) << 4);
  // transposing read of 4 keys x 16 columns by 16 lanes: lane i asks for 8 bytes of key i >> 2 and gets column i of the four keys
  const int vk = (lane & 15) >> 2;
  const int vaddr = P32_TILE + kh * 1024 + vk * 256 + (vk << 6) + (((lane >> 4) & 1) << 5) + ((lane & 3) << 3);
  constexpr int STEP = P32_BN * GROUPS;                      // the groups take a row tile's key tiles in turn
  const int g_first = t_first + P32_BN * group;
  if (g_first < nk) {
    fetch(0, g_first, block_of(entry_of(g_first)));
    if (p.bias_lut) {
      bias_load(g_first);
      bias_store(0);
    }
  }
  int entry = entry_of(g_first + STEP), buf = 0;
  for (int t0 = g_first; t0 - P32_BN * group < nk; t0 += STEP, buf ^= 1) {      // (as often in every group: the barrier is the workgroup's)
    // this wave's part of the tile is there, and it is through with the other buffer
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);                      // vmcnt(0) lgkmcnt(0), where hipcc sees it: it waits for q once, not in every tile
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const bool more = t0 + STEP < nk;
    if (more) {                                              // in flight during this tile's products
      const int blk = block_of(entry);
      entry = entry_of(t0 + 2 * STEP);
      if (p.bias_lut) bias_load(t0 + STEP);
      __builtin_amdgcn_sched_barrier(0);
      fetch(buf ^ 1, t0 + STEP, blk);
    }
    if ((GROUPS == 1 || t0 < nk) && t0 <= ctx + row0 + 31 && !(EXT && t0 + P32_BN <= lo_wave0)) {      // some key of the tile is seen by some row of the wave
      const unsigned char* sb = dba_smem + buf * 2 * P32_TILE;
      // (the order is fixed by hand: left to itself hipcc reads one pair of fragments, waits for it, multiplies, and so on)
      f32x16 s[2];
      u32x4 kf[8][2];
      auto read_k = [&](int k0) {
#pragma unroll
        for (int ks = k0; ks < k0 + 4; ++ks)
#pragma unroll
          for (int b = 0; b < 2; ++b) kf[ks][b] = *reinterpret_cast<const u32x4*>(sb + b * 8192 + (kaddr ^ (ks << 5)));
        __builtin_amdgcn_sched_barrier(0);
      };
      auto multiply_k = [&](int k0) {
#pragma unroll
        for (int ks = k0; ks < k0 + 4; ++ks)
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const f32x16 zero = {};
            s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf[ks][b]), __builtin_bit_cast(bf16x8, qf[ks]), ks == 0 ? zero : s[b], 0, 0, 0);
          }
        __builtin_amdgcn_sched_barrier(0);
      };
      read_k(0);
      read_k(4);
      multiply_k(0);
      multiply_k(4);
      // lane's scores: row l31, keys t0 + 32 b + 8 q + 4 kh + r
      if (EXT && p.softcap > 0.f) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[b][i] = dba_cap2(p, s[b][i] * qs);
        if (p.bias_lut) {
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f32x4 w = *reinterpret_cast<const f32x4*>(bias_lds + buf * QT * 4 * BP + bias_at + 32 * b + 8 * q);
#pragma unroll
              for (int r = 0; r < 4; ++r) s[b][4 * q + r] += w[r];
            }
        }
      } else if (p.bias_lut) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x4 w = *reinterpret_cast<const f32x4*>(bias_lds + buf * QT * 4 * BP + bias_at + 32 * b + 8 * q);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[b][4 * q + r] = __builtin_fmaf(s[b][4 * q + r], qs, w[r]);
          }
      } else {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[b][i] *= qs;
      }
      if (t0 + P32_BN - 1 > ctx + row0) {                    // some key of the tile is ahead of some row of the wave
        const int last = qpos - t0 - 4 * kh;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[b][i] = 32 * b + 8 * (i >> 2) + (i & 3) <= last ? s[b][i] : -1e30f;
      }
      if (EXT && t0 < lo_wave1) {                            // ... or older than what some row of the wave sees
        const int first = lo_row - t0 - 4 * kh;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[b][i] = 32 * b + 8 * (i >> 2) + (i & 3) >= first ? s[b][i] : -1e30f;
      }
      float mx = -1e30f;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[b][i]);
      {                                                      // the other half's largest, without LDS
        const uint32_t mb = __builtin_bit_cast(uint32_t, mx);
        const auto sw = __builtin_amdgcn_permlane32_swap(mb, mb, false, false);
        const uint32_t low = sw[0], high = sw[1];            // (hipcc takes element 0 for either where one is bit-cast in place)
        mx = fmaxf(__builtin_bit_cast(float, low), __builtin_bit_cast(float, high));
      }
      const float m_new = fmaxf(m_run, mx);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      float lsum = 0.f;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[b][i] = __builtin_amdgcn_exp2f(s[b][i] - m_new);      // a masked score is 1e30 below: exactly 0
          lsum += s[b][i];
        }
      l_run = l_run * alpha + lsum;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
      }
      // O^T += V^T P^T, 16 keys a step: k slots 4 h .. + 3 of lane half kh are keys 16 ks + 8 h + 4 kh .. + 3, the ones it has
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const f32x16& e = s[ks >> 1];
        const int i0 = 8 * (ks & 1);
        const u32x4 pf = {pack2_16<true>(e[i0], e[i0 + 1]), pack2_16<true>(e[i0 + 2], e[i0 + 3]), pack2_16<true>(e[i0 + 4], e[i0 + 5]),
                          pack2_16<true>(e[i0 + 6], e[i0 + 7])};
#pragma unroll
        for (int db = 0; db < 4; ++db) {
          const unsigned char* va = sb + (vaddr ^ (db << 6)) + 4 * ks * 1024;
          const dba_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((dba_s16x4 __attribute__((address_space(3)))*)va);
          const dba_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((dba_s16x4 __attribute__((address_space(3)))*)(va + 2048));
          const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, u32x4{l2[0], l2[1], h2[0], h2[1]}),
                                                          __builtin_bit_cast(bf16x8, pf), o[db], 0, 0, 0);
        }
      }
    }
    if (more && p.bias_lut) bias_store(buf ^ 1);
  }
  float l = l_run + __shfl_xor(l_run, 32, 64);
  if constexpr (GROUPS > 1) {                                // the second group's sums join the first's
    f32x4* const ro = reinterpret_cast<f32x4*>(dba_room + p32_lds(QT)) + wave * 16 * 64 + lane;
    float* const rm = reinterpret_cast<float*>(dba_room + p32_lds(QT) + 4 * P32_TILE) + wave * 128 + lane;
    __syncthreads();
    if (group == 1) {
#pragma unroll
      for (int i = 0; i < 16; ++i) ro[64 * i] = f32x4{o[i >> 2][4 * (i & 3)], o[i >> 2][4 * (i & 3) + 1], o[i >> 2][4 * (i & 3) + 2], o[i >> 2][4 * (i & 3) + 3]};
      rm[0] = m_run;
      rm[64] = l;
    }
    __syncthreads();
    if (group == 1) return;
    const float m1 = rm[0], M = fmaxf(m_run, m1), a0 = __builtin_amdgcn_exp2f(m_run - M), a1 = __builtin_amdgcn_exp2f(m1 - M);
    m_run = M;
    l = l * a0 + rm[64] * a1;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const f32x4 x = ro[64 * i];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[i >> 2][4 * (i & 3) + r] = o[i >> 2][4 * (i & 3) + r] * a0 + x[r] * a1;
    }
  }
  if (qrow >= len) return;
  float f = (l > 0.f ? 1.f / l : 0.f) * p.out_scale;
  if (EXT && p.sink) {                                       // one more term of the denominator, without a value
    const float s2 = p.sink[head] * LOG2E, M = fmaxf(m_run, s2), a = __builtin_amdgcn_exp2f(m_run - M);
    f = a / (l * a + __builtin_amdgcn_exp2f(s2 - M)) * p.out_scale;
  }
  if (p.gate && !(FORM != DBA_PLAIN && p.gate_cols)) f *= sigmoid_f(BFloat::to_f32(p.gate[(int64_t)(s0 + qrow) * p.gate_stride + head]));
  uint16_t* op = p.out + (int64_t)(s0 + qrow) * p.out_stride + head * D + 4 * kh;
  const uint16_t* gp = FORM != DBA_PLAIN && p.gate && p.gate_cols ? p.gate + (int64_t)(s0 + qrow) * p.gate_stride + head * D + 4 * kh : nullptr;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c0 = 32 * db + 8 * q;
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = o[db][4 * q + r] * f;
      if (p.vec4) {                                          // rows of out and gate are 8-byte aligned
        if (FORM != DBA_PLAIN && gp) {
          const u16x4 gv = *reinterpret_cast<const u16x4*>(gp + c0);
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] *= sigmoid_f(BFloat::to_f32(gv[r]));
        }
        *reinterpret_cast<u16x4*>(op + c0) = u16x4{BFloat::from_f32(v[0]), BFloat::from_f32(v[1]), BFloat::from_f32(v[2]), BFloat::from_f32(v[3])};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) op[c0 + r] = BFloat::from_f32(FORM != DBA_PLAIN && gp ? v[r] * sigmoid_f(BFloat::to_f32(gp[c0 + r])) : v[r]);
      }
    }
}

template <int DK, int QT, int FORM>
static void launch_prefill_dv(const DBAParams& p, dim3 grid, hipStream_t st) {
  switch (p.vdim) {
    case 32: hipLaunchKernelGGL((dba_prefill_kernel<DK, 32, QT, FORM>), grid, dim3(256), 0, st, p); break;
    case 64: hipLaunchKernelGGL((dba_prefill_kernel<DK, 64, QT, FORM>), grid, dim3(256), 0, st, p); break;
    case 96: hipLaunchKernelGGL((dba_prefill_kernel<DK, 96, QT, FORM>), grid, dim3(256), 0, st, p); break;
    case 128: hipLaunchKernelGGL((dba_prefill_kernel<DK, 128, QT, FORM>), grid, dim3(256), 0, st, p); break;
  }
}

template <int QT, int FORM>
static void launch_prefill_dk(const DBAParams& p, dim3 grid, hipStream_t st) {
  switch (p.dim) {
    case 32: launch_prefill_dv<32, QT, FORM>(p, grid, st); break;
    case 64: launch_prefill_dv<64, QT, FORM>(p, grid, st); break;
    case 96: launch_prefill_dv<96, QT, FORM>(p, grid, st); break;
    case 128: launch_prefill_dv<128, QT, FORM>(p, grid, st); break;
  }
}

template <int QT, int FORM, int GROUPS>
static void launch_prefill32(const DBAParams& p0, int64_t num_tokens, int num_seqs, hipStream_t st) {
  DBAParams p = p0;
  constexpr int R = p32_rows(QT);
  const int64_t most = num_tokens / R + (num_tokens / p.min_len < num_seqs ? num_tokens / p.min_len : num_seqs);     // row tiles there can be
  const int64_t blocks = (most * (p.heads / QT) + 7) / 8 * 8;
  p.snake = GROUPS == 1 && num_seqs == 1 && blocks <= 2 * device_cu_count();
  constexpr size_t lds = GROUPS * p32_lds(QT);
  static bool attr_set_dev[APHRO_MAX_DEVICES] = {}; bool& attr_set = attr_set_dev[device_slot()];
  if (!attr_set)
    attr_set = hipFuncSetAttribute((const void*)dba_prefill32_kernel<QT, FORM, GROUPS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
  hipLaunchKernelGGL((dba_prefill32_kernel<QT, FORM, GROUPS>), dim3((unsigned)blocks), dim3(256 * GROUPS), lds, st, p);
}

template <int FORM>
void dba_prefill_launch(const DBAParams& p0, int64_t num_tokens, int max_q_len, int num_seqs, int max_keys, int max_kv_len, hipStream_t st) {
  // 16-byte loads into LDS want aligned caches (rows are 256 bytes times the kv heads); their 32-bit offsets a block below 4 GiB, or the
  // whole cache where blocks are no multiples of 16 keys
  const int64_t span = (p0.bs_shift >= 4 ? 1 : p0.num_blocks) * p0.block_size * (int64_t)p0.kv_heads * 256;
  if (p0.dim == 128 && p0.vdim == 128 && (((uintptr_t)p0.k_cache | (uintptr_t)p0.v_cache) & 15) == 0 && span < (1ll << 32)) {
    const int per_kv = p0.heads / p0.kv_heads;
    const int qt = per_kv % 4 == 0 ? 4 : per_kv % 2 == 0 ? 2 : 1;
    // Two groups of waves a row tile where a launch lasts as long as its longest chain of key tiles: where the row tiles would leave every CU one workgroup
    // at the most, or two of one segment with chains so unlike that all of them are worth at most 1.31 of the longest to a CU, and 0.86 of it to
    // each.  us, one group / two (the two numbers): 16 heads on 4, fresh, 2800 rows 68 / 52 (0.7, 0.5), 4000 96 / 84 (1.0, 0.5); 2400 behind 4800 keys 189 /
    // 181 (1.0, 0.83), 9600 322 / 328 (1.05, 0.9); 4000 behind 2000 154 / 151 (1.3, 0.67), 4000 211 / 219 (1.5, 0.75); windows: 2400 under 1024 42 / 31
    // (0.9, 0.79), under 512 27 / 30 (1.05, 0.9), behind 2400 under 2048 75 / 81 (1.2, 1), 4000 under 2048 73 / 79 (1.5, 0.74); 32 on 8, 1200
    // fresh 34 / 27, behind 1200 under 1024 44 / 50, 2000 fresh under 1024 43 / 48, three segments of 700 33 / 36.
    const int64_t tiles = (num_tokens + p32_rows(qt) - 1) / p32_rows(qt) * (p0.heads / qt), cus = device_cu_count();
    auto uneven = [&] {                                      // (with max_kv_len, the batch's, for the longest segment's: with longer ones beside it one group is taken)
      const double n = max_q_len, ctx = max(max_kv_len - max_q_len, 0), most = p0.window > 0 ? fmin(ctx + n, p0.window) : ctx + n;
      const double rise = fmin(fmax(most - ctx, 0.0), n);                             // rows whose chains grow
      const double mean = (rise * (ctx + 0.5 * rise) + (n - rise) * most) / (n * most);      // of the longest
      return 2 * n > num_tokens && (p0.chunk == 0 || 2.0 * p0.chunk > n) && mean <= 0.86 && tiles * mean <= 1.31 * cus;
    };
    const bool two = max_keys >= 256 && (tiles <= cus || (tiles <= 2 * cus && uneven()));
#define P32(QT) (two ? launch_prefill32<QT, FORM, 2>(p0, num_tokens, num_seqs, st) : launch_prefill32<QT, FORM, 1>(p0, num_tokens, num_seqs, st))
    if (qt == 4) P32(4);
    else if (qt == 2) P32(2);
    else P32(1);
#undef P32
    return;
  }
  DBAParams p = p0;
  p.max_tiles = (max_q_len + PF_BM - 1) / PF_BM;
  const int qt = (p.heads / p.kv_heads) % 2 == 0 ? 2 : 1;   // two query heads of a kv head per workgroup where they pair up
  const int per_seq = (p.max_tiles * (p.heads / qt) + 7) / 8 * 8;      // a multiple of the XCD count: the numbering repeats per segment
  const dim3 grid((unsigned)per_seq, (unsigned)num_seqs);
  if (qt == 2) launch_prefill_dk<2, FORM>(p, grid, st);
  else launch_prefill_dk<1, FORM>(p, grid, st);
}

// lanes per key row: the smallest power of two that covers both row lengths in 16-byte pieces
static int decode_chl(int dim, int vdim) {
  const int pieces = (max(dim, vdim) + 7) / 8;
  int chl = 2;
  while ((1 << chl) < pieces) ++chl;
  return chl;
}

// query heads a decode workgroup serves: all of a kv head's where they fit (1, 2, 4 or 8, rounded up), else groups of them
static int decode_qh(int heads, int kv_heads, int chl) {
  const int per_kv = heads / kv_heads;
  int qh = 1;
  while (qh < per_kv && qh < 8 && 2 * qh * (1 << chl) <= 64) qh *= 2;
  return qh;
}

template <int FORM>
void dba_decode_launch(const DBAParams& p, int64_t rows, int nsplit, hipStream_t st) {
  const dim3 grid((unsigned)rows, (unsigned)dba_decode_units(p.heads, p.kv_heads, p.dim, p.vdim), (unsigned)nsplit);
  const int chl = decode_chl(p.dim, p.vdim), qh = decode_qh(p.heads, p.kv_heads, chl);
  // rows of the models' width in blocks of whole 16-key tiles, 16-byte pieces aligned, a block's rows within 32-bit offsets
  const bool wide = p.dim == 128 && p.vdim == 128 && p.bs_shift >= 4 && (((uintptr_t)p.k_cache | (uintptr_t)p.v_cache) & 15) == 0 &&
                    (int64_t)p.kv_heads * 128 * 16 < (1ll << 30);
  if (wide) {
    if (qh == 4) hipLaunchKernelGGL((dba_decode128_kernel<4, FORM>), grid, dim3(256), 0, st, p);
    else if (qh == 2) hipLaunchKernelGGL((dba_decode128_kernel<2, FORM>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((dba_decode128_kernel<1, FORM>), grid, dim3(256), 0, st, p);
  } else {
#define DEC(QH, CHL) hipLaunchKernelGGL((dba_decode_kernel<QH, CHL, FORM>), grid, dim3(256), 0, st, p)
#define DEC_BY_CHL(QH)                          \
  switch (chl) {                                \
    case 2: DEC(QH, 2); break;                  \
    case 3: DEC(QH, 3); break;                  \
    case 4: if (QH <= 4) DEC((QH <= 4 ? QH : 1), 4); break; \
    case 5: if (QH <= 2) DEC((QH <= 2 ? QH : 1), 5); break; \
  }
  switch (qh) {
    case 1: DEC_BY_CHL(1); break;
    case 2: DEC_BY_CHL(2); break;
    case 4: DEC_BY_CHL(4); break;
    case 8: DEC_BY_CHL(8); break;
  }
  }
#undef DEC_BY_CHL
#undef DEC
  if (nsplit > 1)
    hipLaunchKernelGGL((dba_merge_kernel<FORM>), dim3((unsigned)rows, (unsigned)p.heads), dim3(64), 0, st, p, nsplit);
}

}  // namespace aphro
