// Gated outer-product memories (outer_memory.hip has the recurrence) over prompt portions, in chunks of 64 tokens on the matrix
// cores.  With G_i the sum of log a over a chunk's tokens up to i and S the state ahead of the chunk:
//     o_i = e^{G_i} S^T q_i + sum_{j <= i} e^{G_i - G_j} b_j (q_i . k_j) v_j,      S' = e^{G_63} S + sum_j e^{G_63 - G_j} b_j k_j v_j^T
// so three launches do what a scan does token by token:
//   1. om_chunk_update: every chunk's own sum U (d x 64 value columns a workgroup) and its decay -- all chunks at once
//   2. om_chunk_carry:  S through the chunks, elementwise; U is replaced by the state ahead of its chunk
//   3. om_chunk_out:    o of every chunk -- all chunks at once
// and mLSTM's running maximum (a recurrence of its own, one number per head and token) is worked out ahead of them by om_gates.
//
// What enters the recurrence is fp32 and stays so.  Decay memories, and inputs that are not bf16, multiply on v_mfma_f32_16x16x4_f32; mLSTM's and the state
// space's bf16 queries, keys and values go to the 16-bit units as they are, against fp32 factors in three bf16 parts (the *16 kernels, several chunks
// of a segment to a workgroup: how many goes by all tokens of the call, so that a segment's last bits may differ with what runs beside it).  G is
// summed in 64 bits, so that a small decay keeps its digits behind a large one.  Only the differences G_i - G_j <= 0 are exponentiated: nothing overflows
// however strong the decay.
//
// What bounds it: the fp32 products (the matrix pipe is busy half of the time in launches 1 and 3) and the states between the chunks
// (written once, read and written once, read once: dim x vdim x 4 bytes a chunk and head).  A scan is bound by the latency of its
// token chain.  One portion of 4096 tokens, scan -> chunks in fp32 -> here: decay 8 x 64 x 128 1106 -> 60 us, mLSTM 4 x 128 x 256 2170 -> 113 -> 64,
// state space 64 x 128 x 64 1476 -> 274 -> 103 (128 heads: 1482 -> 575 -> 211).
// Outputs lie as the products leave them: scores as K Q^T and results as V^T P^T, so that a score's registers are the next product's
// operand and a lane holds four neighbouring value columns of one token.  Row pitches are 4 floats over a multiple of 32: the
// eight lanes that a 16-byte LDS access serves at a time fall on all 32 banks.  The states lie in fragments: as rows of DP, the address unit took four times
// as long over a load (state space 64 heads, 600 / 2000 / 4096 tokens 51 / 73 / 116 -> 46 / 67 / 111 us, decay 16 x 64 x 128, 4096 tokens 92 -> 89).  A
// third of a launch is the way to its first numbers; with a segment's place beside its length, prefix sums without LDS and a fixed decay's
// as multiples 42 / 66 / 103, 87 (89 since silu keeps the last places of its smallest numbers, on a card that took 88.6 before).
#include "outer_memory.h"
#include "chunked_scan.h"

namespace aphro {

constexpr int OMC_COLS = 64;                // value columns of a workgroup
constexpr int OMC_PITCH = CHUNK + 4;

struct OMChunk {
  OuterMemory p;
  int min_len;            // segments shorter than this are the scan's
  int group;              // chunks that a workgroup takes in turn (bf16 inputs' kernels; 1 elsewhere): below, and where states are numbered, a chunk is a group of so many
  int chunk0, span;       // the chunks of these launches (below: [chunks] of one span)
  int vpad;               // vdim rounded up to 16
  float* u;               // [chunks, heads] vpad x DP in fragments (frag8): U, then the state ahead of the chunk
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

// Sums of the log decays up to each lane's token: a fixed decay's are multiples.
template <int MODE>
__device__ __forceinline__ double chunk_decays(double la, int lane, int cnt) {
  if constexpr (MODE == 0) return of_lane(la, 0) * (double)(min(lane, cnt - 1) + 1);
  else return wave_incl_sum(la);
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
  ChunkPlace at;
  if (!locate_chunk(a.chunk0 + blockIdx.x, p, a.min_len, at) || at.slot < 0 || at.slot >= p.num_slots) return;
  const int c = at.c;
  const int h = blockIdx.y, c0 = blockIdx.z * OMC_COLS, hk = MODE == 2 ? h / (p.heads / p.qk_heads) : h;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cnt = min(CHUNK, at.len - c * CHUNK);
  const int64_t row0 = (int64_t)at.start + c * CHUNK;
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
  const double g = chunk_decays<MODE>(la, lane, cnt), gend = of_lane(g, 63);
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
      *reinterpret_cast<f32x4*>(&u[frag8<DP>(ct, wave * DT + dt, li, lg)]) = acc[dt][ct];
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

// The same where keys, queries and values enter as the bf16 numbers they are (mLSTM, state space), a workgroup taking a.group chunks of a segment in
// turn: the states that go through memory are those between groups.  Products are on the 16-bit units, one factor in three bf16 parts.  A wave owns 16 value
// columns: what it multiplies its state and its values with (queries, keys, weights) comes from LDS, the state stays in its registers -- a lane has, of
// one column, the eight neighbouring rows 32 kk + 8 lg + (0..7), which are its part of the next product's operand as they lie (the keys' rows lie in
// LDS in the order that gives this: key_row).  Numbers that are not finite would meet a part that is zero: a chunk with any multiplies in fp32.
// What bounds it: the vector units (splits, weights, the copy to LDS: some 1200 instructions a wave and chunk beside 130 matrix ones).  Against a workgroup
// a chunk, whose states (32 KB each) made 250 of the 370 MB that 64 heads and 2000 tokens moved and whose state products were fp32: state space 64 heads
// 2000 tokens 111 -> 74 us, 4096 216 -> 117, 128 heads 4096 499 -> 211, mLSTM 4 x 128 x 256 4096 95 -> 66; error against 64 bits of outputs 1.6e-7 ->
// 1.2e-7, of states 8.4e-8 -> 8.3e-8.  Without branches at the use of
// every number that may not be finite, and with masks and bits two at a time: 90 -> 74 at the first of these.
constexpr int OMG_PITCH = CHUNK + 8;
constexpr __device__ __forceinline__ int key_row(int d) { return (d & ~31) | ((d & 4) << 2) | ((d & 24) >> 1) | (d & 3); }
// Is a number not finite?  The largest of the bits without sign, two a step.
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void largest_bits(u16x2& m, u32x4 w) {
#pragma unroll
  for (int i = 0; i < 4; ++i) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w[i] & 0x7fff7fffu));
}
__device__ __forceinline__ bool odd_bits(u16x2 m) { return max(m[0], m[1]) >= 0x7f80; }
// Eight neighbouring rows of a lane's token into LDS; row(i) is the place of the i-th.
template <typename F>
__device__ __forceinline__ void put_rows(uint16_t* at, u32x4 w, F row) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    at[row(2 * i) * OMG_PITCH] = (uint16_t)w[i];
    at[row(2 * i + 1) * OMG_PITCH] = (uint16_t)(w[i] >> 16);
  }
}
// split3 of eight finite numbers.
__device__ __forceinline__ void split3_finite(const float (&x)[8], u16x8 (&part)[3]) {
  u32x4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t a0 = __builtin_bit_cast(uint32_t, x[2 * i]), b0 = __builtin_bit_cast(uint32_t, x[2 * i + 1]);
    const float ra = x[2 * i] - __builtin_bit_cast(float, a0 & 0xffff0000u), rb = x[2 * i + 1] - __builtin_bit_cast(float, b0 & 0xffff0000u);
    const uint32_t a1 = __builtin_bit_cast(uint32_t, ra), b1 = __builtin_bit_cast(uint32_t, rb);
    const float la = ra - __builtin_bit_cast(float, a1 & 0xffff0000u), lb = rb - __builtin_bit_cast(float, b1 & 0xffff0000u);
    h[i] = __builtin_amdgcn_perm(b0, a0, 0x07060302u);
    m[i] = __builtin_amdgcn_perm(b1, a1, 0x07060302u);
    l[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, lb), __builtin_bit_cast(uint32_t, la), 0x07060302u);
  }
  part[0] = __builtin_bit_cast(u16x8, h), part[1] = __builtin_bit_cast(u16x8, m), part[2] = __builtin_bit_cast(u16x8, l);
}
// A wave's state S (rows 32 kk + 8 lg + 4 hf + r of its column) after a chunk: S decays by ``all`` and takes the chunk's tokens, values weighted by ws.  The
// tokens' sum starts from zero and meets S once: added to S product by product, S was rounded six times a chunk (error against 64 bits 1.01e-7 for 0.85e-7).
template <int DP>
__device__ __forceinline__ void group_update(f32x4 (&S)[DP / 32][2], const uint16_t* kt, const u16x8 (&v)[CHUNK / 32], const float* ws, float all, bool odd, int li, int lg) {
  float x[CHUNK / 32][8], z = 0.f;                                       // (z is not zero: a weighted value that is not finite)
#pragma unroll
  for (int jj = 0; jj < CHUNK / 32; ++jj) {
    const f32x4 w0 = *reinterpret_cast<const f32x4*>(&ws[32 * jj + 8 * lg]), w1 = *reinterpret_cast<const f32x4*>(&ws[32 * jj + 8 * lg + 4]);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[jj][i] = BFloat::to_f32(v[jj][i]) * (i < 4 ? w0[i] : w1[i - 4]);
      z = fmaf(x[jj][i], 0.f, z);
    }
  }
  const uint16_t* kr = kt + li * OMG_PITCH + 8 * lg;
  f32x4 U[DP / 16] = {};
  if (odd || __any(z != 0.f)) {
#pragma unroll
    for (int jj = 0; jj < CHUNK / 32; ++jj)
#pragma unroll
      for (int kk = 0; kk < DP / 16; ++kk) {
        const u16x8 av = *reinterpret_cast<const u16x8*>(&kr[kk * 16 * OMG_PITCH + 32 * jj]);
#pragma unroll
        for (int m = 0; m < 8; ++m) U[kk] = mfma4(BFloat::to_f32(av[m]), x[jj][m], U[kk]);
      }
  } else {
    u16x8 high[CHUNK / 32];                                              // the first parts: last, when the small ones are in
#pragma unroll
    for (int jj = 0; jj < CHUNK / 32; ++jj) {
      u16x8 part[3];
      split3_finite(x[jj], part);
      high[jj] = part[0];
#pragma unroll
      for (int kb = 0; kb < DP / 16; kb += 4) {
        u16x8 av[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) av[kk] = *reinterpret_cast<const u16x8*>(&kr[(kb + kk) * 16 * OMG_PITCH + 32 * jj]);
#pragma unroll
        for (int n = 2; n >= 1; --n)
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) U[kb + kk] = mfma16(av[kk], part[n], U[kb + kk]);
      }
    }
#pragma unroll
    for (int jj = 0; jj < CHUNK / 32; ++jj)
#pragma unroll
      for (int kk = 0; kk < DP / 16; ++kk) U[kk] = mfma16(*reinterpret_cast<const u16x8*>(&kr[kk * 16 * OMG_PITCH + 32 * jj]), high[jj], U[kk]);
  }
#pragma unroll
  for (int kk = 0; kk < DP / 16; ++kk)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[kk >> 1][kk & 1][r] = fmaf(all, S[kk >> 1][kk & 1][r], U[kk][r]);
}
// The normaliser's number of key row tid.
__device__ __forceinline__ float group_update_n(float sum, const uint16_t* kt, const float* ws, float all, int tid) {
  float add = 0.f;
  for (int t = 0; t < CHUNK; t += 8) {
    const u16x8 x = *reinterpret_cast<const u16x8*>(&kt[key_row(tid) * OMG_PITCH + t]);
#pragma unroll
    for (int i = 0; i < 8; ++i) add += BFloat::to_f32(x[i]) * ws[t + i];
  }
  return all * sum + add;
}
// What a workgroup of the two kernels below works on.  Workgroups that read the same keys and queries -- the heads of a key head, the column blocks of
// a head -- follow each other on one XCD, whose L2 then holds them; pairs of group and key head go round the XCDs.
struct OMGroup {
  int x, h, hk, c0, chunks, tokens;    // group's number in the launch, head, key head, first column, chunks and tokens of the group
  int64_t row0;                        // its first token
};
__host__ __device__ __forceinline__ int om_key_heads(const OuterMemory& p) { return p.mode == 2 ? p.qk_heads : p.heads; }
// A few pairs that do not come out even on the eight XCDs (a key head for all heads, or two): each is divided among the XCDs.  us, one key head for 128 heads
// of 128 x 64, 277 tokens (two or three groups, of which an XCD had one each) 121 -> 87, for
// 64 heads 219 tokens 34.6 -> 27.7, 2725 beside 280 in 25 short segments 137 -> 121.
__host__ __device__ __forceinline__ bool om_split_pairs(int64_t pairs, int subs) { return pairs < 64 && pairs % 8 != 0 && subs >= 8; }
__device__ __forceinline__ bool locate_group(const OMChunk& a, OMGroup& w) {
  const OuterMemory& p = a.p;
  const int key_heads = om_key_heads(p), heads = p.heads / key_heads, blocks = (p.vdim + OMC_COLS - 1) / OMC_COLS;
  const int idx = blockIdx.x >> 3, per = om_split_pairs(a.span * key_heads, heads * blocks) ? (heads * blocks + 7) / 8 : heads * blocks;
  int pair = idx / per, sub = idx % per;
  if (per < heads * blocks) sub += (int)(blockIdx.x & 7) * per;
  else pair = pair * 8 + (int)(blockIdx.x & 7);
  if (pair >= a.span * key_heads || sub >= heads * blocks) return false;
  w.x = pair % a.span, w.hk = pair / a.span, w.h = w.hk * heads + sub / blocks, w.c0 = sub % blocks * OMC_COLS;
  ChunkPlace at;
  if (!locate_chunk(a.chunk0 + w.x, p, a.min_len, at, a.group * CHUNK) || at.slot < 0 || at.slot >= p.num_slots) return false;
  const int first = at.c * a.group * CHUNK;
  w.tokens = min(a.group * CHUNK, at.len - first);
  w.chunks = (w.tokens + CHUNK - 1) / CHUNK;
  w.row0 = (int64_t)at.start + first;
  return true;
}

template <int MODE, int DP, bool VEC>
__global__ __launch_bounds__(256) void om_chunk_update16_kernel(OMChunk a) {
  __shared__ __attribute__((aligned(16))) uint16_t kt[DP * OMG_PITCH];
  __shared__ __attribute__((aligned(16))) uint16_t vt[OMC_COLS * OMG_PITCH];
  __shared__ __attribute__((aligned(16))) float ws[4][CHUNK];
  __shared__ float alls[4];
  const OuterMemory& p = a.p;
  OMGroup g;
  if (!locate_group(a, g)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lg = lane >> 4;
  const int nct = min(OMC_COLS / 16, (p.vdim - g.c0 + 15) >> 4);
  const uint16_t* kb = (const uint16_t*)p.k + (int64_t)g.hk * p.dim;
  const uint16_t* vb = (const uint16_t*)p.v + (int64_t)g.h * p.vdim + g.c0;
  const u32x4 zeros = {};
  u32x4 kx[DP / 32], vx[OMC_COLS / 32];
  auto fetch = [&](int c) {                                              // lane = token; the waves divide the key rows and the columns
    const int64_t row = g.row0 + min(c * CHUNK + lane, g.tokens - 1);
#pragma unroll
    for (int it = 0; it < DP / 32; ++it) kx[it] = __builtin_bit_cast(u32x4, load8_bits<VEC>(kb + row * p.k_stride, wave * (DP / 4) + it * 8, p.dim));
#pragma unroll
    for (int it = 0; it < OMC_COLS / 32; ++it) vx[it] = __builtin_bit_cast(u32x4, load8_bits<VEC>(vb + row * p.v_stride, wave * (OMC_COLS / 4) + it * 8, p.vdim - g.c0));
  };
  fetch(0);
  f32x4 S[DP / 32][2] = {};
  float sn = 0.f;
  float total = 1.f;
  for (int c = 0; c < g.chunks; ++c) {
    if ((c & 3) == 0) {                                                  // the gates of four chunks, one a wave
      double la;
      float b;
      chunk_gate<BFloat, MODE>(a, g.h, g.row0 + (c + wave) * CHUNK, lane, g.tokens - (c + wave) * CHUNK, la, b);
      const double gi = wave_incl_sum(la), gend = of_lane(gi, 63);
      ws[wave][lane] = exp2_d(gend - gi) * b;
      if (lane == 0) alls[wave] = exp2_d(gend);
    }
    if ((c + 1) * CHUNK > g.tokens && c * CHUNK + lane >= g.tokens) {
#pragma unroll
      for (int it = 0; it < DP / 32; ++it) kx[it] = zeros;
#pragma unroll
      for (int it = 0; it < OMC_COLS / 32; ++it) vx[it] = zeros;
    }
    u16x2 top = {};
#pragma unroll
    for (int it = 0; it < DP / 32; ++it) {
      largest_bits(top, kx[it]);
      put_rows(kt + lane, kx[it], [&](int i) { return key_row(wave * (DP / 4) + it * 8 + i); });
    }
#pragma unroll
    for (int it = 0; it < OMC_COLS / 32; ++it)
      put_rows(vt + lane, vx[it], [&](int i) { return wave * (OMC_COLS / 4) + it * 8 + i; });
    bool odd = odd_bits(top);
    odd = __builtin_amdgcn_readfirstlane(__syncthreads_or(odd));
    if (c + 1 < g.chunks) fetch(c + 1);
    total *= alls[c & 3];
    if (wave < nct) {
      u16x8 v[CHUNK / 32];
#pragma unroll
      for (int jj = 0; jj < CHUNK / 32; ++jj) v[jj] = *reinterpret_cast<const u16x8*>(&vt[(wave * 16 + li) * OMG_PITCH + 32 * jj + 8 * lg]);
      group_update<DP>(S, kt, v, ws[c & 3], alls[c & 3], odd, li, lg);
    }
    if (MODE == 1 && g.c0 == 0 && tid < DP) sn = group_update_n(sn, kt, ws[c & 3], alls[c & 3], tid);
    lds_barrier();
  }
  const int64_t at = (int64_t)g.x * p.heads + g.h;
  if (g.c0 == 0 && tid == 0) a.total[at] = total;
  if (MODE == 1 && g.c0 == 0 && tid < DP) a.un[at * DP + tid] = sn;
  if (wave >= nct) return;
  float* u = a.u + (at * a.vpad + g.c0 + wave * 16) * DP + lane * 4;
#pragma unroll
  for (int kk = 0; kk < DP / 32; ++kk)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) *reinterpret_cast<f32x4*>(u + (2 * kk + hf) * 256) = S[kk][hf];
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
  const int unit = a.group * CHUNK;
  if (!span_of(s, (n + unit - 1) / unit, p.q_len, a.min_len, a.chunk0, a.span, begin, nc, first, unit)) return;
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
  const int l = x & 63, f = x >> 6, e = f / (DP / 16) * 16 + (l & 15), d = (f % (DP / 16) >> 1) * 32 + (l >> 4) * 8 + (f & 1) * 4;
  float* sb = p.state_s + ((int64_t)slot * p.heads + h) * p.dim * (int64_t)p.vdim + e;
  f32x4 S = {};
  if (!fresh && e < p.vdim)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (d + i < p.dim) S[i] = sb[(int64_t)(d + i) * p.vdim];
  float* u = a.u + (first * p.heads + h) * a.vpad * (int64_t)DP + 4 * x;
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
  ChunkPlace at;
  if (!locate_chunk(a.chunk0 + blockIdx.x, p, a.min_len, at) || at.slot < 0 || at.slot >= p.num_slots) return;
  const int c = at.c;
  const int h = blockIdx.y, c0 = blockIdx.z * OMC_COLS, hk = MODE == 2 ? h / (p.heads / p.qk_heads) : h;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int cnt = min(CHUNK, at.len - c * CHUNK);
  const int64_t row0 = (int64_t)at.start + c * CHUNK;
  const int64_t row = row0 + min(lane, cnt - 1);
  const ST* kr = (const ST*)p.k + row * p.k_stride + (int64_t)hk * p.dim;
  const ST* vr = (const ST*)p.v + row * p.v_stride + (int64_t)h * p.vdim + c0;
  // the workgroup's keys and values are on their way while the waves multiply with the state; lane = token here
  float kx[DP / 32][8], vx[OMC_COLS / 32][8];
#pragma unroll
  for (int it = 0; it < DP / 32; ++it) load8<T, VEC>(kr, wave * (DP / 4) + it * 8, p.dim, kx[it]);
#pragma unroll
  for (int it = 0; it < OMC_COLS / 32; ++it) load8<T, VEC>(vr, wave * (OMC_COLS / 4) + it * 8, p.vdim - c0, vx[it]);
  if (wave == 0) {                                                       // (while they are)
    double la;
    float b;
    chunk_gate<T, MODE>(a, h, row0, lane, cnt, la, b);
    gs[lane] = chunk_decays<MODE>(la, lane, cnt);
    bs[lane] = b;
  }
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
    const float* sr = st + ct * 16 * DP + lane * 4;
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk) {
      const f32x4 s0 = *reinterpret_cast<const f32x4*>(sr + kk * 512), s1 = *reinterpret_cast<const f32x4*>(sr + kk * 512 + 256);
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

// The outputs of a group of chunks (bf16 inputs; om_chunk_update16_kernel above says how the work lies).  Per chunk: a wave's 16 queries against the keys --
// the weights go to LDS in three bf16 parts, where the keys were --, then every wave's own columns: state times all queries, values times weights, and
// the state after the chunk.  Which wave has which queries goes round: later ones see more tokens.
template <int MODE, int DP, bool VEC>
__global__ __launch_bounds__(256, 2) void om_chunk_out16_kernel(OMChunk a) {
  constexpr int KP = DP + 8, KEYS = CHUNK * KP * 2, PARTS = 3 * CHUNK * OMG_PITCH * 2;
  static_assert(PARTS >= KEYS && PARTS >= CHUNK * (CHUNK + 1) * 4, "");
  __shared__ __attribute__((aligned(16))) unsigned char room[PARTS];     // keys [token][row], then the weights' parts [3][query][token], or fp32 ones
  __shared__ __attribute__((aligned(16))) uint16_t qs[CHUNK * KP];
  __shared__ __attribute__((aligned(16))) uint16_t kt[DP * OMG_PITCH];
  __shared__ __attribute__((aligned(16))) uint16_t vt[OMC_COLS * OMG_PITCH];
  __shared__ double gs[4][CHUNK];
  __shared__ __attribute__((aligned(16))) float bs[4][CHUNK], ws[4][CHUNK];
  __shared__ float alls[4], ns[MODE == 1 ? DP : 1], invs[MODE == 1 ? CHUNK : 1];
  uint16_t* ks = reinterpret_cast<uint16_t*>(room);
  uint16_t* pp = reinterpret_cast<uint16_t*>(room);
  float* ps = reinterpret_cast<float*>(room);
  const OuterMemory& p = a.p;
  OMGroup g;
  if (!locate_group(a, g)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lg = lane >> 4;
  const int nct = min(OMC_COLS / 16, (p.vdim - g.c0 + 15) >> 4);
  const uint16_t* kb = (const uint16_t*)p.k + (int64_t)g.hk * p.dim;
  const uint16_t* qb = (const uint16_t*)p.q + (int64_t)g.hk * p.dim;
  const uint16_t* vb = (const uint16_t*)p.v + (int64_t)g.h * p.vdim + g.c0;
  const u32x4 zeros = {};
  u32x4 kx[DP / 32], qx[DP / 32], vx[OMC_COLS / 32];
  auto fetch = [&](int c) {                                              // lane = token; the waves divide the rows and the columns
    const int64_t row = g.row0 + min(c * CHUNK + lane, g.tokens - 1);
#pragma unroll
    for (int it = 0; it < DP / 32; ++it) kx[it] = __builtin_bit_cast(u32x4, load8_bits<VEC>(kb + row * p.k_stride, wave * (DP / 4) + it * 8, p.dim));
#pragma unroll
    for (int it = 0; it < DP / 32; ++it) qx[it] = __builtin_bit_cast(u32x4, load8_bits<VEC>(qb + row * p.q_stride, wave * (DP / 4) + it * 8, p.dim));
#pragma unroll
    for (int it = 0; it < OMC_COLS / 32; ++it) vx[it] = __builtin_bit_cast(u32x4, load8_bits<VEC>(vb + row * p.v_stride, wave * (OMC_COLS / 4) + it * 8, p.vdim - g.c0));
  };
  fetch(0);
  const int64_t at = (int64_t)g.x * p.heads + g.h;
  f32x4 S[DP / 32][2] = {};
  if (wave < nct) {
    const float* u = a.u + (at * a.vpad + g.c0 + wave * 16) * DP + lane * 4;
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) S[kk][hf] = *reinterpret_cast<const f32x4*>(u + (2 * kk + hf) * 256);
  }
  float sn = 0.f;
  if (MODE == 1 && tid < DP) ns[tid] = sn = a.un[at * DP + tid];
  const float scale = MODE == 1 ? p.q_scale : 1.f, skip = MODE == 2 ? p.skip[g.h] : 0.f;
  const int qt = (wave + g.x + g.h) & 3, qi = qt * 16 + li;
  for (int c = 0; c < g.chunks; ++c) {
    const int c4 = c & 3;
    if (c4 == 0) {                                                       // the gates of four chunks, one a wave
      double la;
      float b;
      chunk_gate<BFloat, MODE>(a, g.h, g.row0 + (c + wave) * CHUNK, lane, g.tokens - (c + wave) * CHUNK, la, b);
      const double gi = wave_incl_sum(la), gend = of_lane(gi, 63);
      gs[wave][lane] = gi;
      bs[wave][lane] = b;
      ws[wave][lane] = exp2_d(gend - gi) * b;
      if (lane == 0) alls[wave] = exp2_d(gend);
    }
    const int cnt = min(CHUNK, g.tokens - c * CHUNK);
    const int64_t row0 = g.row0 + c * CHUNK;
    if (cnt < CHUNK && lane >= cnt) {
#pragma unroll
      for (int it = 0; it < DP / 32; ++it) kx[it] = qx[it] = zeros;
#pragma unroll
      for (int it = 0; it < OMC_COLS / 32; ++it) vx[it] = zeros;
    }
    u16x2 top = {};
#pragma unroll
    for (int it = 0; it < DP / 32; ++it) {
      largest_bits(top, kx[it]);
      largest_bits(top, qx[it]);
      const int d = wave * (DP / 4) + it * 8;
      *reinterpret_cast<u32x4*>(&ks[lane * KP + d]) = kx[it];
      *reinterpret_cast<u32x4*>(&qs[lane * KP + d]) = qx[it];
      put_rows(kt + lane, kx[it], [&](int i) { return key_row(d + i); });
    }
#pragma unroll
    for (int it = 0; it < OMC_COLS / 32; ++it) {
      largest_bits(top, vx[it]);
      put_rows(vt + lane, vx[it], [&](int i) { return wave * (OMC_COLS / 4) + it * 8 + i; });
    }
    bool odd = odd_bits(top);                                            // a number that is not finite
    odd = __builtin_amdgcn_readfirstlane(__syncthreads_or(odd));
    if (c + 1 < g.chunks) fetch(c + 1);
    // the wave's queries against the chunk's tokens up to them
    const double gq = gs[c4][qi];
    f32x4 pr[CHUNK / 16] = {};
    int lj = li;                                                         // (not to be kept as sixteen masks from chunk to chunk)
    asm("" : "+v"(lj));
    float nq = 0.f;                                                      // mLSTM: the lane's part of n . q
    {
      u16x8 q[DP / 32];
#pragma unroll
      for (int kk = 0; kk < DP / 32; ++kk) q[kk] = *reinterpret_cast<const u16x8*>(&qs[qi * KP + 32 * kk + 8 * lg]);
      if constexpr (MODE == 1) {
#pragma unroll
        for (int kk = 0; kk < DP / 32; ++kk)
#pragma unroll
          for (int i = 0; i < 8; ++i) nq += BFloat::to_f32(q[kk][i]) * ns[32 * kk + 8 * lg + i];
        nq *= exp2_d(gq) * scale;
      }
#pragma unroll
      for (int jt = 0; jt < CHUNK / 16; ++jt) {
        if (jt > qt) break;
        const int last = jt == qt ? lj : CHUNK;
        f32x4 sc = {};
#pragma unroll
        for (int kk = 0; kk < DP / 32; ++kk) sc = mfma16(*reinterpret_cast<const u16x8*>(&ks[(jt * 16 + li) * KP + 32 * kk + 8 * lg]), q[kk], sc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = jt * 16 + 4 * lg + r;
          const float w = sc[r] * scale * (exp2_d(gq - gs[c4][j]) * bs[c4][j]);
          pr[jt][r] = 4 * lg + r > last ? 0.f : w;
          if (MODE == 1) nq += pr[jt][r];
          if (MODE == 2 && 4 * lg + r == last) pr[jt][r] += skip;               // skip times the query's own value
        }
      }
    }
    if constexpr (MODE == 1) {
      nq += __shfl_xor(nq, 16, 64);
      nq += __shfl_xor(nq, 32, 64);
      const float em = a.em[(int64_t)g.h * p.num_tokens + row0 + min(qi, cnt - 1)];
      if (lg == 0) invs[qi] = fmaxf(fabsf(nq), em) + 1e-6f;
    }
    lds_barrier();                                                       // every wave is through with the keys
    if (odd) {
#pragma unroll
      for (int jt = 0; jt < CHUNK / 16; ++jt)
        if (jt <= qt)
#pragma unroll
          for (int r = 0; r < 4; ++r) ps[qi * (CHUNK + 1) + jt * 16 + 4 * lg + r] = pr[jt][r];
    } else {
      float z = 0.f;                                                     // not zero: a sum beyond fp32's range
#pragma unroll
      for (int jt = 0; jt < CHUNK / 16; ++jt)
#pragma unroll
        for (int r = 0; r < 4; ++r) z = fmaf(pr[jt][r], 0.f, z);
      const bool all = !__any(z != 0.f);
#pragma unroll
      for (int jp = 0; jp < CHUNK / 32; ++jp) {                          // (products take 32 tokens: zeros up to there)
        if (2 * jp > qt) break;
        const float x[8] = {pr[2 * jp][0], pr[2 * jp][1], pr[2 * jp][2], pr[2 * jp][3], pr[2 * jp + 1][0], pr[2 * jp + 1][1], pr[2 * jp + 1][2], pr[2 * jp + 1][3]};
        u16x8 part[3];
        if (all) split3_finite(x, part);
        else
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            uint16_t t[3];
            split3(x[i], t);
#pragma unroll
            for (int n = 0; n < 3; ++n) part[n][i] = t[n];
          }
#pragma unroll
        for (int n = 0; n < 3; ++n) {
          const u32x4 w = __builtin_bit_cast(u32x4, part[n]);
          uint16_t* at = &pp[(n * CHUNK + qi) * OMG_PITCH + 32 * jp + 4 * lg];
          *reinterpret_cast<u32x2*>(at) = u32x2{w[0], w[1]};
          *reinterpret_cast<u32x2*>(at + 16) = u32x2{w[2], w[3]};
        }
      }
    }
    lds_barrier();
    if (wave < nct) {
      u16x8 v[CHUNK / 32];
#pragma unroll
      for (int jj = 0; jj < CHUNK / 32; ++jj) v[jj] = *reinterpret_cast<const u16x8*>(&vt[(wave * 16 + li) * OMG_PITCH + 32 * jj + 8 * lg]);
      f32x4 acc[CHUNK / 16] = {};
      float eq[CHUNK / 16];
#pragma unroll
      for (int t = 0; t < CHUNK / 16; ++t) eq[t] = exp2_d(gs[c4][t * 16 + li]) * scale;
      float z = 0.f;                                                     // not zero: a state that is not finite
#pragma unroll
      for (int kk = 0; kk < DP / 32; ++kk)
#pragma unroll
        for (int i = 0; i < 8; ++i) z = fmaf(S[kk][i >> 2][i & 3], 0.f, z);
      if (odd || __any(z != 0.f)) {
#pragma unroll
        for (int kk = 0; kk < DP / 32; ++kk)
#pragma unroll
          for (int t = 0; t < CHUNK / 16; ++t) {
            const u16x8 q = *reinterpret_cast<const u16x8*>(&qs[(t * 16 + li) * KP + 32 * kk + 8 * lg]);
#pragma unroll
            for (int m = 0; m < 8; ++m) acc[t] = mfma4(S[kk][m >> 2][m & 3], BFloat::to_f32(q[m]), acc[t]);
          }
      } else {
#pragma unroll
        for (int kk = 0; kk < DP / 32; ++kk) {                           // what the state ahead of the chunk gives
          u16x8 part[3], q[CHUNK / 16];
          const float x[8] = {S[kk][0][0], S[kk][0][1], S[kk][0][2], S[kk][0][3], S[kk][1][0], S[kk][1][1], S[kk][1][2], S[kk][1][3]};
          split3_finite(x, part);
#pragma unroll
          for (int t = 0; t < CHUNK / 16; ++t) q[t] = *reinterpret_cast<const u16x8*>(&qs[(t * 16 + li) * KP + 32 * kk + 8 * lg]);
#pragma unroll
          for (int n = 2; n >= 0; --n)
#pragma unroll
            for (int t = 0; t < CHUNK / 16; ++t) acc[t] = mfma16(part[n], q[t], acc[t]);
        }
      }
#pragma unroll
      for (int t = 0; t < CHUNK / 16; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[t][r] *= eq[t];
      if (!odd) {
#pragma unroll
        for (int jj = 0; jj < CHUNK / 32; ++jj)
#pragma unroll
          for (int n = 2; n >= 0; --n)
#pragma unroll
            for (int t = 2 * jj; t < CHUNK / 16; ++t)
              acc[t] = mfma16(v[jj], *reinterpret_cast<const u16x8*>(&pp[(n * CHUNK + t * 16 + li) * OMG_PITCH + 32 * jj + 8 * lg]), acc[t]);
      } else {
        // zero times a value that is not finite is not zero: a token behind the query must not be multiplied at all
#pragma unroll
        for (int t = 0; t < CHUNK / 16; ++t) {
          const uint16_t* vr = &vt[(wave * 16 + 4 * lg) * OMG_PITCH];
          f32x4 sum = {};
#pragma unroll 1
          for (int j = 0; j <= t * 16 + li; ++j) {
            const float w = ps[(t * 16 + li) * (CHUNK + 1) + j];
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[r] += w * BFloat::to_f32(vr[r * OMG_PITCH + j]);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[t][r] += sum[r];
        }
      }
      const int e = wave * 16 + 4 * lg;
      float* o = p.out + row0 * ((int64_t)p.heads * p.vdim) + (int64_t)g.h * p.vdim + g.c0 + e;
#pragma unroll
      for (int t = 0; t < CHUNK / 16; ++t) {
        const int j = t * 16 + li;
        f32x4 x = acc[t];
        const float inv = MODE == 1 ? invs[j] : 1.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (MODE == 1) x[r] = x[r] / inv;
        }
        if (j >= cnt) continue;
        float* oj = o + (int64_t)j * p.heads * p.vdim;
        if ((p.vdim & 3) == 0) {
          if (g.c0 + e < p.vdim) *reinterpret_cast<f32x4*>(oj) = x;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (g.c0 + e + r < p.vdim) oj[r] = x[r];
        }
      }
      if (c + 1 < g.chunks) group_update<DP>(S, kt, v, ws[c4], alls[c4], odd, li, lg);
    }
    if (c + 1 == g.chunks) return;
    if (MODE == 1 && tid < DP) ns[tid] = sn = group_update_n(sn, kt, ws[c4], alls[c4], tid);
    lds_barrier();
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

// Chunks of a workgroup (bf16 mLSTM and state space): more of them cost parallelism, fewer the traffic of their states.  Measured, us, with 1 / 2 / 4 / 8 /
// 16: state space 64 heads 300 tokens (320 workgroups of one chunk) 38 / 39 / 51, 600 (640) 56 / 50 / 55, 2000 (2048) 109 / 85 / 75 / 90,
// 4096 (4160) 199 / 148 / 126 / 120 / 192; 128 heads 1024 (2176) 111 / 88 / 75 / 112, 4096 (8320) 484 / 294 / 235 / 211 / 200; mLSTM 4 x 128 x 256
// 2000 (512) 50 / 51 / 61, 4096 (1040) 83 / 65 / 78, 16384 (4112) 275 / 209 / 176 / 160 / 238.  Chunks are counted from the tokens: beside a prompt the
// bound over segments would count every decoded sequence as one.
static int om_group_chunks(const OuterMemory& p) {
  if (p.mode == 0 || p.dtype != APHRO_BF16) return 1;
  const int64_t units = (p.num_tokens / CHUNK + 1) * p.heads * ((p.vdim + OMC_COLS - 1) / OMC_COLS);
  return units < 600 ? 1 : units < 1200 ? 2 : units < 4000 ? 4 : 8;
}

template <typename T, int MODE, int DP, bool VEC>
static void om_chunk_launch(OMChunk a, int64_t chunks) {
  const OuterMemory& p = a.p;
  const dim3 grid((unsigned)a.span, (unsigned)p.heads, (unsigned)((p.vdim + OMC_COLS - 1) / OMC_COLS));
  const unsigned pairs = (unsigned)a.span * (unsigned)om_key_heads(p);
  const unsigned subs = (unsigned)(p.heads / om_key_heads(p)) * grid.z;
  const dim3 grid16(om_split_pairs(pairs, (int)subs) ? pairs * ((subs + 7) / 8) * 8 : (pairs + 7) / 8 * 8 * subs);
  const unsigned items = (unsigned)a.vpad * (DP / 4) + (MODE == 1 ? DP : 0);
  if (MODE == 1) hipLaunchKernelGGL((om_gates_kernel<T>), dim3((unsigned)p.num_seqs, (unsigned)p.heads), dim3(1024), 0, p.stream, a);
  for (; a.chunk0 < chunks; a.chunk0 += a.span) {
    constexpr bool B16 = sizeof(typename T::storage) == 2 && MODE != 0;
    if constexpr (B16) hipLaunchKernelGGL((om_chunk_update16_kernel<MODE, DP, VEC>), grid16, dim3(256), 0, p.stream, a);
    else hipLaunchKernelGGL((om_chunk_update_kernel<T, MODE, DP, VEC>), grid, dim3(256), 0, p.stream, a);
    hipLaunchKernelGGL((om_chunk_carry_kernel<MODE, DP>), dim3((items + 63) / 64, (unsigned)p.heads, (unsigned)p.num_seqs), dim3(64), 0, p.stream, a);
    if constexpr (B16) hipLaunchKernelGGL((om_chunk_out16_kernel<MODE, DP, VEC>), grid16, dim3(256), 0, p.stream, a);
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
  int64_t chunks = max_chunks(num_tokens, num_seqs, min_len);
  APHRO_CHECK(chunks <= 0x3fffffff, "outer_memory_chunked: too many tokens");
  a.group = om_group_chunks(p);
  if (a.group > 1) chunks = max_chunks(num_tokens, num_seqs, min_len, a.group * CHUNK);
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
