// The gated delta rule (delta_rule.hip has the recurrence) over prompt portions, in chunks of 64 tokens on the matrix cores.  With g_t the
// decay (per key channel, or the same for all), P_ij = the product of g over tokens j + 1 .. i, Pi_i = P_i,-1 and S the state ahead of the chunk,
//     u_i = beta_i (v_i - S^T (Pi_i k_i) - sum_{j < i} (k_i . P_ij k_j) u_j),   o_i = S^T (Pi_i q_i) + sum_{j <= i} (q_i . P_ij k_j) u_j
//     S' = Pi_63 S + sum_j (P_63,j k_j) u_j^T
// so with L_ij = beta_i (k_i . P_ij k_j) for j < i, and T = (1 + L)^-1 diag(beta):   U = T V - T (Pi K) S.
//   1. gd_chunk_prepare: everything of a chunk and head that does not need S -- T V, W = T (Pi K), Pi Q, (P_63 K)^T, the scores of o -- all
//      chunks at once
//   2. gd_chunk_carry:   U = T V - W S and S' through the chunks of a segment, sixteen value columns a workgroup (columns never meet)
//   3. gd_chunk_out:     o of every chunk -- all chunks at once
// Everything is fp32, products on v_mfma_f32_16x16x4_f32.  The decays enter as products of g, never as differences of logarithms: within
// a block of 16 tokens token by token (the 16 x 16 scores of a block with itself run on the vector ALUs, g folded in on the way), between
// blocks as (from the block's start) x (whole blocks between) x (to the block's end) -- factors of at most one, as exact as the scan's.
//
// A token whose k, beta or g is not finite, and a value that is not, would reach tokens ahead of it in the products (zero times NaN): they are
// entered as a token without effect, and the chunk says from where on outputs and state are NaN (`bad_token`, `bad_value`).  So is a u
// that overflows.
//
// What bounds it: the scan is bound by the latency of its token chain; here launch 2's chain is one of 64-token steps (two products of 64 x
// dim x 16 and two barriers each), launches 1 and 3 have all chunks to fill the chip (launch 1 one workgroup a CU:
// its rows of q, k and g take the LDS).  16 heads of 128 x 128, a decay per channel, one portion: 512 tokens 85 -> 64 us (scan 193), 2000 tokens 198 -> 138,
// 4096 tokens 394 -> 276 (a decay per head 355 -> 261); 32 heads of 64 x 64, 2000 tokens 178 -> 134.  What that took, launches 1 / 2 / 3 at 2000
// tokens 82 / 88 / 39 us: matrices between the launches as rows, of which a load of 16 bytes a lane met another cache line in every lane of
// four, so that the address unit, not the matrix pipe, was waited for (in fragments: launch 2 63, launch 3 30; launch 2's loads between its
// products: 53); decays one after the other, each with a load of its own and log1pf (launch 1: 25 000 cycles of a chunk's 87 000, now 10 000); a block
// with itself without LDS, values loaded ahead: 62.  Left in launch 1: 2 rounds of a workgroup a CU, 64 000 cycles each, half of them waits; in launch 2
// 2 050 of a step's 3 600 cycles are fp32 products.
#include <type_traits>
#include <utility>

#include "delta_rule.h"
#include "chunked_scan.h"

namespace aphro {

constexpr int GDC_P = CHUNK + 4;         // pitch of [.., 64] rows in LDS: 4 floats over a multiple of 32 (chunked_scan.h's access width)

struct GDChunk {
  GatedDelta p;
  int min_len;
  int chunk0, span;        // the chunks of these launches (below: [chunks] of one span)
  int vpad;                // vdim rounded up to 16
  // Matrices lie in the fragments that the waves read, 1 KiB each with a lane's four numbers next to each other: lane (li, lg) = (l % 16, l / 16) of
  // fragment (i, j) has row 16 i + li and columns 16 j + 4 lg + (0..3), or, of an array marked *, of fragment (i, 2 j + u) columns 32 j + 8 lg + 4 u + (0..3).
  float* w;                // [chunks, heads] 64 x DP *   T (Pi K)
  float* qg;               // [chunks, heads] 64 x DP *   Pi Q
  float* kd;               // [chunks, heads] DP x 64     (P_63 K)^T
  float* bm;               // [chunks, heads] 64 x 64     q_i . P_ij k_j, zero above the diagonal of a block with itself, unwritten in later blocks
  float* ut;               // [chunks, heads] vpad x 64   T V, then U
  float* st;               // [chunks, heads] vpad x DP * the state ahead of the chunk
  float* gam;              // [chunks, heads, DP]      Pi_63
  int32_t* bad_token;      // [chunks, heads]          first token that is not finite (64: none)
  int32_t* bad_value;      // [chunks, heads, vpad]    first value, or u, of the column that is not finite (64: none)
};

// x of lane I of the own sixteen.
template <int I>
__device__ __forceinline__ float of_lane16(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + I, 0xf, 0xf, true));
}
// p += sum of x[.] of lane I of the own sixteen times e[.], and q with y.  (hipcc folds the lane's choice into a product, not into an FMA.  The s_nop: what a
// lane's choice reads has to be two steps old.)
template <int I>
__device__ __forceinline__ void fma_of_lane16(float& p, const f32x4& x, float& q, const f32x4& y, const f32x4& e) {
#define GDC_FMA(ACC, X, E) "v_fmac_f32_dpp " ACC ", " X ", " E " row_newbcast:%14 row_mask:0xf bank_mask:0xf\n\t"
  asm("s_nop 1\n\t" GDC_FMA("%0", "%2", "%10") GDC_FMA("%1", "%6", "%10") GDC_FMA("%0", "%3", "%11") GDC_FMA("%1", "%7", "%11")
      GDC_FMA("%0", "%4", "%12") GDC_FMA("%1", "%8", "%12") GDC_FMA("%0", "%5", "%13") GDC_FMA("%1", "%9", "%13")
      : "+v"(p), "+v"(q)
      : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(e[0]), "v"(e[1]), "v"(e[2]), "v"(e[3]), "n"(I));
#undef GDC_FMA
}
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
template <typename F, int... I>
__device__ __forceinline__ void each16_(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }

template <int DP>
constexpr size_t gd_prepare_lds() { return (3 * CHUNK * (DP + 4) + 2 * CHUNK * GDC_P + 4 * DP + CHUNK + 2 * (DP / 16) * CHUNK + CHUNK + 4) * sizeof(float); }

// ---- 1. what a chunk needs no state for --------------------------------------------------------------------------------------------------
// LDS lets one workgroup on a CU: it has a wave per 16 key channels (two per SIMD at 128).
template <typename T, int DP, bool CHANNEL, bool VEC>
__global__ __launch_bounds__(DP * 4) void gd_chunk_prepare_kernel(GDChunk a) {
  typedef typename T::storage ST;
  constexpr int KP = DP + 4, NW = DP / 16, HALVES = NW / 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* kk = lds;                         // [64][KP] k, then k from its block's start, then Pi K
  float* qq = kk + CHUNK * KP;             // [64][KP] q, ...; then V^T [64 columns][GDC_P]
  float* gg = qq + CHUNK * KP;             // [64][KP] g, then k to its block's end
  float* lm = gg + CHUNK * KP;             // [64][GDC_P] L
  float* tm = lm + CHUNK * GDC_P;          // [64][GDC_P] (1 + L)^-1, then T
  float* dd = tm + CHUNK * GDC_P;          // [4][DP] product of a block's g
  float* bet = dd + 4 * DP;                // [64]
  float* red = bet + CHUNK;                // [2][NW][64]
  int* bad_col = (int*)(red + 2 * NW * CHUNK);   // [64]
  int* bad_tok = bad_col + CHUNK;          // [1]
  const GatedDelta& p = a.p;
  ChunkPlace at;
  if (!locate_chunk(a.chunk0 + blockIdx.x, p, a.min_len, at) || at.slot < 0 || at.slot >= p.num_slots) return;
  const int c = at.c;
  const int h = blockIdx.y, hk = h / (p.heads / p.kv_heads);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int cnt = min(CHUNK, at.len - c * CHUNK);
  const int64_t row0 = (int64_t)at.start + c * CHUNK, row = row0 + min(lane, cnt - 1);
  const int64_t unit = (int64_t)blockIdx.x * p.heads + h;
  const bool live = lane < cnt;
  // -- q, k, g, beta: lane = token, the waves divide the key channels
  {
    float q[2][8], k[2][8], g[2][8];
    const ST* qr = (const ST*)p.q + row * p.q_stride + (int64_t)hk * p.dim;
    const ST* kr = (const ST*)p.k + row * p.k_stride + (int64_t)hk * p.dim;
    const ST* ar = (const ST*)p.a + row * p.a_stride + (CHANNEL ? (int64_t)h * p.dim : (int64_t)h);
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int d = wave * 16 + it * 8;
      load8<T, VEC>(qr, d, p.dim, q[it]);
      load8<T, VEC>(kr, d, p.dim, k[it]);
      if constexpr (CHANNEL) load8<T, VEC>(ar, d, p.dim, g[it]);
    }
    float bias[2][8];                                      // (loaded here, not where each is used: sixteen loads to wait for one after the other)
    if constexpr (CHANNEL)
#pragma unroll
      for (int it = 0; it < 2; ++it)
#pragma unroll
        for (int i = 0; i < 8; ++i) bias[it][i] = p.dt_bias[(int64_t)h * p.dim + min(wave * 16 + it * 8 + i, p.dim - 1)];
    const float raw_b = T::to_f32(((const ST*)p.b)[row * p.b_stride + h]);
    const float rate = -expf(p.a_log[h]);
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int i = 0; i < 8; ++i) sq += q[it][i] * q[it][i], sk += k[it][i] * k[it][i];
    red[wave * CHUNK + lane] = sq;
    red[(NW + wave) * CHUNK + lane] = sk;
    if (tid == 0) *bad_tok = CHUNK;
    for (int i = tid; i < CHUNK * GDC_P; i += NW * 64) lm[i] = tm[i] = 0.f;
    __syncthreads();
    sq = sk = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) sq += red[w * CHUNK + lane], sk += red[(NW + w) * CHUNK + lane];
    const float fq = p.q_scale / sqrtf(sq + p.norm_eps), fk = 1.0f / sqrtf(sk + p.norm_eps);
    float beta = live ? sigmoid_f(raw_b) : 0.f, gh = 1.f;
    if constexpr (!CHANNEL) gh = expf(rate * softplus_f(T::to_f32(*ar) + p.dt_bias[h]));
    bool bad = !finite_f(beta);
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int d = wave * 16 + it * 8 + i;
        q[it][i] = live ? q[it][i] * fq : 0.f;
        k[it][i] = live ? k[it][i] * fk : 0.f;
        if constexpr (CHANNEL) {
          const float z = expf(rate * softplus_f(g[it][i] + bias[it][i]));
          g[it][i] = d < p.dim && live ? z : 1.f;
        }
        else g[it][i] = live ? gh : 1.f;
        bad |= !finite_f(k[it][i]) || !finite_f(g[it][i]);
      }
    const uint64_t mask = __ballot(bad && live);
    if (mask && lane == 0) atomicMin(bad_tok, __ffsll((unsigned long long)mask) - 1);
    __syncthreads();
    const bool mute = lane >= *bad_tok;                   // no effect, and what follows is NaN whatever it is
    if (wave == 0) bet[lane] = mute ? 0.f : beta;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int d = wave * 16 + it * 8;
      f32x4 lo, hi;
#pragma unroll
      for (int i = 0; i < 4; ++i) lo[i] = mute ? 0.f : k[it][i], hi[i] = mute ? 0.f : k[it][4 + i];
      *reinterpret_cast<f32x4*>(&kk[lane * KP + d]) = lo;
      *reinterpret_cast<f32x4*>(&kk[lane * KP + d + 4]) = hi;
#pragma unroll
      for (int i = 0; i < 4; ++i) lo[i] = mute ? 1.f : g[it][i], hi[i] = mute ? 1.f : g[it][4 + i];
      *reinterpret_cast<f32x4*>(&gg[lane * KP + d]) = lo;
      *reinterpret_cast<f32x4*>(&gg[lane * KP + d + 4]) = hi;
#pragma unroll
      for (int i = 0; i < 4; ++i) lo[i] = q[it][i], hi[i] = q[it][4 + i];
      *reinterpret_cast<f32x4*>(&qq[lane * KP + d]) = lo;
      *reinterpret_cast<f32x4*>(&qq[lane * KP + d + 4]) = hi;
    }
  }
  __syncthreads();
  if (tid == 0) a.bad_token[unit] = *bad_tok;
  float* bmu = a.bm + unit * CHUNK * CHUNK;
  // -- a block of 16 tokens with itself: a wave takes a block (and, where there are two waves for it, half of the channels); lane = (token j,
  // quarter of those channels), i runs from j on and E = P_ij k_j with it
  {
    float la[16], lb[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) la[i] = lb[i] = 0.f;
    constexpr int PART = DP / 4 / HALVES;
    const int b0 = (wave & 3) * 16, r0 = (wave >> 2) * (DP / 2) + lg * PART;
#pragma unroll 2
    for (int r = r0; r < r0 + PART; r += 4) {
      // a lane's own rows; token i's numbers come from lane i of the sixteen inside the instruction that uses them (read from LDS by every lane: 17 300
      // cycles for 12 700)
      const f32x4 kj = *reinterpret_cast<const f32x4*>(&kk[(b0 + li) * KP + r]);
      const f32x4 gj = *reinterpret_cast<const f32x4*>(&gg[(b0 + li) * KP + r]);
      const f32x4 qj = *reinterpret_cast<const f32x4*>(&qq[(b0 + li) * KP + r]);
      f32x4 e = {0.f, 0.f, 0.f, 0.f};
      each16_([&](auto ii) {
        constexpr int i = decltype(ii)::value;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float d = e[x] * of_lane16<i>(gj[x]);
          e[x] = i == li ? kj[x] : d;
        }
        fma_of_lane16<i>(la[i], kj, lb[i], qj, e);
      }, std::make_integer_sequence<int, 16>{});
    }
    // sums over the quarters; sixteens 0 and 2 keep L, 1 and 3 the scores, of tokens i = 0..7 (sixteens 0 and 1) and 8..15
    float sum[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sum[i] = swap_add32(swap_add16(la[i], lb[i]), swap_add16(la[i + 8], lb[i + 8]));
    const int i0 = (lg >> 1) * 8;
    if constexpr (HALVES == 2) {
      float* half = tm + (b0 + (lane >> 2)) * GDC_P + (lane & 3) * 8;        // eight numbers of a lane, in rows of the block
      if (wave >= 4)
#pragma unroll
        for (int u = 0; u < 2; ++u) *reinterpret_cast<f32x4*>(half + 4 * u) = f32x4{sum[4 * u], sum[4 * u + 1], sum[4 * u + 2], sum[4 * u + 3]};
      __syncthreads();
      if (wave < 4)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(half + 4 * u);
#pragma unroll
          for (int i = 0; i < 4; ++i) sum[4 * u + i] += x[i];
        }
      __syncthreads();
      for (int i = tid; i < CHUNK * 32; i += NW * 64) tm[(i >> 5) * GDC_P + (i & 31)] = 0.f;
    }
    if (wave < 4) {
      if (lg & 1) {
        float* at = bmu + wave * 5 * 256 + (li >> 2) * 64 + (li & 3);
#pragma unroll
        for (int i = 0; i < 8; ++i) at[(i0 + i) * 4] = i0 + i >= li ? sum[i] : 0.f;
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (i0 + i > li) lm[(b0 + i0 + i) * GDC_P + b0 + li] = bet[b0 + i0 + i] * sum[i];
      }
    }
  }
  __syncthreads();
  // -- decays from a block's start and to its end, folded into q and k; thread = (channel, block)
  {
    const int x = tid, r = x % DP, b0 = x / DP * 16;
    float g[16], k[16], f = 1.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) g[i] = gg[(b0 + i) * KP + r], k[i] = kk[(b0 + i) * KP + r];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      f *= g[i];
      kk[(b0 + i) * KP + r] = f * k[i];
      qq[(b0 + i) * KP + r] *= f;
    }
    dd[x] = f;
    f = 1.f;
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      gg[(b0 + i) * KP + r] = f * k[i];
      f *= g[i];
    }
  }
  __syncthreads();
  // -- a block with an earlier one: six pairs (I, J), the whole blocks between them folded into J's side
  for (int x = wave; x < 6; x += NW) {
    const int I = x < 3 ? 3 : x < 5 ? 2 : 1, J = x < 3 ? x : x < 5 ? x - 3 : 0;
    f32x4 al = {}, ab = {};
#pragma unroll
    for (int k8 = 0; k8 < DP / 32; ++k8) {
      const int r = 32 * k8 + 8 * lg;
      f32x4 bj[2], ki[2], qi[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        bj[u] = *reinterpret_cast<const f32x4*>(&gg[(J * 16 + li) * KP + r + 4 * u]);
        ki[u] = *reinterpret_cast<const f32x4*>(&kk[(I * 16 + li) * KP + r + 4 * u]);
        qi[u] = *reinterpret_cast<const f32x4*>(&qq[(I * 16 + li) * KP + r + 4 * u]);
        for (int m = J + 1; m < I; ++m) {
          const f32x4 d = *reinterpret_cast<const f32x4*>(&dd[m * DP + r + 4 * u]);
#pragma unroll
          for (int y = 0; y < 4; ++y) bj[u][y] *= d[y];
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          al = mfma4(ki[u][y], bj[u][y], al);
          ab = mfma4(bj[u][y], qi[u][y], ab);             // (a lane: a query, four neighbouring keys)
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = I * 16 + 4 * lg + r;
      lm[i * GDC_P + J * 16 + li] = bet[i] * al[r];
    }
    *reinterpret_cast<f32x4*>(&bmu[(I * 4 + J) * 256 + lane * 4]) = ab;
  }
  __syncthreads();
  // -- (1 + L)^-1: blocks on the diagonal by substitution (wave = block, lane = column), the others by products, one diagonal after the other
  if (wave < 4) {
    const int b0 = wave * 16;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float sum = i == li ? 1.f : 0.f;
#pragma unroll
      for (int m = 0; m < i; ++m) sum -= lm[(b0 + i) * GDC_P + b0 + m] * x[m];
      x[i] = i < li ? 0.f : sum;
    }
    if (lg == 0)
#pragma unroll
      for (int i = 0; i < 16; ++i) tm[(b0 + i) * GDC_P + b0 + li] = x[i];
  }
  __syncthreads();
  for (int off = 1; off < 4; ++off) {
    if (wave < 4 - off) {
      const int I = wave + off, J = wave;
      f32x4 acc = {};
      for (int m = J; m < I; ++m) {
        const f32x4 l = *reinterpret_cast<const f32x4*>(&lm[(I * 16 + li) * GDC_P + m * 16 + 4 * lg]);
#pragma unroll
        for (int y = 0; y < 4; ++y) acc = mfma4(l[y], tm[(m * 16 + 4 * lg + y) * GDC_P + J * 16 + li], acc);
      }
      const f32x4 t = *reinterpret_cast<const f32x4*>(&tm[(I * 16 + li) * GDC_P + I * 16 + 4 * lg]);
      f32x4 res = {};
#pragma unroll
      for (int y = 0; y < 4; ++y) res = mfma4(t[y], acc[y], res);
#pragma unroll
      for (int r = 0; r < 4; ++r) tm[(I * 16 + 4 * lg + r) * GDC_P + J * 16 + li] = -res[r];
    }
    __syncthreads();
  }
  // -- T = (1 + L)^-1 diag(beta); q and k decayed over whole blocks too; what the other launches read of them leaves
  for (int i = tid; i < CHUNK * CHUNK; i += NW * 64) tm[(i >> 6) * GDC_P + (i & 63)] *= bet[i & 63];
  {
    float* qg = a.qg + unit * CHUNK * DP;
    float* kd = a.kd + unit * DP * CHUNK;
    const int blk = lane >> 4;                              // lane = token; the waves divide the channels
    for (int it = 0; it < 4; ++it) {
      const int r = wave * 16 + it * 4;
      f32x4 pre = {1.f, 1.f, 1.f, 1.f};
      for (int m = 0; m < 3; ++m) {
        const f32x4 d = *reinterpret_cast<const f32x4*>(&dd[m * DP + r]);
#pragma unroll
        for (int y = 0; y < 4; ++y)
          if (m < blk) pre[y] *= d[y];
      }
      f32x4 k = *reinterpret_cast<const f32x4*>(&kk[lane * KP + r]), q = *reinterpret_cast<const f32x4*>(&qq[lane * KP + r]);
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        k[y] *= pre[y];
        q[y] *= pre[y];
      }
      *reinterpret_cast<f32x4*>(&kk[lane * KP + r]) = k;
      *reinterpret_cast<f32x4*>(&qg[frag8<DP>(blk, wave, li, it)]) = q;
    }
    {                                                       // the same of k to the chunk's end: a wave's sixteen channels, four neighbouring tokens a lane
      float suf = 1.f;
      for (int m = 3; m >= 0; --m) {
        f32x4 e;
#pragma unroll
        for (int y = 0; y < 4; ++y) e[y] = gg[(16 * m + 4 * lg + y) * KP + wave * 16 + li] * suf;
        *reinterpret_cast<f32x4*>(&kd[(wave * 4 + m) * 256 + lane * 4]) = e;
        suf *= dd[m * DP + wave * 16 + li];
      }
    }
    for (int r = tid; r < DP; r += NW * 64) a.gam[unit * DP + r] = (dd[r] * dd[DP + r]) * (dd[2 * DP + r] * dd[3 * DP + r]);
  }
  __syncthreads();
  // (the first values are on their way meanwhile)
  constexpr int LOADS = 8 / NW;
  float x[LOADS][8];
  auto values = [&](int c0) {
    const ST* vr = (const ST*)p.v + row * p.v_stride + (int64_t)h * p.vdim + c0;
#pragma unroll
    for (int it = 0; it < LOADS; ++it) load8<T, VEC>(vr, (wave * LOADS + it) * 8, p.vdim - c0, x[it]);
  };
  values(0);
  // -- W^T = (Pi K)^T T^T: a wave's 16 channels x the tokens, four neighbouring channels a lane
  {
    f32x4 acc[4] = {};
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      f32x4 kt;
#pragma unroll
      for (int y = 0; y < 4; ++y) kt[y] = kk[(16 * k4 + 4 * lg + y) * KP + wave * 16 + li];
#pragma unroll
      for (int it = k4; it < 4; ++it) {
        const f32x4 t = *reinterpret_cast<const f32x4*>(&tm[(it * 16 + li) * GDC_P + 16 * k4 + 4 * lg]);
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[it] = mfma4(kt[y], t[y], acc[it]);
      }
    }
    float* w = a.w + unit * CHUNK * DP;
#pragma unroll
    for (int it = 0; it < 4; ++it) *reinterpret_cast<f32x4*>(&w[frag8<DP>(it, wave, li, lg)]) = acc[it];
  }
  // -- T V, 64 value columns at a time: a wave takes 16 columns x the tokens (or every other 16 of them), four neighbouring tokens a lane
  float* vt = qq;
  for (int c0 = 0; c0 < p.vdim; c0 += 64) {
#pragma unroll
    for (int it = 0; it < LOADS; ++it)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int e = (wave * LOADS + it) * 8 + i;
        const float val = live ? x[it][i] : 0.f;
        const bool fine = finite_f(val);
        const uint64_t mask = __ballot(!fine);
        vt[e * GDC_P + lane] = fine ? val : 0.f;
        if (lane == 0) bad_col[e] = mask ? __ffsll((unsigned long long)mask) - 1 : CHUNK;
      }
    __syncthreads();
    if (c0 + 64 < p.vdim) values(c0 + 64);
    if (tid < 64 && c0 + tid < a.vpad) a.bad_value[unit * a.vpad + c0 + tid] = bad_col[tid];
    const int ct = wave & 3;
    if (c0 + ct * 16 < a.vpad) {
      float* ut = a.ut + (unit * a.vpad + c0 + ct * 16) * CHUNK + lane * 4;
#pragma unroll
      for (int i = 0; i < 4 / HALVES; ++i) {
        const int it = HALVES == 2 ? 2 * i + (wave >> 2) : i;
        f32x4 acc = {};
        for (int k4 = 0; k4 <= it; ++k4) {
          const f32x4 vv = *reinterpret_cast<const f32x4*>(&vt[(ct * 16 + li) * GDC_P + 16 * k4 + 4 * lg]);
          const f32x4 t = *reinterpret_cast<const f32x4*>(&tm[(it * 16 + li) * GDC_P + 16 * k4 + 4 * lg]);
#pragma unroll
          for (int y = 0; y < 4; ++y) acc = mfma4(t[y], vv[y], acc);
        }
        *reinterpret_cast<f32x4*>(&ut[it * 256]) = acc;
      }
    }
    __syncthreads();
  }
}

// ---- 2. the state through the chunks ---------------------------------------------------------------------------------------------------
// A workgroup carries sixteen value columns of a (segment, head): the state lies in the waves' registers (a wave's key channels) and once in
// LDS for all; U = T V - W S with 16 tokens a wave, S' with the wave's channels.  The next chunk's operands are on their way meanwhile.
// Heads are the fast index of the grid: with eight XCDs taking workgroups in turn, the column blocks of a head, which read the same operands,
// share an L2.
template <int DP>
struct GDCarry {
  f32x4 w[DP / 32][2], kd[DP / 64][4], gam[DP / 64], ut;
  int bad_token, bad_value;
};

template <int DP>
__global__ __launch_bounds__(256) void gd_chunk_carry_kernel(GDChunk a) {
  constexpr int DT = DP / 64, SP = DP + 4;
  __shared__ __attribute__((aligned(16))) float ss[16 * SP];
  __shared__ __attribute__((aligned(16))) float us[16 * GDC_P];
  const GatedDelta& p = a.p;
  const int s = blockIdx.z, h = blockIdx.x, c0 = blockIdx.y * 16;
  const int n = p.q_len[s], slot = p.slot_of_seq[s];
  if (n < a.min_len || slot < 0 || slot >= p.num_slots) return;
  int begin, nc;
  int64_t first;
  if (!span_of(s, (n + CHUNK - 1) / CHUNK, p.q_len, a.min_len, a.chunk0, a.span, begin, nc, first)) return;
  first += begin, nc -= begin;                             // (chunks are numbered from the span's first from here on)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int col = c0 + li;
  float* sb = p.state + ((int64_t)slot * p.heads + h) * p.dim * (int64_t)p.vdim + col;
  const bool fresh = begin == 0 && p.ctx_len[s] == 0;
  f32x4 S[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = (wave * DT + dt) * 16 + 4 * lg + r;
      S[dt][r] = !fresh && d < p.dim && col < p.vdim ? sb[(int64_t)d * p.vdim] : 0.f;
    }
  // a chunk's operands in pieces: the loads of the next chunk go out between this one's products, as 21 loads in a row hold the wave up for 1 250 cycles
  auto unit_of = [&](int c) { return (first + min(c, nc - 1)) * p.heads + h; };
  auto fetch_w = [&](int64_t unit, GDCarry<DP>& x, int k8, int u) {
    x.w[k8][u] = *reinterpret_cast<const f32x4*>(a.w + unit * CHUNK * DP + wave * 16 * DP + (2 * k8 + u) * 256 + lane * 4);
  };
  auto fetch_kd = [&](int64_t unit, GDCarry<DP>& x, int dt, int k4) {
    x.kd[dt][k4] = *reinterpret_cast<const f32x4*>(a.kd + unit * DP * CHUNK + (wave * DT + dt) * 16 * CHUNK + k4 * 256 + lane * 4);
  };
  auto fetch_rest = [&](int64_t unit, GDCarry<DP>& x) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) x.gam[dt] = *reinterpret_cast<const f32x4*>(a.gam + unit * DP + (wave * DT + dt) * 16 + 4 * lg);
    x.ut = *reinterpret_cast<const f32x4*>(a.ut + (unit * a.vpad + c0) * CHUNK + wave * 256 + lane * 4);
    x.bad_token = a.bad_token[unit];
    x.bad_value = a.bad_value[unit * a.vpad + col];
  };
  auto step = [&](int c, const GDCarry<DP>& x, GDCarry<DP>& y) {
    const int64_t next = unit_of(c + 1);
    const int64_t unit = (first + c) * p.heads + h;
    float* st = a.st + (unit * a.vpad + c0) * DP;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int d = (wave * DT + dt) * 16 + 4 * lg;
      *reinterpret_cast<f32x4*>(&ss[li * SP + d]) = S[dt];
      *reinterpret_cast<f32x4*>(&st[frag8<DP>(0, wave * DT + dt, li, lg)]) = S[dt];
    }
    lds_barrier();
    f32x4 acc[2] = {}, sv[DP / 32][2];
#pragma unroll
    for (int k8 = 0; k8 < DP / 32; ++k8)
#pragma unroll
      for (int u = 0; u < 2; ++u) sv[k8][u] = *reinterpret_cast<const f32x4*>(&ss[li * SP + 32 * k8 + 8 * lg + 4 * u]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k8 = 0; k8 < DP / 32; ++k8)
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
#pragma unroll
        for (int m = i; m < i + 2; ++m)
#pragma unroll
          for (int u = 0; u < 2; ++u) acc[u] = mfma4(x.w[k8][u][m], sv[k8][u][m], acc[u]);
        __builtin_amdgcn_sched_barrier(0);
        fetch_w(next, y, k8, i >> 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    f32x4 uv;
#pragma unroll
    for (int r = 0; r < 4; ++r) uv[r] = x.ut[r] - (acc[0][r] + acc[1][r]);
    *reinterpret_cast<f32x4*>(&us[li * GDC_P + wave * 16 + 4 * lg]) = uv;
    if (!(finite_f(uv[0]) && finite_f(uv[1]) && finite_f(uv[2]) && finite_f(uv[3]))) {      // (overflowed: the state takes it as it is)
#pragma unroll
      for (int r = 3; r >= 0; --r)
        if (!finite_f(uv[r])) {
          atomicMin(&a.bad_value[unit * a.vpad + col], wave * 16 + 4 * lg + r);
          uv[r] = 0.f;
        }
    }
    *reinterpret_cast<f32x4*>(a.ut + (unit * a.vpad + c0) * CHUNK + wave * 256 + lane * 4) = uv;
    lds_barrier();
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[dt][r] *= x.gam[dt][r];
    f32x4 u4[4];
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) u4[k4] = *reinterpret_cast<const f32x4*>(&us[li * GDC_P + 16 * k4 + 4 * lg]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
#pragma unroll
        for (int m = i; m < i + 2; ++m)
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) S[dt] = mfma4(x.kd[dt][k4][m], u4[k4][m], S[dt]);
        __builtin_amdgcn_sched_barrier(0);
        if (DT == 2 || i == 0) fetch_kd(next, y, DT == 2 ? i >> 1 : 0, k4);
        if (k4 == 3 && i == 0) fetch_rest(next, y);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (x.bad_token < CHUNK || x.bad_value < CHUNK)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) S[dt] = f32x4{NAN, NAN, NAN, NAN};
  };
  GDCarry<DP> x0, x1;
  {
    const int64_t unit = unit_of(0);
#pragma unroll
    for (int k8 = 0; k8 < DP / 32; ++k8) fetch_w(unit, x0, k8, 0), fetch_w(unit, x0, k8, 1);
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) fetch_kd(unit, x0, dt, k4);
    fetch_rest(unit, x0);
  }
  for (int c = 0; c < nc; c += 2) {
    step(c, x0, x1);
    if (c + 1 >= nc) break;
    step(c + 1, x1, x0);
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = (wave * DT + dt) * 16 + 4 * lg + r;
      if (d < p.dim && col < p.vdim) sb[(int64_t)d * p.vdim] = S[dt][r];
    }
}

// ---- 3. every chunk's outputs -------------------------------------------------------------------------------------------------------------
// wave = 16 tokens x 64 value columns; every operand comes as four or eight neighbouring numbers of a row, no LDS.
template <int DP>
__global__ __launch_bounds__(256) void gd_chunk_out_kernel(GDChunk a) {
  const GatedDelta& p = a.p;
  ChunkPlace at;
  if (!locate_chunk(a.chunk0 + blockIdx.x, p, a.min_len, at) || at.slot < 0 || at.slot >= p.num_slots) return;
  const int c = at.c;
  const int h = blockIdx.y, c0 = blockIdx.z * 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int cnt = min(CHUNK, at.len - c * CHUNK);
  const int64_t unit = (int64_t)blockIdx.x * p.heads + h;
  const int qt = (wave + blockIdx.x + blockIdx.y) & 3, tok = qt * 16 + li;       // (later tokens see more: the long tiles go round the SIMDs)
  const int nct = min(4, (p.vdim - c0 + 15) >> 4);
  f32x4 q[DP / 32][2], b[4];
#pragma unroll
  for (int k8 = 0; k8 < DP / 32; ++k8)
#pragma unroll
    for (int u = 0; u < 2; ++u) q[k8][u] = *reinterpret_cast<const f32x4*>(a.qg + unit * CHUNK * DP + qt * 16 * DP + (2 * k8 + u) * 256 + lane * 4);
#pragma unroll
  for (int jt = 0; jt < 4; ++jt)
    if (jt <= qt) b[jt] = *reinterpret_cast<const f32x4*>(a.bm + unit * CHUNK * CHUNK + (qt * 4 + jt) * 256 + lane * 4);
  const int bad_token = a.bad_token[unit];
  float* o = p.out + ((int64_t)at.start + c * CHUNK + tok) * ((int64_t)p.heads * p.vdim) + (int64_t)h * p.vdim + c0;
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    if (ct >= nct) break;
    const int64_t colrow = unit * a.vpad + c0 + ct * 16;
    f32x4 acc = {}, acc2 = {};
#pragma unroll
    for (int k8 = 0; k8 < DP / 32; ++k8) {
      const float* sp = a.st + colrow * DP + k8 * 512 + lane * 4;
      const f32x4 s0 = *reinterpret_cast<const f32x4*>(sp), s1 = *reinterpret_cast<const f32x4*>(sp + 256);
#pragma unroll
      for (int y = 0; y < 4; ++y) acc = mfma4(s0[y], q[k8][0][y], acc);
#pragma unroll
      for (int y = 0; y < 4; ++y) acc2 = mfma4(s1[y], q[k8][1][y], acc2);
    }
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) {
      if (jt > qt) break;
      const f32x4 u = *reinterpret_cast<const f32x4*>(a.ut + colrow * CHUNK + jt * 256 + lane * 4);
#pragma unroll
      for (int y = 0; y < 4; ++y) acc = mfma4(u[y], b[jt][y], acc);
    }
    if (tok >= cnt) continue;
    const int e = ct * 16 + 4 * lg;
    const i32x4 bad = *reinterpret_cast<const i32x4*>(&a.bad_value[unit * a.vpad + c0 + e]);
    f32x4 x;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      x[r] = acc[r] + acc2[r];
      if (tok >= bad_token || tok >= bad[r]) x[r] = NAN;
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

// Sizes of the workspace's parts for so many chunks, in floats.
static void gd_chunk_parts(const GatedDelta& p, int64_t chunks, int64_t (&n)[9]) {
  const int64_t units = chunks * p.heads, dp = p.dim <= 64 ? 64 : 128, vpad = (p.vdim + 15) / 16 * 16;
  n[0] = n[1] = n[2] = units * CHUNK * dp;
  n[3] = units * CHUNK * CHUNK;
  n[4] = units * vpad * CHUNK;
  n[5] = units * vpad * dp;
  n[6] = units * dp;
  n[7] = (units + 3) / 4 * 4;
  n[8] = units * vpad;
}
static int64_t gd_chunk_floats(const GatedDelta& p, int64_t chunks) {
  int64_t n[9], sum = 0;
  gd_chunk_parts(p, chunks, n);
  for (int64_t x : n) sum += x;
  return sum;
}

template <typename T, int DP, bool CHANNEL, bool VEC>
static int gd_chunk_launch(GDChunk a, int64_t chunks) {
  const GatedDelta& p = a.p;
  constexpr size_t lds = gd_prepare_lds<DP>();
  static bool attr_set_dev[APHRO_MAX_DEVICES] = {};
  bool& attr_set = attr_set_dev[device_slot()];
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)gd_chunk_prepare_kernel<T, DP, CHANNEL, VEC>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
      set_error("gated_delta_chunked: cannot raise the dynamic LDS limit");
      return APHRO_ERR_LAUNCH;
    }
    attr_set = true;
  }
  const unsigned span = (unsigned)a.span;
  for (; a.chunk0 < chunks; a.chunk0 += a.span) {
    hipLaunchKernelGGL((gd_chunk_prepare_kernel<T, DP, CHANNEL, VEC>), dim3(span, (unsigned)p.heads), dim3(DP * 4), lds, p.stream, a);
    hipLaunchKernelGGL((gd_chunk_carry_kernel<DP>), dim3((unsigned)p.heads, (unsigned)a.vpad / 16, (unsigned)p.num_seqs), dim3(256), 0, p.stream, a);
    hipLaunchKernelGGL((gd_chunk_out_kernel<DP>), dim3(span, (unsigned)p.heads, (unsigned)((p.vdim + 63) / 64)), dim3(256), 0, p.stream, a);
  }
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

}  // namespace aphro

using namespace aphro;

extern "C" int64_t aphro_gated_delta_chunked_workspace(int num_seqs, int64_t num_tokens, int heads, int dim, int vdim, int min_len) {
  if (num_seqs <= 0 || num_tokens <= 0 || heads <= 0 || dim <= 0 || dim > 128 || vdim <= 0 || min_len <= 0) return 0;
  GatedDelta p = {};
  p.num_seqs = num_seqs, p.num_tokens = num_tokens, p.heads = heads, p.dim = dim, p.vdim = vdim;
  return span_workspace(max_chunks(num_tokens, num_seqs, num_seqs == 1 ? 1 : min_len), [&](int64_t n) { return gd_chunk_floats(p, n); });
}

extern "C" int aphro_gated_delta_chunked(float* out, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                                         int64_t v_stride, const void* b, int64_t b_stride, const void* a, int64_t a_stride,
                                         const float* a_log, const float* dt_bias, float* state, const int32_t* slot_of_seq,
                                         int num_slots, const int32_t* q_start, const int32_t* q_len, const int32_t* ctx_len,
                                         int num_seqs, int64_t num_tokens, int heads, int kv_heads, int dim, int vdim, int channel_decay,
                                         float q_scale, float norm_eps, int min_len, float* workspace, int64_t workspace_bytes,
                                         int dtype, void* stream) {
  if (num_tokens == 0 || num_seqs == 0) return APHRO_OK;
  GDChunk x = {};
  x.p = {out, q, k, v, b, a, q_stride, k_stride, v_stride, b_stride, a_stride, a_log, dt_bias, state, slot_of_seq, num_slots,
         q_start, q_len, ctx_len, num_seqs, num_tokens, heads, kv_heads, dim, vdim, channel_decay, q_scale, norm_eps, dtype, (hipStream_t)stream};
  const GatedDelta& p = x.p;
  const int rc = gated_delta_check(p);
  if (rc != APHRO_OK) return rc;
  APHRO_CHECK(dim <= 128 && min_len > 0 && num_seqs > 0 && num_seqs <= 65535, "gated_delta_chunked: dim %d (<= 128), %d segments (<= 65535) from %d tokens on", dim, num_seqs, min_len);
  if (num_seqs == 1) min_len = 1;
  const int64_t chunks = max_chunks(num_tokens, num_seqs, min_len);
  APHRO_CHECK(chunks <= 0x3fffffff, "gated_delta_chunked: too many tokens");
  const int64_t span = span_chunks(chunks, workspace_bytes, [&](int64_t m) { return gd_chunk_floats(p, m); });
  APHRO_CHECK(((uintptr_t)out & 15) == 0 && (chunks == 0 || (workspace && ((uintptr_t)workspace & 15) == 0 && span > 0)),
              "gated_delta_chunked: a workspace of %lld bytes at least, 16-byte aligned, is needed", (long long)gd_chunk_floats(p, 1) * 4);
  int64_t n[9];
  gd_chunk_parts(p, span, n);
  x.chunk0 = 0, x.span = (int)span;
  x.min_len = min_len;
  x.vpad = (vdim + 15) / 16 * 16;
  float* at = workspace;
  float** parts[7] = {&x.w, &x.qg, &x.kd, &x.bm, &x.ut, &x.st, &x.gam};
  for (int i = 0; i < 7; ++i) *parts[i] = at, at += n[i];
  x.bad_token = (int32_t*)at;
  x.bad_value = x.bad_token + n[7];
  if (num_seqs > 1) {                                       // (a single segment: chunks, whatever its length)
    const int rs = gated_delta_scan_launch(p, min_len, min_len > 32);
    if (rs != APHRO_OK || chunks == 0) return rs;
  }
  const int elem = dtype == APHRO_BF16 ? 2 : 4;
  const bool vec = rows_of_16_bytes(q, q_stride, dim, elem) && rows_of_16_bytes(k, k_stride, dim, elem) && rows_of_16_bytes(v, v_stride, vdim, elem) &&
                   (!channel_decay || rows_of_16_bytes(a, a_stride, dim, elem));
#define GDC_LAUNCH(DP, CH) (vec ? gd_chunk_launch<T, DP, CH, true>(x, chunks) : gd_chunk_launch<T, DP, CH, false>(x, chunks))
  MIX_DISPATCH_DTYPE(dtype, {
    if (dim <= 64) return channel_decay ? GDC_LAUNCH(64, true) : GDC_LAUNCH(64, false);
    return channel_decay ? GDC_LAUNCH(128, true) : GDC_LAUNCH(128, false);
  });
#undef GDC_LAUNCH
  return APHRO_OK;
}
