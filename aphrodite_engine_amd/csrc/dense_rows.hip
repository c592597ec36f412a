// 16-bit matrix product for few rows, out[M <= 192, N] = x[M, K] . w[N, K]^T (f16 / bf16, fp32 sums): the unquantised linears and heads of
// decode steps and short prompt portions.  Bound by reading w once; what an implementation can lose is (1) x, which every column tile
// reads again, and (2) chips that a narrow w does not fill.
//   * A workgroup owns 64 or 128 rows of w and ALL rows of x, so x crosses L2 M / 64 or M / 128 times as often as w.  (A first form with one
//     16-row tile of w per workgroup and fragments straight from global memory read x 2-4 times as often as w: 36 us where this one
//     takes 23 on [4096, 11008] with 32 rows.)
//   * Both operands go through LDS in steps of 64 k by LDS-DMA, 8 rows of a full 128-byte line per instruction, 2 to 5 steps ahead; chunk
//     j of row r lies at j ^ (r & 7), which leaves the fragment reads without bank conflicts.  One barrier a step.
//   * Few column tiles: K is split over workgroups, each slice's sums go to a slab, a second small launch adds the slabs in order (no state
//     between calls, the same bits every time).
//   * Optional bias, fp32 results (rounded through the 16-bit type: what .float() of the 16-bit product holds), or a gated activation
//     act(x . gate^T) * (x . up^T) over w = [gate; up]: a 16-row MFMA tile then holds 8 gate and 8 up rows of the same 8 columns, and the
//     two halves of a wave exchange their sums in registers.
// Measured against torch's product (hipBLASLt), us, bf16, weights from memory, graph replay:
//   [N, K] \ M         16            32            64            128           185
//   [4096, 11008]   22.0 / 37.6   23.0 / 29.6   25.4 / 33.9   30.3 / 59.4   35.5 / 49.3
//   [2048, 7680]    12.6 / 13.5   13.2 / 17.0   14.2 / 23.1   17.8 / 21.3   22.3 / 27.3
//   [6144, 4096]    15.2 / 14.6   15.9 / 15.5   18.3 / 18.2   21.1 / 25.6   25.9 / 26.2
//   [11264, 2048]   12.4 / 14.9   13.2 / 15.0   15.4 / 16.2   21.2 / 18.8   26.9 / 26.5
//   [22016, 4096]   39.5 / 50.5   40.5 / 40.8   43.2 / 43.1   51.2 / 44.7   57.6 / 58.2   (gated: without the 3.5 us of an activation launch)
//   [128256, 4096]  177 / 186     184 / 195     188 / 208     206 / 233     240 / 294
// and the call costs the host a third of torch's 24 us.  From 193 rows on two row tiles re-read w and the library is ahead.
#include "mixers/mixers_common.h"

namespace aphro {

struct DenseRowsParams {
  const uint16_t* a;
  const uint16_t* w;
  const uint16_t* bias;     // [N] or null; not with an activation
  void* out;                // [M, ldo] 16-bit, or fp32 if out_f32
  float* slabs;             // [ksplit][M][rows of w], only if ksplit > 1
  int M, N, K;              // N: columns of out
  int lda, ldw, ldo;
  int tiles_n, ksplit;
  int out_f32;
};

typedef __attribute__((address_space(3))) void* dr_lds_ptr;

template <typename T>
__device__ __forceinline__ f32x4 dr_mfma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (__is_same(T, Half))
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// ACT: -1 none, 0 silu, 1 gelu (tanh)
template <int ACT>
__device__ __forceinline__ float dr_act(float g) {
  if constexpr (ACT == 0) return silu_f(g);
  else return gelu_tanh_f(g);
}

// four neighbouring columns of one row
template <typename T>
__device__ __forceinline__ void dr_store(const DenseRowsParams& p, int m, int n, f32x4 v) {
  if (p.bias) {
    const u16x4 b = *reinterpret_cast<const u16x4*>(p.bias + n);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] += T::to_f32(b[r]);
  }
  u16x4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = T::from_f32(v[r]);
  if (p.out_f32) {
    f32x4 f;
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = T::to_f32(o[r]);
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + (size_t)m * p.ldo + n) = f;
  } else {
    *reinterpret_cast<u16x4*>(reinterpret_cast<uint16_t*>(p.out) + (size_t)m * p.ldo + n) = o;
  }
}

// MT: 16-row tiles of x; NT: 64 NT rows of w; WR: groups of four waves that divide x's rows; NS: LDS stages.
template <typename T, int MT, int NT, int WR, int NS, int ACT>
__global__ __launch_bounds__(256 * WR) void dense_rows_kernel(DenseRowsParams p) {
  constexpr int MTW = MT / WR, BN = 64 * NT, BM = 16 * MT, NW = 4 * WR;
  constexpr int WI = BN / 8 / NW, XI = (BM / 8 + NW - 1) / NW, LPS = WI + XI, STAGE = (BN + BM) * 128;
  static_assert(MT % WR == 0 && NS >= 2, "");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15, wc = wave & 3, wr = wave >> 2;
  int lin;                                            // contiguous ranges of tiles per XCD
  {
    const int n = gridDim.x, q = n / 8, r = n % 8, xcd = blockIdx.x % 8, k = blockIdx.x / 8;
    lin = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + k;
  }
  const int tn = lin % p.tiles_n, ks = lin / p.tiles_n;
  const int S = p.K / 64, s0 = ks * S / p.ksplit, n = (ks + 1) * S / p.ksplit - s0;
  // first output column of the tile; row r of the tile's BN is row wrow(r) of w behind wbase (rows past the end: the last one, not stored)
  const int n0 = tn * (ACT < 0 ? BN : BN / 2);
  auto wrow = [&](int r) {
    if constexpr (ACT < 0) return min(r, p.N - n0 - 1);
    return ((r >> 3) & 1) * p.N + min((r >> 4) * 8 + (r & 7), p.N - n0 - 1);
  };
  const uint32_t last_row = ACT < 0 ? (uint32_t)(min(p.N - n0, BN) - 1) : (uint32_t)(2 * p.N - 1 - n0);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.w) + (size_t)n0 * p.ldw, 0,
                                                                      (last_row * (uint32_t)p.ldw + (uint32_t)p.K) * 2u, 0x00020000);
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a), 0,
                                                                      ((uint32_t)(p.M - 1) * (uint32_t)p.lda + (uint32_t)p.K) * 2u, 0x00020000);
  int vw[WI], vx[XI];
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = (wave + NW * i) * 8 + (lane >> 3);
    vw[i] = wrow(r) * p.ldw * 2 + (((lane & 7) ^ (r & 7)) << 4);
  }
#pragma unroll
  for (int i = 0; i < XI; ++i) {                      // (where the waves outnumber the pieces, two of them fetch the same one)
    const int r = ((wave + NW * i) % (2 * MT)) * 8 + (lane >> 3);
    vx[i] = min(r, p.M - 1) * p.lda * 2 + (((lane & 7) ^ (r & 7)) << 4);
  }
  auto issue = [&](int s, int slot) {
    unsigned char* st = smem + slot * STAGE;
    const int so = (s0 + s) * 128;
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int v = vw[i];                            // (a local copy: see wna16_gemm_large.hip)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (dr_lds_ptr)(st + (wave + NW * i) * 1024), 16, v, so, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int v = vx[i];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (dr_lds_ptr)(st + BN * 128 + ((wave + NW * i) % (2 * MT)) * 1024), 16, v, so, 0, 0);
    }
  };
  f32x4 acc[NT][MTW];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < MTW; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int sw[2] = {(g ^ (c & 7)) << 4, ((4 + g) ^ (c & 7)) << 4};
  const int wbase = (16 * wc + c) * 128, xbase = BN * 128 + (wr * MTW * 16 + c) * 128;
  for (int d = 0; d < NS - 1; ++d)
    if (d < n) issue(d, d);
  int slot = 0, fetch = NS - 1;
  for (int s = 0; s < n; ++s) {
    // step s has landed when at most the loads of the NS - 2 steps behind it are outstanding; past the barrier every wave is through
    // with step s - 1, whose stage the loads issued now take
    if (s + NS - 2 < n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * LPS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + NS - 1 < n) issue(s + NS - 1, fetch);
    const unsigned char* st = smem + slot * STAGE;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      u32x4 wf[NT], xf[MTW];
#pragma unroll
      for (int t = 0; t < NT; ++t) wf[t] = *reinterpret_cast<const u32x4*>(st + wbase + t * 8192 + sw[u]);
#pragma unroll
      for (int i = 0; i < MTW; ++i) xf[i] = *reinterpret_cast<const u32x4*>(st + xbase + i * 2048 + sw[u]);
#pragma unroll
      for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t][i] = dr_mfma<T>(wf[t], xf[i], acc[t][i]);
    }
    slot = slot + 1 == NS ? 0 : slot + 1;
    fetch = fetch + 1 == NS ? 0 : fetch + 1;
  }
  // D: lane (g, c) has rows 4 g .. + 3 of the w tile for row c of the x tile
#pragma unroll
  for (int i = 0; i < MTW; ++i) {
    const int m = (wr * MTW + i) * 16 + c;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 v = acc[t][i];
      if constexpr (ACT < 0) {
        const int col = n0 + t * 64 + 16 * wc + 4 * g;
        if (m < p.M && col < p.N) {
          if (p.ksplit > 1) *reinterpret_cast<f32x4*>(p.slabs + ((size_t)ks * p.M + m) * p.N + col) = v;
          else dr_store<T>(p, m, col, v);
        }
      } else {
        const int col = n0 + t * 32 + 8 * wc + 4 * (g & 1);     // lanes g < 2 hold the gate's sums, the others the up ones'
        if (p.ksplit > 1) {
          if (m < p.M && col < p.N) *reinterpret_cast<f32x4*>(p.slabs + ((size_t)ks * p.M + m) * 2 * p.N + (g >> 1) * p.N + col) = v;
        } else {
          f32x4 up;
#pragma unroll
          for (int r = 0; r < 4; ++r) up[r] = __shfl_xor(v[r], 32, 64);
          if (g < 2 && m < p.M && col < p.N) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = dr_act<ACT>(v[r]) * up[r];
            dr_store<T>(p, m, col, v);
          }
        }
      }
    }
  }
}

// The K slices' slabs, added in order, four columns a thread.
template <typename T, int ACT>
__global__ __launch_bounds__(256) void dense_rows_reduce_kernel(DenseRowsParams p) {
  const int n4 = p.N >> 2;
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= n4 * p.M) return;
  const int m = q / n4, col = (q - m * n4) * 4;
  const int W = ACT < 0 ? p.N : 2 * p.N;
  auto total = [&](int at) {
    const float* src = p.slabs + (size_t)m * W + at;
    f32x4 s = *reinterpret_cast<const f32x4*>(src);
    for (int k = 1; k < p.ksplit; ++k) s += *reinterpret_cast<const f32x4*>(src + (size_t)k * p.M * W);
    return s;
  };
  f32x4 v = total(col);
  if constexpr (ACT >= 0) {
    const f32x4 up = total(p.N + col);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = dr_act<ACT>(v[r]) * up[r];
  }
  dr_store<T>(p, m, col, v);
}

struct DenseRowsPlan { int mt, nt, ksplit; };

// Which tile, and over how many workgroups K is split (us of [N, K] with M rows, both sides measured):
//  * 128 rows of w once that gives 160 workgroups: [22016, 4096], 64 rows of x: 43.2 against 45; up to 32 rows of x and many tiles 64
//    rows are ahead ([32000, 2048], 16: 26.5 against 27.4; [128256, 4096], 32: 184 against 187).
//  * 160 tiles of 64 rows and more: K in one piece ([11264, 2048], 16: 12.4, split 14.5).
//  * else one workgroup a CU, or two where one a CU would leave more than an eighth of the CUs idle ([6144, 4096], 16: 5 slices 15.2);
//    a slice has at least 4 steps of 64 k.
//  * from 65 rows of x on, 128 rows of w also with K split while a slice keeps 12 steps: [4096, 11008], 128: 30.3 against 33.5.
static void dense_rows_plan(int64_t M, int64_t N, int64_t K, bool gated, DenseRowsPlan& plan) {
  const int64_t rows = gated ? 2 * N : N;
  const int t64 = (int)((rows + 63) / 64), t128 = (int)((rows + 127) / 128), steps = (int)(K / 64);
  const int mt = (int)((M + 15) / 16);
  auto split = [&](int tiles, bool two) {
    int k = 256 / tiles;
    if (two && (k < 1 || tiles * k < 224)) k = 512 / tiles;
    k = k > steps / 4 ? steps / 4 : k;
    return k < 1 ? 1 : k > 16 ? 16 : k;
  };
  plan.mt = mt <= 4 ? mt : (mt + 1) / 2 * 2;
  if (mt <= 4) {
    plan.nt = t128 >= 160 && (mt > 2 || t64 < 480) ? 2 : 1;
    plan.ksplit = t64 >= 160 ? 1 : split(t64, true);
  } else if (t128 >= 160 || t64 >= 160) {
    plan.nt = t128 >= 160 ? 2 : 1;
    plan.ksplit = 1;
  } else {
    const int k2 = split(t128, false);
    plan.nt = steps / k2 >= 12 ? 2 : 1;
    plan.ksplit = plan.nt == 2 ? k2 : split(t64, true);
  }
}

template <typename T, int MT, int NT, int WR, int NS, int ACT>
static int dense_rows_launch(const DenseRowsParams& p, hipStream_t st) {
  constexpr size_t lds = (size_t)NS * (64 * NT + 16 * MT) * 128;
  auto kern = dense_rows_kernel<T, MT, NT, WR, NS, ACT>;
  if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
    set_error("dense_rows: cannot raise the dynamic LDS limit to %zu", lds);
    return APHRO_ERR_LAUNCH;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_n * p.ksplit)), dim3(256 * WR), lds, st, p);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

// Stages: as many as let two workgroups share a CU's 160 KB (64 rows of w: three or two); where 256 CUs' worth of 128-row tiles is all there
// is ([22016, 4096], 65 rows and more), one workgroup of eight waves a CU with deeper stages.
template <typename T, int ACT>
static int dense_rows_dispatch(const DenseRowsParams& p, const DenseRowsPlan& plan, hipStream_t st) {
  const bool many = p.tiles_n >= 512;
  if (plan.nt == 1) {
    switch (plan.mt) {
      case 1: return dense_rows_launch<T, 1, 1, 1, 5, ACT>(p, st);
      case 2: return dense_rows_launch<T, 2, 1, 1, 6, ACT>(p, st);
      case 3: return dense_rows_launch<T, 3, 1, 1, 5, ACT>(p, st);
      case 4: return dense_rows_launch<T, 4, 1, 1, 5, ACT>(p, st);
      case 6: return dense_rows_launch<T, 6, 1, 1, 3, ACT>(p, st);
      case 8: return dense_rows_launch<T, 8, 1, 1, 3, ACT>(p, st);
      case 10: return dense_rows_launch<T, 10, 1, 1, 3, ACT>(p, st);
      default: return dense_rows_launch<T, 12, 1, 1, 3, ACT>(p, st);
    }
  }
  switch (plan.mt) {
    case 1: return dense_rows_launch<T, 1, 2, 1, 4, ACT>(p, st);
    case 2: return dense_rows_launch<T, 2, 2, 1, 4, ACT>(p, st);
    case 3: return dense_rows_launch<T, 3, 2, 1, 3, ACT>(p, st);
    case 4: return dense_rows_launch<T, 4, 2, 1, 3, ACT>(p, st);
    case 6: return many ? dense_rows_launch<T, 6, 2, 1, 2, ACT>(p, st) : dense_rows_launch<T, 6, 2, 1, 3, ACT>(p, st);
    case 8: return many ? dense_rows_launch<T, 8, 2, 1, 2, ACT>(p, st) : dense_rows_launch<T, 8, 2, 2, 3, ACT>(p, st);
    case 10: return many ? dense_rows_launch<T, 10, 2, 1, 2, ACT>(p, st) : dense_rows_launch<T, 10, 2, 2, 4, ACT>(p, st);
    default: return many ? dense_rows_launch<T, 12, 2, 1, 2, ACT>(p, st) : dense_rows_launch<T, 12, 2, 2, 4, ACT>(p, st);
  }
}

template <typename T, int ACT>
static int dense_rows_run(DenseRowsParams p, const DenseRowsPlan& plan, hipStream_t st) {
  p.tiles_n = (int)(((ACT < 0 ? (int64_t)p.N : 2 * (int64_t)p.N) + 64 * plan.nt - 1) / (64 * plan.nt));
  p.ksplit = plan.ksplit;
  if (const int rc = dense_rows_dispatch<T, ACT>(p, plan, st); rc != APHRO_OK || plan.ksplit == 1) return rc;
  hipLaunchKernelGGL((dense_rows_reduce_kernel<T, ACT>), dim3((unsigned)((p.M * (p.N >> 2) + 255) / 256)), dim3(256), 0, st, p);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

}  // namespace aphro

using namespace aphro;

extern "C" int64_t aphro_dense_rows_slab_floats(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int act) {
  constexpr int64_t LIMIT = 0x7fffffffll;
  const int64_t rows = act >= 0 ? 2 * N : N;
  if (M < 1 || M > 192 || N < 8 || N % 8 != 0 || K < 64 || K % 64 != 0 || lda < K || ldw < K || lda % 8 != 0 || ldw % 8 != 0 || act > 1) return -1;
  // (byte offsets inside x, and inside a tile of w -- with an activation, inside all of w -- are 32-bit)
  if (lda > LIMIT || ldw > LIMIT || N > (LIMIT >> 4) || (M * lda + K) * 2 > LIMIT) return -1;
  if (((act >= 0 ? rows : 128) * ldw + K) * 2 > LIMIT) return -1;
  DenseRowsPlan plan;
  dense_rows_plan(M, N, K, act >= 0, plan);
  return plan.ksplit > 1 ? plan.ksplit * M * rows : 0;
}

extern "C" int aphro_dense_rows(void* out, int64_t ldo, const void* x, int64_t lda, const void* weight, int64_t ldw, const void* bias,
                                float* slabs, int64_t slab_floats, int64_t M, int64_t N, int64_t K, int act, int out_f32, int dtype,
                                void* stream) {
  APHRO_CHECK(dtype == APHRO_F16 || dtype == APHRO_BF16, "dense_rows: dtype must be f16 or bf16");
  const int64_t need = aphro_dense_rows_slab_floats(M, N, K, lda, ldw, act);
  APHRO_CHECK(need >= 0, "dense_rows: M=%ld N=%ld K=%ld lda=%ld ldw=%ld is not served", (long)M, (long)N, (long)K, (long)lda, (long)ldw);
  APHRO_CHECK(((uintptr_t)x % 16) == 0 && ((uintptr_t)weight % 16) == 0 && ((uintptr_t)out % (out_f32 ? 16 : 8)) == 0 && ldo >= N && ldo % 4 == 0 &&
                  ldo <= 0x7fffffff && ((uintptr_t)bias % 8) == 0,
              "dense_rows: 16-byte aligned operands and 8-byte aligned (fp32: 16) output rows required");
  APHRO_CHECK(act < 0 || bias == nullptr, "dense_rows: no bias with an activation");
  APHRO_CHECK(need == 0 || (slabs != nullptr && slab_floats >= need && ((uintptr_t)slabs % 16) == 0), "dense_rows: %ld floats of slabs needed", (long)need);
  DenseRowsPlan plan;
  dense_rows_plan(M, N, K, act >= 0, plan);
  DenseRowsParams p;
  p.a = (const uint16_t*)x; p.w = (const uint16_t*)weight; p.bias = (const uint16_t*)bias; p.out = out; p.slabs = slabs;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.lda = (int)lda; p.ldw = (int)ldw; p.ldo = (int)ldo; p.out_f32 = out_f32;
  hipStream_t st = (hipStream_t)stream;
#define DR_ACT(TT) (act < 0 ? dense_rows_run<TT, -1>(p, plan, st) : act == 0 ? dense_rows_run<TT, 0>(p, plan, st) : dense_rows_run<TT, 1>(p, plan, st))
  return dtype == APHRO_F16 ? DR_ACT(Half) : DR_ACT(BFloat);
#undef DR_ACT
}
