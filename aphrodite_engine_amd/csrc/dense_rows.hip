// 16-bit matrix product for few rows, out[M <= 192, N] = x[M, K] . w[N, K]^T (f16 / bf16, fp32 sums): the unquantised linears and heads of
// decode steps and short prompt portions.  Bound by reading w once; what an implementation can lose is (1) x, which every column tile
// reads again, and (2) chips that a narrow w does not fill.
//   * A workgroup owns 64 or 128 rows of w and ALL rows of x, so x crosses L2 M / 64 or M / 128 times as often as w.  (A first form with one
//     16-row tile of w per workgroup and fragments straight from global memory read x 2-4 times as often as w: 36 us where this one
//     takes 23 on [4096, 11008] with 32 rows.)
//   * Both operands go through LDS in steps of 64 k by LDS-DMA, 8 rows of a full 128-byte line per instruction, 1 to 5 steps ahead; chunk
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
// and the call costs the host a third of torch's 24 us.  From 193 rows on two row tiles re-read w and the library is ahead, from 65 rows on
// with some wide weights too: aphro_dense_rows_preferred.
#include "dense_rows.h"
#include "mixers/mixers_common.h"

namespace aphro {

struct DenseRowsParams {
  RowsOperands op;
  const uint16_t* bias;     // [N] or null; not with an activation
  void* out;                // [M, ldo] 16-bit, or fp32 if out_f32
  float* slabs;             // [ksplit][M][rows of w], only if ksplit > 1
  int ldo, out_f32;
};

template <typename T>
struct DenseRowsProduct {
  template <int NT, int MTW>
  static __device__ __forceinline__ void step(const unsigned char* st, int wbase, int xbase, const int (&sw)[2], f32x4 (&acc)[NT][MTW]) {
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
        for (int t = 0; t < NT; ++t) {
          if constexpr (__is_same(T, Half))
            acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, wf[t]), __builtin_bit_cast(f16x8, xf[i]), acc[t][i], 0, 0, 0);
          else
            acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[t]), __builtin_bit_cast(bf16x8, xf[i]), acc[t][i], 0, 0, 0);
        }
    }
  }
};

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

template <typename T, int MT, int NT, int WR, int NS, int ACT, bool STREAM>
__global__ __launch_bounds__(256 * WR) void dense_rows_kernel(DenseRowsParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  RowsTile<DenseRowsProduct<T>, MT, NT, WR, NS, (ACT >= 0), STREAM> tile;
  tile.run(p.op, smem);
  const int M = p.op.M, N = p.op.N, ks = tile.ks, g = tile.g;
#pragma unroll
  for (int i = 0; i < MT / WR; ++i) {
    const int m = (tile.wr * (MT / WR) + i) * 16 + tile.c;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 v = tile.acc[t][i];
      if constexpr (ACT < 0) {
        const int col = tile.n0 + t * 64 + 16 * tile.wc + 4 * g;
        if (m < M && col < N) {
          if (p.op.ksplit > 1) *reinterpret_cast<f32x4*>(p.slabs + ((size_t)ks * M + m) * N + col) = v;
          else dr_store<T>(p, m, col, v);
        }
      } else {
        const int col = tile.n0 + t * 32 + 8 * tile.wc + 4 * (g & 1);     // lanes g < 2 hold the gate's sums, the others the up ones'
        if (p.op.ksplit > 1) {
          if (m < M && col < N) *reinterpret_cast<f32x4*>(p.slabs + ((size_t)ks * M + m) * 2 * N + (g >> 1) * N + col) = v;
        } else {
          f32x4 up;
#pragma unroll
          for (int r = 0; r < 4; ++r) up[r] = __shfl_xor(v[r], 32, 64);
          if (g < 2 && m < M && col < N) {
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
  const int N = p.op.N, M = p.op.M, n4 = N >> 2;
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= n4 * M) return;
  const int m = q / n4, col = (q - m * n4) * 4;
  const int W = ACT < 0 ? N : 2 * N;
  auto total = [&](int at) {
    const float* src = p.slabs + (size_t)m * W + at;
    f32x4 s = *reinterpret_cast<const f32x4*>(src);
    for (int k = 1; k < p.op.ksplit; ++k) s += *reinterpret_cast<const f32x4*>(src + (size_t)k * M * W);
    return s;
  };
  f32x4 v = total(col);
  if constexpr (ACT >= 0) {
    const f32x4 up = total(N + col);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = dr_act<ACT>(v[r]) * up[r];
  }
  dr_store<T>(p, m, col, v);
}

// Whether a w that passes the caches once (weights_streamed) takes the non-temporal hint (RowsTile) above 48 rows of x, up to which it does: with 40
// steps of 64 k a slice and more, up to 128 rows.  us without / with it, f16, weights from memory: [128256, 4096], 16 / 64 / 96 / 192 rows 187 / 198 / 212 / 254 and 167 / 192 / 211 / 253;
// [28672, 4096], 16 / 64 / 128 / 150 rows 50.5 / 51.4 / 57.9 / 59.5 and 46.7 / 47.9 / 56.8 / 60.1; [10240, 8192], 42 steps, 32 / 65 / 128 rows 38.1 /
// 37.9 / 42.6 and 35.2 / 35.5 / 41.8.  Short slices lose with many rows: [4096, 14336], 28 steps, 16 / 48 / 96 / 128 rows 24.9 / 26.8 / 30.4 / 33.2
// and 22.1 / 25.3 / 32.2 / 35.6; [6144, 4096], 12 steps, 16 / 64 / 128 rows 14.3 / 17.6 / 20.5 and 13.5 / 19.0 / 23.4.  (FP8, half the bytes of x a step,
// is ahead or level with it everywhere: fp8_gemm_rows.hip.)  Weights that stay in the last-level cache from call to call, 180 to 260 MB in all, without /
// with it, 16 and 48 rows: [2048, 2048] 8.1 / 8.1 and 9.5 / 9.5, [4096, 4096] 9.8 / 10.8 and 10.9 / 12.7, [11008, 4096] 15.4 / 19.8 and 20.5 / 24.7,
// [32000, 2048] 21.1 / 27.1 and 22.2 / 28.7; one more of the latter, from memory, 30.6 / 27.7 and 31.8 / 29.9.  FP8 [28672, 4096], 64 rows 20.7 / 29.2.
inline bool dense_rows_stream(const RowsOperands& op) { return op.M <= 48 || (op.M <= 128 && op.row_bytes >= 40 * 128 * op.ksplit); }

template <typename T, int ACT>
static int dense_rows_run(DenseRowsParams p, const RowsPlan& plan, bool streamed, hipStream_t st) {
  p.op.tiles_n = (int)(((ACT < 0 ? (int64_t)p.op.N : 2 * (int64_t)p.op.N) + 64 * plan.nt - 1) / (64 * plan.nt));
  p.op.ksplit = plan.ksplit;
  const int rc = rows_dispatch<(ACT < 0)>(plan, p.op.tiles_n, [&](auto mt, auto nt, auto wr, auto ns) {
    constexpr int MT = decltype(mt)::value, NT = decltype(nt)::value, WR = decltype(wr)::value, NS = decltype(ns)::value;
    constexpr size_t lds = RowsTile<DenseRowsProduct<T>, MT, NT, WR, NS, (ACT >= 0), true>::LDS;
    auto kern = dense_rows_kernel<T, MT, NT, WR, NS, ACT, false>;
    if constexpr (MT <= 8) {
      if (streamed && dense_rows_stream(p.op)) kern = dense_rows_kernel<T, MT, NT, WR, NS, ACT, true>;
    }
    if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
      set_error("dense_rows: cannot raise the dynamic LDS limit to %zu", lds);
      return (int)APHRO_ERR_LAUNCH;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(p.op.tiles_n * p.op.ksplit)), dim3(256 * WR), lds, st, p);
    APHRO_LAUNCH_CHECK();
    return (int)APHRO_OK;
  });
  if (rc != APHRO_OK || plan.ksplit == 1) return rc;
  hipLaunchKernelGGL((dense_rows_reduce_kernel<T, ACT>), dim3((unsigned)((p.op.M * (p.op.N >> 2) + 255) / 256)), dim3(256), 0, st, p);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

}  // namespace aphro

using namespace aphro;

extern "C" int64_t aphro_dense_rows_slab_floats(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int act) {
  if (act > 1 || N % 8 != 0 || K > (1 << 30) || lda > (1 << 30) || ldw > (1 << 30) || lda % 8 != 0 || ldw % 8 != 0 ||
      !rows_fits(M, N, 2 * K, 2 * lda, 2 * ldw, act >= 0))
    return -1;
  const int64_t rows = act >= 0 ? 2 * N : N;
  const RowsPlan plan = rows_plan(M, rows, 2 * K, act < 0);
  return plan.ksplit > 1 ? plan.ksplit * M * rows : 0;
}

// Whether the product is the faster one, by the GPU's time, against the library's.  Up to 64 rows of x, narrow weights (the library's host time
// alone is what those take) and sliced K it is, or within a tenth.  Where K is in one piece, w large and rows many, it is not
//  * with 64-column tiles, which bring x through LDS twice as often: [12288, 4096], 65 / 128 / 192 rows 31.5 / 37.0 / 48.6 us, library 30.3 / 33.0 /
//    41.8, [18944, 3584], 96 rows 49 and 37;
//  * with 128-column tiles that leave more than a tenth of the CUs idle in their last round, from 97 rows on: [22016, 4096], 128 / 160 rows 53 / 58,
//    library 47 / 53, [28672, 4096] 59 / 62 and 55 / 58, [57344, 8192] 199 / 207 and 191 / 191 (at 65 and 80 rows 45 / 47 and 46 / 46, 54 / 55 and 54 /
//    64, 183 / 188 and 186 / 178); where more than a third idle, from 65 on ([37888, 3584], 65 / 80 rows 68 / 70 and 65 / 62).
// [32000, 4096] to [32000, 5120], [62000, 4096], [128256, 4096] and [128256, 8192] fill the CUs: ahead of the library or level with it.
extern "C" int aphro_dense_rows_preferred(int64_t M, int64_t N, int64_t K) {
  if (!rows_fits(M, N, 2 * K, 2 * K, 2 * K, false)) return 0;
  if (M <= 64 || K < 2560 || N * K < 40000000) return 1;
  const RowsPlan plan = rows_plan(M, N, 2 * K, true);
  if (plan.ksplit > 1) return 1;
  if (plan.nt == 1) return 0;
  const int64_t tiles = (N + 127) / 128, cus = (tiles + 255) / 256 * 256;
  return M > 96 ? tiles * 10 >= cus * 9 : tiles * 3 >= cus * 2;
}

extern "C" int aphro_dense_rows(void* out, int64_t ldo, const void* x, int64_t lda, const void* weight, int64_t ldw, const void* bias,
                                float* slabs, int64_t slab_floats, int64_t M, int64_t N, int64_t K, int act, int out_f32, int dtype,
                                void* stream) {
  const bool streamed = weights_streamed(weights_flags(dtype), (size_t)(act >= 0 ? 2 * N : N) * K * 2);
  APHRO_CHECK(dtype == APHRO_F16 || dtype == APHRO_BF16, "dense_rows: dtype must be f16 or bf16");
  const int64_t need = aphro_dense_rows_slab_floats(M, N, K, lda, ldw, act);
  APHRO_CHECK(need >= 0, "dense_rows: M=%ld N=%ld K=%ld lda=%ld ldw=%ld is not served", (long)M, (long)N, (long)K, (long)lda, (long)ldw);
  APHRO_CHECK(((uintptr_t)x % 16) == 0 && ((uintptr_t)weight % 16) == 0 && ((uintptr_t)out % (out_f32 ? 16 : 8)) == 0 && ldo >= N && ldo % 4 == 0 &&
                  ldo <= 0x7fffffff && ((uintptr_t)bias % 8) == 0,
              "dense_rows: 16-byte aligned operands and 8-byte aligned (fp32: 16) output rows required");
  APHRO_CHECK(act < 0 || bias == nullptr, "dense_rows: no bias with an activation");
  APHRO_CHECK(need == 0 || (slabs != nullptr && slab_floats >= need && ((uintptr_t)slabs % 16) == 0), "dense_rows: %ld floats of slabs needed", (long)need);
  DenseRowsParams p;
  p.op.a = (const uint8_t*)x; p.op.w = (const uint8_t*)weight; p.op.M = (int)M; p.op.N = (int)N; p.op.row_bytes = (int)(2 * K);
  p.op.lda = (int)(2 * lda); p.op.ldw = (int)(2 * ldw);
  p.bias = (const uint16_t*)bias; p.out = out; p.slabs = slabs; p.ldo = (int)ldo; p.out_f32 = out_f32;
  const RowsPlan plan = rows_plan(M, act >= 0 ? 2 * N : N, 2 * K, act < 0);
  hipStream_t st = (hipStream_t)stream;
#define DR_ACT(TT) (act < 0 ? dense_rows_run<TT, -1>(p, plan, streamed, st) : act == 0 ? dense_rows_run<TT, 0>(p, plan, streamed, st) : dense_rows_run<TT, 1>(p, plan, streamed, st))
  return dtype == APHRO_F16 ? DR_ACT(Half) : DR_ACT(BFloat);
#undef DR_ACT
}
