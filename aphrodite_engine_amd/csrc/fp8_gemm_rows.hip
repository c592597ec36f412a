// FP8 W8A8 product for 33 to 192 rows: the tile of dense_rows.h with v_mfma_scale_f32_16x16x128_f8f6f4 (unit E8M0 scales), a step of 128 bytes a
// row being one product.  A lane takes 16-byte chunks g and 4 + g of its row in both operands -- any bijection between (lane group, byte)
// and k is a valid operand order.  Bound by reading w once.  Results are scaled and rounded here, or left as raw fp32 slabs for a fused consumer
// (fp8_gemm.hip's contract); a slab per K slice, added in order.
// Measured, us, weights from memory, graph replay, [N, K] with 64 / 128 / 192 rows; in brackets the kernels before (fp8_gemm.hip's two passes of 32
// rows, from 65 on the prompt kernel); raw slabs last:
//   [28672, 4096]   30.7 / 32.5 / 36.8  (59.7 / 33.4 / 38.2)      27.8 / 30.8 / 35.0
//   [4096, 14336]   18.7 / 22.2 / 27.1  (36.8 / 25.3 / 30.4)      13.3 / 17.0 / 21.1
//   [6144, 4096]    14.4 / 17.9 / 19.8  (17.0 / 18.8 / 22.9)       9.2 / 12.4 / 14.5
//   [4096, 4096]    11.1 / 14.8 / 18.9  (12.7 / 19.2 / 22.8)       7.0 /  9.1 / 10.4
// (raw slabs: with the non-temporal hint on w's loads, as where weights_streamed; without it 29.5 / 32.3 / 36.6, 14.0 / 17.5 / 21.3, 9.3 / 12.3 / 14.6 and 7.1 / 9.3 / 10.4)
// (a result in 16 bits over several K slices pays a second launch; the same bits as before at every shape measured)
#include "dense_rows.h"

namespace aphro {

struct Fp8RowsParams {
  RowsOperands op;
  const float* a_scales;
  const float* b_scales;
  const uint16_t* bias;
  uint16_t* out;            // [M, N], or null: the raw sums go to slabs
  float* slabs;             // [ksplit][M][N]
  int a_per_token, b_per_channel;
};

typedef int fr_i32x8 __attribute__((ext_vector_type(8)));

struct Fp8RowsProduct {
  static __device__ __forceinline__ fr_i32x8 fragment(const unsigned char* row, const int (&sw)[2]) {
    const u32x4 lo = *reinterpret_cast<const u32x4*>(row + sw[0]), hi = *reinterpret_cast<const u32x4*>(row + sw[1]);
    return fr_i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
  }
  template <int NT, int MTW>
  static __device__ __forceinline__ void step(const unsigned char* st, int wbase, int xbase, const int (&sw)[2], f32x4 (&acc)[NT][MTW]) {
    fr_i32x8 wf[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) wf[t] = fragment(st + wbase + t * 8192, sw);
#pragma unroll
    for (int i = 0; i < MTW; ++i) {
      const fr_i32x8 xf = fragment(st + xbase + i * 2048, sw);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[t], xf, acc[t][i], 0, 0, 0, 127, 0, 127);
    }
  }
};

struct __attribute__((packed, aligned(4))) Fp8RowsQuad { float x[4]; };

// scales (and bias) of four neighbouring columns
template <typename T>
struct Fp8RowsColumns {
  float scale[4], bias[4];
  __device__ __forceinline__ void load(const Fp8RowsParams& p, int n) {
    if (p.b_per_channel) {
      const Fp8RowsQuad q = *reinterpret_cast<const Fp8RowsQuad*>(p.b_scales + n);
#pragma unroll
      for (int r = 0; r < 4; ++r) scale[r] = q.x[r];
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) scale[r] = p.b_scales[0];
    }
    if (p.bias)
#pragma unroll
      for (int r = 0; r < 4; ++r) bias[r] = T::to_f32(p.bias[n + r]);
  }
};

template <typename T>
__device__ __forceinline__ void fr_store(const Fp8RowsParams& p, int m, int n, float as, const Fp8RowsColumns<T>& cols, f32x4 v) {
  u16x4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float x = as * (cols.scale[r] * v[r]);
    asm("" : "+v"(x));                                 // (rounded to fp32 before the bias or the conversion, as the op's formula says)
    o[r] = from_f32_exact<T>(p.bias ? x + cols.bias[r] : x);
  }
  *reinterpret_cast<u16x4*>(p.out + (size_t)m * p.op.N + n) = o;
}

template <typename T, int MT, int NT, int WR, int NS, bool STREAM>
__global__ __launch_bounds__(256 * WR) void fp8_gemm_rows_kernel(Fp8RowsParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  RowsTile<Fp8RowsProduct, MT, NT, WR, NS, false, STREAM> tile;
  tile.run(p.op, smem);
  constexpr int MTW = MT / WR;
  const int m0 = tile.wr * MTW * 16 + tile.c, n0 = tile.n0 + 16 * tile.wc + 4 * tile.g, M = p.op.M, N = p.op.N;
  if (p.out == nullptr || p.op.ksplit > 1) {
    float* slab = p.slabs + (size_t)tile.ks * M * N;
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (m0 + 16 * i < M && n0 + 64 * t < N) *reinterpret_cast<f32x4*>(slab + (size_t)(m0 + 16 * i) * N + n0 + 64 * t) = tile.acc[t][i];
    return;
  }
  // (all scales at once: fetched in front of each store they cost 4 of 34 us on [28672, 4096])
  Fp8RowsColumns<T> cols[NT];
  float as[MTW];
#pragma unroll
  for (int t = 0; t < NT; ++t) cols[t].load(p, min(n0 + 64 * t, N - 4));
#pragma unroll
  for (int i = 0; i < MTW; ++i) as[i] = p.a_scales[p.a_per_token ? min(m0 + 16 * i, M - 1) : 0];
#pragma unroll
  for (int i = 0; i < MTW; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if (m0 + 16 * i < M && n0 + 64 * t < N) fr_store<T>(p, m0 + 16 * i, n0 + 64 * t, as[i], cols[t], tile.acc[t][i]);
}

template <typename T>
__global__ __launch_bounds__(256) void fp8_rows_reduce_kernel(Fp8RowsParams p) {
  const int N = p.op.N, n4 = N >> 2;
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= n4 * p.op.M) return;
  const int m = q / n4, col = (q - m * n4) * 4;
  Fp8RowsColumns<T> cols;
  cols.load(p, col);
  const float as = p.a_scales[p.a_per_token ? m : 0];
  const float* src = p.slabs + (size_t)m * N + col;
  f32x4 s = *reinterpret_cast<const f32x4*>(src);
  for (int k = 1; k < p.op.ksplit; ++k) s += *reinterpret_cast<const f32x4*>(src + (size_t)k * p.op.M * N);
  fr_store<T>(p, m, col, as, cols, s);
}

template <typename T>
static int fp8_rows_run(const Fp8RowsParams& p, const RowsPlan& plan, bool streamed, hipStream_t st) {
  const int rc = rows_dispatch<false>(plan, p.op.tiles_n, [&](auto mt, auto nt, auto wr, auto ns) {
    constexpr int MT = decltype(mt)::value, NT = decltype(nt)::value, WR = decltype(wr)::value, NS = decltype(ns)::value;
    if constexpr (MT < 3) {
      set_error("fp8_gemm_rows: fewer than 33 rows");
      return (int)APHRO_ERR_INVALID;
    } else {
      constexpr size_t lds = RowsTile<Fp8RowsProduct, MT, NT, WR, NS, false, true>::LDS;
      auto kern = streamed ? fp8_gemm_rows_kernel<T, MT, NT, WR, NS, true> : fp8_gemm_rows_kernel<T, MT, NT, WR, NS, false>;
      if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
        set_error("fp8_gemm_rows: cannot raise the dynamic LDS limit to %zu", lds);
        return (int)APHRO_ERR_LAUNCH;
      }
      hipLaunchKernelGGL(kern, dim3((unsigned)(p.op.tiles_n * p.op.ksplit)), dim3(256 * WR), lds, st, p);
      APHRO_LAUNCH_CHECK();
      return (int)APHRO_OK;
    }
  });
  if (rc != APHRO_OK || plan.ksplit == 1 || p.out == nullptr) return rc;
  hipLaunchKernelGGL((fp8_rows_reduce_kernel<T>), dim3((unsigned)((p.op.M * (p.op.N >> 2) + 255) / 256)), dim3(256), 0, st, p);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

}  // namespace aphro

using namespace aphro;

extern "C" int aphro_fp8_gemm_rows_ksplit(int64_t M, int64_t N, int64_t K) {
  if (M <= 32 || N % 16 != 0 || K % 128 != 0 || !rows_fits(M, N, K, K, K, false)) return 0;
  return rows_plan(M, N, K).ksplit;
}

// Whether aphro_scaled_mm_fp8 is the faster op for 65 rows and more: wherever it is served ([6144, 4096], the closest, 65 / 128 / 160 / 192 rows:
// 14.1 / 17.8 / 18.1 / 19.6 us, the prompt kernel 16.8 / 18.5 / 21.0 / 22.6).
extern "C" int aphro_fp8_gemm_rows_preferred(int64_t M, int64_t N, int64_t K) { return M > 64 && aphro_fp8_gemm_rows_ksplit(M, N, K) > 0; }

extern "C" int aphro_fp8_gemm_rows(const void* a, const void* w, const float* a_scales, const float* b_scales, const void* bias, void* out,
                                   float* slabs, size_t slabs_bytes, int64_t M, int64_t N, int64_t K, int a_scale_per_token,
                                   int b_scale_per_channel, int dtype, void* stream) {
  const bool streamed = weights_streamed(weights_flags(dtype), (size_t)N * K);
  APHRO_CHECK(dtype == APHRO_F16 || dtype == APHRO_BF16, "fp8_gemm_rows: output dtype must be f16 or bf16");
  const int split = aphro_fp8_gemm_rows_ksplit(M, N, K);
  APHRO_CHECK(split > 0, "fp8_gemm_rows: M=%ld N=%ld K=%ld is not served", (long)M, (long)N, (long)K);
  APHRO_CHECK(((uintptr_t)a % 16) == 0 && ((uintptr_t)w % 16) == 0 && ((uintptr_t)out % 8) == 0 && ((uintptr_t)slabs % 16) == 0,
              "fp8_gemm_rows: 16-byte aligned operands and slabs, 8-byte aligned output required");
  APHRO_CHECK(out == nullptr || (a_scales && b_scales), "fp8_gemm_rows: scales needed");
  if (out == nullptr || split > 1) {
    const size_t need = (size_t)split * M * N * sizeof(float);
    if (slabs == nullptr || slabs_bytes < need) {
      set_error("fp8_gemm_rows: workspace %zu < %zu bytes", slabs_bytes, need);
      return APHRO_ERR_WORKSPACE;
    }
  }
  const RowsPlan plan = rows_plan(M, N, K);
  Fp8RowsParams p;
  p.op.a = (const uint8_t*)a; p.op.w = (const uint8_t*)w; p.op.M = (int)M; p.op.N = (int)N;
  p.op.row_bytes = p.op.lda = p.op.ldw = (int)K;
  p.op.tiles_n = (int)((N + 64 * plan.nt - 1) / (64 * plan.nt));
  p.op.ksplit = plan.ksplit;
  p.a_scales = a_scales; p.b_scales = b_scales; p.bias = (const uint16_t*)bias; p.out = (uint16_t*)out; p.slabs = slabs;
  p.a_per_token = a_scale_per_token; p.b_per_channel = b_scale_per_channel;
  return dtype == APHRO_F16 ? fp8_rows_run<Half>(p, plan, streamed, (hipStream_t)stream) : fp8_rows_run<BFloat>(p, plan, streamed, (hipStream_t)stream);
}
