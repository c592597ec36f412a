// Shared by the kernels of libaphrodite_mi355x_mixers.so: dtype dispatch and block reductions.  wave = 64 lanes.
#pragma once
#include "../common.h"
#include "../../../include/aphrodite_mi355x_mixers.h"

namespace aphro {

// Activation / weight storage of this library: bf16 or fp32 (APHRO_BF16 / APHRO_F32).  fp32 is a true 32-bit path:
// no reduced-precision product anywhere.
#define MIX_DISPATCH_DTYPE(dtype, ...)                                             \
  do {                                                                             \
    if ((dtype) == APHRO_BF16) { typedef ::aphro::BFloat T; __VA_ARGS__; }          \
    else if ((dtype) == APHRO_F32) { typedef ::aphro::Float T; __VA_ARGS__; }       \
    else { ::aphro::set_error("dtype %d: this library serves bf16 (1) and fp32 (2)", (int)(dtype)); return APHRO_ERR_INVALID; } \
  } while (0)

// sum over a workgroup of up to 16 waves; every thread gets the total.  red: >= 16 floats of LDS.
__device__ __forceinline__ float wg_sum(float v, float* red) {
  v = wave_sum(v);
  const int nw = (blockDim.x + 63) >> 6;
  if (nw == 1) return v;
  __syncthreads();                     // a previous use of red may still be read
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
  for (int w = 0; w < nw; ++w) t += red[w];
  return t;
}

// the same for an ``red`` that nothing in the kernel has used before: one barrier instead of two
__device__ __forceinline__ float wg_sum_once(float v, float* red) {
  v = wave_sum(v);
  const int nw = (blockDim.x + 63) >> 6;
  if (nw == 1) return v;
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
  for (int w = 0; w < nw; ++w) t += red[w];
  return t;
}

// Sums over groups of 2^LOG adjacent lanes with DPP moves (no LDS round trip): quad permutes for 2 and 4, the half-row and
// row mirrors for 8 and 16 (after the quad steps every lane of a quad holds the quad's total, so the mirror partner brings
// in the other half); every lane of a group ends with the group's total.  Wider groups finish with ds_bpermute shuffles.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
template <int LOG>
__device__ __forceinline__ float group_sum(float v) {
  if (LOG >= 1) v += dpp_f<0xB1>(v);       // quad_perm [1, 0, 3, 2]
  if (LOG >= 2) v += dpp_f<0x4E>(v);       // quad_perm [2, 3, 0, 1]
  if (LOG >= 3) v += dpp_f<0x141>(v);      // row_half_mirror
  if (LOG >= 4) v += dpp_f<0x140>(v);      // row_mirror
  if (LOG >= 5) v += __shfl_xor(v, 16, 64);
  if (LOG >= 6) v += __shfl_xor(v, 32, 64);
  return v;
}

// 8 numbers as they lie in memory (16 bytes of bf16, 32 of fp32): rows in flight take no more registers than that
template <typename T>
struct Chunk8 {
  u32x4 v[sizeof(typename T::storage) / 2];
  __device__ __forceinline__ void load(const typename T::storage* p) {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(typename T::storage) / 2); ++i) v[i] = reinterpret_cast<const u32x4*>(p)[i];
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(typename T::storage) / 2); ++i) v[i] = u32x4{0, 0, 0, 0};
  }
  __device__ __forceinline__ void store(typename T::storage* p) const {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(typename T::storage) / 2); ++i) reinterpret_cast<u32x4*>(p)[i] = v[i];
  }
  __device__ __forceinline__ void floats(float* o) const {
    if constexpr (sizeof(typename T::storage) == 2) {
      const u16x8 x = __builtin_bit_cast(u16x8, v[0]);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = T::to_f32(x[j]);
    } else {
      const f32x4 a = __builtin_bit_cast(f32x4, v[0]), b = __builtin_bit_cast(f32x4, v[1]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        o[j] = a[j];
        o[4 + j] = b[j];
      }
    }
  }
};

// Sums over the four rows of 16 lanes of a wave, scattered: of four values a lane, the lane ends with the total of one over the lanes of its
// column (lane % 16), without a shuffle through LDS: of value scatter_index4(lane).  (A bit cast of a vector's element, without the
// conversion in between, reads element 0 whatever its index.)
__device__ __forceinline__ float swap_add32(float a, float b) {          // lower half: a of both halves, upper half: b
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ float swap_add16(float a, float b) {          // even rows: a of the two rows, odd rows: b
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
// the value whose total a lane ends with
__device__ __forceinline__ float scatter_sum4(const float (&v)[4]) { return swap_add16(swap_add32(v[0], v[1]), swap_add32(v[2], v[3])); }
__device__ __forceinline__ int scatter_index4(int lane) { return ((lane >> 5) & 1) | ((lane >> 3) & 2); }

// NI neighbouring floats of LDS, in the widest pieces that NI allows
template <int NI>
__device__ __forceinline__ void lds_row(const float* p, float (&o)[NI]) {
  if constexpr (NI % 4 == 0) {
#pragma unroll
    for (int i = 0; i < NI; i += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(p + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[i + j] = x[j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < NI; i += 2) {
      const f32x2 x = *reinterpret_cast<const f32x2*>(p + i);
      o[i] = x[0];
      o[i + 1] = x[1];
    }
  }
}

// out [rows, n] = x / rms(x over its group) * out_scale * weight * act(gate), x fp32 dense, groups of neighbouring columns; weight [n], or
// [group] shared by the groups (``shared``), or NULL; gate [rows, n] or NULL, act 0 sigmoid, 1 silu.  False: not a form that the launch serves
// (groups of whole 8s up to 8192, 16-byte pieces).
bool group_rms_norm_launch(void* out, int64_t out_stride, const float* x, const void* weight, bool shared, const void* gate, int64_t gate_stride,
                           int64_t rows, int n, int group, float eps, float out_scale, int act, int dtype, hipStream_t stream);

// n / (1 + e^-z): the reciprocal's product, one correction and the hardware's rules for zeros, infinities and NaN, without a division's scaling (ten
// instructions for seven), and with a division's bits wherever n is not scaled: the reciprocal is a quarter's, as that of 2^126 and more would be
// taken for zero.  Every 257th of all floats: a division's bits.  Where the vector units bound: decay memories of 4096 tokens, 16 heads, 86.6 -> 83.9 us, a
// convolution of 2024 rows 18.5 -> 17.6, with both sides scaled (six instructions, two bits less below 4.7e-38; the seventh: 88.6 -> 88.9 on one card).
__device__ __forceinline__ float over_1_exp_f(float n, float z) {
  const float d = 1.0f + __expf(-z), r = 0.25f * __builtin_amdgcn_rcpf(0.25f * d), q = n * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, d, n), r, q), d, n);
}
__device__ __forceinline__ float sigmoid_f(float z) { return over_1_exp_f(1.0f, z); }
__device__ __forceinline__ float silu_f(float z) { return over_1_exp_f(z, z); }
__device__ __forceinline__ float gelu_tanh_f(float z) {
  const float u = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  return 0.5f * z * (1.0f + tanhf(u));
}
// log(1 + e^z) = max(z, 0) + 2 atanh(h / 2), h = x / (1 + x / 2), x = e^-|z|: h in two numbers, atanh by its series in h^2 (coefficients fitted by least
// squares over h <= 2 / 3, 1e-10), the sum with what its first step rounds away (z = infinity leaves NaN there: -1 for it).  No branch.  Error against 64 bits, of the result, x 2^-24, largest and root mean square, log1pf(expf(z)) / here: over
// [-20, 20] 2.26, 0.495 / 2.26, 0.491; [-1, -0.1] 1.80, 0.549 / 1.88, 0.551; [-0.1, 0.1] 1.66, 0.528 / 1.49, 0.479; [0.1, 1] 1.61, 0.517 / 1.39, 0.464.
__device__ __forceinline__ float softplus_f(float z) {
  const float x = expf(-fabsf(z)), d = fmaf(x, 0.5f, 1.f), dl = fmaf(x, 0.5f, 1.f - d), r = __builtin_amdgcn_rcpf(d);
  const float h = x * r, hl = fmaf(-h, dl, fmaf(-h, d, x)) * r, t = h * h;
  const float s = fmaf(fmaf(fmaf(fmaf(0.12120297f / 1024, t, 0.10722389f / 256), t, 0.14307591f / 64), t, 0.19999473f / 16), t, 0.33333337f / 4);
  const float m = fmaxf(z, 0.f), a = fmaxf(m, h), b = fminf(m, h), sum = a + b;
  return sum + (fmaxf(b - (sum - a), -1.f) + fmaf(h * t, s, hl));
}
// log(sigmoid(z)) without overflow on either side
__device__ __forceinline__ float log_sigmoid_f(float z) {
  return fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
}

}  // namespace aphro
