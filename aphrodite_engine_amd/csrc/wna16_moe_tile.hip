// Grouped W4A16 expert GEMM for PROMPT-sized batches on gfx950 (the marlin_gemm_moe role, kernels/moe/marlin_moe_ops.cu, where an expert
// has dozens of rows or more), and the routing in front of it.  wna16_gemm_kernel (wna16_gemm.hip) serves decode-sized batches: one
// 16-row m-tile a workgroup, every weight read and unpacked once per 16 rows.
//
//   * tile = 64 WM rows of ONE expert (a block of moe_align) x 256 columns, 4 WM waves of 64 x 64, K tile 64.
//     D^T[n][m] = W^T[n][k] . A^T[k][m] with v_mfma_f32_32x32x16_f16 as in wna16_gemm_large.hip: an exllama dword is a lane's weight fragment.
//   * the weights enter the product as the integers q - z (exact in f16); a group's fp32 sum is multiplied by the group's scale in fp32 and
//     added to the total -- the decode kernel's numerics, no rounding of a weight.  That costs one FMA per accumulator element and group
//     (64 per 128 k of 32 MFMAs) and saves the multiply of every dword.
//   * activations go global -> LDS with direct-to-LDS loads, 128-byte rows XOR-swizzled on the source address; the first GEMM GATHERS them:
//     the row's token comes from the sorted slots, nothing is copied in front.  Three or four stages of activations and packed weights, one
//     raw barrier per K tile; scales and zero points of the workgroup's columns in LDS for its whole K range.
//   * epilogue: SiluAndMul of interleaved (gate, up) columns into 16-bit rows (first GEMM), or the fp32 total (second; K slices as
//     further slabs, summed by moe_combine).
//   * workgroups go eight row blocks x all column tiles at a time, contiguous ranges per XCD: an XCD's L2 sees a few column tiles'
//     weights and eight blocks' activations at once.
// Bound by the matrix pipe and the vector ALUs together (9 VALU a dword in each of the two waves that share its columns, one FMA an
// accumulator element and group).  Mixtral-8x7B's two GEMMs: 160 tokens 451 -> 258 us, 3000 tokens 6900 -> 2500 us, 0.85 PFLOP/s of the
// useful work (padding to blocks is another 4 to 8 %).  On the way, 3000 tokens: scale converts behind a run-time branch 3260, this
// pipeline with three stages 2670, with four 2480 us.
#include <type_traits>

#include "common.h"

namespace aphro {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;

struct MoeTileParams {
  const uint16_t* a;          // f16 [rows, lda]
  const int32_t* slots;       // gather: sorted slots, row = slot / topk; NULL: rows as they are
  const uint32_t* qw;         // [E, K/8, N]
  const uint32_t* qz;         // [E, G, N/8]
  const uint16_t* sc;         // [E, G, N]
  const int32_t* expert_ids;  // [blocks]
  const int32_t* num_post_pad;
  uint16_t* act;              // SiluAndMul output f16 [m_pad, N / 2], or
  float* out;                 // [ksplit, m_pad, N]
  uint32_t a_bytes;           // of a, its last row to K
  int numel, topk, lda, N, K, group_size, zero_offset;
  int m_pad, ksplit;
};

__device__ __forceinline__ uint32_t mt_and_or(uint32_t a, uint32_t mask, uint32_t orv) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(mask), "v"(orv));
  return r;
}
// one exllama dword -> 8 integers q - z as f16, exact
__device__ __forceinline__ f16x8 mt_dq8(uint32_t w, f16x2 zh, f16x2 zh16) {
  const f16x2 inv16 = {(f16)0.0625f, (f16)0.0625f};
  const uint32_t magic = 0x64006400u;
  const uint32_t q0 = mt_and_or(w, 0x000f000fu, magic);
  const uint32_t q1 = mt_and_or(w, 0x00f000f0u, magic);
  const uint32_t w8 = w >> 8;
  const uint32_t q2 = mt_and_or(w8, 0x000f000fu, magic);
  const uint32_t q3 = mt_and_or(w8, 0x00f000f0u, magic);
  const f16x2 d0 = __builtin_bit_cast(f16x2, q0) - zh;
  const f16x2 d1 = __builtin_bit_cast(f16x2, q1) * inv16 + zh16;
  const f16x2 d2 = __builtin_bit_cast(f16x2, q2) - zh;
  const f16x2 d3 = __builtin_bit_cast(f16x2, q3) * inv16 + zh16;
  u32x4 r = {__builtin_bit_cast(uint32_t, d0), __builtin_bit_cast(uint32_t, d1), __builtin_bit_cast(uint32_t, d2),
             __builtin_bit_cast(uint32_t, d3)};
  return __builtin_bit_cast(f16x8, r);
}

constexpr int MT_BN = 256, MT_BK = 64;
// LDS stages: four for the workgroup that fills a CU by itself (two K tiles in flight behind the one that is multiplied), three for the
// 64-row one, so that two of them share a CU.
constexpr int mt_stages(int wm) { return wm == 2 ? 4 : 3; }
constexpr size_t mt_lds(int wm, size_t groups) {
  return (size_t)mt_stages(wm) * (64 * wm * MT_BK * 2 + MT_BK / 8 * MT_BN * 4) + groups * (MT_BN * 2 + MT_BN / 8 * 4);
}

// G128: groups of 128 k, the K loop's own step; else (128 x 2^n) a step may continue a group.
template <int WM, bool SILU, bool BF16, bool G128>
__global__ __launch_bounds__(WM * 256) void wna16_moe_tile_kernel(MoeTileParams p) {
  constexpr int NWAVE = 4 * WM, BM = 64 * WM, STAGES = mt_stages(WM);
  constexpr int A_STAGE = BM * MT_BK * 2, B_STAGE = (MT_BK / 8) * MT_BN * 4, STAGE = A_STAGE + B_STAGE;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int kh = lane >> 5, l31 = lane & 31;
  // ---- which tile ---------------------------------------------------------------------------------------------------------------
  const int nblk = *p.num_post_pad / BM, tiles_n = p.N / MT_BN, total = nblk * tiles_n;
  if ((int)blockIdx.x >= total) return;
  int lin;
  {
    const int q = total / 8, r = total % 8, xcd = blockIdx.x % 8, k = blockIdx.x / 8;
    lin = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + k;
  }
  const int grp8 = lin / (8 * tiles_n), rem = lin - grp8 * 8 * tiles_n, nb8 = min(8, nblk - grp8 * 8);
  const int blk = grp8 * 8 + rem % nb8, n0 = rem / nb8 * MT_BN, m0 = blk * BM;
  const int e = p.expert_ids[blk];
  if (e < 0) return;
  const int klen = p.K / p.ksplit, k_begin = blockIdx.y * klen, ktiles = klen / MT_BK;
  const int G_all = p.K / p.group_size, g_begin = k_begin / p.group_size, G = klen / p.group_size;
  const uint32_t* qw = p.qw + (size_t)e * (p.K >> 3) * p.N;
  const uint32_t* qz = p.qz + ((size_t)e * G_all + g_begin) * (p.N >> 3) + (n0 >> 3);
  const uint16_t* sc = p.sc + ((size_t)e * G_all + g_begin) * p.N + n0;
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(qw), 0, (uint32_t)((size_t)(p.K >> 3) * p.N * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a), 0, p.a_bytes, 0x00020000);
  // ---- scales and zero points of the columns for the K range ----------------------------------------------------------------------
  uint16_t* meta_sc = reinterpret_cast<uint16_t*>(smem + STAGES * STAGE);
  uint32_t* meta_z = reinterpret_cast<uint32_t*>(smem + STAGES * STAGE + G * MT_BN * 2);
  for (int i = threadIdx.x; i < G * (MT_BN / 8); i += NWAVE * 64) {
    const int g = i / (MT_BN / 8), j = i % (MT_BN / 8);
    reinterpret_cast<u32x4*>(meta_sc)[i] = *reinterpret_cast<const u32x4*>(sc + (size_t)g * p.N + j * 8);
    meta_z[i] = qz[(size_t)g * (p.N >> 3) + j];
  }
  // ---- staging --------------------------------------------------------------------------------------------------------------------
  constexpr int A_PER_WAVE = BM / 8 / NWAVE, B_PER_WAVE = B_STAGE / 1024 / NWAVE;
  uint32_t a_voff[A_PER_WAVE];
#pragma unroll
  for (int i = 0; i < A_PER_WAVE; ++i) {
    const int row = (wave * A_PER_WAVE + i) * 8 + (lane >> 3);
    const int slot = (lane & 7) ^ ((row >> 1) & 7);
    int src = m0 + row;
    if (p.slots != nullptr) {
      const int sl = p.slots[src];
      src = ((uint32_t)sl < (uint32_t)p.numel ? sl : 0) / p.topk;               // (a padding row multiplies some token's row; nobody reads the result)
    }
    a_voff[i] = ((uint32_t)src * (uint32_t)p.lda + slot * 8) * 2;
  }
  const int b_row_bytes = p.N * 4;
  auto stage = [&](int st, int kt) {
    unsigned char* sa = smem + st * STAGE;
#pragma unroll
    for (int i = 0; i < A_PER_WAVE; ++i) {
      const int voff = (int)a_voff[i];                      // (a local copy: see wna16_gemm_large.hip)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_ptr)(sa + (wave * A_PER_WAVE + i) * 1024), 16, voff,
                                               (k_begin + kt * MT_BK) * 2, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < B_PER_WAVE; ++i) {
      const int row = wave * B_PER_WAVE + i;                // one packed row of 256 columns per instruction
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void_ptr)(sa + A_STAGE + row * 1024), 16, n0 * 4 + lane * 16,
                                               (k_begin / 8 + kt * 8 + row) * b_row_bytes, 0, 0);
    }
  };
  f32x16 tot[2][2], acc[2][2];
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) tot[nb][mb][r] = 0.f;

  constexpr int DMA_PER_TILE = A_PER_WAVE + B_PER_WAVE;
  stage(0, 0);
  stage(1, 1);                                               // (a K range holds whole groups: two tiles at least)
  __syncthreads();                                           // scales and zero points are published, tiles 0 and 1 are there
  if (STAGES == 4 && ktiles > 2) stage(2, 2);
  // A step is 16 k.  While its MFMAs run the next step's activations come from LDS and its weights -- read two steps ahead, a pair of
  // steps at a time -- are unpacked, across the tiles' borders too.  Halfway through a tile the next one has to be there: with four stages
  // it has landed once at most one tile's loads are outstanding (the tile after it), with three when none is.  Past the barrier every wave
  // is through with the tile BEFORE this one, whose stage the next tile to be fetched takes.
  auto cross = [&](int kt) {
    if (kt + 1 >= ktiles) return;
    if (STAGES == 4 && kt + 2 < ktiles) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(DMA_PER_TILE) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (kt + STAGES - 1 < ktiles) stage((kt + STAGES - 1) % STAGES, kt + STAGES - 1);
  };
  f16x2 zh[2], zh16[2];
  auto zeros = [&](int grp) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int col = wn * 64 + nb * 32 + l31;
      const int z = (int)((meta_z[grp * (MT_BN / 8) + (col >> 3)] >> ((col & 7) * 4)) & 0xf) + p.zero_offset;
      const f16 a16 = __builtin_bit_cast(f16, (uint16_t)(0x6400 | z));        // 1024 + z
      const f16 b16 = (f16)(float)(-64 - z);
      zh[nb] = f16x2{a16, a16};
      zh16[nb] = f16x2{b16, b16};
    }
  };
  // fragment addresses: rows 32 apart keep the swizzle, a step moves the 16-byte slot
  const uint32_t a_base = (uint32_t)(wm * 64 + l31) * 128u, a_swz = (uint32_t)((l31 >> 1) & 7);
  const uint32_t b_base = (uint32_t)(A_STAGE + (kh * MT_BN + wn * 64 + l31) * 4);
  auto read_a = [&](int kt, int j, u32x4 (&a2)[2]) {
    const unsigned char* sa = smem + kt % STAGES * STAGE;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) a2[mb] = *reinterpret_cast<const u32x4*>(sa + a_base + mb * 4096 + (((uint32_t)(2 * j + kh) ^ a_swz) << 4));
  };
  auto read_w = [&](int kt, int j, uint32_t (&w2)[2]) {
    const unsigned char* sa = smem + kt % STAGES * STAGE;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) w2[nb] = *reinterpret_cast<const uint32_t*>(sa + b_base + (2 * j * MT_BN + nb * 32) * 4);
  };
  u32x4 af[2][2];
  uint32_t wraw[4][2];
  f16x8 wf[2][2];
  int grp = 0, in_group = 0;
  zeros(0);
  read_a(0, 0, af[0]);
  read_w(0, 0, wraw[0]);
  read_w(0, 1, wraw[1]);
#pragma unroll
  for (int nb = 0; nb < 2; ++nb) wf[0][nb] = mt_dq8(wraw[0][nb], zh[nb], zh16[nb]);
  const int steps_per_group = G128 ? 1 : p.group_size / (2 * MT_BK);
  for (int kt = 0; kt < ktiles; kt += 2) {
    const bool last = G128 || in_group + 1 == steps_per_group;      // the group ends with this pair of tiles
    f16x4 s4[2][4];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int t = kt + (j >> 2);                          // (behind the last tile the fragments are what lies in the stage: never multiplied)
      if ((j & 3) == 2) cross(t);
      if ((j & 1) == 0) {
        read_w((j & 3) == 0 ? t : t + 1, (j + 2) & 3, wraw[(j + 2) & 3]);
        read_w((j & 3) == 0 ? t : t + 1, (j + 3) & 3, wraw[(j + 3) & 3]);
      }
      read_a((j & 3) == 3 ? t + 1 : t, (j + 1) & 3, af[(j + 1) & 1]);
      if (j == 4 && last) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            s4[nb][q] = *reinterpret_cast<const f16x4*>(meta_sc + grp * MT_BN + wn * 64 + nb * 32 + 8 * q + 4 * kh);
      }
      if (j == 7 && last && kt + 2 < ktiles) zeros(grp + 1);
      if (j == 0 && (G128 || in_group == 0)) {
        const f32x16 zero = {};
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
            acc[nb][mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[0][nb], __builtin_bit_cast(f16x8, af[0][mb]), zero, 0, 0, 0);
      } else {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
            acc[nb][mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[j & 1][nb], __builtin_bit_cast(f16x8, af[j & 1][mb]), acc[nb][mb], 0, 0, 0);
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) wf[(j + 1) & 1][nb] = mt_dq8(wraw[(j + 1) & 3][nb], zh[nb], zh16[nb]);
    }
    if (last) {
      // the group's sums join the total: lane's columns of a quad are nb * 32 + 8 q + 4 kh + (0..3)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float sv = BF16 ? bf16_bits_to_f32(__builtin_bit_cast(u16x4, s4[nb][q])[r]) : (float)s4[nb][q][r];
              tot[nb][mb][4 * q + r] = __builtin_fmaf(sv, acc[nb][mb][4 * q + r], tot[nb][mb][4 * q + r]);
            }
      in_group = 0;
      ++grp;
    } else {
      ++in_group;
    }
  }
  if constexpr (!SILU) {
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
      float* prow = p.out + ((size_t)blockIdx.y * p.m_pad + m0 + wm * 64 + mb * 32 + l31) * p.N + n0 + wn * 64;
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<f32x4*>(prow + nb * 32 + 8 * q + 4 * kh) =
              f32x4{tot[nb][mb][4 * q], tot[nb][mb][4 * q + 1], tot[nb][mb][4 * q + 2], tot[nb][mb][4 * q + 3]};
    }
  } else {
    // a quad's four columns are two (gate, up) pairs -> two activations = one dword; 64 rows x 64 bytes in the wave's LDS region, 16-byte
    // chunks XOR-ed with (row >> 2) & 3, out as whole 64-byte row segments (wna16_gemm_large.hip)
    __syncthreads();
    unsigned char* region = smem + wave * 4096;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = mb * 32 + l31, c4 = nb * 8 + 2 * q + kh;
          uint16_t o[2];
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const float gate = tot[nb][mb][4 * q + 2 * t], up = tot[nb][mb][4 * q + 2 * t + 1];
            if constexpr (BF16)
              o[t] = bf16_bits_to_f16_bits_sat(silu_mul_bits<BFloat>(BFloat::to_f32(BFloat::from_f32(gate)), BFloat::to_f32(BFloat::from_f32(up))));
            else
              o[t] = silu_mul_bits<Half>(Half::to_f32(Half::from_f32(gate)), Half::to_f32(Half::from_f32(up)));
          }
          *reinterpret_cast<uint32_t*>(region + row * 64 + ((((c4 >> 2) ^ ((row >> 2) & 3)) << 4) | ((c4 & 3) << 2))) =
              (uint32_t)o[0] | ((uint32_t)o[1] << 16);
        }
    const int64_t ldc = p.N / 2;
    uint16_t* c = p.act + (int64_t)(m0 + wm * 64) * ldc + (n0 + wn * 64) / 2;
    const int r16 = lane >> 2, c16 = lane & 3;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = i * 16 + r16;
      *reinterpret_cast<u32x4*>(c + (int64_t)row * ldc + c16 * 8) =
          *reinterpret_cast<const u32x4*>(region + row * 64 + ((c16 ^ ((row >> 2) & 3)) << 4));
    }
  }
}

__global__ void moe_rows_to_f16_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int64_t rows, int K, int64_t lda) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (i >= rows * K) return;
  u16x8 v = *reinterpret_cast<const u16x8*>(in + i / K * lda + i % K);
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = bf16_bits_to_f16_bits_sat(v[j]);
  *reinterpret_cast<u16x8*>(out + i) = v;
}

template <int WM, bool SILU, bool BF16, bool G128>
static int moe_tile_launch_t(const MoeTileParams& p, int64_t blocks, hipStream_t st) {
  const size_t lds = mt_lds(WM, (size_t)(p.K / p.group_size / p.ksplit));
  APHRO_CHECK(lds <= 160 * 1024, "wna16_moe_tile: %zu bytes of LDS", lds);
  static bool attr_set_dev[APHRO_MAX_DEVICES] = {};
  bool& attr_set = attr_set_dev[device_slot()];
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)wna16_moe_tile_kernel<WM, SILU, BF16, G128>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess) {
      set_error("wna16_moe_tile: cannot raise the dynamic LDS limit");
      return APHRO_ERR_LAUNCH;
    }
    attr_set = true;
  }
  hipLaunchKernelGGL((wna16_moe_tile_kernel<WM, SILU, BF16, G128>), dim3((unsigned)(blocks * (p.N / MT_BN)), (unsigned)p.ksplit), dim3(WM * 256), lds, st, p);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}
template <int WM, bool SILU>
static int moe_tile_launch(const MoeTileParams& p, int64_t blocks, bool bf16, hipStream_t st) {
  if (p.group_size == 128) return bf16 ? moe_tile_launch_t<WM, SILU, true, true>(p, blocks, st) : moe_tile_launch_t<WM, SILU, false, true>(p, blocks, st);
  return bf16 ? moe_tile_launch_t<WM, SILU, true, false>(p, blocks, st) : moe_tile_launch_t<WM, SILU, false, false>(p, blocks, st);
}

}  // namespace aphro

using namespace aphro;

// K slices of the second GEMM for `blocks` row blocks: enough workgroups for the chip to be full a few times over, whole groups per slice,
// no more groups than the LDS holds beside the stages -- for 64-row blocks in half of it, so that two workgroups share a CU, as far as four
// slices do that.  0: the shape is not served.
static int moe_tile_ksplit(int64_t blocks, int64_t N, int64_t K, int64_t groups, int block_m, int silu) {
  if (groups <= 0 || K % groups != 0 || N % MT_BN != 0 || (block_m != 64 && block_m != 128)) return 0;
  if (K / groups % 128 != 0 || K / 8 * N * 4 > 0xffffffffll) return 0;
  const int64_t tiles = blocks * (N / MT_BN), cus = device_cu_count();
  int ks = 1;
  for (;;) {
    const size_t lds = mt_lds(block_m / 64, (size_t)(groups / ks));
    const bool must = lds > 160 * 1024, want = !silu && ks < 4 && (tiles * ks < 2 * cus || (block_m == 64 && lds > 80 * 1024));
    if (!must && !want) break;
    if (groups % (2 * ks) != 0) return must ? 0 : ks;
    ks *= 2;
  }
  return silu && ks > 1 ? 0 : ks;
}

extern "C" int aphro_wna16_moe_tile_ksplit(int64_t blocks, int64_t N, int64_t K, int64_t groups, int block_m, int silu) {
  return moe_tile_ksplit(blocks, N, K, groups, block_m, silu);
}

extern "C" int aphro_wna16_moe_tile(const void* a, int64_t rows, int64_t lda, const int32_t* sorted_slots, int64_t numel, int topk,
                                    const uint32_t* q_weight, const uint32_t* qzeros, const void* scales, const int32_t* expert_ids,
                                    const int32_t* num_tokens_post_pad, void* act, float* out, int64_t m_pad, int64_t N, int64_t K,
                                    int64_t groups, int ksplit, int block_m, int zero_offset, int dtype, void* stream) {
  APHRO_CHECK(dtype == APHRO_F16 || dtype == APHRO_BF16, "wna16_moe_tile: dtype must be f16 or bf16");
  APHRO_CHECK(a && q_weight && qzeros && scales && expert_ids && num_tokens_post_pad && (act != nullptr) != (out != nullptr), "wna16_moe_tile: null argument");
  APHRO_CHECK(block_m == 64 || block_m == 128, "wna16_moe_tile: blocks of 64 or 128 rows");
  APHRO_CHECK(m_pad > 0 && m_pad % block_m == 0 && topk >= 1, "wna16_moe_tile: m_pad=%ld is no multiple of %d", (long)m_pad, block_m);
  APHRO_CHECK(groups > 0 && K % groups == 0 && (K / groups) % 128 == 0 && N % MT_BN == 0 && ksplit >= 1 && groups % ksplit == 0 && (act == nullptr || ksplit == 1),
              "wna16_moe_tile: shape N=%ld K=%ld groups=%ld slices=%d is not served", (long)N, (long)K, (long)groups, ksplit);
  APHRO_CHECK(lda % 8 == 0 && lda >= K && ((uintptr_t)a % 16) == 0 && ((uintptr_t)scales % 16) == 0 && ((uintptr_t)q_weight % 16) == 0,
              "wna16_moe_tile: rows of 16 bytes");
  APHRO_CHECK((size_t)rows * lda * 2 < 0xffffffffull && K / 8 * N * 4 <= 0xffffffffll && m_pad / block_m * (N / MT_BN) <= 0x7fffffff,
              "wna16_moe_tile: operand exceeds 4 GiB");
  APHRO_CHECK(sorted_slots != nullptr ? numel >= 1 && (numel - 1) / topk < rows : m_pad <= rows, "wna16_moe_tile: rows outside the activations");
  MoeTileParams p;
  p.a_bytes = (uint32_t)(((rows - 1) * lda + K) * 2);
  p.a = (const uint16_t*)a; p.slots = sorted_slots; p.qw = q_weight; p.qz = qzeros; p.sc = (const uint16_t*)scales;
  p.expert_ids = expert_ids; p.num_post_pad = num_tokens_post_pad; p.act = (uint16_t*)act; p.out = out;
  p.numel = (int)numel; p.topk = topk; p.lda = (int)lda; p.N = (int)N; p.K = (int)K; p.group_size = (int)(K / groups);
  p.zero_offset = zero_offset; p.m_pad = (int)m_pad; p.ksplit = ksplit;
  const int64_t blocks = m_pad / block_m;
  hipStream_t st = (hipStream_t)stream;
  const bool bf = dtype == APHRO_BF16;
  if (block_m == 128) return act ? moe_tile_launch<2, true>(p, blocks, bf, st) : moe_tile_launch<2, false>(p, blocks, bf, st);
  return act ? moe_tile_launch<1, true>(p, blocks, bf, st) : moe_tile_launch<1, false>(p, blocks, bf, st);
}

// bf16 rows as the f16 the matrix cores multiply (saturating), dense.
extern "C" int aphro_moe_rows_to_f16(const void* a, void* out, int64_t rows, int64_t K, int64_t lda, void* stream) {
  APHRO_CHECK(a && out && K % 8 == 0 && lda % 8 == 0 && ((uintptr_t)a % 16) == 0 && K <= 0x7fffffff, "moe_rows_to_f16: rows of 16 bytes");
  if (rows == 0) return APHRO_OK;
  hipLaunchKernelGGL(moe_rows_to_f16_kernel, dim3((unsigned)((rows * K / 8 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (const uint16_t*)a,
                     (uint16_t*)out, rows, (int)K, lda);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}
