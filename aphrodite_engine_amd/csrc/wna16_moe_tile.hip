// Grouped W4A16 expert GEMM for PROMPT-sized batches on gfx950 (the marlin_gemm_moe role, kernels/moe/marlin_moe_ops.cu, where an expert
// has dozens of rows or more), and the routing in front of it.  wna16_gemm_kernel (wna16_gemm.hip) serves decode-sized batches: one
// 16-row m-tile a workgroup, every weight read and unpacked once per 16 rows.
//
//   * tile = up to 128 rows of ONE expert (a block of moe_align) x 256 columns, 8 waves of all the rows x 32 columns, K tile 64: a weight is
//     unpacked once and multiplied with every row.  D^T[n][m] = W^T[n][k] . A^T[k][m] with v_mfma_f32_32x32x16_f16 as in
//     wna16_gemm_large.hip: an exllama dword is a lane's weight fragment.  32-row pieces behind an expert's rows are left out: the code is
//     there for one to four of them.
//   * the weights enter the product as the integers q - z (exact in f16); a group's fp32 sum is multiplied by the group's scale in fp32 and
//     added to the total -- the decode kernel's numerics, no rounding of a weight.  That costs one FMA per accumulator element and group
//     (16 a product of eight) and saves the multiply of every dword.
//   * activations go global -> LDS with direct-to-LDS loads, 128-byte rows XOR-swizzled on the source address; the first GEMM GATHERS them:
//     the row's token comes from the sorted slots, nothing is copied in front.  Four stages of activations and packed weights, one raw barrier
//     per K tile; one piece or two have too few products for an LDS read's latency, so they read three steps ahead, with a barrier for two
//     tiles.  Scales and zero points of the workgroup's columns in LDS.
//   * epilogue: SiluAndMul of interleaved (gate, up) columns into 16-bit rows (first GEMM), or the fp32 total (second; K slices as
//     further slabs, summed by moe_combine).
//   * workgroups go eight row blocks x all column tiles at a time, contiguous ranges per XCD: an XCD's L2 sees a few column tiles'
//     weights and eight blocks' activations at once.
// Bound by the matrix pipe and the vector ALUs together: 9 operations a dword for one to four products and two a product for the groups' sums
// (waves of 64 x 64, which unpacked every dword twice, had 4.5 and two).  Mixtral-8x7B's experts, us, those waves / these: 100 tokens 259 / 198, 362
// 452 / 387, 1366 1263 / 1117, 3000 2591 / 2334, 4096 3568 / 3108 (0.93 PFLOP/s of the useful work).  4096 tokens without the groups' sums 1.09 of
// it, without the unpacking 1.08, without LDS reads 1.15, with products and weights' loads alone 1.45.  On the way: the groups' sums
// between the next group's first products instead of behind the last ones 15 to 25 % slower (both waves of a SIMD are then short of vector
// operations at once), five stages as fast as four, waves that ask for weights only beside ones that ask for activations only 10 % slower.
#include <type_traits>
#include <utility>

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
  const int32_t* row_slots;   // sorted slots of the rows, numel and more: padding; NULL: not known
};

__device__ __forceinline__ uint32_t mt_and_or(uint32_t a, uint32_t mask, uint32_t orv) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(mask), "v"(orv));
  return r;
}
constexpr int MT_BN = 256, MT_BK = 64;
constexpr int MT_W_STAGE = MT_BK / 8 * MT_BN * 4;
// One workgroup a CU with up to 128 rows, or two with up to 64 (TWO).  Behind the stages: scales and zero points, of so many groups at a time.
constexpr int mt_rows(bool two) { return two ? 64 : 128; }
constexpr int mt_meta(bool two) { return (two ? 3 : 4) * (mt_rows(two) * MT_BK * 2 + MT_W_STAGE); }
constexpr int mt_groups(bool two) { return two ? 48 : 96; }
constexpr size_t mt_lds(bool two, int64_t groups) { return (size_t)mt_meta(two) + (groups < mt_groups(two) ? groups : mt_groups(two)) * (MT_BN * 2 + MT_BN / 8 * 4); }
// 64-row blocks: two workgroups a CU in front of the activation (us, 100 / 160 / 220 tokens of Mixtral-8x7B: 125 / 156 / 167, one 135 / 175 / 190), one
// with fewer K slices behind it (two slices 58 / 79 / 95, two workgroups and four slices 58 / 89 / 111).
constexpr bool mt_two(int bm, bool silu) { return bm == 64 && silu; }

// f(integral_constant 0), .. f(integral_constant N - 1)
template <typename F, int... I>
__device__ __forceinline__ void mt_unroll_(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void mt_unroll(F&& f) { mt_unroll_(f, std::make_integer_sequence<int, N>{}); }

// Rows m0 .. m0 + 32 MB - 1, all of expert e, by 256 columns.  A wave's 32 columns are multiplied with all of the rows: each weight is unpacked
// once, and an unpacked one serves MB products.
template <int MB, bool TWO, bool SILU, bool BF16, bool G128>
__device__ __forceinline__ void moe_tile(const MoeTileParams& p, unsigned char* smem, int m0, int n0, int e) {
  // Few rows: fragments read three steps of 16 k ahead (one step's products cover an LDS read's latency from three blocks on), and one barrier for
  // two K tiles, three pairs of stages.  K tiles in LDS: SLOTS of UNIT tiles of SUB bytes.
  constexpr bool FEW = !TWO && MB <= 2;
  constexpr int GROUPS = mt_groups(TWO), META = mt_meta(TWO);
  constexpr int AHEAD = FEW ? 3 : 1, W_AHEAD = FEW ? 3 : 2, RING = AHEAD + 1;
  constexpr int A_BYTES = FEW ? MB * 4096 : mt_rows(TWO) * MT_BK * 2, SUB = A_BYTES + MT_W_STAGE, UNIT = FEW ? 2 : 1, SLOTS = TWO || FEW ? 3 : 4, SLOT = UNIT * SUB;
  static_assert(SLOTS * SLOT <= META, "");
  constexpr int A_LOADS = (MB + 1) / 2, LOADS = A_LOADS + 1;   // DMA instructions of a wave and K tile: 8 rows of activations, a packed row of weights
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kh = lane >> 5, l31 = lane & 31;
  const int klen = p.K / p.ksplit, k_begin = blockIdx.y * klen, ktiles = klen / MT_BK;
  const int G_all = p.K / p.group_size, g_begin = k_begin / p.group_size, G = klen / p.group_size;
  const uint32_t* qz = p.qz + ((size_t)e * G_all + g_begin) * (p.N >> 3) + (n0 >> 3);
  const uint16_t* sc = p.sc + ((size_t)e * G_all + g_begin) * p.N + n0;
  const uint32_t* qw = p.qw + (size_t)e * (p.K >> 3) * p.N;
  // ---- staging --------------------------------------------------------------------------------------------------------------------
  uint32_t a_voff[A_LOADS];
#pragma unroll
  for (int i = 0; i < A_LOADS; ++i) {
    const int row = (wave + 8 * i) % (4 * MB) * 8 + (lane >> 3);          // (where the waves outnumber the pieces, two of them fetch the same one)
    int src = m0 + row;
    if (p.slots != nullptr) {
      const int sl = p.slots[src];
      src = ((uint32_t)sl < (uint32_t)p.numel ? sl : 0) / p.topk;         // (a padding row multiplies some token's row; nobody reads the result)
    }
    a_voff[i] = ((uint32_t)src * (uint32_t)p.lda + ((lane & 7) ^ ((row >> 1) & 7)) * 8) * 2;
  }
  const uint32_t b_voff = (uint32_t)n0 * 4u + lane * 16u, b_step = (uint32_t)p.N * 32u;
  uint32_t a_off = (uint32_t)k_begin * 2u, b_off = (uint32_t)(k_begin / 8 + wave) * (uint32_t)p.N * 4u;
  int to_load = ktiles;                                      // K tiles from the next load's on; behind the last it is fetched again, and nobody reads it
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a), 0, p.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(qw), 0, (uint32_t)((size_t)(p.K >> 3) * p.N * 4), 0x00020000);
  auto load_a = [&](uint32_t st, int i) {
    const int voff = (int)a_voff[i];                         // (a local copy: see wna16_gemm_large.hip)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_ptr)(smem + st + (wave + 8 * i) % (4 * MB) * 1024), 16, voff, (int)a_off, 0, 0);
  };
  auto load_w = [&](uint32_t st) {
    const int voff = (int)b_voff;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void_ptr)(smem + st + A_BYTES + wave * 1024), 16, voff, (int)b_off, 0, 0);
  };
  auto advance = [&] {
    const bool more = to_load > 1;
    to_load -= more ? 1 : 0;
    a_off += more ? MT_BK * 2 : 0;
    b_off += more ? b_step : 0u;
  };
#pragma unroll
  for (int t = 0; t < (FEW ? SLOTS * UNIT : SLOTS - 1); ++t) {
    load_w(t * SUB);
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) load_a(t * SUB, i);
    asm volatile("" ::: "memory");                           // (the counted waits rely on the order of the loads)
    advance();
  }
  // ---- scales and zero points of the columns, up to GROUPS groups at a time ------------------------------------------------------
  uint16_t* meta_sc = reinterpret_cast<uint16_t*>(smem + META);
  uint32_t* meta_z = reinterpret_cast<uint32_t*>(smem + META + min(G, GROUPS) * MT_BN * 2);
  auto stage_meta = [&](int g0) {
    const int n = min(G - g0, GROUPS);
    for (int i = threadIdx.x; i < n * (MT_BN / 8); i += 512) {
      const int g = g0 + i / (MT_BN / 8), j = i % (MT_BN / 8);
      reinterpret_cast<u32x4*>(meta_sc)[i] = *reinterpret_cast<const u32x4*>(sc + (size_t)g * p.N + j * 8);
      meta_z[i] = qz[(size_t)g * (p.N >> 3) + j];
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  stage_meta(0);                                             // (the first tiles are there too)
  f32x16 tot[MB], acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) tot[mb][r] = acc[mb][r] = 0.f;
  const int col = wave * 32 + l31;
  f16x2 zh, zh16;
  auto zeros = [&](int grp) {
    const int z = (int)((meta_z[grp * (MT_BN / 8) + (col >> 3)] >> ((col & 7) * 4)) & 0xf) + p.zero_offset;
    const f16 a16 = __builtin_bit_cast(f16, (uint16_t)(0x6400 | z));          // 1024 + z
    const f16 b16 = (f16)960.f - a16;                                         // -64 - z
    zh = f16x2{a16, a16};
    zh16 = f16x2{b16, b16};
  };
  // fragment addresses: rows 32 apart keep the swizzle, a step moves the 16-byte slot
  uint32_t a_read[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) a_read[j] = (uint32_t)l31 * 128u + (((uint32_t)(2 * j + kh) ^ (uint32_t)((l31 >> 1) & 7)) << 4);
  const uint32_t w_read = (uint32_t)(A_BYTES + (kh * MT_BN + col) * 4);
  u32x4 af[RING][MB];
  uint32_t wraw[4];
  f16x8 wf[2];
  auto read_a = [&](uint32_t st, int j, int mb) { af[j & (RING - 1)][mb] = *reinterpret_cast<const u32x4*>(smem + st + a_read[j & 3] + mb * 4096); };
  auto read_w = [&](uint32_t st, int j) { wraw[j & 3] = *reinterpret_cast<const uint32_t*>(smem + st + w_read + (j & 3) * (2 * MT_BN * 4)); };
  // an exllama dword -> 8 integers q - z as f16, exact, in pieces of 3 operations
  f16x2 d0, d1, d2, d3;
  uint32_t w8, q0, q1, q2, q3;
  auto unpack = [&](int j, int piece) {
    const f16x2 inv16 = {(f16)0.0625f, (f16)0.0625f};
    const uint32_t magic = 0x64006400u, w = wraw[j & 3];
    if (piece == 0) {
      q0 = mt_and_or(w, 0x000f000fu, magic);
      q1 = mt_and_or(w, 0x00f000f0u, magic);
      w8 = w >> 8;
    } else if (piece == 1) {
      q2 = mt_and_or(w8, 0x000f000fu, magic);
      q3 = mt_and_or(w8, 0x00f000f0u, magic);
      d0 = __builtin_bit_cast(f16x2, q0) - zh;
    } else {
      d1 = __builtin_bit_cast(f16x2, q1) * inv16 + zh16;
      d2 = __builtin_bit_cast(f16x2, q2) - zh;
      d3 = __builtin_bit_cast(f16x2, q3) * inv16 + zh16;
      wf[j & 1] = __builtin_bit_cast(f16x8, u32x4{__builtin_bit_cast(uint32_t, d0), __builtin_bit_cast(uint32_t, d1), __builtin_bit_cast(uint32_t, d2),
                                                  __builtin_bit_cast(uint32_t, d3)});
    }
  };
  // a group's sums join the total: the lane's columns of a quad are 8 q + 4 kh + (0..3)
  f16x4 s4[4];
  auto read_scales = [&](int grp) {
#pragma unroll
    for (int q = 0; q < 4; ++q) s4[q] = *reinterpret_cast<const f16x4*>(meta_sc + grp * MT_BN + wave * 32 + 8 * q + 4 * kh);
  };
  auto fold = [&](int mb) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float sv = BF16 ? bf16_bits_to_f32(__builtin_bit_cast(u16x4, s4[q])[r]) : (float)s4[q][r];
        tot[mb][4 * q + r] = __builtin_fmaf(sv, acc[mb][4 * q + r], tot[mb][4 * q + r]);
      }
  };
  int grp = 0, in_group = 0, meta_g0 = 0;            // of the staged groups; the first staged one
  uint32_t before = (SLOTS - 1) * SLOT, here = 0;            // slots of the tiles ahead of those being multiplied, and of those
  zeros(0);
#pragma unroll
  for (int j = 0; j < W_AHEAD; ++j) read_w(0, j);
#pragma unroll
  for (int j = 0; j < AHEAD; ++j)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) read_a(0, j, mb);
#pragma unroll
  for (int i = 0; i < 3; ++i) unpack(0, i);
  const int pairs_per_group = G128 ? 1 : p.group_size / (2 * MT_BK);
  // A step is 16 k: MB products.  Meanwhile a later step's activations and weights come from LDS and the next one's weights are unpacked, across
  // the tiles' borders too.  Before the first read of the next tiles they have to be there: they have landed once at most one slot's loads (the
  // next but one's; with four slots the one's behind the next) are outstanding.  Past the barrier every wave is through with the slot that the loads
  // issued now take: the one before, and where few rows are read far ahead the one being multiplied.  (Behind the last tile the fragments are
  // what lies in LDS: never multiplied.)
  for (int kt = 0; kt < ktiles; kt += 2) {
    const bool last = G128 || in_group + 1 == pairs_per_group;       // the group ends with this pair of tiles
    mt_unroll<8>([&](auto step) {
      constexpr int J = decltype(step)::value, H = J & 3;
      constexpr bool CROSS = FEW ? J == 5 : H == 2;
      if constexpr (CROSS) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(TWO ? 0 : UNIT * LOADS) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
      const uint32_t next = here == (SLOTS - 1) * SLOT ? 0 : here + SLOT;
      // where step J + n lies
      constexpr bool A_NEXT = FEW ? J + AHEAD >= 8 : H + AHEAD >= 4, W_NEXT = FEW ? J + W_AHEAD >= 8 : H + W_AHEAD >= 4;
      constexpr uint32_t A_SUB = FEW ? ((J + AHEAD) >> 2 & 1) * SUB : 0, W_SUB = FEW ? ((J + W_AHEAD) >> 2 & 1) * SUB : 0;
      if constexpr (J == 7) {
        if (last) {
          if (__builtin_expect(grp + 1 == GROUPS && meta_g0 + GROUPS < G, 0)) {
            // the staged groups are through (the last one's scales are in registers once every wave is here)
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            meta_g0 += GROUPS;
            grp -= GROUPS;
            stage_meta(meta_g0);
          }
          zeros(min(grp + 1, min(G - meta_g0, GROUPS) - 1));
        }
      }
      mt_unroll<MB>([&](auto block) {
        constexpr int B = decltype(block)::value;
        if constexpr (J == 0 && G128) {
          const f32x16 zero = {};
          acc[B] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[0], __builtin_bit_cast(f16x8, af[0][B]), zero, 0, 0, 0);
        } else {
          acc[B] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[J & 1], __builtin_bit_cast(f16x8, af[J & (RING - 1)][B]), acc[B], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        read_a((A_NEXT ? next : here) + A_SUB, J + AHEAD, B);
        if constexpr (B == 0) read_w((W_NEXT ? next : here) + W_SUB, J + W_AHEAD);
        if constexpr (CROSS || (FEW && J == 7)) {
          const uint32_t to = FEW ? here + (J == 7 ? SUB : 0) : before;
          if constexpr (B == MB / 2) load_a(to, 0);
          if constexpr (B == MB - 1) load_w(to);
          if constexpr (B == MB - 1 && A_LOADS > 1) load_a(to, A_LOADS - 1);
        }
        if constexpr (FEW ? (J == 6 && B == 0) || (J == 7 && B == MB - 1) : H == 3 && B == 0) advance();
        if constexpr (J == 5 && B == MB - 1) read_scales(grp);
        // (three pieces over MB slots)
        mt_unroll<3>([&](auto piece) {
          if constexpr (decltype(piece)::value * MB / 3 == B) unpack(J + 1, decltype(piece)::value);
        });
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (FEW ? J == 7 : H == 3) {
        before = here;
        here = next;
      }
    });
    if (last) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        fold(mb);
        if constexpr (!G128) {
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;
        }
      }
      in_group = 0;
      ++grp;
    } else {
      ++in_group;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int c0 = n0 + wave * 32;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int64_t row = m0 + mb * 32 + l31;
    if constexpr (!SILU) {
      float* prow = p.out + ((size_t)blockIdx.y * p.m_pad + row) * p.N + c0 + 4 * kh;
#pragma unroll
      for (int q = 0; q < 4; ++q) *reinterpret_cast<f32x4*>(prow + 8 * q) = f32x4{tot[mb][4 * q], tot[mb][4 * q + 1], tot[mb][4 * q + 2], tot[mb][4 * q + 3]};
    } else {
      // a quad's four columns are two (gate, up) pairs -> two activations = one dword; the lane that holds the quad's other half hands
      // its dword over, so that every lane stores four activations of its row twice
      uint32_t o[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint16_t h[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const float gate = tot[mb][4 * q + 2 * t], up = tot[mb][4 * q + 2 * t + 1];
          if constexpr (BF16)
            h[t] = bf16_bits_to_f16_bits_sat(silu_mul_bits<BFloat>(BFloat::to_f32(BFloat::from_f32(gate)), BFloat::to_f32(BFloat::from_f32(up))));
          else
            h[t] = silu_mul_bits<Half>(Half::to_f32(Half::from_f32(gate)), Half::to_f32(Half::from_f32(up)));
        }
        o[q] = (uint32_t)h[0] | ((uint32_t)h[1] << 16);
      }
      uint16_t* arow = p.act + row * (p.N / 2) + c0 / 2 + 4 * kh;
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(o[q], o[q + 1], false, false));
        *reinterpret_cast<u32x2*>(arow + 4 * q) = x;
      }
    }
  }
}

// G128: groups of 128 k, the K loop's own step; else (128 x 2^n) a step may continue a group.  BM: rows of a block.
template <int BM, bool SILU, bool BF16, bool G128>
__global__ __launch_bounds__(512, mt_two(BM, SILU) ? 4 : 2) void wna16_moe_tile_kernel(MoeTileParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // ---- which tile ---------------------------------------------------------------------------------------------------------------
  const int nblk = *p.num_post_pad / BM, tiles_n = p.N / MT_BN, total = nblk * tiles_n;
  if ((int)blockIdx.x >= total) return;
  int lin;
  {
    const int q = total / 8, r = total % 8, xcd = blockIdx.x % 8, k = blockIdx.x / 8;
    lin = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + k;
  }
  const int grp8 = lin / (8 * tiles_n), rem = lin - grp8 * 8 * tiles_n, nb8 = min(8, nblk - grp8 * 8);
  const int blk = grp8 * 8 + rem % nb8, n0 = rem / nb8 * MT_BN;
  const int e = __builtin_amdgcn_readfirstlane(p.expert_ids[blk]);
  if (e < 0) return;
  const int m0 = blk * BM;
  // 32-row blocks that hold a row: padding follows an expert's rows
  int mbs = BM / 32;
  if (p.row_slots != nullptr)
    while (mbs > 1 && __builtin_amdgcn_readfirstlane(p.row_slots[m0 + 32 * (mbs - 1)]) >= p.numel) --mbs;
  if constexpr (BM == 128) {
    if (mbs == 4) return moe_tile<4, mt_two(BM, SILU), SILU, BF16, G128>(p, smem, m0, n0, e);
    if (mbs == 3) return moe_tile<3, mt_two(BM, SILU), SILU, BF16, G128>(p, smem, m0, n0, e);
  }
  if (mbs == 2) moe_tile<2, mt_two(BM, SILU), SILU, BF16, G128>(p, smem, m0, n0, e);
  else moe_tile<1, mt_two(BM, SILU), SILU, BF16, G128>(p, smem, m0, n0, e);
}

__global__ void moe_rows_to_f16_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int64_t rows, int K, int64_t lda) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (i >= rows * K) return;
  u16x8 v = *reinterpret_cast<const u16x8*>(in + i / K * lda + i % K);
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = bf16_bits_to_f16_bits_sat(v[j]);
  *reinterpret_cast<u16x8*>(out + i) = v;
}

template <int BM, bool SILU, bool BF16, bool G128>
static int moe_tile_launch_t(const MoeTileParams& p, int64_t blocks, hipStream_t st) {
  const size_t lds = mt_lds(mt_two(BM, SILU), p.K / p.group_size / p.ksplit);

  APHRO_CHECK(lds <= 160 * 1024, "wna16_moe_tile: %zu bytes of LDS", lds);
  static bool attr_set_dev[APHRO_MAX_DEVICES] = {};
  bool& attr_set = attr_set_dev[device_slot()];
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)wna16_moe_tile_kernel<BM, SILU, BF16, G128>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess) {
      set_error("wna16_moe_tile: cannot raise the dynamic LDS limit");
      return APHRO_ERR_LAUNCH;
    }
    attr_set = true;
  }
  hipLaunchKernelGGL((wna16_moe_tile_kernel<BM, SILU, BF16, G128>), dim3((unsigned)(blocks * (p.N / MT_BN)), (unsigned)p.ksplit), dim3(512), lds, st, p);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}
template <int BM, bool SILU>
static int moe_tile_launch(const MoeTileParams& p, int64_t blocks, bool bf16, hipStream_t st) {
  if (p.group_size == 128) return bf16 ? moe_tile_launch_t<BM, SILU, true, true>(p, blocks, st) : moe_tile_launch_t<BM, SILU, false, true>(p, blocks, st);
  return bf16 ? moe_tile_launch_t<BM, SILU, true, false>(p, blocks, st) : moe_tile_launch_t<BM, SILU, false, false>(p, blocks, st);
}

}  // namespace aphro

using namespace aphro;

// K slices of the second GEMM for up to `blocks` row blocks, of which padding takes some four: the mean of the rounds of workgroups over the CUs
// with and without a started one counting as whole, each round 1 us per K tile and 6 us around them, and the slabs.  Mixtral-8x7B, us with one /
// two / four: 100 tokens 104 / 61 / 66, 362 183 / 116 / 123, 700 205 / 208 / 219, 1000 361 / 296 / 283, 3000 823 / 763 / 775.  A slice has 179 groups
// at most in blocks of 64 rows and 102 in blocks of 128: more have not been measured (the kernel would stage them in turn).  0: the shape is not served.
static int moe_tile_ksplit(int64_t blocks, int64_t N, int64_t K, int64_t groups, int block_m, int silu) {
  if (groups <= 0 || K % groups != 0 || N % MT_BN != 0 || (block_m != 64 && block_m != 128)) return 0;
  if (K / groups % 128 != 0 || K / 8 * N * 4 > 0xffffffffll) return 0;
  const int64_t cus = device_cu_count(), most = block_m == 64 ? 179 : 102;
  const int64_t tiles = (blocks * 4 / 5 > blocks - 4 ? blocks * 4 / 5 : blocks - 4) * (N / MT_BN);
  int best = 0;
  int64_t best_ns = 0;
  for (int ks = 1; ks <= (silu ? 1 : 256) && groups % ks == 0; ks *= 2) {
    if (groups / ks > most) continue;
    const int64_t whole = (tiles * ks + cus - 1) / cus, part = tiles * ks > cus ? tiles * ks * 100 / cus : 100;
    const int64_t ns = (whole * 100 + part) * (K / MT_BK / ks * 1000 + 6000) / 200 + (silu ? 0 : ks * blocks * block_m * N / 1000);
    if (best == 0 || ns < best_ns) { best = ks; best_ns = ns; }
    if (ks >= 4) break;
  }
  return best;
}

extern "C" int aphro_wna16_moe_tile_ksplit(int64_t blocks, int64_t N, int64_t K, int64_t groups, int block_m, int silu) {
  return moe_tile_ksplit(blocks, N, K, groups, block_m, silu);
}

static int moe_tile(const void* a, int64_t rows, int64_t lda, const int32_t* sorted_slots, const int32_t* row_slots, int64_t numel, int topk,
                    const uint32_t* q_weight, const uint32_t* qzeros, const void* scales, const int32_t* expert_ids,
                    const int32_t* num_tokens_post_pad, void* act, float* out, int64_t m_pad, int64_t N, int64_t K, int64_t groups, int ksplit,
                    int block_m, int zero_offset, int dtype, void* stream) {
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
  p.row_slots = row_slots;
  const int64_t blocks = m_pad / block_m;
  hipStream_t st = (hipStream_t)stream;
  const bool bf = dtype == APHRO_BF16;
  if (block_m == 128) return act ? moe_tile_launch<128, true>(p, blocks, bf, st) : moe_tile_launch<128, false>(p, blocks, bf, st);
  return act ? moe_tile_launch<64, true>(p, blocks, bf, st) : moe_tile_launch<64, false>(p, blocks, bf, st);
}

extern "C" int aphro_wna16_moe_tile(const void* a, int64_t rows, int64_t lda, const int32_t* sorted_slots, int64_t numel, int topk,
                                    const uint32_t* q_weight, const uint32_t* qzeros, const void* scales, const int32_t* expert_ids,
                                    const int32_t* num_tokens_post_pad, void* act, float* out, int64_t m_pad, int64_t N, int64_t K,
                                    int64_t groups, int ksplit, int block_m, int zero_offset, int dtype, void* stream) {
  return moe_tile(a, rows, lda, sorted_slots, nullptr, numel, topk, q_weight, qzeros, scales, expert_ids, num_tokens_post_pad, act, out,
                  m_pad, N, K, groups, ksplit, block_m, zero_offset, dtype, stream);
}

// The same for callers that know which rows are padding: row_slots [padded rows], numel and more behind an expert's rows.  32-row pieces of
// padding are not computed.
extern "C" int aphro_wna16_moe_tile_padded(const void* a, int64_t rows, int64_t lda, const int32_t* sorted_slots, const int32_t* row_slots,
                                           int64_t numel, int topk, const uint32_t* q_weight, const uint32_t* qzeros,
                                           const void* scales, const int32_t* expert_ids, const int32_t* num_tokens_post_pad, void* act, float* out,
                                           int64_t m_pad, int64_t N, int64_t K, int64_t groups, int ksplit, int block_m, int zero_offset, int dtype,
                                           void* stream) {
  APHRO_CHECK(row_slots && numel >= 1, "wna16_moe_tile_padded: null argument");
  return moe_tile(a, rows, lda, sorted_slots, row_slots, numel, topk, q_weight, qzeros, scales, expert_ids, num_tokens_post_pad, act, out,
                  m_pad, N, K, groups, ksplit, block_m, zero_offset, dtype, stream);
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
