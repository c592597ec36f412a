// W4A16 (GPTQ / AWQ-repacked int4) GEMM for 65 rows and more on gfx950: large decode batches and prompts up to a few thousand tokens, where
// the 256-row tiles of wna16_gemm_large.hip are half empty or too few for the chip.
//
//   * tile = 32 MB rows (MB = 3, 4, 5: the height fits the batch) x 128 columns, K tile 128, 8 waves: 2 column groups of 64 x 4 K groups
//     of 32.  D^T[n][m] = W^T[n][k] . A^T[k][m] with v_mfma_f32_32x32x16_f16, an exllama dword being a lane's weight fragment; every
//     dword is fetched and unpacked by ONE wave of the chip per row tile, for all its rows: 13 VALU against MB MFMAs of 32 cycles.
//     The four K groups meet in LDS at the end, in fixed order.
//   * weights, scales and zero points go global -> VGPR (8 bytes a lane: two adjacent columns, so that a lane ends with 8 adjacent columns
//     of its row); the activations go direct to LDS, 256-byte rows XOR-swizzled on the source address.  Four stages, three tiles ahead.
//   * int4 -> f16 in registers with the numerics of wna16_gemm_large.hip: (q - z) exact, one rounding in the multiply by the group scale.
//   * a step's MFMAs run while the next step's fragments are read and unpacked, and the loads go out BETWEEN the MFMAs: all eight
//     waves' at once, behind the barrier, made the waves wait for the address unit with the matrix cores idle (28672 x 4096, 150 rows:
//     48.9 -> 41.8 us).
//   * K slices write the accumulators as they lie in the registers, 1 KiB a store; a second kernel sums them in the order of K.
//   * what a wave issues is the other limit: with the scalar arithmetic of a tile's addresses (57 operations), its zero points' 64-bit
//     addresses and the fragment reads of a step in one place, the first four waves of a CU needed 1 205 cycles a tile alone, and the
//     other four, behind them, as many again beside their MFMAs.  Running offsets, groups by one multiplication and one MFMA, one read or
//     load and three or four operations of the unpacking a slot: 19 scalar operations of 143 in all.
// Bound by MFMAs, which pull the clock to 1.65 GHz: 1 670 cycles per K tile of 160 rows (1 900 before), 1 280 of them MFMA.
// Layer of Llama-3-8B at 150 rows, four GEMMs with their slab sums: 192 -> 114 us (qkv 40.4 -> 24, o 27.3 -> 17, gate_up 76 -> 42,
// down 48 -> 31); at 65 rows 128 -> 79; at 1300 rows 756 -> 629 us.
#include <type_traits>
#include <utility>

#include "common.h"
#include "row_norm.h"
#include "wna16_rows.h"

namespace aphro {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;

__device__ __forceinline__ uint32_t rw_and_or(uint32_t a, uint32_t mask, uint32_t orv) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(mask), "v"(orv));
  return r;
}
// f(integral_constant 0), .. f(integral_constant N - 1)
template <typename F, int... I>
__device__ __forceinline__ void rw_unroll_(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void rw_unroll(F&& f) { rw_unroll_(f, std::make_integer_sequence<int, N>{}); }

constexpr int RW_BN = 128, RW_BK = 128, RW_STAGES = 4;
constexpr int rw_pass(int mb) { return (mb + 1) / 2; }      // 32-row blocks whose K groups meet in LDS at a time
constexpr int RW_EXACT_GROUPS = 64;                         // of a K slice, whose scales EXACT keeps in LDS behind the stages
constexpr size_t rw_lds(int mb, bool exact = false) {
  if (exact) return (size_t)RW_STAGES * mb * 32 * RW_BK * 2 + RW_EXACT_GROUPS * RW_BN * 2;
  const size_t stages = (size_t)RW_STAGES * mb * 32 * RW_BK * 2, meet = (size_t)8 * 3 * rw_pass(mb) * 2048;
  return stages > meet ? stages : meet;
}

// Slabs of K slices are images of the accumulators: [ksplit][tile][32-row block][16-column group] of 2 KiB, a lane's two quads 1 KiB apart.
__device__ __forceinline__ size_t rw_image(const Wna16RowsParams& p, int MB, int ks, int tile, int mb, int group) {
  return (((size_t)ks * (p.tiles_m * p.tiles_n) + tile) * MB + mb) * 4096 + (size_t)group * 512;
}

// EXACT: the numerics of the decode kernels -- the integers q - z enter the products, and a K tile's fp32 sum is added times its group's
// fp32 scale, one FMA an accumulator element (with the f16 scale as it is: v_fma_mix_f32).  An accumulator's columns are other lanes'
// weights, so the scales come from LDS, 16 bytes a quad.  Twice the accumulators, so two 32-row blocks at most.  float16, 65 / 128 rows, 4096 x 4096:
// 15.0 / 17.3 us, error against 64 bits 2.08e-4, a float16 result's own rounding; the form that rounds weights 15.5 / 23 us, 2.87e-4; the
// decode kernel, two passes of 64 rows, 17.3 / 22.0 us.
template <int MB, bool BF16, bool STRIP, bool EXACT>
__global__ __launch_bounds__(512) void wna16_gemm_rows_kernel(Wna16RowsParams p) {
  static_assert(!EXACT || (MB <= 2 && !BF16), "registers; bf16 stays with the decode kernels");
  constexpr int STAGE = MB * 32 * RW_BK * 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 1, kg = wave >> 1;
  const int kh = lane >> 5, l31 = lane & 31;
  // ---- which tile: contiguous ranges per XCD, the column tiles of one K slice and row tile next to each other -------------------
  int lin;
  {
    const int n = gridDim.x, q = n / 8, r = n % 8, xcd = blockIdx.x % 8, k = blockIdx.x / 8;
    lin = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + k;
  }
  const int tn = lin % p.tiles_n, rest = lin / p.tiles_n, tm = rest % p.tiles_m, ks = rest / p.tiles_m;
  const int m0 = tm * MB * 32, n0 = tn * RW_BN;
  const int T = p.K / RW_BK, t0 = ks * T / p.ksplit, t1 = (ks + 1) * T / p.ksplit;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a) + (size_t)m0 * p.lda, 0,
                                                                (uint32_t)((size_t)(p.M - m0) * p.lda * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.qw), 0, (uint32_t)((size_t)(p.K >> 3) * p.N * 4), 0x00020000);
  // ---- activations: one DMA instruction = 4 rows of 256 B, rows 32 apart from one to the next; LDS slot s of row r holds the row's
  // slot s ^ (r & 15).  Rows from M on read zeros (the buffer ends there); 32-row blocks that begin behind M read the last one that does
  // not, because a scalar offset past the buffer's end is not certain to fail the range check.  Nobody stores either. ------------------
  const int row0 = wave * 4 + (lane >> 4), last_block = (p.M - m0 - 1) >> 5;
  const int a_voff = (int)((uint32_t)row0 * (uint32_t)p.lda * 2u + (((lane & 15) ^ (row0 & 15)) << 4));
  // ---- weights: the lane's columns are col and col + 1 (MFMA row i of block nb is column 2 i + nb) -------------------------------
  const int col = n0 + wn * 64 + 2 * l31;
  uint32_t w_voff, mult = 0;
  if constexpr (STRIP) w_voff = wna16_strip_col(p.strip, col & ~3, mult) + (uint32_t)(col & 3) + mult * (64u * (uint32_t)kh + 16u * (uint32_t)kg);
  else w_voff = (uint32_t)((kg * 4 + kh) * p.N + col);
  w_voff *= 4u;
  const uint32_t mult4 = mult * 4u;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.sc), 0, (uint32_t)(p.K / p.group_size * p.N * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.qz), 0, (uint32_t)(p.K / p.group_size * (p.N >> 3) * 4), 0x00020000);
  const int sc_voff = col * 2, z_voff = (col >> 3) * 4;
  const int zshift = (col & 7) * 4;
  const int first_k = t0 * RW_BK + kg * 32, first_grp = first_k / p.group_size, first_in = first_k - first_grp * p.group_size;
  // Where the next load fetches, scalar: k of the wave's part (its group by a multiplication), the tiles until a chunk of the strip-major copy or
  // the slice ends.
  const uint32_t sc_row = (uint32_t)p.N * 2u;
  uint32_t k_load = (uint32_t)(t0 * RW_BK + kg * 32), sc_off, z_off;
  uint32_t w_off, w_vrun = w_voff, a_run = (uint32_t)a_voff + (uint32_t)t0 * (RW_BK * 2);
  int t_load = t0, event;
  auto place = [&] {
    if constexpr (STRIP) {
      uint32_t chunk, R;
      wna16_strip_row(p.strip, (uint32_t)t_load * 16u, chunk, R);
      w_off = chunk * 4u;
      w_vrun = w_voff + __umul24(mult4, R);
      event = min(p.strip.nseg - (int)(R >> 8), t1 - t_load);
    } else {
      w_off = (uint32_t)t_load * 64u * (uint32_t)p.N;
      event = t1 - t_load;
    }
  };
  auto groups = [&] {
    const uint32_t g = (uint32_t)(((uint64_t)k_load * p.inv_group) >> 32);
    sc_off = g * sc_row;
    z_off = sc_off >> 2;
  };
  place();
  groups();
  u32x2 wr[3][2];
  uint32_t scr[3], zr[3];
  auto load_meta = [&](auto set) {
    constexpr int S = decltype(set)::value;
    if constexpr (!EXACT) scr[S] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, sc_voff, (int)sc_off, 0);
    zr[S] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rz, z_voff, (int)z_off, 0);
  };
  auto load_w = [&](auto set, int j) {
    constexpr int S = decltype(set)::value;
    if constexpr (STRIP)
      wr[S][j] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rb, (int)(j ? w_vrun + mult4 * 128u : w_vrun), (int)w_off, 0));
    else
      wr[S][j] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rb, (int)w_voff, (int)w_off + 2 * j * p.N * 4, 0));
  };
  auto load_a = [&](uint32_t st, int i) {
    const int voff = (int)a_run;                           // (a local copy: see wna16_gemm_large.hip)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_ptr)(smem + st + (i * 8 + wave) * 1024), 16, voff,
                                             (int)((uint32_t)min(i, last_block) * 64u * (uint32_t)p.lda), 0, 0);
  };
  auto advance_groups = [&] { k_load += RW_BK; groups(); };
  auto advance_tile = [&] {
    ++t_load;
    a_run += RW_BK * 2;
    if constexpr (STRIP) w_vrun += mult4 * 256u;
    else w_off += 64u * (uint32_t)p.N;
    if (__builtin_expect(--event == 0, 0)) {
      if (t_load == t1) {                                    // the slice's end: the last tile again, which nobody reads
        --t_load;
        k_load -= RW_BK;
        a_run -= RW_BK * 2;
        if constexpr (STRIP) w_vrun -= mult4 * 256u;
        else w_off -= 64u * (uint32_t)p.N;
        groups();
        event = 1;
      } else {
        place();
      }
    }
  };
  // EXACT: one tile on, behind the slice's end not, without a branch (one among the sums costs registers, here more than there are)
  auto stay = [&] {
    t_load = min(t_load + 1, t1 - 1);
    k_load = (uint32_t)(t_load * RW_BK + kg * 32);
    a_run = (uint32_t)a_voff + (uint32_t)t_load * (RW_BK * 2);
    place();
    groups();
  };
  auto load = [&](auto set, uint32_t st) {
    load_w(set, 0);
    load_w(set, 1);
    load_meta(set);
#pragma unroll
    for (int i = 0; i < MB; ++i) load_a(st, i);
  };
  constexpr int LOADS = MB + (EXACT ? 3 : 4);              // memory instructions of one load()
  f32x16 acc[2][MB], total[EXACT ? 2 : 1][EXACT ? MB : 1];
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[nb][mb][r] = 0.f;
        if constexpr (EXACT) total[nb][mb][r] = 0.f;
      }
  // EXACT: scales of the slice's groups, [group][128 columns]; the accumulators' columns 16 q + 8 kh + 2 r + nb are 16 bytes for a quad
  constexpr int SC_LOADS = RW_EXACT_GROUPS * (RW_BN / 2) / 512;
  unsigned char* sc_lds = smem + RW_STAGES * STAGE;
  const int slice_grp = t0 * RW_BK / p.group_size;
  uint32_t sc_reg[SC_LOADS];
  if constexpr (EXACT) {
    const int dwords = ((t1 * RW_BK - 1) / p.group_size + 1 - slice_grp) * (RW_BN / 2);
    const uint32_t* src = reinterpret_cast<const uint32_t*>(p.sc + (size_t)slice_grp * p.N + n0);
#pragma unroll
    for (int i = 0; i < SC_LOADS; ++i) {
      const int x = threadIdx.x + 512 * i;
      sc_reg[i] = x < dwords ? src[(size_t)(x >> 6) * (p.N >> 1) + (x & 63)] : 0u;
    }
    asm volatile("" ::: "memory");                         // (ahead of the loads that are counted)
  }
  const int grp_step = RW_BK / p.group_size, grp_rest = RW_BK - grp_step * p.group_size;
  int tile_grp = first_grp, tile_in = first_in;             // of the tile being multiplied
  auto fold = [&] {
    const unsigned char* row = sc_lds + (tile_grp - slice_grp) * (RW_BN * 2) + wn * 128 + kh * 16;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f16x8 s8 = *reinterpret_cast<const f16x8*>(row + q * 32);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            total[EXACT ? nb : 0][EXACT ? mb : 0][4 * q + r] =
                __builtin_fmaf(acc[nb][mb][4 * q + r], (float)s8[2 * r + nb], total[EXACT ? nb : 0][EXACT ? mb : 0][4 * q + r]);
    }
    tile_grp += grp_step;
    tile_in += grp_rest;
    if (tile_in >= p.group_size) { tile_in -= p.group_size; ++tile_grp; }
  };
  // ---- K loop.  While a step's (16 k) MFMAs run, the next step's activations come from LDS and its weights are unpacked, across the
  // tiles' borders too: halfway through a tile the next one has to be there -----------------------------------------------------------
  u32x4 af[2][MB];
  f16x8 wf[2][2];
  f16x2 zh[2], zh16[2], sv[2];
  const uint32_t a_base = (uint32_t)l31 * 256u;
  const uint32_t a_read[2] = {a_base + (((uint32_t)(kg * 4 + kh) ^ (uint32_t)(l31 & 15)) << 4),
                              a_base + (((uint32_t)(kg * 4 + 2 + kh) ^ (uint32_t)(l31 & 15)) << 4)};
  auto read_a = [&](uint32_t st, int j, int mb) { af[j][mb] = *reinterpret_cast<const u32x4*>(smem + st + a_read[j] + mb * 8192); };
  auto meta = [&](auto set, int nb) {
    constexpr int S = decltype(set)::value;
    uint16_t sb = 0;
    if constexpr (!EXACT) sb = (uint16_t)(nb ? scr[S] >> 16 : scr[S]);
    const int z = (int)((zr[S] >> (zshift + 4 * nb)) & 0xf) + p.zero_offset;
    const f16 s16 = BF16 ? (f16)bf16_bits_to_f32(sb) : __builtin_bit_cast(f16, sb);
    const f16 a16 = __builtin_bit_cast(f16, (uint16_t)(0x6400 | z));       // 1024 + z
    const f16 b16 = (f16)960.f - a16;                                      // -64 - z
    sv[nb] = f16x2{s16, s16};
    zh[nb] = f16x2{a16, a16};
    zh16[nb] = f16x2{b16, b16};
  };
  f16x2 diff[2][4];
  uint32_t high[2], biased[2][4];
  // the weights of a step, an exllama dword a column: (1024 + q) - (1024 + z), exact, and times the scale (one rounding; EXACT: not here), in
  // pieces of 3 or 4 operations
  auto unpack_piece = [&](auto set, auto step, auto piece) {
    constexpr int S = decltype(set)::value, J = decltype(step)::value, P = decltype(piece)::value, nb = P >> 2, q = P & 3;
    const f16x2 inv16 = {(f16)0.0625f, (f16)0.0625f};
    const uint32_t magic = 0x64006400u;
    const uint32_t w = wr[S][J][nb];
    if constexpr (q == 0) {
      biased[nb][0] = rw_and_or(w, 0x000f000fu, magic);
      biased[nb][1] = rw_and_or(w, 0x00f000f0u, magic);
      high[nb] = w >> 8;
    } else if constexpr (q == 1) {
      biased[nb][2] = rw_and_or(high[nb], 0x000f000fu, magic);
      biased[nb][3] = rw_and_or(high[nb], 0x00f000f0u, magic);
      diff[nb][0] = __builtin_bit_cast(f16x2, biased[nb][0]) - zh[nb];
    } else if constexpr (q == 2) {
      diff[nb][1] = __builtin_bit_cast(f16x2, biased[nb][1]) * inv16 + zh16[nb];
      diff[nb][2] = __builtin_bit_cast(f16x2, biased[nb][2]) - zh[nb];
      diff[nb][3] = __builtin_bit_cast(f16x2, biased[nb][3]) * inv16 + zh16[nb];
    } else {
      f16x2 d[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = EXACT ? diff[nb][i] : diff[nb][i] * sv[nb];
      wf[J][nb] = __builtin_bit_cast(f16x8, u32x4{__builtin_bit_cast(uint32_t, d[0]), __builtin_bit_cast(uint32_t, d[1]),
                                                  __builtin_bit_cast(uint32_t, d[2]), __builtin_bit_cast(uint32_t, d[3])});
    }
  };
  auto unpack = [&](auto set, auto step) {
    rw_unroll<8>([&](auto piece) { unpack_piece(set, step, piece); });
  };
  auto multiply = [&](auto step, int i) {
    constexpr int J = decltype(step)::value;
    const f32x16 zero = {};
    const int mb = i >> 1, nb = i & 1;
    acc[nb][mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[J][nb], __builtin_bit_cast(f16x8, af[J][mb]), EXACT && J == 0 ? zero : acc[nb][mb], 0, 0, 0);
  };
  uint32_t before = 3 * STAGE, here = 0;                   // stages of the tile ahead of the one being multiplied, and of that one
  auto tile = [&](auto set, auto more) {
    constexpr int S = decltype(set)::value, SLOTS = 2 * MB;
    constexpr bool MORE = decltype(more)::value;
    constexpr std::integral_constant<int, 0> step0{};
    constexpr std::integral_constant<int, 1> step1{};
    constexpr std::integral_constant<int, (S + 1) % 3> next{};
    if constexpr (MORE && EXACT) stay();
    // A slot: one MFMA and what fits its 64 cycles (two waves share a matrix pipe).  First 16 k: the others' fragments are read, their
    // weights unpacked; scalars one tile on.
    rw_unroll<SLOTS>([&](auto slot) {
      constexpr int I = decltype(slot)::value, P0 = I * 8 / SLOTS, P1 = (I + 1) * 8 / SLOTS;
      multiply(step0, I);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (I < MB) read_a(here, 1, I);
      if constexpr (MORE && !EXACT && I == 1) advance_groups();
      if constexpr (MORE && !EXACT && I == 3) advance_tile();
      rw_unroll<P1 - P0>([&](auto i) { unpack_piece(set, step1, std::integral_constant<int, P0 + decltype(i)::value>{}); });
      __builtin_amdgcn_sched_barrier(0);
    });
    // the next tile has landed once at most the loads of the one behind it are outstanding; past the barrier every wave is through with the
    // tile BEFORE this one, whose stage the loads issued now take
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(LOADS) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const uint32_t fetch = before;
    before = here;
    here = here == 3 * STAGE ? 0 : here + STAGE;
    __builtin_amdgcn_sched_barrier(0);
    // the loads go out between the MFMAs: all waves' at once would wait for one another with the matrix cores idle
    rw_unroll<SLOTS>([&](auto slot) {
      constexpr int I = decltype(slot)::value, P0 = I < 1 ? 0 : (I - 1) * 8 / (SLOTS - 1), P1 = I * 8 / (SLOTS - 1);
      multiply(step1, I);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (I < MB) read_a(here, 0, I);
      if constexpr (MORE && I < 2) load_w(set, I);
      if constexpr (MORE && I == 2) load_meta(set);
      if constexpr (I == 1) meta(next, 0);
      if constexpr (I == SLOTS / 2) meta(next, 1);
      if constexpr (MORE && I >= SLOTS - MB) load_a(fetch, I - (SLOTS - MB));
      rw_unroll<P1 - P0>([&](auto i) { unpack_piece(next, step0, std::integral_constant<int, P0 + decltype(i)::value>{}); });
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (EXACT) {
      fold();
      __builtin_amdgcn_sched_barrier(0);                   // (the next tile's sums would be a second set of accumulators)
    }
  };
  constexpr std::integral_constant<int, 0> set0{};
  constexpr std::integral_constant<int, 1> set1{};
  constexpr std::integral_constant<int, 2> set2{};
  auto advance = [&] {
    if constexpr (EXACT) {
      stay();
    } else {
      advance_groups();
      advance_tile();
    }
  };
  load(set0, 0);
  asm volatile("" ::: "memory");                           // (the counted waits rely on the order of the loads)
  advance();
  load(set1, STAGE);
  asm volatile("" ::: "memory");
  advance();
  load(set2, 2 * STAGE);
  if constexpr (EXACT) {
#pragma unroll
    for (int i = 0; i < SC_LOADS; ++i) reinterpret_cast<uint32_t*>(sc_lds)[threadIdx.x + 512 * i] = sc_reg[i];
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(2 * LOADS) : "memory");
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) read_a(0, 0, mb);
  meta(set0, 0);
  meta(set0, 1);
  unpack(set0, std::integral_constant<int, 0>{});
  int left = t1 - t0;
  for (; left >= 3; left -= 3) {
    tile(set0, std::true_type{});
    tile(set1, std::true_type{});
    tile(set2, std::true_type{});
  }
  // the last one or two tiles, whose loads the loop has issued
  if (left > 0) tile(set0, std::false_type{});
  if (left > 1) tile(set1, std::false_type{});
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  // ---- the four K groups meet in LDS: the wave of group g ends with quad g of every block, columns 16 g + 8 kh + 2 r + nb ----------
  constexpr int RM = rw_pass(MB);
  auto& sum = [&]() -> f32x16 (&)[2][MB] {
    if constexpr (EXACT) return total;
    else return acc;
  }();
#pragma unroll
  for (int m1 = 0; m1 < MB; m1 += RM) {
    __syncthreads();
    f32x4 own[2][RM];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q != kg) {
        unsigned char* dst = smem + (size_t)(((q * 2 + wn) * 3 + (kg ^ q) - 1) * RM) * 2048 + lane * 16;
#pragma unroll
        for (int i = 0; i < RM; ++i)
          if (m1 + i < MB)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
              const f32x16& x = sum[nb][m1 + i < MB ? m1 + i : 0];
              *reinterpret_cast<f32x4*>(dst + (i * 2 + nb) * 1024) = f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
            }
      } else {
#pragma unroll
        for (int i = 0; i < RM; ++i)
          if (m1 + i < MB)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
              const f32x16& x = sum[nb][m1 + i < MB ? m1 + i : 0];
              own[nb][i] = f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
            }
      }
    }
    __syncthreads();
    const unsigned char* src = smem + (size_t)((kg * 2 + wn) * 3 * RM) * 2048 + lane * 16;
    // (v0 + v1) + (v2 + v3) whichever group the wave is: a column's bits do not depend on its place
#pragma unroll
    for (int i = 0; i < RM; ++i)
      if (m1 + i < MB)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          f32x4 v[3];
#pragma unroll
          for (int s = 0; s < 3; ++s) v[s] = *reinterpret_cast<const f32x4*>(src + (size_t)((s * RM + i) * 2 + nb) * 1024);
#pragma unroll
          for (int r = 0; r < 4; ++r) own[nb][i][r] = (own[nb][i][r] + v[0][r]) + (v[1][r] + v[2][r]);
        }
#pragma unroll
    for (int i = 0; i < RM; ++i) {
      if (m1 + i >= MB) continue;
      const int row = m0 + (m1 + i) * 32 + l31;
      if (row >= p.M) continue;
      const int c0 = n0 + wn * 64 + 16 * kg + 8 * kh;
      const f32x4 x = own[0][i], y = own[1][i];
      if (p.ksplit > 1 && p.row_slabs) {                     // rows of N, which a norm or a rotation reads whole
        float* o = p.partial + ((size_t)ks * p.tiles_m * (MB * 32) + row) * p.N + c0;
        *reinterpret_cast<f32x4*>(o) = f32x4{x[0], y[0], x[1], y[1]};
        *reinterpret_cast<f32x4*>(o + 4) = f32x4{x[2], y[2], x[3], y[3]};
      } else if (p.ksplit > 1) {
        float* o = p.partial + rw_image(p, MB, ks, tm * p.tiles_n + tn, m1 + i, wn * 4 + kg) + lane * 4;
        *reinterpret_cast<f32x4*>(o) = x;
        *reinterpret_cast<f32x4*>(o + 256) = y;
      } else if (p.silu) {
        using T16 = std::conditional_t<BF16, BFloat, Half>;
        u16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = silu_mul_bits<T16>(T16::to_f32(T16::from_f32(x[r])), T16::to_f32(T16::from_f32(y[r])));
        *reinterpret_cast<u16x4*>(p.c + (size_t)row * (p.N / 2) + c0 / 2) = o;
      } else {
        const u32x4 o = {pack2_16<BF16>(x[0], y[0]), pack2_16<BF16>(x[1], y[1]), pack2_16<BF16>(x[2], y[2]), pack2_16<BF16>(x[3], y[3])};
        *reinterpret_cast<u32x4*>(p.c + (size_t)row * p.N + c0) = o;
      }
    }
  }
}

// The slabs summed in the order of K, one wave per image, and rounded (SiluAndMul behind it as in the kernel itself).
template <bool BF16>
__global__ __launch_bounds__(256) void wna16_rows_reduce_kernel(Wna16RowsParams p, int MB) {
  const int lane = threadIdx.x & 63, kh = lane >> 5, l31 = lane & 31;
  const int img = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int group = img & 7, rest = img >> 3, mb = rest % MB, tile = rest / MB;
  const int row = (tile / p.tiles_n * MB + mb) * 32 + l31;
  if (row >= p.M) return;
  const float* src = p.partial + rw_image(p, MB, 0, tile, mb, group) + lane * 4;
  const size_t slab = (size_t)p.tiles_m * p.tiles_n * MB * 4096;
  f32x4 x = *reinterpret_cast<const f32x4*>(src), y = *reinterpret_cast<const f32x4*>(src + 256);
#pragma unroll 4
  for (int s = 1; s < p.ksplit; ++s) {
    x += *reinterpret_cast<const f32x4*>(src + s * slab);
    y += *reinterpret_cast<const f32x4*>(src + s * slab + 256);
  }
  const int c0 = tile % p.tiles_n * RW_BN + group * 16 + kh * 8;
  if (p.silu) {
    using T16 = std::conditional_t<BF16, BFloat, Half>;
    u16x4 a;
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = silu_mul_bits<T16>(T16::to_f32(T16::from_f32(x[r])), T16::to_f32(T16::from_f32(y[r])));
    *reinterpret_cast<u16x4*>(p.c + (size_t)row * (p.N / 2) + c0 / 2) = a;
    return;
  }
  const u32x4 o = {pack2_16<BF16>(x[0], y[0]), pack2_16<BF16>(x[1], y[1]), pack2_16<BF16>(x[2], y[2]), pack2_16<BF16>(x[3], y[3])};
  *reinterpret_cast<u32x4*>(p.c + (size_t)row * p.N + c0) = o;
}

// The slabs summed as above and rounded, added to the residual, rounded, and normed: a workgroup a row, the bits of wna16_rows_reduce_kernel
// and fused_add_rms_norm (rms_norm_kernel) in one launch instead of two of 5 us.  Bound by the latency of its loads and the sum over the row.
// int4 steps, us before / after: 150 rows, 16 layers 4230 / 4180, 90 rows, 8 layers 1395 / 1363, prompt of 250, 4 layers 962 / 946, of 900 2257 / 2252.
template <typename T>
__global__ void wna16_rows_norm_kernel(Wna16RowsParams p, int pad_rows) {
  __shared__ float red[16];
  const size_t row = blockIdx.x;
  const int nv = p.N >> 3;
  const size_t slab = (size_t)pad_rows * p.N;
  float v[2][8], ss = 0.f;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int i = threadIdx.x + it * blockDim.x;
    if (i < nv) {
      const float* src = p.partial + row * p.N + 8 * i;
      uint16_t* rp = p.residual + row * p.N + 8 * i;
      const u16x8 b = *reinterpret_cast<const u16x8*>(rp);
      f32x4 x = *reinterpret_cast<const f32x4*>(src), y = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll 4
      for (int s = 1; s < p.ksplit; ++s) {
        x += *reinterpret_cast<const f32x4*>(src + s * slab);
        y += *reinterpret_cast<const f32x4*>(src + s * slab + 4);
      }
      u16x8 r;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        r[j] = T::from_f32(T::to_f32(T::from_f32(j < 4 ? x[j] : y[j - 4])) + T::to_f32(b[j]));
        v[it][j] = T::to_f32(r[j]);
      }
      *reinterpret_cast<u16x8*>(rp) = r;
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += v[it][j] * v[it][j];
    }
  }
  ss = block_sum(ss, red);
  const float inv = __frsqrt_rn(ss / (float)p.N + p.norm_eps);
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int i = threadIdx.x + it * blockDim.x;
    if (i < nv) {
      const u16x8 w = *reinterpret_cast<const u16x8*>(p.norm_weight + 8 * i);
      u16x8 r;
#pragma unroll
      for (int j = 0; j < 8; ++j) r[j] = T::from_f32(T::to_f32(T::from_f32(v[it][j] * inv)) * T::to_f32(w[j]));
      *reinterpret_cast<u16x8*>(p.c + row * p.N + 8 * i) = r;
    }
  }
}

static uint32_t rw_inv_group(int64_t gs) { return (uint32_t)((0x100000000ll + gs - 1) / gs); }
// whether k * inv_group >> 32 is k / group_size for all k < K: but for odd groups of a K of 65536 and more it always is
static bool rw_groups_exact(int64_t K, int64_t gs) { return (rw_inv_group(gs) * gs - 0x100000000ll) * K < 0x100000000ll; }

// Tile height and K slices by the time they are expected to take (MI355X, ns; within 10 % of what was measured for 65 .. 4096 rows of
// Llama-3-8B's and -70B's matrices): rounds of workgroups over the CUs, each 170 + 200 per 32-row block and K tile and 4.7 us around
// them, a last one that is not full 0.74 of that and 0.26 by how full it is (few workgroups run at a higher clock and have the memory to
// themselves; 0.7 and 0.3 fit better by 0.1 %, but take fewer than four slices at 150 rows of 4096 x 4096 with one group per column, whose
// workspace is promised), and the slabs written and read again at 2.2 TB/s behind 3 us.  Of the forms measured for 150 to 4096 rows of 28672 x 4096, 6144 x
// 4096, 4096 x 4096 and 4096 x 14336 the one taken is 0.2 % behind the best on average (a last round counted whole: 2.2 %).  us: 6144 x 4096,
// 150 rows: five blocks and four slices 24.3, three and two 21.1; 900 rows, five blocks in 1.1 rounds 69.8, three in 1.9 59.6; 4096 x 14336, 150
// rows: one slice 82, two 49, four 32; 4096 x 4096, 150 rows: five blocks and four slices 20.6, three and three 18.2.
Wna16RowsPlan wna16_rows_plan(int64_t M, int64_t N, int64_t K, int64_t gs, int64_t slab_bytes, int64_t other_ns) {
  Wna16RowsPlan best = {0, 1, false};
  if (M <= 64 || M > 4096 || N % RW_BN || K % RW_BK || gs % 64 || !rw_groups_exact(K, gs)) return best;
  const int cus = device_cu_count();
  const int64_t T = K / RW_BK;
  int64_t best_ns = other_ns;
  for (int mb = 3; mb <= 5; ++mb) {
    const int64_t tiles_m = (M + mb * 32 - 1) / (mb * 32), tiles = tiles_m * (N / RW_BN);
    for (int ks = 1; ks <= 16 && (ks == 1 || T / ks >= 4); ++ks) {
      const int64_t slabs = tiles_m * mb * 32 * N * 4 * ks;
      if (ks > 1 && slabs > slab_bytes) break;
      const int64_t full = tiles * ks / cus, rest = tiles * ks % cus, round = (T + ks - 1) / ks * (170 + 200 * mb) + 4700;
      const int64_t ns = full * round + (rest ? round * (74 * cus + 26 * rest) / (100 * cus) : 0) + (ks > 1 ? 3000 + slabs * 45 / 100000 : 0);
      if (best_ns < 0 || ns < best_ns) { best = {mb, ks, false}; best_ns = ns; }
    }
  }
  return best;
}

// The EXACT form, 65 to 128 rows: two tiles of 64.  K slices by the time they are expected to take, as above; a slice's groups fit its LDS.
Wna16RowsPlan wna16_rows_plan_exact(int64_t M, int64_t N, int64_t K, int64_t gs, int64_t slab_bytes) {
  Wna16RowsPlan best = {0, 1, true};
  if (M <= 64 || M > 128 || N % RW_BN || K % RW_BK || gs % 64 || !rw_groups_exact(K, gs)) return best;
  const int cus = device_cu_count();
  const int64_t T = K / RW_BK, tiles = 2 * (N / RW_BN);
  int64_t best_ns = -1;
  for (int ks = 1; ks <= 16 && (ks == 1 || T / ks >= 4); ++ks) {
    const int64_t slabs = 128 * N * 4 * ks;
    if (ks > 1 && slabs > slab_bytes) break;
    bool fits = true;
    for (int i = 0; i < ks; ++i) fits = fits && ((i + 1) * T / ks * RW_BK - 1) / gs - i * T / ks * RW_BK / gs < RW_EXACT_GROUPS;
    if (!fits) continue;
    const int64_t ns = (tiles * ks + cus - 1) / cus * ((T + ks - 1) / ks * 700 + 4700) + (ks > 1 ? 3000 + slabs * 45 / 100000 : 0);
    if (best_ns < 0 || ns < best_ns) { best = {2, ks, true}; best_ns = ns; }
  }
  return best;
}

template <int MB, bool BF16, bool STRIP, bool EXACT>
static int rows_launch(Wna16RowsParams p, hipStream_t st) {
  p.tiles_m = (p.M + MB * 32 - 1) / (MB * 32);
  p.tiles_n = p.N / RW_BN;
  p.inv_group = rw_inv_group(p.group_size);
  static bool attr_set_dev[APHRO_MAX_DEVICES] = {}; bool& attr_set = attr_set_dev[device_slot()];
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)wna16_gemm_rows_kernel<MB, BF16, STRIP, EXACT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            160 * 1024) != hipSuccess) {
      set_error("wna16_gemm_rows: cannot raise the dynamic LDS limit");
      return APHRO_ERR_LAUNCH;
    }
    attr_set = true;
  }
  hipLaunchKernelGGL((wna16_gemm_rows_kernel<MB, BF16, STRIP, EXACT>), dim3(p.tiles_m * p.tiles_n * p.ksplit), dim3(512), rw_lds(MB, EXACT), st, p);
  APHRO_LAUNCH_CHECK();
  if (p.ksplit > 1 && p.norm_weight) {
    using T16 = std::conditional_t<BF16, BFloat, Half>;
    hipLaunchKernelGGL(wna16_rows_norm_kernel<T16>, dim3(p.M), dim3(norm_threads(p.N)), 0, st, p, p.tiles_m * MB * 32);
    APHRO_LAUNCH_CHECK();
  } else if (p.ksplit > 1 && !p.row_slabs) {
    hipLaunchKernelGGL(wna16_rows_reduce_kernel<BF16>, dim3(p.tiles_m * p.tiles_n * MB * 2), dim3(256), 0, st, p, MB);
    APHRO_LAUNCH_CHECK();
  }
  return APHRO_OK;
}

template <int MB>
static int rows_launch_mb(const Wna16RowsParams& p, hipStream_t st) {
  if (p.bf16) return p.strip.on ? rows_launch<MB, true, true, false>(p, st) : rows_launch<MB, true, false, false>(p, st);
  return p.strip.on ? rows_launch<MB, false, true, false>(p, st) : rows_launch<MB, false, false, false>(p, st);
}

size_t wna16_rows_slab_bytes(const Wna16RowsPlan& plan, int64_t M, int64_t N) {
  const int64_t bm = plan.mb * 32;
  return plan.mb > 0 && plan.ksplit > 1 ? (size_t)((M + bm - 1) / bm * bm * N * 4 * plan.ksplit) : 0;
}

int wna16_rows_launch(const Wna16RowsParams& p, const Wna16RowsPlan& plan, hipStream_t st) {
  if (plan.exact) return p.strip.on ? rows_launch<2, false, true, true>(p, st) : rows_launch<2, false, false, true>(p, st);
  if (plan.mb == 3) return rows_launch_mb<3>(p, st);
  if (plan.mb == 4) return rows_launch_mb<4>(p, st);
  return rows_launch_mb<5>(p, st);
}

}  // namespace aphro
