// Prompt attention over rows of 128: a workgroup owns 128 / QT consecutive query rows of QT heads of one kv head (QT = 4, 2, 1: as many as divide its
// heads), a wave 32 rows of one head, so that a K or V tile fetched once serves 128 rows and a 300-token prompt still has a workgroup for a third of the CUs.
//   * S^T = K Q^T and O^T = V^T P^T on 32x32x16 products: a lane holds 32 of the 64 scores of one row, its probabilities are the second product's
//     operand where they lie.
//   * K and V tiles of 64 keys go from memory to LDS without a stop in registers, two buffers, one barrier a tile; LDS slot s of key j holds K's
//     16-byte piece s ^ (j & 15), V's s ^ 4 (j & 3): fragment reads and transposing reads find their banks free.  Keys past the sequence's end are
//     fetched as zeros (the buffer ends there) and masked.
//   * the scale is the exponential's FMA; LONG (from 4096 keys on): one step of the online softmax a tile, and the maximum moves only for rows that are
//     past it by more than 2^8, else a step is 32 keys and its largest probability 1 up to the rounding of the scaled maximum, which the FMA's product
//     does not share; a row's sum and its values take the same probability, before it is 16 bits (error against 64 bits, of the result's size, bf16: steps
//     of 32 keys 0.00206 at 3000 keys and 0.00209 at 8192, LONG 0.00212 and 0.00215, the kernel that it replaced there 0.00215).
//   * GROUPS = 2: two such groups of waves take the key tiles in turn, each in LDS of its own, and their sums meet at the end: half the chain.
// Bound by a tile's chain of steps where a workgroup is alone on its CU (1.2 us: 32 products, the softmax), else by issue and power: at 8192 tokens the
// matrix pipe is busy 60 % of the SIMDs' cycles, the vector ALUs 53 %, LDS 30 %, at 1.7 GHz.  us before / here, 32 heads on 8, causal, bf16, the two in turn
// on one card (others take 507 to 532 for 8192 tokens, 536 in f16, 491 for numbers a third as large: power): against
// 64-row workgroups with V transposed number by number, 300 tokens 18.8 / 12.0; against 128-row ones, 1000 tokens 45.5 / 23.6; against one wave
// a SIMD with 64 rows of the whole register file (deleted), 4096 tokens 174 / 159, 8192 601 / 558, 5000 261 / 210, two of 4096 324 / 276, 8 heads on one
// 250 / 161.  Below 64 keys the first kernel of flash_attn.hip is the faster (six of 26 tokens 6.1 / 7.4).
// No gain: loads hidden from hipcc, which otherwise waits for the next tile in front of the transposing reads (three of 1000 tokens 53 / 55); loads between
// the products (8192 tokens, on a faster card, 531 / 534); the next tile's scores between this one's exponentials (530 / 531); row sums as a product with ones (531 / 550).
#include "common.h"
#include "flash_attn_common.h"

#include <type_traits>

namespace aphro {

typedef short fas_s16x4 __attribute__((ext_vector_type(4)));

constexpr float FAS_LAZY = 8.f;                               // log2 of what a row may be past its maximum before it moves (LONG)
constexpr int FAS_BN = 64, FAS_TILE = FAS_BN * 256;          // keys of a tile, bytes of its K (or V) rows

template <typename T, int QT, bool LONG, int GROUPS>
__global__ __launch_bounds__(256 * GROUPS, 2) void flash_attn_short_kernel(FAParams p) {
  constexpr bool BF = __is_same(T, BFloat);
  constexpr int HD = 128, R = 128 / QT;
  extern __shared__ __attribute__((aligned(16))) unsigned char fas_room[];       // a group: [2 buffers][K | V]
  const int lane = threadIdx.x & 63, kh = lane >> 5, l31 = lane & 31;
  const int group = GROUPS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x & 255) >> 6);     // of the group's four
  unsigned char* const smem = fas_room + group * 4 * FAS_TILE;
  const int unit = blockIdx.x, seq = blockIdx.z;             // heads unit QT ..; a kv head's workgroups share an XCD where eight divides the units
  const int s0 = p.cu_seqlens[seq], qlen = p.cu_seqlens[seq + 1] - s0;
  const int k0 = p.cu_seqlens_k ? p.cu_seqlens_k[seq] : s0, len = p.cu_seqlens_k ? p.cu_seqlens_k[seq + 1] - k0 : qlen;
  const int off = len - qlen;                                // query row i sits at key position i + off
  const int tile = (qlen + R - 1) / R - 1 - (int)blockIdx.y; // the longest key ranges first
  if (tile < 0) return;
  const int head = unit * QT + wave % QT, kvh = unit * QT / (p.num_heads / p.num_kv_heads);
  const int q0 = tile * R, row0 = q0 + 32 * (wave / QT), qrow = row0 + l31;
  const float sc2 = p.scale * 1.44269504088896f;             // scores in units of ln 2: the exponentials are exp2
  const float slope2 = p.alibi ? p.alibi[head] * 1.44269504088896f : 0.f;
  u32x4 qf[8];
  {
    const uint16_t* qp = (const uint16_t*)p.q + (int64_t)(s0 + min(qrow, qlen - 1)) * p.q_stride + head * HD + 8 * kh;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = *reinterpret_cast<const u32x4*>(qp + 16 * ks);
  }
  const int nk = p.causal ? min(len, q0 + R + off) : len;    // keys the tile's last row sees
  const uint16_t* kbase = (const uint16_t*)p.k + (int64_t)k0 * p.k_stride + kvh * HD;
  const uint16_t* vbase = (const uint16_t*)p.v + (int64_t)k0 * p.v_stride + kvh * HD;
  const uint32_t k_row = (uint32_t)p.k_stride * 2, v_row = (uint32_t)p.v_stride * 2;
  // a wave fetches 16 keys of a tile, four an instruction, lane -> key lane >> 4; lane offsets are the tile's, its first key is the buffer's
  const int lrow = 16 * wave + (lane >> 4);
  int klane[4], vlane[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    klane[j] = (lrow + 4 * j) * (int)k_row + (((lane & 15) ^ (4 * j + (lane >> 4))) << 4);
    vlane[j] = (lrow + 4 * j) * (int)v_row + (((lane & 15) ^ ((lane >> 4) << 2)) << 4);
  }
  const bool near = (int64_t)len * (k_row > v_row ? k_row : v_row) < (1ll << 31);      // 32-bit offsets reach every key
  const __amdgpu_buffer_rsrc_t rk0 = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kbase), 0, near ? (uint32_t)(len - 1) * k_row + HD * 2 : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t rv0 = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(vbase), 0, near ? (uint32_t)(len - 1) * v_row + HD * 2 : 0, 0x00020000);
  auto fetch = [&](int buf, int t0) __attribute__((always_inline)) {
    unsigned char* dst = smem + buf * 2 * FAS_TILE + wave * 4096;
    if (near && t0 + FAS_BN <= len) {
      const int ks = t0 * (int)k_row, vs = t0 * (int)v_row;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rk0, (fa_lds_ptr)(dst + j * 1024), 16, klane[j], ks, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv0, (fa_lds_ptr)(dst + FAS_TILE + j * 1024), 16, vlane[j], vs, 0, 0);
      }
      return;
    }
    const int64_t kleft = (int64_t)(len - 1 - t0) * k_row + HD * 2, vleft = (int64_t)(len - 1 - t0) * v_row + HD * 2;      // a buffer from the tile's first key on
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kbase) + (int64_t)t0 * p.k_stride, 0, (uint32_t)min(kleft, (int64_t)0x7fffffff), 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(vbase) + (int64_t)t0 * p.v_stride, 0, (uint32_t)min(vleft, (int64_t)0x7fffffff), 0x00020000);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (fa_lds_ptr)(dst + j * 1024), 16, klane[j], 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (fa_lds_ptr)(dst + FAS_TILE + j * 1024), 16, vlane[j], 0, 0, 0);
    }
  };
  f32x16 o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float m_run = -1e28f, l_run = 0.f;                         // above a masked score: a row without a visible key so far adds nothing
  const int kaddr = l31 * 256 + ((kh ^ (l31 & 15)) << 4);
  // transposing read of 4 keys x 16 columns by 16 lanes: lane i asks for 8 bytes of key i >> 2 and gets column i of the four keys
  const int vk = (lane & 15) >> 2;
  const int vaddr = FAS_TILE + kh * 1024 + vk * 256 + (vk << 6) + (((lane >> 4) & 1) << 5) + ((lane & 3) << 3);
  constexpr int STEP = FAS_BN * GROUPS;                      // the groups take the key tiles in turn
  int t0 = FAS_BN * group, buf = 0;
  if (t0 < nk) fetch(0, t0);
  for (; t0 - FAS_BN * group < nk; t0 += STEP, buf ^= 1) {    // (as often in every group: the barrier is the workgroup's)
    // this wave's part of the tile is there, and it is through with the other buffer
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);                      // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t0 + STEP < nk) fetch(buf ^ 1, t0 + STEP);           // in flight during this tile's products
    if ((GROUPS > 1 && t0 >= nk) || (p.causal && t0 > row0 + 31 + off)) continue;      // no row of the wave sees the tile (uniform; the barrier is the loop's)
    const unsigned char* sb = smem + buf * 2 * FAS_TILE;
    f32x16 s[2];
    u32x4 kf[8][2];
    // (the order is fixed by hand: left to itself hipcc reads one pair of fragments, waits for it, multiplies, and so on)
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
#pragma unroll
      for (int b = 0; b < 2; ++b) kf[ks][b] = *reinterpret_cast<const u32x4*>(sb + b * 8192 + (kaddr ^ (ks << 5)));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const f32x16 zero = {};
        s[b] = fa_mfma32<T>(kf[ks][b], qf[ks], ks == 0 ? zero : s[b]);
      }
    __builtin_amdgcn_sched_barrier(0);
    // lane's scores: row l31, keys t0 + 32 b + 8 q + 4 kh + r
    float f2 = sc2;
    if (slope2 != 0.f || !(sc2 > 0.f)) {                                     // ALiBi: slope times (key - query)
      const float d0 = (float)(t0 + 4 * kh - qrow - off);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[b][i] = s[b][i] * sc2 + slope2 * (d0 + (float)(32 * b + 8 * (i >> 2) + (i & 3)));
      f2 = 1.f;
    }
    if (t0 + FAS_BN > len || (p.causal && t0 + FAS_BN - 1 > row0 + off)) {
      const int last = (p.causal ? min(len - 1, qrow + off) : len - 1) - t0 - 4 * kh;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[b][i] = 32 * b + 8 * (i >> 2) + (i & 3) <= last ? s[b][i] : -INFINITY;
    }
    // The scores are the products' results: what reads them first is where hipcc sees it, as it keeps the wait states between a product and its reader only
    // there.  (One instruction for three numbers, without the canonicalising v_max that fmaxf has in front; a NaN makes its row NaN, as it does
    // without.)
    auto max3 = [](float a, float b, float c) __attribute__((always_inline)) { return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c); };
    // a step of the online softmax: NB blocks of 32 keys from block b0 on; the running maximum moves for rows that are past it by more than 2^lazy
    auto softmax = [&](auto nb, int b0, float lazy) __attribute__((always_inline)) {
      constexpr int NB = decltype(nb)::value;
      float m4[2 * NB];
#pragma unroll
      for (int c = 0; c < 2 * NB; ++c) {
        const int b = b0 + (c >> 1), i0 = 8 * (c & 1);
        m4[c] = max3(s[b][i0], s[b][i0 + 1], s[b][i0 + 2]);
        m4[c] = max3(m4[c], s[b][i0 + 3], s[b][i0 + 4]);
        m4[c] = max3(m4[c], s[b][i0 + 5], s[b][i0 + 6]);
        m4[c] = __builtin_elementwise_maximum(m4[c], s[b][i0 + 7]);
      }
      float mx = __builtin_elementwise_maximum(m4[0], m4[1]);
      if constexpr (NB == 2) mx = max3(mx, m4[2], m4[3]);
      const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, mx), __builtin_bit_cast(unsigned, mx), false, false);
      const unsigned low = sw[0], high = sw[1];
      mx = fmaxf(__builtin_bit_cast(float, low), __builtin_bit_cast(float, high)) * f2;      // both halves' keys
      if (__builtin_amdgcn_ballot_w64(mx > m_run + lazy) != 0) {
        const float m_new = mx > m_run + lazy ? mx : m_run;
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
      }
      float lsum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = b0; b < b0 + NB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[b][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][i], f2, -m_run));     // a masked score: exactly 0
          lsum[i & 3] += s[b][i];
        }
      l_run += (lsum[0] + lsum[1]) + (lsum[2] + lsum[3]);
    };
    // O^T += V^T P^T, 16 keys a product: k slots 4 h .. + 3 of lane half kh are keys 16 ks + 8 h + 4 kh .. + 3, the ones it has
    auto add_values = [&](int ks0, int ks1) __attribute__((always_inline)) {
#pragma unroll
      for (int ks = ks0; ks < ks1; ++ks) {
        const int i0 = 8 * (ks & 1), b = ks >> 1;
        const u32x4 pf = {pack2_16<BF>(s[b][i0], s[b][i0 + 1]), pack2_16<BF>(s[b][i0 + 2], s[b][i0 + 3]), pack2_16<BF>(s[b][i0 + 4], s[b][i0 + 5]),
                          pack2_16<BF>(s[b][i0 + 6], s[b][i0 + 7])};
#pragma unroll
        for (int db = 0; db < 4; ++db) {
          const unsigned char* va = sb + (vaddr ^ (db << 6)) + 4 * ks * 1024;
          const fas_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((fas_s16x4 __attribute__((address_space(3)))*)va);
          const fas_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((fas_s16x4 __attribute__((address_space(3)))*)(va + 2048));
          const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
          o[db] = fa_mfma32<T>(u32x4{l2[0], l2[1], h2[0], h2[1]}, pf, o[db]);
        }
      }
    };
    if constexpr (LONG) {
      softmax(std::integral_constant<int, 2>{}, 0, FAS_LAZY);
      add_values(0, 4);
    } else {
      softmax(std::integral_constant<int, 1>{}, 0, 0.f);
      add_values(0, 2);
      softmax(std::integral_constant<int, 1>{}, 1, 0.f);
      add_values(2, 4);
    }
  }
  float l = l_run + __shfl_xor(l_run, 32, 64);
  if constexpr (GROUPS > 1) {                                // the second group's sums join the first's
    f32x4* const ro = reinterpret_cast<f32x4*>(fas_room + 4 * FAS_TILE) + wave * 16 * 64 + lane;
    float* const rm = reinterpret_cast<float*>(fas_room) + wave * 128 + lane;
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
    l = l * a0 + rm[64] * a1;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const f32x4 x = ro[64 * i];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[i >> 2][4 * (i & 3) + r] = o[i >> 2][4 * (i & 3) + r] * a0 + x[r] * a1;
    }
  }
  if (qrow >= qlen) return;
  const float f = l > 0.f ? 1.f / l : 0.f;
  uint16_t* op = (uint16_t*)p.out + (int64_t)(s0 + qrow) * p.o_stride + head * HD + 4 * kh;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<u32x2*>(op + 32 * db + 8 * q) =
          u32x2{pack2_16<BF>(o[db][4 * q] * f, o[db][4 * q + 1] * f), pack2_16<BF>(o[db][4 * q + 2] * f, o[db][4 * q + 3] * f)};
}

template <typename T, int QT, bool LONG, int GROUPS>
static void fa_short_launch_g(const FAParams& p, int batch, int max_query_len, hipStream_t st) {
  constexpr int rows = 128 / QT;
  constexpr size_t lds = (size_t)GROUPS * 4 * FAS_TILE;
  auto kern = flash_attn_short_kernel<T, QT, LONG, GROUPS>;
  if constexpr (lds > 64 * 1024) {
    static bool attr_set_dev[APHRO_MAX_DEVICES] = {}; bool& attr_set = attr_set_dev[device_slot()];
    if (!attr_set) attr_set = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
  }
  const dim3 grid((unsigned)(p.num_heads / QT), (unsigned)((max_query_len + rows - 1) / rows), (unsigned)batch);
  hipLaunchKernelGGL(kern, grid, dim3(256 * GROUPS), lds, st, p);
}

template <typename T>
static void fa_short_launch_t(const FAParams& p, int batch, int max_query_len, int max_key_len, hipStream_t st) {
  const int per_kv = p.num_heads / p.num_kv_heads, qt = per_kv % 4 == 0 ? 4 : per_kv % 2 == 0 ? 2 : 1, rows = 128 / qt;
  // Two groups of waves a row tile where a launch lasts as long as its longest chain of key tiles: where the row tiles would leave every CU one workgroup
  // at the most, or two of which one prompt's have anything from one key tile to all.  us, one group / two, 32 heads on 8: 600 tokens 18.6 /
  // 16.4, 1500 40.8 / 32.6, 2000 55.3 / 51.7, two of 500 17.0 / 15.7; 8 heads on one, 8192 tokens 187 / 160, 4 on one, 16384 356 / 290.
  // Behind cached keys a prompt's chains are the more alike the more keys there are, and two workgroups of one group that share a CU are then the faster
  // (gather included): 32 on 8, 1300 rows behind 650 / 1300 / 2600 / 20800 keys 62 / 58, 78 / 82, 114 / 125, 596 / 645; 1480 behind 740 / 990 / 2220
  // 68.4 / 67.5, 74.7 / 75.8, 110 / 117.  Long chains bear more: 8 on one, 4800 behind 4800 / 7200 / 14400 194 / 182, 240 / 247, 420 / 444, and where the
  // CUs have two nearly all over any number: 6800 rows behind 6800 / 27200 313 / 297, 883 / 868.
  const int64_t tiles = (int64_t)batch * ((max_query_len + rows - 1) / rows) * (p.num_heads / qt), cus = device_cu_count();
  const int64_t cached = max((int64_t)max_key_len - max_query_len, (int64_t)0);
  const bool uneven = 3 * cached <= 2 * (int64_t)max_query_len || (max_key_len >= 8192 && (3 * cached <= 4 * (int64_t)max_query_len || 5 * tiles >= 8 * cus));
  const bool two = max_key_len >= 256 && (tiles <= cus || (batch == 1 && p.causal && tiles <= 2 * cus && uneven));
  const bool lng = max_key_len >= 1024 && max_key_len >= knobs().fa_v4_min_keys;
#define APHRO_FAS(QT)                                                                                                                            \
  (two ? (lng ? fa_short_launch_g<T, QT, true, 2>(p, batch, max_query_len, st) : fa_short_launch_g<T, QT, false, 2>(p, batch, max_query_len, st)) \
       : (lng ? fa_short_launch_g<T, QT, true, 1>(p, batch, max_query_len, st) : fa_short_launch_g<T, QT, false, 1>(p, batch, max_query_len, st)))
  if (qt == 4) APHRO_FAS(4);
  else if (qt == 2) APHRO_FAS(2);
  else APHRO_FAS(1);
#undef APHRO_FAS
}

bool fa_short_launch(const FAParams& p, int dtype, int batch, int max_query_len, int max_key_len, hipStream_t st) {
  const int64_t span = (int64_t)FAS_BN * 2 * (p.k_stride > p.v_stride ? p.k_stride : p.v_stride);      // a tile's lane offsets
  if (max_key_len < FAS_BN || p.window > 0 || span >= (1ll << 30) || batch > 65535 || (p.o_stride & 3) || ((uintptr_t)p.out & 7)) return false;
  if (dtype == APHRO_F16) fa_short_launch_t<Half>(p, batch, max_query_len, max_key_len, st);
  else fa_short_launch_t<BFloat>(p, batch, max_query_len, max_key_len, st);
  return true;
}

}  // namespace aphro
