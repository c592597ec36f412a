// Prompt attention over rows of 128, below the key counts of the fourth generation (flash_attn_v4.hip): a workgroup owns 128 / QT consecutive
// query rows of QT heads of one kv head (QT = 4, 2, 1: as many as divide its heads), a wave 32 rows of one head, so that a K or V tile fetched once serves 128 rows and a 300-token prompt still makes hundreds of workgroups.
//   * S^T = K Q^T and O^T = V^T P^T on 32x32x16 products: a lane holds 32 of the 64 scores of one row, its probabilities are the second product's
//     operand where they lie.
//   * K and V tiles of 64 keys go from memory to LDS without a stop in registers, two buffers, one barrier a tile; LDS slot s of key j holds K's
//     16-byte piece s ^ (j & 15), V's s ^ 4 (j & 3): fragment reads and transposing reads find their banks free.  Keys past the sequence's end are
//     fetched as zeros (the buffer ends there) and masked.
//   * the output is rescaled only when some row's maximum moved.
// Bound by a tile's chain of steps (1.5 us: 32 products, two softmaxes), and by the launch for the shortest.  us before / here (32 heads on 8,
// causal): against 64-row workgroups with V transposed number by number, below 512 keys, 300 tokens 18.8 / 13.7, five prompts of 107 to 430 39.4 /
// 20.4; against the second generation's 128 rows a workgroup, 1000 tokens 45.5 / 30.8, five of 600 61.9 / 39.1, three of 1000 94 / 53; against the
// third's 256 rows (deleted), 1111 tokens 45.2 / 35.5, 3000 116.7 / 101.8, three of 1500 107 / 90, six of 1300 161 / 128.  The fourth: 4096 tokens
// 176 / 187, 8192 596 / 604, but 5000 267 / 247: the line at 4096 keys does not look at how full the last of its 256-row tiles is.  Below 64 keys the
// first is the faster (six of 26 tokens 6.1 / 7.4).
// Loads hidden from hipcc, which otherwise waits for the next tile in front of the transposing reads: no faster (three of 1000 tokens 53 / 55).
#include "common.h"
#include "flash_attn_common.h"

namespace aphro {

typedef short fas_s16x4 __attribute__((ext_vector_type(4)));

constexpr int FAS_BN = 64, FAS_TILE = FAS_BN * 256;          // keys of a tile, bytes of its K (or V) rows

template <typename T, int QT>
__global__ __launch_bounds__(256, 2) void flash_attn_short_kernel(FAParams p) {
  constexpr bool BF = __is_same(T, BFloat);
  constexpr int HD = 128, R = 128 / QT;
  __shared__ __attribute__((aligned(16))) unsigned char smem[4 * FAS_TILE];      // [2 buffers][K | V]
  const int lane = threadIdx.x & 63, kh = lane >> 5, l31 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
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
  const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kbase), 0, (uint32_t)(len - 1) * k_row + HD * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(vbase), 0, (uint32_t)(len - 1) * v_row + HD * 2, 0x00020000);
  // a wave fetches 16 keys of a tile, four an instruction, lane -> key lane >> 4
  auto fetch = [&](int buf, int t0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int key = 16 * wave + 4 * j + (lane >> 4);
      unsigned char* dst = smem + buf * 2 * FAS_TILE + wave * 4096 + j * 1024;
      const int ko = (int)((uint32_t)(t0 + key) * k_row + (((lane & 15) ^ (4 * j + (lane >> 4))) << 4));
      const int vo = (int)((uint32_t)(t0 + key) * v_row + (((lane & 15) ^ ((lane >> 4) << 2)) << 4));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (fa_lds_ptr)dst, 16, ko, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (fa_lds_ptr)(dst + FAS_TILE), 16, vo, 0, 0, 0);
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
  fetch(0, 0);
  int buf = 0;
  for (int t0 = 0; t0 < nk; t0 += FAS_BN, buf ^= 1) {
    // this wave's part of the tile is there, and it is through with the other buffer
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (t0 + FAS_BN < nk) fetch(buf ^ 1, t0 + FAS_BN);       // in flight during this tile's products
    if (p.causal && t0 > row0 + 31 + off) continue;          // no row of the wave sees the tile (uniform; the barrier is the loop's)
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
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[b][i] *= sc2;
    if (slope2 != 0.f) {                                     // ALiBi: slope times (key - query)
      const float d0 = (float)(t0 + 4 * kh - qrow - off);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[b][i] += slope2 * (d0 + (float)(32 * b + 8 * (i >> 2) + (i & 3)));
    }
    if (t0 + FAS_BN > len || (p.causal && t0 + FAS_BN - 1 > row0 + off)) {
      const int last = (p.causal ? min(len - 1, qrow + off) : len - 1) - t0 - 4 * kh;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[b][i] = 32 * b + 8 * (i >> 2) + (i & 3) <= last ? s[b][i] : -1e30f;
    }
    // 32 keys a step of the online softmax, as in the first two generations: a step's largest probability is 1, exactly
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      // (four partial maxima and sums: a chain of 16 dependent steps would be waited for)
      float mx4[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) mx4[i] = fmaxf(fmaxf(s[b][i], s[b][4 + i]), fmaxf(s[b][8 + i], s[b][12 + i]));
      float mx = fmaxf(fmaxf(mx4[0], mx4[1]), fmaxf(mx4[2], mx4[3]));
      const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, mx), __builtin_bit_cast(unsigned, mx), false, false);
      mx = fmaxf(__builtin_bit_cast(float, (unsigned)sw[0]), __builtin_bit_cast(float, (unsigned)sw[1]));      // both halves' keys
      const float m_new = fmaxf(m_run, mx);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      float lsum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[b][i] = __builtin_amdgcn_exp2f(s[b][i] - m_new);   // a masked score is 1e30 below: exactly 0
        lsum[i & 3] += s[b][i];
      }
      l_run = l_run * alpha + ((lsum[0] + lsum[1]) + (lsum[2] + lsum[3]));
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
      }
      // O^T += V^T P^T, 16 keys a product: k slots 4 h .. + 3 of lane half kh are keys 16 ks + 8 h + 4 kh .. + 3, the ones it has
#pragma unroll
      for (int ks = 2 * b; ks < 2 * b + 2; ++ks) {
        const int i0 = 8 * (ks & 1);
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
    }
  }
  const float l = l_run + __shfl_xor(l_run, 32, 64);
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

template <typename T>
static void fa_short_launch_t(const FAParams& p, int batch, int max_query_len, hipStream_t st) {
  const int per_kv = p.num_heads / p.num_kv_heads, qt = per_kv % 4 == 0 ? 4 : per_kv % 2 == 0 ? 2 : 1, rows = 128 / qt;
  const dim3 grid((unsigned)(p.num_heads / qt), (unsigned)((max_query_len + rows - 1) / rows), (unsigned)batch);
  if (qt == 4) hipLaunchKernelGGL((flash_attn_short_kernel<T, 4>), grid, dim3(256), 0, st, p);
  else if (qt == 2) hipLaunchKernelGGL((flash_attn_short_kernel<T, 2>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((flash_attn_short_kernel<T, 1>), grid, dim3(256), 0, st, p);
}

bool fa_short_launch(const FAParams& p, int dtype, int batch, int max_query_len, int max_key_len, hipStream_t st) {
  const int64_t span = (int64_t)(max_key_len + 2 * FAS_BN) * 2 * (p.k_stride > p.v_stride ? p.k_stride : p.v_stride);      // offsets, tiles past the end too
  if (max_key_len < FAS_BN || p.window > 0 || span >= (1ll << 31) || batch > 65535 || (p.o_stride & 3) || ((uintptr_t)p.out & 7)) return false;
  if (dtype == APHRO_F16) fa_short_launch_t<Half>(p, batch, max_query_len, st);
  else fa_short_launch_t<BFloat>(p, batch, max_query_len, st);
  return true;
}

}  // namespace aphro
