// The tile of the few-rows products (dense_rows.hip: 16-bit, fp8_gemm_rows.hip: FP8): D = w-tile . x^T for up to 192 rows of x, both operands
// through LDS in steps of 128 bytes a row.  What bounds it and why it is cut this way: dense_rows.hip.
#pragma once
#include <utility>

#include "common.h"

namespace aphro {

struct RowsOperands {
  const uint8_t* a;         // [M] rows, lda bytes apart
  const uint8_t* w;         // [N] rows (with a gated activation [2 N]), ldw bytes apart
  int M, N;                 // N: columns of the result
  int row_bytes, lda, ldw;  // row_bytes: K's, a multiple of 128
  int tiles_n, ksplit;
};

typedef __attribute__((address_space(3))) void* rows_lds_ptr;

struct RowsPlan { int mt, nt, ksplit; };

// Which tile, and over how many workgroups K is split (us of [N, K] bf16 with M rows, both sides measured):
//  * 128 rows of w once that gives 160 workgroups: [22016, 4096], 64 rows of x: 43.2 against 45; up to 32 rows of x and many tiles 64
//    rows are ahead ([32000, 2048], 16: 26.5 against 27.4; [128256, 4096], 32: 184 against 187).
//  * 160 tiles of 64 rows and more: K in one piece ([11264, 2048], 16: 12.4, split 14.5).
//  * else one workgroup a CU, or two where one a CU would leave more than an eighth of the CUs idle ([6144, 4096], 16: 5 slices 15.2);
//    a slice has at least 4 steps.
//  * from 65 rows of x on, 128 rows of w also with K split while a slice keeps 10 steps: [4096, 11008], 128: 30.3 against 33.5; and in place of
//    K in one piece where that gives work to more CUs ([10240, 8192], 65 / 128 / 192: 57 / 67 / 90 in one piece of 64 rows, 39 / 43 / 54 in
//    three of 128).
//  * from 129 rows of x on a 64-row tile's stages leave room for one workgroup a CU (rows_dispatch), so that more than 256 of them run in two
//    rounds: no second workgroup a CU, and 128 rows of w above 256 tiles.  FP8, raw sums, 129 / 160 / 192 rows: [6144, 4096] 15.2 / 16.6 / 18.3 in 5
//    slices, 12.5 / 13.2 / 14.6 in 2; [17408, 4096] 39.6 / 41.1 / 45.5 by 64, 29.3 / 30.5 / 31.4 by 128.
//  * 16-bit products of 65 to 160 rows of x on weights of two rounds and more of 256 rows a workgroup, the last nine tenths full, K >= 2560: those
//    (``wide``), which read x through LDS half as often ([128256, 4096], 65 / 96 / 128 / 160 rows 192 / 198 / 208 / 229 by 128 rows, 176 / 180 / 184 /
//    212 here; 176 rows 243 / 256; rounds less full lose: [32768, 4096], 128 rows 64 / 82, [151552, 2048], 150 rows 165 / 174).
inline RowsPlan rows_plan(int64_t M, int64_t w_rows, int64_t row_bytes, bool wide = false) {
  RowsPlan plan;
  const int t64 = (int)((w_rows + 63) / 64), t128 = (int)((w_rows + 127) / 128), steps = (int)(row_bytes / 128);
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
    return plan;
  }
  const int t256 = (int)((w_rows + 255) / 256), rounds = (t256 + 255) / 256;
  if (wide && plan.mt <= 10 && rounds >= 2 && t256 * 10 >= rounds * 256 * 9 && row_bytes >= 40 * 128) {
    plan.nt = 4;
    plan.ksplit = 1;
    return plan;
  }
  const bool lone = plan.mt > 8;
  const int k2 = split(t128, false);
  const bool long_slices = steps / k2 >= 10;
  if (t128 >= 160 || (lone && t64 > 256)) {
    plan.nt = 2;
    plan.ksplit = 1;
  } else if (t64 >= 160 && (t128 * k2 <= t64 || !long_slices)) {
    plan.nt = plan.ksplit = 1;
  } else {
    plan.nt = long_slices ? 2 : 1;
    plan.ksplit = long_slices ? k2 : split(t64, !lone);
  }
  return plan;
}

// Byte offsets inside x, and inside a tile of w (with an activation: inside all of w) are 32-bit.
inline bool rows_fits(int64_t M, int64_t N, int64_t row_bytes, int64_t lda, int64_t ldw, bool gated) {
  constexpr int64_t LIMIT = 0x7fffffffll;
  return M >= 1 && M <= 192 && N >= 4 && N <= (LIMIT >> 4) && row_bytes >= 128 && row_bytes % 128 == 0 && lda >= row_bytes && ldw >= row_bytes &&
         lda <= LIMIT && ldw <= LIMIT && M * lda + row_bytes <= LIMIT && (gated ? 2 * N : 128) * ldw + row_bytes <= LIMIT;
}

// Tr: the products.  MT: 16-row tiles of x; NT: 64 NT rows of w; WR: groups of four waves that divide x's rows; NS: LDS stages.  GATED: a
// 16-row tile of w is 8 rows of the first half and the 8 rows of the second half that go with them.  STREAM: w is fetched with the non-temporal
// hint, which keeps it out of the caches that it passes once (a plain read of 1 GB by 256 to 1024 workgroups: 6.2 TB/s, with the hint 7.0).
template <typename Tr, int MT, int NT, int WR, int NS, bool GATED, bool STREAM>
struct RowsTile {
  static constexpr int MTW = MT / WR, BN = 64 * NT, BM = 16 * MT, NW = 4 * WR;
  static constexpr int WI = BN / 8 / NW, XI = (BM / 8 + NW - 1) / NW, LPS = WI + XI, STAGE = (BN + BM) * 128;
  static constexpr size_t LDS = (size_t)NS * STAGE;
  static_assert(MT % WR == 0 && NS >= 2, "");
  int lane, g, c, wc, wr;   // lane group and column of the MFMA layouts; the wave's 16 rows of w and its part of x's rows
  int ks, n0;               // K slice; first output column
  f32x4 acc[NT][MTW];       // lane (g, c): rows 4 g .. + 3 of the w tile, row c of the x tile

  __device__ __forceinline__ void run(const RowsOperands& p, unsigned char* smem) {
    lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    g = lane >> 4; c = lane & 15; wc = wave & 3; wr = wave >> 2;
    int lin;                                            // contiguous ranges of tiles per XCD
    {
      const int n = gridDim.x, q = n / 8, r = n % 8, xcd = blockIdx.x % 8, k = blockIdx.x / 8;
      lin = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + k;
    }
    ks = lin / p.tiles_n;
    n0 = (lin % p.tiles_n) * (GATED ? BN / 2 : BN);
    const int S = p.row_bytes / 128, s0 = ks * S / p.ksplit, n = (ks + 1) * S / p.ksplit - s0;
    // row r of the tile's BN is row wrow(r) of w behind row n0 (rows past the end: the last one, not stored)
    auto wrow = [&](int r) {
      if constexpr (!GATED) return min(r, p.N - n0 - 1);
      return ((r >> 3) & 1) * p.N + min((r >> 4) * 8 + (r & 7), p.N - n0 - 1);
    };
    const uint32_t last_row = GATED ? (uint32_t)(2 * p.N - 1 - n0) : (uint32_t)(min(p.N - n0, BN) - 1);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w) + (size_t)n0 * p.ldw, 0,
                                                                        last_row * (uint32_t)p.ldw + (uint32_t)p.row_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.a), 0,
                                                                        (uint32_t)(p.M - 1) * (uint32_t)p.lda + (uint32_t)p.row_bytes, 0x00020000);
    int vw[WI], vx[XI];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int r = (wave + NW * i) * 8 + (lane >> 3);
      vw[i] = wrow(r) * p.ldw + (((lane & 7) ^ (r & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) {                      // (where the waves outnumber the pieces, two of them fetch the same one)
      const int r = ((wave + NW * i) % (2 * MT)) * 8 + (lane >> 3);
      vx[i] = min(r, p.M - 1) * p.lda + (((lane & 7) ^ (r & 7)) << 4);
    }
    auto issue = [&](int s, int slot) {
      unsigned char* st = smem + slot * STAGE;
      const int so = (s0 + s) * 128;
#pragma unroll
      for (int i = 0; i < WI; ++i) {
        const int v = vw[i];                            // (a local copy: see wna16_gemm_large.hip)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (rows_lds_ptr)(st + (wave + NW * i) * 1024), 16, v, so, 0, STREAM ? 2 : 0);
      }
#pragma unroll
      for (int i = 0; i < XI; ++i) {
        const int v = vx[i];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (rows_lds_ptr)(st + BN * 128 + ((wave + NW * i) % (2 * MT)) * 1024), 16, v, so, 0, 0);
      }
    };
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
      // with step s - 1 -- its fragments are in registers (lgkmcnt: nothing else keeps a product, and the wait for its operands, ahead of the
      // barrier) -- whose stage the loads issued now take
      if (s + NS - 2 < n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NS - 2) * LPS) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (s + NS - 1 < n) issue(s + NS - 1, fetch);
      Tr::template step<NT, MTW>(smem + slot * STAGE, wbase, xbase, sw, acc);
      slot = slot + 1 == NS ? 0 : slot + 1;
      fetch = fetch + 1 == NS ? 0 : fetch + 1;
    }
  }
};

// f(MT, NT, WR, NS) for a plan (WIDE: of those that may have 256 rows of w).  Stages: as many as let two workgroups share a CU's 160 KB; from 129 rows of x on, three with 64 rows of w, and one
// workgroup a CU (two stages and two workgroups: [6144, 4096] FP8, 160 rows, 5 slices 13.7 us, this in 2 slices 13.2).  128-row tiles that all
// run at once with one workgroup a CU ([22016, 4096], 65 rows and more) get eight waves and deeper stages, more tiles than CUs two stages:
// bf16 [37888, 3584], 65 / 160 rows 73 / 99 us deep, 68 / 93 with two; [62000, 4096], 65 / 160 rows 111 / 133 and 115 / 126.
template <bool WIDE, typename F>
int rows_dispatch(const RowsPlan& plan, int tiles_n, F&& f) {
#define ROWS(MT, NT, WR, NS) f(std::integral_constant<int, MT>{}, std::integral_constant<int, NT>{}, std::integral_constant<int, WR>{}, std::integral_constant<int, NS>{})
  const bool many = tiles_n >= 512 || (tiles_n > 256 && (plan.mt > 8 || tiles_n < 448));
  if (plan.nt == 1) {
    switch (plan.mt) {
      case 1: return ROWS(1, 1, 1, 5);
      case 2: return ROWS(2, 1, 1, 6);
      case 3: return ROWS(3, 1, 1, 5);
      case 4: return ROWS(4, 1, 1, 5);
      case 6: return ROWS(6, 1, 1, 3);
      case 8: return ROWS(8, 1, 1, 3);
      case 10: return ROWS(10, 1, 1, 3);
      default: return ROWS(12, 1, 1, 3);
    }
  }
  if constexpr (WIDE) {
    if (plan.nt == 4) {
      switch (plan.mt) {
        case 6: return ROWS(6, 4, 2, 3);
        case 8: return ROWS(8, 4, 2, 3);
        default: return ROWS(10, 4, 2, 3);
      }
    }
  }
  switch (plan.mt) {
    case 1: return ROWS(1, 2, 1, 4);
    case 2: return ROWS(2, 2, 1, 4);
    case 3: return ROWS(3, 2, 1, 3);
    case 4: return ROWS(4, 2, 1, 3);
    case 6: return many ? ROWS(6, 2, 1, 2) : ROWS(6, 2, 1, 3);
    case 8: return many ? ROWS(8, 2, 1, 2) : ROWS(8, 2, 2, 3);
    case 10: return many ? ROWS(10, 2, 1, 2) : ROWS(10, 2, 2, 4);
    default: return many ? ROWS(12, 2, 1, 2) : ROWS(12, 2, 2, 4);
  }
#undef ROWS
}

}  // namespace aphro
