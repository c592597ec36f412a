// W4A16 (GPTQ / AWQ-repacked int4) decode GEMM for M <= 32 on gfx950 with the ACTIVATIONS RESIDENT IN REGISTERS -- round 3.
//
// Same role as wna16_gemm.hip's fast kernel (the reference's exllama kernel gemm_half_q_half_gptq_4bit_kernel,
// kernels/quantization/gptq/q_gemm.cu:190-326, and the gptq_marlin_gemm role at small M), same arithmetic -- and, for a
// configuration with the same K partition (4 waves x NSEG segments, same K slices), the same BITS: per 128-k group
// acc = sum a'.q.2^-24 through v_mfma_f32_16x16x32_f16 on subnormal operands, c += s.(2^24 acc - z.rowsum) in fp32, the
// waves' partial sums added in wave order.  What changes is the shape of the work ("resident" kernel):
//
//   * ONE workgroup per CU, every workgroup the same amount of work: the grid is (N / CW) column STRIPS x K slices = 256
//     for the Llama-3-8B projections (gate_up: 256 strips of 112 columns; down: 64 strips of 64 x 4 slices).  The 64-column
//     tile grid of wna16_gemm.hip puts 448 workgroups on 256 CUs for gate_up: 192 CUs do two, 64 do one.
//   * a wave keeps the A fragments of its whole K range in registers (NSEG x 32 VGPRs at 32 rows; up to 256 of the 512 a
//     wave owns at one wave per SIMD) and walks over the strip's column PASSES (64 columns = one 16-byte load per lane and
//     k-step; a last pass of 16/32/48 columns): the activations go through the vector L1 ONCE per workgroup instead of
//     once per 64 columns.  Measured on the round-2 kernel: without its A loads 14.0 us instead of 19.3 (gate_up) -- a
//     CU's miss path carries ~50 GB/s whatever the source, and A (L2 hits) was taking 2/3 of the bytes.
//   * the pre-scale of the A fragments (x 1/16 on the k that meet in-place nibbles) and the row sums are done once, in
//     the first pass, and kept.
//   * the weight stream of a wave is ONE long sequence of loads over all its passes, DEPTH k-steps ahead in a register
//     ring (16 KiB in flight per wave at DEPTH 16); straight-line code (every index is a template constant) so that hipcc
//     counts vmcnt exactly.
//   * optional STRIP-MAJOR weight layout (strip_layout = 1, aphro_wna16_strip_relayout): the 16-byte pieces a wave reads
//     are stored in the order it reads them, so every load instruction is one lane-linear 1 KiB (or 256 REM bytes) piece
//     and a workgroup's share of the matrix is one contiguous range.  The [K/8, N] exllama layout (strip_layout = 0) is
//     read as 256-byte row pieces, exactly like the round-2 kernel.
//   * K reduction over the waves through LDS as a [wave][row][column] tile; the output leaves as whole rows: 16 bytes per
//     thread for the fp32 slabs / the 16-bit result, one 16-byte fragment piece per thread for the SiluAndMul + pack form.
#include <mutex>
#include <utility>

#include "common.h"

namespace aphro {

struct Wna16ResParams {
  const uint16_t* apk;    // fragment-major f16 activations (pack_a_kernel / the fused producers)
  const uint32_t* qw;     // [K/8, N] exllama order, or strip-major (strip_layout)
  const uint32_t* qz;     // [G, N/8]
  const uint16_t* sc;     // [G, N]
  uint16_t* c;            // [M, N] when ksplit == 1 and neither of the two below
  float* partial;         // [ksplit][M][N] fp32 slabs (ksplit > 1 or force_partial)
  uint16_t* act_packed;   // SiluAndMul + pack epilogue (interleaved gate / up columns), ksplit == 1 only
  int M, N, K;
  int gshift;             // log2(group_size / 128)
  int zero_offset;
  int ksplit;             // grid.y
  int force_partial;
  int strip_layout;
  int is_bf16;            // scales / output in bf16 (the activations were widened to f16 when packed)
  const uint16_t* a;      // AROW instantiations: row-major f16 activations [M, lda] read in place (no pack launch)
  int lda;
  unsigned* counter;      // one launch for [M, N] with K slices: tickets per strip (zero between launches), see the epilogue
  int strips, xcd_shift, strips_per_xcd;   // res_set_placement
};

// Workgroup -> (strip, K slice).  Workgroups are dealt round-robin to the 8 XCDs; the host (res_set_placement) works the
// divisions out once per launch -- done here they were ~120 instructions of v_rcp / readfirstlane chains in front of the
// first weight load of every K-sliced launch (profiles/r5_decode_experiments.txt (2)).
__device__ __forceinline__ void res_place(const Wna16ResParams& p, int& strip, int& ky) {
  const int S = p.strips;
  if (p.xcd_shift >= 0) {                 // K slices: slice y owns 8 / ksplit XCDs (each L2 fetches only its slice of A)
    const int L = blockIdx.y * S + blockIdx.x, xcd = L & 7, idx = L >> 3;
    ky = xcd >> p.xcd_shift;
    strip = (xcd & ((1 << p.xcd_shift) - 1)) * p.strips_per_xcd + idx;
  } else {                                // every XCD one contiguous run of strips
    strip = (S & 7) == 0 ? (int)(blockIdx.x & 7) * (S >> 3) + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    ky = blockIdx.y;
  }
}

static void res_set_placement(Wna16ResParams& p, int strips) {
  p.strips = strips;
  p.xcd_shift = -1;
  p.strips_per_xcd = 0;
  const int ks = p.ksplit;
  if (ks > 1 && 8 % ks == 0 && strips % (8 / ks) == 0) {
    const int per = 8 / ks;               // 4, 2, 1
    p.xcd_shift = per == 4 ? 2 : per == 2 ? 1 : 0;
    p.strips_per_xcd = strips / per;
  }
}

template <int B, int E, typename F>
__device__ __forceinline__ void res_static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    res_static_for<B + 1, E>(f);
  }
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t res_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

// write-through (system-scope) store and coherent loads for the in-launch K-slice reduce (same primitives as the split
// form of paged_attention.hip).  Eight 16-byte loads in flight, the wait INSIDE the statement.
__device__ __forceinline__ void res_st_wt(float* p, f32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void res_ld_coh8(f32x4 (&v)[8], const float* const (&p)[8]) {
  asm volatile(
      "global_load_dwordx4 %0, %8, off sc0 sc1\n\tglobal_load_dwordx4 %1, %9, off sc0 sc1\n\t"
      "global_load_dwordx4 %2, %10, off sc0 sc1\n\tglobal_load_dwordx4 %3, %11, off sc0 sc1\n\t"
      "global_load_dwordx4 %4, %12, off sc0 sc1\n\tglobal_load_dwordx4 %5, %13, off sc0 sc1\n\t"
      "global_load_dwordx4 %6, %14, off sc0 sc1\n\tglobal_load_dwordx4 %7, %15, off sc0 sc1\n\t"
      "s_waitcnt vmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
      : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7])
      : "memory");
}

typedef __attribute__((address_space(3))) void* res_lds_ptr;

// AROW: hipcc does not order a ds_read after the `buffer_load ... lds` that fills its source, so the wait is written by
// hand: the number of vector-memory instructions issued after the last staging load of segment s and before its
// fragments are read (loads return in order: vmcnt(that number) = "segment s has landed", everything younger stays in
// flight).  Mirrors the issue order of the kernel below exactly -- straight-line code, every term a constant.
template <int MT, int NSEG, int NP4, int REM, int DEPTH, int AD>
constexpr int res_vm_after_stage(int s) {
  constexpr int NPASS = NP4 + (REM > 0 ? 1 : 0), NST = NPASS * NSEG * 4;
  auto nmeta = [](int q) { return (q / NSEG < NP4) ? 2 : (REM == 3 ? 5 : 2); };
  auto block = [&](int I, bool w, bool a, bool m) {      // the issue block of k-step I (which of its three parts)
    const int pass = I / (NSEG * 4), sg = (I / 4) % NSEG, u = I % 4, q = pass * NSEG + sg;
    int n = 0;
    if (w && I + DEPTH < NST) n += 1;
    if (a && pass == 0 && u == 0 && sg + AD < NSEG) n += 4 * MT;
    if (m && u == 0 && q + 1 < NPASS * NSEG) n += nmeta(q + 1);
    return n;
  };
  int n = 0;
  if (s < AD) {       // staged in the prologue: the later prologue stages, the first weights, the blocks of steps 0 .. 4 s
    n += (AD - 1 - s) * 4 * MT + (DEPTH < NST ? DEPTH : NST);
    for (int I = 0; I <= 4 * s; ++I) n += block(I, true, true, true);
  } else {            // staged in the block of step 4 (s - AD): its metadata, then the blocks up to step 4 s
    n += block(4 * (s - AD), false, false, true);
    for (int I = 4 * (s - AD) + 1; I <= 4 * s; ++I) n += block(I, true, true, true);
  }
  return n > 63 ? 63 : n;
}

struct ResMeta {          // RAW scale / zero words of one (pass, segment): untouched until the segment is consumed
  uint32_t sc[3];
  uint32_t z0, z1;
};

// Columns of a strip: CW = 64 NP4 + 16 REM.  Pass p < NP4: lane (g, c) owns columns 64 p + 4 c + t (t < 4); the last pass
// (REM > 0): columns 64 NP4 + REM c + t (t < REM).  Wave w of K slice y owns segments [(y NWV + w) NSEG, + NSEG).
template <int MT, int NWV, int NSEG, int NP4, int REM, int DEPTH, int ADEPTH, bool KEEP_RS, bool AROW = false>
__global__ __launch_bounds__(NWV * 64, NWV <= 4 ? 1 : 2) void wna16_gemm_resident_kernel(Wna16ResParams p) {
  constexpr int NPASS = NP4 + (REM > 0 ? 1 : 0);
  constexpr int NST = NPASS * NSEG * 4;             // k-steps of a wave over all passes
  constexpr int CW = 64 * NP4 + 16 * REM;
  constexpr int CWP = CW + 4;                       // LDS row pitch (floats): 16-byte aligned rows, conflict-free reads
  constexpr int ROWS = 16 * MT;
  constexpr int RING = DEPTH + 1;
  constexpr int AD = ADEPTH < NSEG ? ADEPTH : NSEG;
  // AROW (row-major activations, the op-level form): a wave stages its A segments through LDS -- coalesced
  // `buffer_load ... lds` of 4 rows x 256 bytes per instruction (8 full cache lines; the 16-row fragment gather straight
  // from the rows touches 32 lines per instruction and cost +7 us at 32 rows), slots XOR-swizzled by the row so that the
  // fragment reads (16 rows, one 16-byte chunk each, per 16 lanes) are bank-conflict free.  NBUF segments per wave, in
  // the wave's own slice of `red` (its reduction tile is written after its last staged segment has been read).
  constexpr int NBUF = AD + 1;
  constexpr int SEGB = ROWS * 256;                  // bytes of one staged segment: [row][16 chunks of 8 k]
  constexpr int WP = (AROW && NBUF * SEGB / 4 > ROWS * CWP) ? NBUF * SEGB / 4 : ROWS * CWP;   // floats per wave
  extern __shared__ __attribute__((aligned(16))) float red[];   // [NWV][WP]: [ROWS][CWP] tiles
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4;
  const int c = lane & 15;
  // workgroups are dealt round-robin to the 8 XCDs: give every XCD one contiguous run of strips (neighbouring strips
  // share cache lines at their edges when a strip's row piece is not a multiple of 128 bytes)
  // With K slices (grid.y > 1) all strips of slice y read the same activation rows: slice y goes to 8 / grid.y XCDs, so
  // that each XCD's L2 fetches only its slice of A (same placement as wna16_gemm.hip's xcd_remap).
  const int S = p.strips;
  int strip, ky;
  res_place(p, strip, ky);
  const int seg0 = (ky * NWV + wave) * NSEG;
  const int cb = strip * CW;
  const int mtiles = (p.M + 15) >> 4;

  const __amdgpu_buffer_rsrc_t rw = res_rsrc(p.qw, (uint32_t)((size_t)(p.K >> 3) * p.N * 4));
  const __amdgpu_buffer_rsrc_t ra = AROW ? res_rsrc(p.a, (uint32_t)(((size_t)(p.M - 1) * p.lda + p.K) * 2))
                                         : res_rsrc(p.apk, (uint32_t)((size_t)(p.K >> 7) * 4 * mtiles * 1024));
  const int ngroups = (p.K >> 7) >> p.gshift;
  const __amdgpu_buffer_rsrc_t rs_ = res_rsrc(p.sc, (uint32_t)((size_t)ngroups * p.N * 2));
  const __amdgpu_buffer_rsrc_t rz = res_rsrc(p.qz, (uint32_t)((size_t)ngroups * (p.N >> 3) * 4));

  // weight addressing: voffset per lane (one for the 64-column passes, one for the last pass), SGPR offset
  // sbase + pass offset + s * SS + u * SU
  int voff_w4, voff_wr, sbase, ss4, su4, ssr, sur, poff4, poffr;
  if (p.strip_layout) {
    constexpr int WAVE_BYTES = NSEG * 4 * 64 * (16 * NP4 + 4 * REM);
    sbase = ((ky * S + strip) * NWV + wave) * WAVE_BYTES;
    voff_w4 = lane * 16; voff_wr = lane * 4 * REM;
    ss4 = 4096; su4 = 1024; ssr = 1024 * REM; sur = 256 * REM;
    poff4 = NSEG * 4096; poffr = NP4 * NSEG * 4096;
  } else {
    sbase = seg0 * 16 * p.N * 4;
    voff_w4 = (4 * g * p.N + cb + 4 * c) * 4; voff_wr = (4 * g * p.N + cb + 64 * NP4 + REM * c) * 4;
    ss4 = ssr = 16 * p.N * 4; su4 = sur = p.N * 4;
    poff4 = 256; poffr = 0;
  }
  int voff_a[AROW ? 4 * MT : MT];
  if constexpr (AROW) {
    // staging instruction `it`: lane -> slot row 4 it + lane / 16 (rows past M read row M - 1: never stored), chunk
    // (lane % 16) ^ (slot row % 16); lands lane-linear in LDS = [slot row][swizzled chunk]
#pragma unroll
    for (int it = 0; it < 4 * MT; ++it) {
      const int srow = 4 * it + (lane >> 4);
      voff_a[it] = min(srow, p.M - 1) * p.lda * 2 + (((lane & 15) ^ (srow & 15)) << 4);
    }
  } else {
#pragma unroll
    for (int i = 0; i < MT; ++i) voff_a[i] = (min(i, mtiles - 1) * 64 + lane) * 16;
  }
  unsigned char* const astage = reinterpret_cast<unsigned char*>(red) + (size_t)wave * WP * 4;
  const int abytes = mtiles * 1024;
  // metadata addressing
  const int col4 = cb + 4 * c;                      // first column of the lane in pass 0 (pass p: + 64 p)
  const int colr = cb + 64 * NP4 + REM * c;         // first column of the lane in the last pass
  const int voff_s4 = col4 * 2, voff_z4 = (col4 >> 3) * 4, zshift4 = (col4 & 7) * 4;
  const int voff_sr = colr * 2, voff_zr0 = (colr >> 3) * 4, voff_zr1 = ((colr + (REM > 0 ? REM - 1 : 0)) >> 3) * 4;
  const int zshiftr = (colr & 7) * 4;
  const float zoff = (float)p.zero_offset;
  const f16x8 ones = {(f16)1.f, (f16)1.f, (f16)16.f, (f16)16.f, (f16)1.f, (f16)1.f, (f16)16.f, (f16)16.f};
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

  u32x4 af[NSEG][4][MT];
  f32x4 rsk[KEEP_RS ? NSEG : 1][MT];
  f32x4 cacc[MT][4], acc[MT][4], rs[MT];
  u32x4 wr[RING];
  ResMeta meta[2];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    rs[i] = zero4;
#pragma unroll
    for (int t = 0; t < 4; ++t) { cacc[i][t] = zero4; acc[i][t] = zero4; }
  }

  auto load_w = [&](auto I_) -> u32x4 {
    constexpr int I = decltype(I_)::value;
    constexpr int pass = I / (NSEG * 4), s = (I / 4) % NSEG, u = I % 4;
    if constexpr (pass < NP4) {
      return __builtin_amdgcn_raw_buffer_load_b128(rw, voff_w4, sbase + pass * poff4 + s * ss4 + u * su4, 2);
    } else {
      const int so = sbase + poffr + s * ssr + u * sur;
      if constexpr (REM == 3) {
        typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
        const u32x3 v = __builtin_amdgcn_raw_buffer_load_b96(rw, voff_wr, so, 2);
        return u32x4{v[0], v[1], v[2], 0u};
      } else if constexpr (REM == 2) {
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rw, voff_wr, so, 2);
        return u32x4{v[0], v[1], 0u, 0u};
      } else {
        return u32x4{__builtin_amdgcn_raw_buffer_load_b32(rw, voff_wr, so, 2), 0u, 0u, 0u};
      }
    }
  };
  auto load_a = [&](auto S_) {
    constexpr int s = decltype(S_)::value;
    if constexpr (AROW) {
#pragma unroll
      for (int it = 0; it < 4 * MT; ++it) {
        const int vo = voff_a[it];    // (local copy: see wna16_gemm_large.hip on the hipcc host-stub bug)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (res_lds_ptr)(astage + (s % NBUF) * SEGB + it * 1024), 16, vo,
                                                 (seg0 + s) * 256, 0, 0);
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const int vo = voff_a[i];
          af[s][u][i] = __builtin_amdgcn_raw_buffer_load_b128(ra, vo, ((seg0 + s) * 4 + u) * abytes, 0);
        }
    }
  };
  auto fetch_a = [&](auto S_) {     // AROW: the staged segment -> fragments (lane (g, c): row 16 i + c, chunk 4 g + u)
    constexpr int s = decltype(S_)::value;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < MT; ++i)
        af[s][u][i] = *reinterpret_cast<const u32x4*>(astage + (s % NBUF) * SEGB + (16 * i + c) * 256 + (((4 * g + u) ^ c) << 4));
  };
  auto load_meta = [&](auto Q_) {   // Q = pass * NSEG + s
    constexpr int Q = decltype(Q_)::value;
    constexpr int pass = Q / NSEG, s = Q % NSEG;
    ResMeta& m = meta[Q & 1];
    const int grp = (seg0 + s) >> p.gshift;
    const int so_s = grp * p.N * 2, so_z = grp * (p.N >> 3) * 4;
    if constexpr (pass < NP4) {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rs_, voff_s4, so_s + pass * 128, 0);
      m.sc[0] = v[0]; m.sc[1] = v[1];
      m.z0 = __builtin_amdgcn_raw_buffer_load_b32(rz, voff_z4, so_z + pass * 32, 0);
    } else {
      if constexpr (REM == 2) {
        m.sc[0] = __builtin_amdgcn_raw_buffer_load_b32(rs_, voff_sr, so_s, 0);
      } else {
#pragma unroll
        for (int t = 0; t < REM; ++t) m.sc[t] = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs_, voff_sr, so_s + 2 * t, 0);
      }
      m.z0 = __builtin_amdgcn_raw_buffer_load_b32(rz, voff_zr0, so_z, 0);
      if constexpr (REM == 3) m.z1 = __builtin_amdgcn_raw_buffer_load_b32(rz, voff_zr1, so_z, 0);
    }
  };

  // ---- prologue: metadata of the first group, the first AD segments of A, the first DEPTH weight steps --------------
  load_meta(std::integral_constant<int, 0>{});
  if constexpr (AROW) __builtin_amdgcn_sched_barrier(0);      // (AROW: the issue ORDER is what res_vm_after_stage counts)
  res_static_for<0, AD>([&](auto S_) { load_a(S_); });
  if constexpr (AROW) __builtin_amdgcn_sched_barrier(0);
  res_static_for<0, (DEPTH < NST ? DEPTH : NST)>([&](auto I_) { wr[decltype(I_)::value % RING] = load_w(I_); });
  __builtin_amdgcn_sched_barrier(0);

  res_static_for<0, NST>([&](auto I_) {
    constexpr int I = decltype(I_)::value;
    constexpr int pass = I / (NSEG * 4), s = (I / 4) % NSEG, u = I % 4;
    constexpr bool LAST = pass >= NP4;
    constexpr int VEC = LAST ? REM : 4;
    constexpr int Q = pass * NSEG + s;
    // ---- issue: weights DEPTH steps ahead, A AD segments ahead (first pass only), metadata one segment ahead ---------
    if constexpr (I + DEPTH < NST) wr[(I + DEPTH) % RING] = load_w(std::integral_constant<int, I + DEPTH>{});
    if constexpr (AROW && pass == 0 && u == 0) __builtin_amdgcn_sched_barrier(0);
    if constexpr (pass == 0 && u == 0 && s + AD < NSEG) load_a(std::integral_constant<int, (s + AD < NSEG ? s + AD : 0)>{});
    if constexpr (AROW && pass == 0 && u == 0) __builtin_amdgcn_sched_barrier(0);
    if constexpr (u == 0 && Q + 1 < NPASS * NSEG) load_meta(std::integral_constant<int, (Q + 1 < NPASS * NSEG ? Q + 1 : 0)>{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (AROW && pass == 0 && u == 0) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(res_vm_after_stage<MT, NSEG, NP4, REM, DEPTH, AD>(s)) : "memory");
      fetch_a(std::integral_constant<int, s>{});
    }
    // ---- A fragments: nibbles 2,3,6,7 of a word are taken in place (bits 4-7 of each half) and weigh 16x, so those k
    // of the fragment carry 1/16 (once: the scaled fragment is what stays resident) ------------------------------------
    f16x8 a[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      u32x4 av = af[s][u][i];
      if constexpr (pass == 0) {
        // (sixteenths() takes 2 to 6 registers more here, of all that there are, and spills; the s_nop: what a product reads has to be two states old)
        asm("v_pk_mul_f16 %0, %2, %4\n\tv_pk_mul_f16 %1, %3, %4\n\ts_nop 1" : "=&v"(av[1]), "=v"(av[3]) : "v"(av[1]), "v"(av[3]), "s"(0x2c002c00u));
        af[s][u][i] = av;
      }
      a[i] = __builtin_bit_cast(f16x8, av);
      if constexpr (pass == 0 || !KEEP_RS)
        rs[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], ones, u == 0 ? zero4 : rs[i], 0, 0, 0);
    }
    const u32x4 wq = wr[I % RING];
#pragma unroll
    for (int t = 0; t < VEC; ++t) {
      const uint32_t wv = wq[t];
      const uint32_t w8 = wv >> 8;
      const u32x4 bq = {wv & 0x000f000fu, wv & 0x00f000f0u, w8 & 0x000f000fu, w8 & 0x00f000f0u};
      const f16x8 b = __builtin_bit_cast(f16x8, bq);
#pragma unroll
      for (int i = 0; i < MT; ++i)
        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b, u == 0 ? zero4 : acc[i][t], 0, 0, 0);
    }
    if constexpr (u == 3) {
      if constexpr (KEEP_RS) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          if constexpr (pass == 0) rsk[s][i] = rs[i]; else rs[i] = rsk[s][i];
        }
      }
      // ---- group epilogue (fp32): c += s * (2^24 * acc - z * rowsum) ---------------------------------------------------
      const ResMeta& m = meta[Q & 1];
      uint32_t zbits;
      if constexpr (!LAST) zbits = m.z0 >> zshift4;
      else if constexpr (REM == 3) zbits = __builtin_amdgcn_alignbit(m.z1, m.z0, zshiftr);
      else zbits = m.z0 >> zshiftr;
#pragma unroll
      for (int t = 0; t < VEC; ++t) {
        const float z = (float)((zbits >> (4 * t)) & 0xf) + zoff;
        uint16_t sb;
        if constexpr (!LAST) sb = (uint16_t)(m.sc[t >> 1] >> (16 * (t & 1)));
        else if constexpr (REM == 2) sb = (uint16_t)(m.sc[0] >> (16 * t));
        else sb = (uint16_t)m.sc[t];
        const float sf = p.is_bf16 ? bf16_bits_to_f32(sb) : f16_bits_to_f32(sb);
        const float s24 = sf * 16777216.f;
        const float nzs = -z * sf;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          // (945 v_fma_f32 in the gate_up instantiation; 437 v_pk_fma_f32, which the library is built without, measured the same to
          //  +-0.1 us on all four projections, profiles/r5_decode_experiments.txt)
          cacc[i][t] = __builtin_elementwise_fma(acc[i][t], f32x4{s24, s24, s24, s24}, cacc[i][t]);
          cacc[i][t] = __builtin_elementwise_fma(rs[i], f32x4{nzs, nzs, nzs, nzs}, cacc[i][t]);
        }
      }
      if constexpr (s == NSEG - 1) {
        // ---- the pass is complete: this wave's partial sums go to its LDS tile, the accumulators start over ------------
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float* dst = &red[wave * WP + (16 * i + 4 * g + r) * CWP + (LAST ? 64 * NP4 + REM * c : 64 * pass + 4 * c)];
            if constexpr (!LAST) {
              *reinterpret_cast<f32x4*>(dst) = f32x4{cacc[i][0][r], cacc[i][1][r], cacc[i][2][r], cacc[i][3][r]};
            } else {
#pragma unroll
              for (int t = 0; t < REM; ++t) dst[t] = cacc[i][t][r];
            }
          }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int t = 0; t < 4; ++t) cacc[i][t] = zero4;
      }
    }
  });
  __syncthreads();

  // ---- K reduction over the waves (wave order: the summation order of wna16_gemm.hip) + store ---------------------------
  const int tid = threadIdx.x;
  if (p.act_packed != nullptr) {
    // SiluAndMul + pack (columns 2j / 2j+1 = gate_j / up_j): a unit = 16 columns of one row = 8 output features = one
    // 16-byte piece of the consumer's fragment-major buffer; consecutive threads take consecutive rows (256 B runs)
    constexpr int UNITS = ROWS * (CW / 16);
    for (int unit = tid; unit < UNITS; unit += NWV * 64) {
      const int ch = unit / ROWS, row = unit % ROWS;
      float v[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 sum = zero4;
#pragma unroll
        for (int w2 = 0; w2 < NWV; ++w2) sum += *reinterpret_cast<const f32x4*>(&red[w2 * WP + row * CWP + 16 * ch + 4 * q]);
        v[4 * q] = sum[0]; v[4 * q + 1] = sum[1]; v[4 * q + 2] = sum[2]; v[4 * q + 3] = sum[3];
      }
      uint16_t o[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (p.is_bf16) {
          o[q] = bf16_bits_to_f16_bits_sat(silu_mul_bits<BFloat>(BFloat::to_f32(BFloat::from_f32(v[2 * q])), BFloat::to_f32(BFloat::from_f32(v[2 * q + 1]))));
        } else {
          o[q] = silu_mul_bits<Half>(Half::to_f32(Half::from_f32(v[2 * q])), Half::to_f32(Half::from_f32(v[2 * q + 1])));
        }
      }
      const int j0 = (cb + 16 * ch) >> 1;
      uint16_t* dst = p.act_packed + ((((size_t)(j0 >> 7) * 4 + ((j0 & 31) >> 3)) * mtiles + (row >> 4)) * 64 + ((j0 & 127) >> 5) * 16 + (row & 15)) * 8;
      if (row < p.M)
        *reinterpret_cast<u32x4*>(dst) = u32x4{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16),
                                               (uint32_t)o[4] | ((uint32_t)o[5] << 16), (uint32_t)o[6] | ((uint32_t)o[7] << 16)};
    }
  } else if (AROW && p.counter != nullptr) {      // (AROW instantiations only: the packed forms keep their code as it was.
    // An epilogue-specialised instantiation per output form was tried on top: same box, gate_up 19.9-20.3 us against 19.5
    // for this generic kernel in tools/resident_bench.py -- smaller code is not faster here, the schedule hipcc finds is)
    // ---- [M, N] out of ONE launch although K is sliced over workgroups (the op-level form: no reduce launch).  Each slice
    // stores its fp32 tile write-through (the slices of a strip sit on different XCDs = different L2s), takes a ticket;
    // the last arriver adds the slices IN SLICE ORDER (= splitk_reduce_kernel's order: the bits do not depend on who
    // arrives last), rounds and stores.  No fences (an agent-scope release / acquire writes back / invalidates the whole
    // L2): write-through stores, a wait for their completion, a relaxed ticket, coherent loads.
    constexpr int UNITS = ROWS * (CW / 4);
    constexpr int NT = NWV * 64;
    for (int unit = tid; unit < UNITS; unit += NT) {
      const int row = unit / (CW / 4), c4 = unit % (CW / 4);
      f32x4 sum = zero4;
#pragma unroll
      for (int w2 = 0; w2 < NWV; ++w2) sum += *reinterpret_cast<const f32x4*>(&red[w2 * WP + row * CWP + 4 * c4]);
      if (row < p.M) res_st_wt(p.partial + ((size_t)ky * p.M + row) * p.N + cb + 4 * c4, sum);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* flag = reinterpret_cast<int*>(red);          // (every wave is past its reads of the tile)
    if (tid == 0) {
      const unsigned old = __hip_atomic_fetch_add(p.counter + strip, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = old == (unsigned)p.ksplit - 1u;
    }
    __syncthreads();
    if (*flag == 0) return;
    if (tid == 0) __hip_atomic_store(p.counter + strip, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    constexpr int PER = (UNITS + NT - 1) / NT;      // units per thread
    auto reduce_batches = [&](auto SPU_) {            // SPU slices per unit (ksplit rounded up), 8 / SPU units per 8-load batch
      constexpr int SPU = decltype(SPU_)::value, UPC = 8 / SPU;
      for (int u0 = 0; u0 < PER; u0 += UPC) {
        const float* ptr[8];
        f32x4 v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int unit = tid + (u0 + j / SPU) * NT, z = j % SPU;
          const bool ok = unit < UNITS && z < p.ksplit;
          const int row = ok ? min(unit / (CW / 4), p.M - 1) : 0, c4 = ok ? unit % (CW / 4) : 0;
          ptr[j] = p.partial + ((size_t)(ok ? z : 0) * p.M + row) * p.N + cb + 4 * c4;
        }
        res_ld_coh8(v, ptr);
#pragma unroll
        for (int q = 0; q < UPC; ++q) {
          const int unit = tid + (u0 + q) * NT;
          const int row = unit / (CW / 4), c4 = unit % (CW / 4);
          f32x4 sum = v[q * SPU];
#pragma unroll
          for (int z = 1; z < SPU; ++z)
            if (z < p.ksplit) sum += v[q * SPU + z];
          uint16_t o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = p.is_bf16 ? BFloat::from_f32(sum[e]) : Half::from_f32(sum[e]);
          if (unit < UNITS && row < p.M)
            *reinterpret_cast<u32x2*>(p.c + (size_t)row * p.N + cb + 4 * c4) =
                u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
        }
      }
    };
    if (p.ksplit <= 2) reduce_batches(std::integral_constant<int, 2>{});
    else if (p.ksplit <= 4) reduce_batches(std::integral_constant<int, 4>{});
    else reduce_batches(std::integral_constant<int, 8>{});
  } else if (p.ksplit > 1 || p.force_partial) {
    constexpr int UNITS = ROWS * (CW / 4);          // 4 columns of one row: 16 bytes of fp32
    for (int unit = tid; unit < UNITS; unit += NWV * 64) {
      const int row = unit / (CW / 4), c4 = unit % (CW / 4);
      f32x4 sum = zero4;
#pragma unroll
      for (int w2 = 0; w2 < NWV; ++w2) sum += *reinterpret_cast<const f32x4*>(&red[w2 * WP + row * CWP + 4 * c4]);
      if (row < p.M) *reinterpret_cast<f32x4*>(p.partial + ((size_t)ky * p.M + row) * p.N + cb + 4 * c4) = sum;
    }
  } else {
    constexpr int UNITS = ROWS * (CW / 8);          // 8 columns of one row: 16 bytes of f16 / bf16
    for (int unit = tid; unit < UNITS; unit += NWV * 64) {
      const int row = unit / (CW / 8), c8 = unit % (CW / 8);
      f32x4 s0 = zero4, s1 = zero4;
#pragma unroll
      for (int w2 = 0; w2 < NWV; ++w2) {
        s0 += *reinterpret_cast<const f32x4*>(&red[w2 * WP + row * CWP + 8 * c8]);
        s1 += *reinterpret_cast<const f32x4*>(&red[w2 * WP + row * CWP + 8 * c8 + 4]);
      }
      uint16_t o[8];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        o[q] = p.is_bf16 ? BFloat::from_f32(s0[q]) : Half::from_f32(s0[q]);
        o[4 + q] = p.is_bf16 ? BFloat::from_f32(s1[q]) : Half::from_f32(s1[q]);
      }
      if (row < p.M)
        *reinterpret_cast<u32x4*>(p.c + (size_t)row * p.N + cb + 8 * c8) =
            u32x4{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16),
                  (uint32_t)o[4] | ((uint32_t)o[5] << 16), (uint32_t)o[6] | ((uint32_t)o[7] << 16)};
    }
  }
}

// K reduction over the waves (LDS tile [wave][row][column], of sums times 2^-24) + the three output forms.
template <int MT, int NWV, int NP4, int REM, int NTHREADS = NWV * 64>
__device__ __forceinline__ void res_reduce_store(const Wna16ResParams& p, float* red, int WP, int ky, int cb, int mtiles,
                                                 int row0 = 0) {
  constexpr int CW = 64 * NP4 + 16 * REM;
  constexpr int CWP = CW + 4;
  constexpr int ROWS = 16 * MT;
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  const int tid = threadIdx.x;
  if (p.act_packed != nullptr) {
    constexpr int UNITS = ROWS * (CW / 16);
    for (int unit = tid; unit < UNITS; unit += NTHREADS) {
      const int ch = unit / ROWS, row = unit % ROWS;
      float v[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 sum = zero4;
#pragma unroll
        for (int w2 = 0; w2 < NWV; ++w2) sum += *reinterpret_cast<const f32x4*>(&red[w2 * WP + row * CWP + 16 * ch + 4 * q]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * q + e] = sum[e] * 16777216.f;
      }
      uint16_t o[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (p.is_bf16) {
          o[q] = bf16_bits_to_f16_bits_sat(silu_mul_bits<BFloat>(BFloat::to_f32(BFloat::from_f32(v[2 * q])), BFloat::to_f32(BFloat::from_f32(v[2 * q + 1]))));
        } else {
          o[q] = silu_mul_bits<Half>(Half::to_f32(Half::from_f32(v[2 * q])), Half::to_f32(Half::from_f32(v[2 * q + 1])));
        }
      }
      const int j0 = (cb + 16 * ch) >> 1;
      uint16_t* dst = p.act_packed + ((((size_t)(j0 >> 7) * 4 + ((j0 & 31) >> 3)) * mtiles + ((row0 + row) >> 4)) * 64 + ((j0 & 127) >> 5) * 16 + (row & 15)) * 8;
      if (row0 + row < p.M)
        *reinterpret_cast<u32x4*>(dst) = u32x4{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16),
                                               (uint32_t)o[4] | ((uint32_t)o[5] << 16), (uint32_t)o[6] | ((uint32_t)o[7] << 16)};
    }
  } else if (p.ksplit > 1 || p.force_partial) {
    constexpr int UNITS = ROWS * (CW / 4);
    for (int unit = tid; unit < UNITS; unit += NTHREADS) {
      const int row = unit / (CW / 4), c4 = unit % (CW / 4);
      f32x4 sum = zero4;
#pragma unroll
      for (int w2 = 0; w2 < NWV; ++w2) sum += *reinterpret_cast<const f32x4*>(&red[w2 * WP + row * CWP + 4 * c4]);
      if (row0 + row < p.M) *reinterpret_cast<f32x4*>(p.partial + ((size_t)ky * p.M + row0 + row) * p.N + cb + 4 * c4) = sum * 16777216.f;
    }
  } else {
    constexpr int UNITS = ROWS * (CW / 8);
    for (int unit = tid; unit < UNITS; unit += NTHREADS) {
      const int row = unit / (CW / 8), c8 = unit % (CW / 8);
      f32x4 s0 = zero4, s1 = zero4;
#pragma unroll
      for (int w2 = 0; w2 < NWV; ++w2) {
        s0 += *reinterpret_cast<const f32x4*>(&red[w2 * WP + row * CWP + 8 * c8]);
        s1 += *reinterpret_cast<const f32x4*>(&red[w2 * WP + row * CWP + 8 * c8 + 4]);
      }
      s0 *= 16777216.f;
      s1 *= 16777216.f;
      uint16_t o[8];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        o[q] = p.is_bf16 ? BFloat::from_f32(s0[q]) : Half::from_f32(s0[q]);
        o[4 + q] = p.is_bf16 ? BFloat::from_f32(s1[q]) : Half::from_f32(s1[q]);
      }
      if (row0 + row < p.M)
        *reinterpret_cast<u32x4*>(p.c + (size_t)(row0 + row) * p.N + cb + 8 * c8) =
            u32x4{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16),
                  (uint32_t)o[4] | ((uint32_t)o[5] << 16), (uint32_t)o[6] | ((uint32_t)o[7] << 16)};
    }
  }
}

// The single-pass STREAM kernel (round 4): same grid, K partition and arithmetic as the resident kernel above (bit-identical
// slabs / packed results), but every k-step covers ALL the strip's columns, so a wave uses each A fragment exactly once:
// nothing is resident, the A fragments of k-step I ride in the same register ring as its weights (D k-steps ahead).
// Strip-major weights and packed activations only.  (The round-4 norm-in-consumer and LDS-ring forms of this kernel were lab
// material -- measured slower, profiles/r4_norm_in_consumer.txt, r4_gemm_lab.txt -- and left the tree in round 5; git
// history: commit 9b85643.)
// Kernel arguments: what the first loads need (weight / activation pointers, placement, sizes) comes FIRST and as scalars, so
// that -amdgpu-kernarg-preload-count (Makefile) has the dispatcher deliver it in SGPRs -- a by-value struct is fetched by
// s_load at entry, one scalar-cache miss in front of every address (profiles/r5_decode_experiments.txt (2)).  p_in carries the rest;
// its copies of the leading fields are not read.
// Everything a group adds carries the products' factor 2^-24 (weights enter them as subnormals) until the waves have met: the scale then
// goes into the FMA as the f16 it is (v_fma_mix_f32), zero points convert a byte at a time and are scaled in the FMA that adds their
// offset, and bf16 is an instantiation.  All factors are powers of two: the resident kernel's bits.  That is 2843 VALU instead of 3502 in gate_up's
// two-tile instance (3032 with packed fp32, which the library is built without); Llama-3-8B, 16 layers, a decode step of 1 / 32 rows
// 992.8 / 1407.9 -> 982.8 / 1401.8 us with the norm's squares as FMAs (fused_decode.hip).  The row sums keep ones that are normal
// numbers: with 2^-24 in their place the sums' last bits changed.
// Two m-tiles: 256 registers, so that the two halves of 33..64 rows share a CU.  (Left free, gate_up's instance takes 257 where fp32 has no packed
// instructions: Llama-3-8B, 16 layers, a decode step of 33 / 64 rows 2333 / 2640 us, so 1978 / 2262.)
template <int MT, int NWV, int NSEG, int NP4, int REM, int D, bool BF16>
__global__ __launch_bounds__(NWV * 64, MT) void wna16_gemm_stream_kernel(const uint32_t* qw, const uint16_t* apk, int strips,
                                                                        int xcd_shift, int strips_per_xcd, int ksplit, int M,
                                                                        int N, int K, int gshift, const uint16_t* sc,
                                                                        const uint32_t* qz, Wna16ResParams p_in) {
  Wna16ResParams p = p_in;
  p.qw = qw; p.apk = apk; p.strips = strips; p.xcd_shift = xcd_shift; p.strips_per_xcd = strips_per_xcd; p.ksplit = ksplit;
  p.M = M; p.N = N; p.K = K; p.gshift = gshift; p.sc = sc; p.qz = qz;
  p.is_bf16 = BF16;
  constexpr int NST = NSEG * 4;
  constexpr int CW = 64 * NP4 + 16 * REM;
  constexpr int CWP = CW + 4;
  constexpr int ROWS = 16 * MT;
  constexpr int NT = 4 * NP4 + REM;
  constexpr int DD = D < NST ? D : NST;
  constexpr int RING = DD + 1;
  constexpr int WP = ROWS * CWP;
  extern __shared__ __attribute__((aligned(16))) float red[];     // [NWV][ROWS][CWP]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4;
  const int c = lane & 15;
  const int S = p.strips;
  int strip, ky;
  res_place(p, strip, ky);
  const int seg0 = (ky * NWV + wave) * NSEG;
  const int cb = strip * CW;
  const int mtiles = (p.M + 15) >> 4;
  const __amdgpu_buffer_rsrc_t rw = res_rsrc(p.qw, (uint32_t)((size_t)(p.K >> 3) * p.N * 4));
  const __amdgpu_buffer_rsrc_t ra = res_rsrc(p.apk, (uint32_t)((size_t)(p.K >> 7) * 4 * mtiles * 1024));
  const int ngroups = (p.K >> 7) >> p.gshift;
  const __amdgpu_buffer_rsrc_t rs_ = res_rsrc(p.sc, (uint32_t)((size_t)ngroups * p.N * 2));
  const __amdgpu_buffer_rsrc_t rz = res_rsrc(p.qz, (uint32_t)((size_t)ngroups * (p.N >> 3) * 4));
  // strip-major weights only (this kernel is reached through the fused decode path, which re-lays its weights)
  constexpr int WAVE_BYTES = NSEG * 4 * 64 * (16 * NP4 + 4 * REM);
  const int sbase = ((ky * S + strip) * NWV + wave) * WAVE_BYTES;
  const int voff_w4 = lane * 16, voff_wr = lane * 4 * REM;
  constexpr int poff4 = NSEG * 4096, poffr = NP4 * NSEG * 4096;
  // 33..64 rows: gridDim.z = 2 -- blockIdx.z picks a 32-row half; the two workgroups of a strip are the 32-row kernel twice,
  // co-resident on a CU (<= 256 VGPRs each: two waves per SIMD, what one workgroup cannot afford).  Both halves of a strip
  // land on the same XCD (x + S (y + ksplit z)), but the second reader of a weight line finds it in that L2 only part of
  // the time: FETCH_SIZE says 97.6 MB per launch on the 4096 x 28672 gate_up (61.5 MB algorithmic: 1.6 x) and 33.7 MB on
  // the 8192 x 7168 shard (1.1 x) -- profiles/r4_norm_in_consumer.txt (6)
  const int mt0 = (int)blockIdx.z * MT;
  int voff_a[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) voff_a[i] = (min(mt0 + i, mtiles - 1) * 64 + lane) * 16;
  const int abytes = mtiles * 1024;
  const int col4 = cb + 4 * c;
  const int colr = cb + 64 * NP4 + REM * c;
  const int voff_s4 = col4 * 2, voff_z4 = (col4 >> 3) * 4, zshift4 = (col4 & 7) * 4;
  const int voff_sr = colr * 2, voff_zr0 = (colr >> 3) * 4, voff_zr1 = ((colr + (REM > 0 ? REM - 1 : 0)) >> 3) * 4;
  const int zshiftr = (colr & 7) * 4;
  const float nzoff = (float)p.zero_offset * -0x1p-24f;
  const f16x8 ones = {(f16)1.f, (f16)1.f, (f16)16.f, (f16)16.f, (f16)1.f, (f16)1.f, (f16)16.f, (f16)16.f};
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

  struct Meta { uint32_t sc[NP4 > 0 ? 2 * NP4 : 1], z[NP4 > 0 ? NP4 : 1], scr[3], zr0, zr1; };
  Meta meta[2];
  f32x4 cacc[MT][NT], acc[MT][NT], rs[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    rs[i] = zero4;
#pragma unroll
    for (int t = 0; t < NT; ++t) { cacc[i][t] = zero4; acc[i][t] = zero4; }
  }
  u32x4 ar[RING][MT], wr4[RING][NP4 > 0 ? NP4 : 1], wrr[RING];
  auto load_a = [&](auto I_) {
    constexpr int I = decltype(I_)::value;
    constexpr int s = I / 4, u = I % 4, B = I % RING;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int vo = voff_a[i];
      ar[B][i] = __builtin_amdgcn_raw_buffer_load_b128(ra, vo, ((seg0 + s) * 4 + u) * abytes, 0);
    }
  };
  auto load_w = [&](auto I_) {
    constexpr int I = decltype(I_)::value;
    constexpr int s = I / 4, u = I % 4, B = I % RING;
#pragma unroll
    for (int pp = 0; pp < NP4; ++pp)
      wr4[B][pp] = __builtin_amdgcn_raw_buffer_load_b128(rw, voff_w4, sbase + pp * poff4 + s * 4096 + u * 1024, 2);
    const int so = sbase + poffr + s * 1024 * REM + u * 256 * REM;
    if constexpr (REM == 3) {
      typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
      const u32x3 v = __builtin_amdgcn_raw_buffer_load_b96(rw, voff_wr, so, 2);
      wrr[B] = u32x4{v[0], v[1], v[2], 0u};
    } else if constexpr (REM == 2) {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rw, voff_wr, so, 2);
      wrr[B] = u32x4{v[0], v[1], 0u, 0u};
    } else if constexpr (REM == 1) {
      wrr[B] = u32x4{__builtin_amdgcn_raw_buffer_load_b32(rw, voff_wr, so, 2), 0u, 0u, 0u};
    }
  };
  auto load_meta = [&](auto Q_) {
    constexpr int Q = decltype(Q_)::value;
    Meta& m = meta[Q & 1];
    const int grp = (seg0 + Q) >> p.gshift;
    const int so_s = grp * p.N * 2, so_z = grp * (p.N >> 3) * 4;
#pragma unroll
    for (int pp = 0; pp < NP4; ++pp) {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rs_, voff_s4, so_s + pp * 128, 0);
      m.sc[2 * pp] = v[0]; m.sc[2 * pp + 1] = v[1];
      m.z[pp] = __builtin_amdgcn_raw_buffer_load_b32(rz, voff_z4, so_z + pp * 32, 0);
    }
    if constexpr (REM == 2) {
      m.scr[0] = __builtin_amdgcn_raw_buffer_load_b32(rs_, voff_sr, so_s, 0);
    } else if constexpr (REM > 0) {
#pragma unroll
      for (int t = 0; t < REM; ++t) m.scr[t] = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs_, voff_sr, so_s + 2 * t, 0);
    }
    if constexpr (REM > 0) m.zr0 = __builtin_amdgcn_raw_buffer_load_b32(rz, voff_zr0, so_z, 0);
    if constexpr (REM == 3) m.zr1 = __builtin_amdgcn_raw_buffer_load_b32(rz, voff_zr1, so_z, 0);
  };

  auto load_step = [&](auto I_) { load_a(I_); load_w(I_); };
  load_meta(std::integral_constant<int, 0>{});
  res_static_for<0, DD>([&](auto I_) { load_step(I_); });
  __builtin_amdgcn_sched_barrier(0);

  res_static_for<0, NST>([&](auto I_) {
    constexpr int I = decltype(I_)::value;
    constexpr int s = I / 4, u = I % 4, B = I % RING;
    if constexpr (I + DD < NST) {
      load_step(std::integral_constant<int, (I + DD < NST ? I + DD : 0)>{});
    }
    if constexpr (u == 0 && s + 1 < NSEG) load_meta(std::integral_constant<int, (s + 1 < NSEG ? s + 1 : 0)>{});
    __builtin_amdgcn_sched_barrier(0);
    f16x8 a[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      a[i] = sixteenths(ar[B][i]);
      rs[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], ones, u == 0 ? zero4 : rs[i], 0, 0, 0);
    }
    res_static_for<0, NT>([&](auto T_) {
      constexpr int t = decltype(T_)::value;
      uint32_t wv;
      if constexpr (t < 4 * NP4) wv = wr4[B][t / 4][t % 4];
      else wv = wrr[B][t - 4 * NP4];
      const uint32_t w8 = wv >> 8;
      const u32x4 bq = {wv & 0x000f000fu, wv & 0x00f000f0u, w8 & 0x000f000fu, w8 & 0x00f000f0u};
      const f16x8 b = __builtin_bit_cast(f16x8, bq);
#pragma unroll
      for (int i = 0; i < MT; ++i)
        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b, u == 0 ? zero4 : acc[i][t], 0, 0, 0);
    });
    if constexpr (u == 3) {
      const Meta& m = meta[s & 1];
      // even and odd nibbles as bytes, which convert in one instruction each
      uint32_t z4[NP4 > 0 ? NP4 : 1][2], zr[2] = {0u, 0u};
#pragma unroll
      for (int pp = 0; pp < NP4; ++pp) {
        const uint32_t zb = m.z[pp] >> zshift4;
        z4[pp][0] = zb & 0x0f0fu;
        z4[pp][1] = (zb >> 4) & 0x0f0fu;
      }
      if constexpr (REM > 0) {
        uint32_t zb;
        if constexpr (REM == 3) zb = __builtin_amdgcn_alignbit(m.zr1, m.zr0, zshiftr);
        else zb = m.zr0 >> zshiftr;
        zr[0] = zb & 0x0f0fu;
        zr[1] = (zb >> 4) & 0x0f0fu;
      }
      res_static_for<0, NT>([&](auto T_) {
        constexpr int t = decltype(T_)::value, tr = t < 4 * NP4 ? t % 4 : t - 4 * NP4;
        uint32_t zb, word;          // the word that holds the column's scale
        bool high;
        if constexpr (t < 4 * NP4) {
          zb = z4[t / 4][tr & 1];
          word = m.sc[2 * (t / 4) + (tr >> 1)], high = t & 1;
        } else {
          zb = zr[tr & 1];
          if constexpr (REM == 2) word = m.scr[0], high = tr;
          else word = m.scr[tr], high = false;
        }
        const float nz = __builtin_fmaf((float)((zb >> (8 * (tr >> 1))) & 0xffu), -0x1p-24f, nzoff);
        float sf;
        if constexpr (BF16) sf = __builtin_bit_cast(float, high ? word & 0xffff0000u : word << 16);
        else sf = f16_bits_to_f32((uint16_t)(high ? word >> 16 : word));
        const float nzs = nz * sf;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          cacc[i][t] = __builtin_elementwise_fma(acc[i][t], f32x4{sf, sf, sf, sf}, cacc[i][t]);
          cacc[i][t] = __builtin_elementwise_fma(rs[i], f32x4{nzs, nzs, nzs, nzs}, cacc[i][t]);
        }
      });
      __builtin_amdgcn_sched_barrier(0);
    }
  });
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* row = &red[wave * WP + (16 * i + 4 * g + r) * CWP];
#pragma unroll
      for (int pp = 0; pp < NP4; ++pp)
        *reinterpret_cast<f32x4*>(row + 64 * pp + 4 * c) = f32x4{cacc[i][4 * pp][r], cacc[i][4 * pp + 1][r], cacc[i][4 * pp + 2][r], cacc[i][4 * pp + 3][r]};
#pragma unroll
      for (int t = 0; t < REM; ++t) row[64 * NP4 + REM * c + t] = cacc[i][4 * NP4 + t][r];
    }
  __syncthreads();
  res_reduce_store<MT, NWV, NP4, REM>(p, red, WP, ky, cb, mtiles, 16 * mt0);
}

// [K/8, N] exllama order -> strip-major: the 16-byte (last pass: 4 REM-byte) pieces in the order the waves read them.
// One thread per strip-major dword.  INVERSE: the same permutation backwards (strip-major -> [K/8, N]): what a caller that
// keeps ONLY the strip-major copy runs for the kernels that do not read it (aphro_wna16_strip_unrelayout).
template <bool INVERSE>
__global__ void wna16_strip_relayout_kernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int N, int K,
                                            int nwv, int nseg, int np4, int rem, int ksplit) {
  const int64_t total = (int64_t)(K >> 3) * N;
  const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= total) return;
  const int cw = 64 * np4 + 16 * rem;
  const int S = N / cw;
  const int lane_dw = 4 * np4 + rem;                 // dwords per lane per (s, u) over all passes
  const int64_t wave_dw = (int64_t)nseg * 4 * 64 * lane_dw;
  int64_t r = d;
  const int64_t widx = r / wave_dw; r -= widx * wave_dw;       // ((ky * S + strip) * nwv + wave)
  const int wave = (int)(widx % nwv);
  const int strip = (int)((widx / nwv) % S);
  const int ky = (int)(widx / nwv / S);
  int pass, s, u, lane, t;
  const int64_t p4_dw = (int64_t)np4 * nseg * 4 * 256;
  if (r < p4_dw) {
    pass = (int)(r / (nseg * 1024)); r %= nseg * 1024;
    s = (int)(r / 1024); r %= 1024;
    u = (int)(r / 256); r %= 256;
    lane = (int)(r / 4); t = (int)(r % 4);
  } else {
    r -= p4_dw;
    pass = np4;
    s = (int)(r / (256 * rem)); r %= 256 * rem;
    u = (int)(r / (64 * rem)); r %= 64 * rem;
    lane = (int)(r / rem); t = (int)(r % rem);
  }
  const int g = lane >> 4, c = lane & 15;
  const int seg = (ky * nwv + wave) * nseg + s;
  const int row = seg * 16 + 4 * g + u;
  const int col = strip * cw + (pass < np4 ? 64 * pass + 4 * c + t : 64 * np4 + rem * c + t);
  if constexpr (INVERSE) out[(size_t)row * N + col] = in[d];
  else out[d] = in[(size_t)row * N + col];
}

}  // namespace aphro

using namespace aphro;

struct ResConfig { int nwv, nseg, np4, rem, ksplit; };

// The configuration serving (M, N, K, group size), or nwv == 0.  One workgroup per CU with equal work where the shape
// allows it: strips x K slices as close to the CU count as the divisibility permits.
//   APHRO_WNA16_RES_CFG="nwv,nseg,np4,rem" picks an instantiated configuration by hand (lab / tests).
static bool res_instantiated(int nwv, int nseg, int np4, int rem);
static bool res_stream_instantiated(int nwv, int nseg, int np4, int rem);
static ResConfig res_plan32(int64_t M, int64_t N, int64_t K, int64_t gs);
// 33..64 rows (round 4): the plan of the 32-row class, launched with gridDim.z = 2 -- stream-kernel plans only
static ResConfig res_plan(int64_t M, int64_t N, int64_t K, int64_t gs) {
  if (M <= 32) return res_plan32(M, N, K, gs);
  ResConfig none = {0, 0, 0, 0, 0};
  if (M > 64 || APHRO_LAB_ENV_INT("APHRO_WNA16_NO_ROW_HALVES", 0)) return none;
  const ResConfig cf = res_plan32(32, N, K, gs);
  return cf.nwv != 0 && res_stream_instantiated(cf.nwv, cf.nseg, cf.np4, cf.rem) ? cf : none;
}
static ResConfig res_plan32(int64_t M, int64_t N, int64_t K, int64_t gs) {
  ResConfig none = {0, 0, 0, 0, 0};
  if (M < 1 || M > 32 || K % 128 != 0 || gs % 128 != 0 || N % 16 != 0) return none;
  const int64_t gq = gs >> 7;
  if ((gq & (gq - 1)) != 0 || (K / 8) * N * 4 >= (int64_t)0xffffffff) return none;
  const int segs = (int)(K / 128);
  auto fits = [&](int nwv, int nseg, int np4, int rem) -> int {   // K slices, or 0
    const int cw = 64 * np4 + 16 * rem;
    if (!res_instantiated(nwv, nseg, np4, rem) || N % cw != 0 || segs % (nwv * nseg) != 0) return 0;
    return segs / (nwv * nseg);
  };
  if (knobs().res_cfg_set != 0) {
    if (knobs().res_cfg_set > 0) {
      const int* rc4 = knobs().res_cfg;
      const int ks = fits(rc4[0], rc4[1], rc4[2], rc4[3]);
      if (ks > 0 && ks <= 16) return ResConfig{rc4[0], rc4[1], rc4[2], rc4[3], ks};
    }
    return none;
  }
  // candidates in order of preference per shape class; the first that fits and fills >= 3/4 of the CUs wins
  // ({4, 4, 1, 3}: round 4, the 8192 x 7168 gate_up of a 70B TP-8 shard -- 64 strips of 112 columns x 4 K slices)
  static const int cand[][4] = {{4, 8, 1, 3}, {4, 4, 1, 3}, {4, 7, 1, 0}, {4, 8, 1, 0}, {4, 4, 1, 0}, {4, 2, 1, 0}, {4, 4, 0, 3}};
  // (round 6: 48-column strips for qkv -- 128 x 2 = 256 workgroups instead of 96 x 2 = 192 -- measured null in the step:
  // 2.5415 / 2.5557 against 2.5513 / 2.5460 ms, profiles/r6_decode_experiments.txt; the plan stays at 64 columns)
  for (const auto& cd : cand) {
    const int ks = fits(cd[0], cd[1], cd[2], cd[3]);
    if (ks <= 0 || ks > 8) continue;
    const int64_t wgs = N / (64 * cd[2] + 16 * cd[3]) * ks;
    if (wgs >= 192 && wgs <= 256) return ResConfig{cd[0], cd[1], cd[2], cd[3], ks};
  }
  return none;
}

template <int MT, int NWV, int NSEG, int NP4, int REM, int DEPTH, int ADEPTH, bool KEEP_RS, bool AROW = false>
static int res_launch(const Wna16ResParams& p, hipStream_t st) {
  constexpr int CW = 64 * NP4 + 16 * REM;
  constexpr int AD = ADEPTH < NSEG ? ADEPTH : NSEG;
  constexpr size_t TILE = (size_t)16 * MT * (CW + 4) * sizeof(float), STAGE = (size_t)(AD + 1) * 16 * MT * 256;
  const size_t lds = (size_t)NWV * (AROW && STAGE > TILE ? STAGE : TILE);
  auto kern = wna16_gemm_resident_kernel<MT, NWV, NSEG, NP4, REM, DEPTH, ADEPTH, KEEP_RS, AROW>;
  if (lds > 64 * 1024) {   // per device and cheap: set every time (a process-wide flag misses a second GPU)
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
      set_error("wna16_gemm_resident: cannot raise the dynamic LDS limit to %zu", lds);
      return APHRO_ERR_LAUNCH;
    }
  }
  const dim3 grid((unsigned)(p.N / CW), (unsigned)p.ksplit);
  Wna16ResParams q = p;
  res_set_placement(q, (int)grid.x);
  hipLaunchKernelGGL(kern, grid, dim3(NWV * 64), lds, st, q);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

template <int MT, int NWV, int NSEG, int NP4, int REM, int D, bool BF16>
static int res_launch_stream_t(const Wna16ResParams& p, hipStream_t st) {
  constexpr int CW = 64 * NP4 + 16 * REM;
  constexpr size_t LDS = (size_t)NWV * 16 * MT * (CW + 4) * sizeof(float);
  static_assert(LDS <= 160 * 1024, "the K-reduce tile exceeds the LDS");
  auto kern = wna16_gemm_stream_kernel<MT, NWV, NSEG, NP4, REM, D, BF16>;
  if (LDS > 64 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS) != hipSuccess) {
    set_error("wna16_gemm_stream: cannot raise the dynamic LDS limit to %zu", LDS);
    return APHRO_ERR_LAUNCH;
  }
  const dim3 grid((unsigned)(p.N / CW), (unsigned)p.ksplit, (unsigned)(p.M > 32 ? 2 : 1));
  Wna16ResParams q = p;
  res_set_placement(q, (int)grid.x);
  hipLaunchKernelGGL(kern, grid, dim3(NWV * 64), LDS, st, q.qw, q.apk, q.strips, q.xcd_shift, q.strips_per_xcd, q.ksplit, q.M, q.N,
                     q.K, q.gshift, q.sc, q.qz, q);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}

template <int MT, int NWV, int NSEG, int NP4, int REM, int D>
static int res_launch_stream(const Wna16ResParams& p, hipStream_t st) {
  return p.is_bf16 ? res_launch_stream_t<MT, NWV, NSEG, NP4, REM, D, true>(p, st) : res_launch_stream_t<MT, NWV, NSEG, NP4, REM, D, false>(p, st);
}

// ---- the instantiated configurations ------------------------------------------------------------------------------------
#ifndef RES_DEPTH
#define RES_DEPTH 8
#endif
#ifndef RES_ADEPTH
#define RES_ADEPTH 2
#endif
// stream kernel (nwv, nseg, np4, rem, k-steps in flight): the plans of the configs[1] projections, each at the depth that
// measured best (tools/reslab.hip, profiles/r4_gemm_lab.txt (8): gate_up 3 / 4 / 5 / 6 -> 14.9 / 15.2 / 15.3 / 16.1 us against
// 15.5-16.0 for the two-pass kernel; down 5 / 6 / 7 -> 9.92 / 9.84 / 10.12 against 10.2; qkv 5 / 6 / 7 -> 6.62 / 6.65 / 6.94
// against 7.0; o 4 / 6 / 8 -> 4.98 / 5.09 / 5.20 against 5.58 for wna16_gemm_kernel)
#define RES_STREAM_CONFIGS(X) \
  X(4, 8, 1, 3, 4)            \
  X(4, 7, 1, 0, 6)            \
  X(4, 4, 1, 0, 6)            \
  X(4, 2, 1, 0, 4)            \
  X(4, 4, 1, 3, 4)
#define RES_KEEP_RS(x) (x)
#define RES_CONFIGS(X) \
  X(4, 8, 1, 3)        \
  X(4, 7, 1, 0)        \
  X(4, 8, 1, 0)        \
  X(4, 4, 1, 0)        \
  X(4, 2, 1, 0)        \
  X(4, 4, 0, 3)        \
  X(4, 4, 1, 3)

// row-major activations read in place (the op-level gptq_gemm in one launch): the same plans
#define RES_AROW_CONFIGS(X) \
  X(4, 8, 1, 3)             \
  X(4, 7, 1, 0)             \
  X(4, 8, 1, 0)             \
  X(4, 4, 1, 0)             \
  X(4, 2, 1, 0)             \
  X(4, 4, 0, 3)             \
  X(4, 4, 1, 3)

static bool res_instantiated(int nwv, int nseg, int np4, int rem) {
#define X(a, b, c, d) if (nwv == a && nseg == b && np4 == c && rem == d) return true;
  RES_CONFIGS(X)
#undef X
  return false;
}

static bool res_stream_instantiated(int nwv, int nseg, int np4, int rem) {
#define X(a, b, c, d, r) if (nwv == a && nseg == b && np4 == c && rem == d) return true;
  RES_STREAM_CONFIGS(X)
#undef X
  return false;
}

static int res_dispatch(const Wna16ResParams& p, const ResConfig& cf, hipStream_t st) {
  const int mt = p.M > 16 ? 2 : 1;
  if (p.M > 32 && !(p.a == nullptr && p.strip_layout)) {
    set_error("wna16_gemm_resident: %d rows are served on packed activations and strip-major weights only", p.M);
    return APHRO_ERR_INVALID;
  }
  if (p.a == nullptr && p.strip_layout) {
    // packed activations on strip-major weights: the single-pass stream kernel where it is instantiated
    // (APHRO_WNA16_STREAM=0: the two-pass resident kernel, 32 rows at most)
    const bool stream = knobs().wna16_stream != 0;
#define X(a, b, c, d, r)                                                                 \
    if (stream && cf.nwv == a && cf.nseg == b && cf.np4 == c && cf.rem == d)             \
      return mt == 2 ? res_launch_stream<2, a, b, c, d, r>(p, st) : res_launch_stream<1, a, b, c, d, r>(p, st);
    RES_STREAM_CONFIGS(X)
#undef X
  }
  if (p.M > 32) {    // (the two-pass kernel has no second row half -- rows 32.. would stay unwritten)
    set_error("wna16_gemm_resident: %d rows need a stream-kernel plan (configuration %d,%d,%d,%d, APHRO_WNA16_STREAM=0?)", p.M,
              cf.nwv, cf.nseg, cf.np4, cf.rem);
    return APHRO_ERR_INVALID;
  }
  if (p.a != nullptr) {   // row-major activations read in place: the configurations res_plan picks by itself
#define X(a, b, c, d)                                                                                    \
    if (cf.nwv == a && cf.nseg == b && cf.np4 == c && cf.rem == d) {                                     \
      constexpr bool KR = RES_KEEP_RS((c + (d > 0 ? 1 : 0)) > 1);                                                   \
      return mt == 2 ? res_launch<2, a, b, c, d, RES_DEPTH, RES_ADEPTH, KR, true>(p, st)          \
                     : res_launch<1, a, b, c, d, RES_DEPTH, RES_ADEPTH, KR, true>(p, st);         \
    }
    RES_AROW_CONFIGS(X)
#undef X
    set_error("wna16_gemm_resident: configuration %d,%d,%d,%d has no row-major instantiation", cf.nwv, cf.nseg, cf.np4, cf.rem);
    return APHRO_ERR_INVALID;
  }
#define X(a, b, c, d)                                                                       \
  if (cf.nwv == a && cf.nseg == b && cf.np4 == c && cf.rem == d) {                          \
    constexpr bool KR = RES_KEEP_RS((c + (d > 0 ? 1 : 0)) > 1);                                        \
    return mt == 2 ? res_launch<2, a, b, c, d, RES_DEPTH, RES_ADEPTH, KR>(p, st)            \
                   : res_launch<1, a, b, c, d, RES_DEPTH, RES_ADEPTH, KR>(p, st);           \
  }
  RES_CONFIGS(X)
#undef X
  set_error("wna16_gemm_resident: configuration %d,%d,%d,%d is not instantiated", cf.nwv, cf.nseg, cf.np4, cf.rem);
  return APHRO_ERR_INVALID;
}

// K slices the resident kernel produces for this shape (fp32 slabs when > 1), 0: shape not served.
extern "C" int aphro_wna16_resident_ksplit(int64_t M, int64_t N, int64_t K, int64_t groups) {
  if (groups <= 0 || K % groups != 0) return 0;
  const ResConfig cf = res_plan(M, N, K, K / groups);
  return cf.nwv ? cf.ksplit : 0;
}

// Decode GEMM on packed activations with the resident kernel.  Exactly one output: act_packed (gate_up form: interleaved
// gate / up columns, SiluAndMul + pack epilogue, one K slice), slabs (fp32 [ksplit][M][N] for a fused consumer) or c
// ([M, N] in `dtype`, one K slice).  strip_layout: q_weight was re-laid by aphro_wna16_strip_relayout for THIS shape.
extern "C" int aphro_wna16_gemm_resident(const void* a_packed, const uint32_t* q_weight, const uint32_t* qzeros,
                                         const void* scales, void* c, float* slabs, size_t slabs_bytes, void* act_packed,
                                         int64_t M, int64_t N, int64_t K, int64_t groups, int zero_offset, int dtype,
                                         int strip_layout, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  APHRO_CHECK(dtype == APHRO_F16 || dtype == APHRO_BF16, "wna16_gemm_resident: dtype must be f16 or bf16");
  APHRO_CHECK(groups > 0 && K % groups == 0, "wna16_gemm_resident: bad groups");
  const ResConfig cf = res_plan(M, N, K, K / groups);
  APHRO_CHECK(cf.nwv != 0, "wna16_gemm_resident: shape M=%ld N=%ld K=%ld groups=%ld is not served", (long)M, (long)N, (long)K, (long)groups);
  APHRO_CHECK(((uintptr_t)a_packed % 16) == 0 && ((uintptr_t)q_weight % 16) == 0, "wna16_gemm_resident: 16-byte alignment required");
  Wna16ResParams p;
  p.apk = (const uint16_t*)a_packed; p.qw = q_weight; p.qz = qzeros; p.sc = (const uint16_t*)scales;
  p.c = (uint16_t*)c; p.partial = slabs; p.act_packed = (uint16_t*)act_packed;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.zero_offset = zero_offset; p.ksplit = cf.ksplit;
  p.gshift = 0;
  for (int64_t q = (K / groups) >> 7; q > 1; q >>= 1) ++p.gshift;
  p.force_partial = 0; p.strip_layout = strip_layout ? 1 : 0; p.is_bf16 = dtype == APHRO_BF16;
  p.a = nullptr; p.lda = 0; p.counter = nullptr;
  if (act_packed != nullptr) {
    APHRO_CHECK(cf.ksplit == 1 && N % 256 == 0, "wna16_gemm_resident: the SiluAndMul form needs one K slice and N/2 %% 128 == 0 (N=%ld)", (long)N);
    p.c = nullptr; p.partial = nullptr;
  } else if (slabs != nullptr) {
    APHRO_CHECK(slabs_bytes >= (size_t)cf.ksplit * M * N * sizeof(float), "wna16_gemm_resident: slabs too small");
    p.force_partial = 1; p.c = nullptr;
  } else {
    APHRO_CHECK(c != nullptr && cf.ksplit == 1, "wna16_gemm_resident: this shape needs the slab form (%d K slices)", cf.ksplit);
  }
  return res_dispatch(p, cf, st);
}

// Tickets of the one-launch K-slice reduce, per device: zero between launches (the last arriver of a strip resets its
// ticket).  hipMalloc'ed on first use, never during a stream capture.  The op-level GEMMs of a process are stream-ordered
// (one compute stream per worker, as in the reference): two of them running CONCURRENTLY on one device would share tickets.
static unsigned* g_res_counter[APHRO_MAX_DEVICES];
static constexpr int RES_COUNTERS = 4096;

static unsigned* res_counters(hipStream_t st) {
  static std::mutex mu;                        // host threads racing on the first call allocate once
  std::lock_guard<std::mutex> lock(mu);
  unsigned*& cnt = g_res_counter[device_slot()];
  if (cnt == nullptr) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return nullptr;
    if (hipMalloc((void**)&cnt, RES_COUNTERS * sizeof(unsigned)) != hipSuccess) { cnt = nullptr; return nullptr; }
    if (hipMemset(cnt, 0, RES_COUNTERS * sizeof(unsigned)) != hipSuccess) { (void)hipFree(cnt); cnt = nullptr; return nullptr; }
  }
  return cnt;
}

// 1: aphro_wna16_gemm_rowmajor serves this call (f16 activations, M <= 32, a shape the resident kernel tiles).
extern "C" int aphro_wna16_gemm_rowmajor_supported(int64_t M, int64_t N, int64_t K, int64_t groups, int dtype) {
  if (dtype != APHRO_F16 || M > 32 || groups <= 0 || K % groups != 0 || knobs().wna16_op_no_resident) return 0;
  const ResConfig cf = res_plan(M, N, K, K / groups);
  if (cf.nwv == 0 || N / (64 * cf.np4 + 16 * cf.rem) > RES_COUNTERS) return 0;
#define X(a, b, c, d) if (cf.nwv == a && cf.nseg == b && cf.np4 == c && cf.rem == d) return 1;
  RES_AROW_CONFIGS(X)
#undef X
  return 0;
}

// The op-level decode GEMM in ONE launch: c[M, N] = a[M, K] (row-major f16, row pitch lda) x int4 weights -- no activation
// pack launch (the kernel gathers its A fragments from the rows), no split-K reduce launch (last-arriver reduce inside the
// kernel).  workspace: ksplit x M x N floats when the shape is K-sliced (aphro_wna16_workspace_bytes covers it).
// Returns APHRO_ERR_WORKSPACE without launching anything when the tickets cannot be allocated (first call under a stream
// capture) or the workspace is too small: the caller takes the three-launch path (aphro_gptq_gemm does).
extern "C" int aphro_wna16_gemm_rowmajor(const void* a, int64_t lda, const uint32_t* q_weight, const uint32_t* qzeros,
                                         const void* scales, void* c, void* workspace, size_t workspace_bytes, int64_t M,
                                         int64_t N, int64_t K, int64_t groups, int zero_offset, int dtype,
                                         int strip_layout, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  APHRO_CHECK(aphro_wna16_gemm_rowmajor_supported(M, N, K, groups, dtype), "wna16_gemm_rowmajor: M=%ld N=%ld K=%ld groups=%ld dtype=%d is not served",
              (long)M, (long)N, (long)K, (long)groups, dtype);
  APHRO_CHECK(((uintptr_t)a % 16) == 0 && lda % 8 == 0 && lda >= K && ((uintptr_t)q_weight % 16) == 0 && ((uintptr_t)c % 16) == 0,
              "wna16_gemm_rowmajor: 16-byte alignment required (lda %% 8 == 0)");
  APHRO_CHECK(((size_t)(M - 1) * lda + K) * 2 < 0xffffffffull, "wna16_gemm_rowmajor: activations exceed one buffer descriptor");
  const ResConfig cf = res_plan(M, N, K, K / groups);
  Wna16ResParams p;
  p.apk = nullptr; p.qw = q_weight; p.qz = qzeros; p.sc = (const uint16_t*)scales;
  p.c = (uint16_t*)c; p.partial = nullptr; p.act_packed = nullptr;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.zero_offset = zero_offset; p.ksplit = cf.ksplit;
  p.gshift = 0;
  for (int64_t q = (K / groups) >> 7; q > 1; q >>= 1) ++p.gshift;
  p.force_partial = 0; p.strip_layout = strip_layout ? 1 : 0; p.is_bf16 = 0;
  p.a = (const uint16_t*)a; p.lda = (int)lda; p.counter = nullptr;
  if (cf.ksplit > 1) {
    const size_t need = (size_t)cf.ksplit * M * N * sizeof(float);
    if (workspace == nullptr || workspace_bytes < need || ((uintptr_t)workspace % 16) != 0) {
      set_error("wna16_gemm_rowmajor: workspace %zu < %zu bytes", workspace_bytes, need);
      return APHRO_ERR_WORKSPACE;
    }
    p.counter = res_counters(st);
    if (p.counter == nullptr) {
      set_error("wna16_gemm_rowmajor: tickets not allocated (first call under a stream capture)");
      return APHRO_ERR_WORKSPACE;
    }
    p.partial = (float*)workspace;
  }
  return res_dispatch(p, cf, st);
}

// Load-time relayout of a [K/8, N] exllama-ordered int4 matrix into the strip-major order of the configuration
// res_plan picks for (M, N, K, groups).  out != in.
static int strip_relayout_impl(const uint32_t* in, uint32_t* out, int64_t M, int64_t N, int64_t K, int64_t groups, bool inverse,
                               void* stream) {
  APHRO_CHECK(groups > 0 && K % groups == 0 && in != out && in && out, "wna16_strip_relayout: bad arguments");
  const ResConfig cf = res_plan(M, N, K, K / groups);
  APHRO_CHECK(cf.nwv != 0, "wna16_strip_relayout: shape M=%ld N=%ld K=%ld is not served by the resident kernel", (long)M, (long)N, (long)K);
  const int64_t total = (K / 8) * N;
  const dim3 grid((unsigned)((total + 255) / 256));
  if (inverse)
    hipLaunchKernelGGL(wna16_strip_relayout_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, in, out, (int)N, (int)K,
                       cf.nwv, cf.nseg, cf.np4, cf.rem, cf.ksplit);
  else
    hipLaunchKernelGGL(wna16_strip_relayout_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, in, out, (int)N, (int)K,
                       cf.nwv, cf.nseg, cf.np4, cf.rem, cf.ksplit);
  APHRO_LAUNCH_CHECK();
  return APHRO_OK;
}
extern "C" int aphro_wna16_strip_relayout(const uint32_t* q_weight, uint32_t* out, int64_t M, int64_t N, int64_t K,
                                          int64_t groups, void* stream) {
  return strip_relayout_impl(q_weight, out, M, N, K, groups, false, stream);
}
// The permutation backwards: strip-major (as aphro_wna16_strip_relayout wrote it for the same M class, N, K, groups) ->
// [K/8, N] exllama order.  out != strip.  For a caller that keeps only the strip-major copy resident.
extern "C" int aphro_wna16_strip_unrelayout(const uint32_t* strip, uint32_t* out, int64_t M, int64_t N, int64_t K,
                                            int64_t groups, void* stream) {
  return strip_relayout_impl(strip, out, M, N, K, groups, true, stream);
}
// The strip-major geometry of (M class, N, K, groups): geom[5] = {waves, 128-k segments per wave, 64-column passes,
// 16-column remainder units, K slices}.  1: served, 0: no strip-major form for the shape (geom untouched).  What the
// prompt-sized kernels (wna16_gemm_large.hip) address the strip-major copy with.
extern "C" int aphro_wna16_strip_geometry(int64_t M, int64_t N, int64_t K, int64_t groups, int* geom) {
  if (groups <= 0 || K % groups != 0) return 0;
  const ResConfig cf = res_plan(M, N, K, K / groups);
  if (cf.nwv == 0) return 0;
  if (geom) { geom[0] = cf.nwv; geom[1] = cf.nseg; geom[2] = cf.np4; geom[3] = cf.rem; geom[4] = cf.ksplit; }
  return 1;
}
