// Lab harness for the prefill attention kernels: the library sources compiled standalone (tools/run_fa_lab.sh).
// Times the two kernels of head size 128 -- flash_attn_short.hip's and the fourth generation's, each forced on by its key count
// (APHRO_FA_V4_MIN_KEYS) -- on the same random input (T tokens, Hq 32 / Hkv 8, causal; T >= 1024) and compares their outputs element by
// element.
#include "bin/csrc_lab/flash_attn.hip"
#include "bin/csrc_lab/flash_attn_v4.hip"
#include "bin/csrc_lab/flash_attn_short.hip"
#include "bin/csrc_lab/runtime.hip"
#include <cmath>
#include <cstring>
#include <vector>
int main(int argc, char** argv) {
  const int T = argc > 1 ? atoi(argv[1]) : 8192, Hq = 32, Hkv = 8, D = 128;
  if (T < 1024) { printf("fewer than 1024 tokens: the fourth generation does not run\n"); return 1; }
  const int dt = argc > 2 ? atoi(argv[2]) : APHRO_F16;
  const size_t row = (size_t)(Hq + 2 * Hkv) * D;
  std::vector<uint16_t> h(T * row);
  uint32_t st = 12345;
  for (auto& x : h) {
    st = st * 1664525u + 1013904223u;
    const float f = (((st >> 8) & 0xffff) / 65536.f - 0.5f) * 4.f;
    if (dt == APHRO_F16) { _Float16 v = (_Float16)f; x = *(uint16_t*)&v; }
    else { uint32_t u; memcpy(&u, &f, 4); x = (uint16_t)(u >> 16); }
  }
  uint16_t *qkv, *out, *out_short; int32_t* cu;
  const size_t on = (size_t)T * Hq * D;
  hipMalloc(&qkv, h.size() * 2); hipMalloc(&out, on * 2); hipMalloc(&out_short, on * 2); hipMalloc(&cu, 8);
  hipMemcpy(qkv, h.data(), h.size() * 2, hipMemcpyHostToDevice);
  const int32_t hc[2] = {0, T}; hipMemcpy(cu, hc, 8, hipMemcpyHostToDevice);
  auto run = [&](uint16_t* o) { return aphro_flash_attn_varlen(o, qkv, qkv + Hq * D, qkv + (Hq + Hkv) * D, cu, 1, T, Hq, Hkv, D, row, row, row, 0.0883883f, 1, nullptr, dt, nullptr); };
  auto bench = [&](const char* name, uint16_t* o) {
    hipMemset(o, 0xff, on * 2);
    if (run(o) != 0) { printf("error: %s\n", aphro_last_error()); exit(1); }
    if (hipDeviceSynchronize() != hipSuccess) { printf("%s: kernel fault\n", name); exit(1); }
    for (int i = 0; i < 40; ++i) run(o);            // the first ~50 ms of MFMA-heavy work run below the clocks the chip then holds
    hipDeviceSynchronize();
    hipEvent_t a, b; hipEventCreate(&a); hipEventCreate(&b);
    hipEventRecord(a); for (int i = 0; i < 20; ++i) run(o); hipEventRecord(b); hipEventSynchronize(b);
    float ms; hipEventElapsedTime(&ms, a, b); ms /= 20;
    printf("%s T=%d %s: %.3f ms  %.1f TFLOP/s (causal flops)\n", name, T, dt == APHRO_F16 ? "f16" : "bf16", ms,
           4.0 * T * T * D * Hq / 2 / (ms * 1e-3) / 1e12);
  };
  setenv("APHRO_FA_V4_MIN_KEYS", "1073741824", 1); aphro_reload_env();
  bench("flash_attn_short ", out_short);
  setenv("APHRO_FA_V4_MIN_KEYS", "1024", 1); aphro_reload_env();
  bench("fourth generation", out);
  std::vector<uint16_t> a(on), b(on);
  hipMemcpy(a.data(), out_short, on * 2, hipMemcpyDeviceToHost);
  hipMemcpy(b.data(), out, on * 2, hipMemcpyDeviceToHost);
  auto tof = [&](uint16_t x) { if (dt == APHRO_F16) { _Float16 v; memcpy(&v, &x, 2); return (float)v; } uint32_t u = (uint32_t)x << 16; float f; memcpy(&f, &u, 4); return f; };
  double worst = 0; size_t bad = 0, nan = 0, wi = 0;
  for (size_t i = 0; i < on; ++i) {
    const float x = tof(a[i]), y = tof(b[i]);
    if (y != y) { ++nan; continue; }
    const double d = fabs((double)x - y);
    if (d > worst) { worst = d; wi = i; }
    if (d > 2e-2 * (dt == APHRO_F16 ? 1 : 4)) ++bad;
  }
  printf("fourth generation vs flash_attn_short: worst abs diff %.3e at token %zu head %zu d %zu (%.4f vs %.4f), %zu beyond tolerance, %zu NaN\n",
         worst, wi / (Hq * D), (wi / D) % Hq, wi % D, tof(a[wi]), tof(b[wi]), bad, nan);
  return 0;
}
