// v_mfma_f32_16x16x4_f32 against the chain of four fused multiply-adds over k
// that the prefill attention takes it for: 16 x 16 results per wave, each
// compared bit for bit with fmaf on the host, in the operand and result layout
// the kernel uses (A lane l: row l%16, k = l/16; B lane l: column l%16, k =
// l/16; D lane l register i: row 4*(l/16) + i, column l%16).
//   mfma_check <distribution>
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int WAVES = 4096;

__global__ void __launch_bounds__(64) k_mfma(const float* a, const float* b, const float* c, float* d) {
  const size_t w = blockIdx.x, lane = threadIdx.x;
  const f32x4 acc = *reinterpret_cast<const f32x4*>(c + (w * 64 + lane) * 4);
  *reinterpret_cast<f32x4*>(d + (w * 64 + lane) * 4) =
      __builtin_amdgcn_mfma_f32_16x16x4f32(a[w * 64 + lane], b[w * 64 + lane], acc, 0, 0, 0);
}

#define OK(e)                                                   \
  if (const hipError_t err = (e)) {                             \
    std::printf("%s: %s\n", #e, hipGetErrorString(err));        \
    return 1;                                                   \
  }

int main(int argc, char** argv) {
  const int dist = argc > 1 ? std::atoi(argv[1]) : 0;
  const size_t n = size_t{WAVES} * 64;
  std::vector<float> a(n), b(n), c(4 * n), d(4 * n);
  std::mt19937 g(7 + dist);
  std::normal_distribution<float> nd;
  // +-1.x * 2^e, e uniform in [lo, hi] (below -126: denormal)
  auto wide = [&](int lo, int hi) {
    const int e = lo + static_cast<int>(g() % static_cast<unsigned>(hi - lo + 1));
    return std::ldexp(1.0f + static_cast<float>(g() & 0x7fffff) / 8388608.0f, e) * (g() & 1 ? 1.0f : -1.0f);
  };
  for (size_t i = 0; i < n; ++i) {
    switch (dist) {
      case 0: a[i] = nd(g), b[i] = nd(g); break;                        // scores
      case 1: a[i] = wide(-40, 40), b[i] = wide(-40, 40); break;        // widely spread
      case 2: a[i] = wide(-149, 0), b[i] = wide(-10, 10); break;        // softmax terms down to denormals
      case 3: a[i] = wide(-85, -60), b[i] = wide(-85, -60); break;      // products that underflow
      case 4: a[i] = std::fabs(wide(-126, 0)), b[i] = wide(-149, -120); break;  // denormal values
      default: a[i] = nd(g), b[i] = 1.0f + 1e-6f * nd(g); break;        // sums that cancel (c below)
    }
  }
  for (size_t w = 0; w < WAVES; ++w)
    for (int l = 0; l < 64; ++l)
      for (int i = 0; i < 4; ++i) {
        const int row = 4 * (l / 16) + i, col = l % 16;
        float v = 0.0f;
        if (dist == 0) v = nd(g);
        if (dist == 1) v = wide(-80, 80);
        if (dist == 2 || dist == 4) v = g() & 1 ? 0.0f : wide(-149, -100);
        if (dist == 3) v = g() & 1 ? 0.0f : wide(-149, -130);
        if (dist >= 5) {
          double s = 0.0;
          for (int k = 0; k < 4; ++k) s += static_cast<double>(a[w * 64 + 16 * k + row]) * b[w * 64 + 16 * k + col];
          v = static_cast<float>(-s);
        }
        c[(w * 64 + l) * 4 + i] = v;
      }
  float *da, *db, *dc, *dd;
  OK(hipMalloc(&da, n * 4));
  OK(hipMalloc(&db, n * 4));
  OK(hipMalloc(&dc, n * 16));
  OK(hipMalloc(&dd, n * 16));
  OK(hipMemcpy(da, a.data(), n * 4, hipMemcpyHostToDevice));
  OK(hipMemcpy(db, b.data(), n * 4, hipMemcpyHostToDevice));
  OK(hipMemcpy(dc, c.data(), n * 16, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_mfma, dim3(WAVES), dim3(64), 0, 0, da, db, dc, dd);
  OK(hipGetLastError());
  OK(hipMemcpy(d.data(), dd, n * 16, hipMemcpyDeviceToHost));
  size_t bad = 0, denormal = 0;
  for (size_t w = 0; w < WAVES; ++w)
    for (int l = 0; l < 64; ++l)
      for (int i = 0; i < 4; ++i) {
        const size_t o = (w * 64 + l) * 4 + i;
        const int row = 4 * (l / 16) + i, col = l % 16;
        float v = c[o];
        for (int k = 0; k < 4; ++k) v = std::fmaf(a[w * 64 + 16 * k + row], b[w * 64 + 16 * k + col], v);
        denormal += std::fpclassify(v) == FP_SUBNORMAL;
        if (std::memcmp(&v, &d[o], 4) && bad++ < 5) std::printf("wave %zu lane %d register %d: %a, chain %a\n", w, l, i, d[o], v);
      }
  std::printf("distribution %d: %zu results, %zu denormal, %zu differ\n", dist, 4 * n, denormal, bad);
  return bad ? 1 : 0;
}
