// Prints which kernel and tiles a quantised projection takes, by the rules that the launches
// use (engine-mlx_amd/csrc/qmatmul_plan.hpp): one line "kernel mt nt" per input line
// "M N K group bits ldx scale_offset cus" (scale_offset: bytes of scales and biases past a 16-byte
// boundary; qgemm_dq_staged: qgemm_dq with its scales through LDS).
#include <cstdio>

#include "qmatmul_plan.hpp"

int main() {
  static const char* const names[] = {"gemv1", "qmv_ks", "qgemm_ks", "qmv", "qmvx", "qgemm_dq", "qmm"};
  long long m, n, k, gs, bits, ldx, off, cus;
  while (std::scanf("%lld %lld %lld %lld %lld %lld %lld %lld", &m, &n, &k, &gs, &bits, &ldx, &off, &cus) == 8) {
    ema::QmmArgs a{};
    a.s = a.b = reinterpret_cast<const uint8_t*>(static_cast<uintptr_t>(4096 + off));
    a.ldx = ldx;
    a.M = (int)m;
    a.N = (int)n;
    a.K = (int)k;
    a.G = (int)(k / gs);
    const ema::QmmRoute r = ema::qmm_route(a, (int)gs, (int)bits, (int)cus);
    const bool staged = r.kernel == ema::QmmKernel::qgemm_dq && ema::dq_stages_scales(a, r.mt);
    std::printf("%s%s %d %d\n", names[(int)r.kernel], staged ? "_staged" : "", r.mt, r.nt);
  }
  return 0;
}
