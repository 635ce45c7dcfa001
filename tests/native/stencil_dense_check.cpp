// Host check: the dense row weights of the bounded x pass (weights of
// f(q) - f(0), q = -5..-1, 1..5) against the row-by-row stencils d1/d2 on all
// 11 row kinds, and the interior rows with working-precision coefficients
// (d1_in, d2_in) against d1/d2 bit for bit.  Exits non-zero on a mismatch.
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdio>
#undef __device__
#define __device__
#undef __constant__
#define __constant__
#define __builtin_amdgcn_sbfe(v, off, w) (((int)((unsigned)(v) << (32 - (off) - (w)))) >> (32 - (w)))
#include "sg_stencil.h"
using namespace sg;

int main() {
  Params P{};
  for (int k = 0; k < 5; k++) { P.ac[k] = 1.1 + k; P.sc[k] = 2.3 + k; P.s1[k] = 3.7 + k; P.s2[k] = 4.1 + k; }
  for (int k = 0; k < 4; k++) { P.c1[k] = 5.3 + k; P.c2[k] = 6.7 + k; P.c5[k] = 7.1 + k; P.s5[k] = 8.9 + k; }
  for (int k = 0; k < 3; k++) { P.c4[k] = 9.2 + k; P.s4[k] = 10.1 + k; }
  for (int k = 0; k < 2; k++) { P.c3[k] = 11.3 + k; P.s3[k] = 12.7 + k; }
  P.ovdel[0] = 0.7; P.ovdl2[0] = 0.49;
  for (int k = 0; k < 5; k++) { P.id.ac[k] = P.ac[k]; P.id.sc[k] = P.sc[k]; }
  P.id.ovdel[0] = P.ovdel[0]; P.id.ovdl2[0] = P.ovdl2[0];
  double fv[17];
  for (int q = 0; q < 17; q++) fv[q] = std::sin(0.37 * q + 0.1) * 3.0 + q * 0.01;
  auto at = [&](int kk) { return fv[kk]; };
  const int modes[11] = {0, 1, 2, 3, 4, 5, 11, 12, 13, 14, 15};
  int bad = 0;
  for (int mode : modes) {
    Sten S;
    S.mode = mode;
    const double a1 = d1<true>(P, S, 0, at), a2 = d2<true>(P, S, 0, at);
    const int row = row_of_mode(mode);
    double w5[10], w[20];
    row_weights(P, row, w5);
    row_dense(w5, row, w);
    double b1 = 0.0, b2 = 0.0, m1 = 0.0, m2 = 0.0;
    for (int q = 0; q < 10; q++) {
      const double f = fv[8 + (q < 5 ? q - 5 : q - 4)] - fv[8];
      b1 += w[q] * f;
      b2 += w[10 + q] * f;
      m1 += std::fabs(w[q] * f);
      m2 += std::fabs(w[10 + q] * f);
    }
    b1 *= P.ovdel[0];
    b2 *= P.ovdl2[0];
    // both sum at most 20 terms: within 40 roundings of the sum of magnitudes
    const double e1 = 40 * 2.2e-16 * m1 * P.ovdel[0], e2 = 40 * 2.2e-16 * m2 * P.ovdl2[0];
    const bool ok = std::fabs(a1 - b1) <= e1 && std::fabs(a2 - b2) <= e2;
    std::printf("mode %2d row %2d d1 %.17g %.17g d2 %.17g %.17g %s\n", mode, row, a1, b1, a2, b2, ok ? "ok" : "MISMATCH");
    bad += !ok;
  }
  Sten S;
  S.mode = 0;
  const bool in = d1_in(P.id, 0, at) == d1<false>(P, S, 0, at) && d2_in(P.id, 0, at) == d2<false>(P, S, 0, at);
  std::printf("interior rows %s\n", in ? "ok" : "MISMATCH");
  return bad + !in;
}
