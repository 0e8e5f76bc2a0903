// Four-step twiddles of the compiled passes (ldm_twiddle.h), every (s, q) of a
// column's progression against W_L^e evaluated directly.
//
// Bound: a factor's components are below 1 and rounded once, 2^-25 each, so the
// factor is off by at most sqrt(2) 2^-25 and the product of two by 2 sqrt(2) 2^-25;
// the FP64 powers add at most R + IT products of 2^-52 (1e-14).
#include <cmath>
#include <cstdio>

#include "ldm_twiddle.h"

static double2 w(long long e, long long L) {
  const long double a = -2.0L * 3.14159265358979323846264338327950288L * (long double)(e % L) / (long double)L;
  return make_double2((double)cosl(a), (double)sinl(a));
}

static double g_worst = 0.0;

template <int IT, int R>
static void check(long long L, long long n1, long long ds) {
  const long long dq = n1 / R, n2 = L / n1;
  for (long long m = 0; m < n2; m += (n2 > 97 ? n2 / 97 : 1))
    for (long long j0 = 0; j0 < ds; j0 += (ds > 5 ? ds / 5 : 1)) {
      TwProg<IT, R> t;
      // the three factors as the kernels form them: products of the table halves
      auto halves = [&](long long e) { return cmul64(w(e >> 10 << 10, L), w(e & 1023, L)); };
      t.set(halves(m * j0), halves(m * ds), halves(m * dq));
      for (int s = 0; s < IT; ++s)
        for (int q = 0; q < R; ++q) {
          const double2 p = cmul64(make_double2(t.ws[s].x, t.ws[s].y), make_double2(t.wq[q].x, t.wq[q].y));
          const double2 x = w(m * (j0 + s * ds + q * dq), L);
          g_worst = std::fmax(g_worst, std::hypot(p.x - x.x, p.y - x.y));
        }
    }
}

int main() {
  for (int k = 0; k < 2; ++k) {
    const long long n2 = k ? 2048 : 64;
    check<1, 16>(256 * n2, 256, 16);
    check<2, 8>(512 * n2, 512, 32);
    check<3, 4>(320 * n2, 320, 32);
    check<2, 8>(640 * n2, 640, 64);
    check<1, 16>(768 * n2, 768, 48);
    check<4, 4>(1024 * n2, 1024, 64);
  }
  std::printf("worst %.3e\n", g_worst);
  return g_worst <= 2.0 * std::sqrt(2.0) * std::ldexp(1.0, -25) + 1e-13 ? 0 : 1;
}
