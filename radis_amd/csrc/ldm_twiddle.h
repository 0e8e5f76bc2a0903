// Four-step twiddles of the compiled FFT passes.
#pragma once
#include "ldm_job.h"

__host__ __device__ inline double2 cmul64(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}

// Twiddles W_L^(m * (j0 + s*DS + q*DQ)) of one thread's last-stage outputs
// (s < IT thread passes, q < R legs; m fixed per thread) as
// (base * A^s) * C^q from three table values, so an output costs one complex
// product instead of two table gathers.  Tables and powers are FP64 and rounded
// once: a power's error is its base's times the exponent, and from FP32 tables
// the twiddles were off by 0.8 to 2.9e-7 rms (R = 4 to 16), more than the
// butterflies of a whole transform; now 3.3e-8.  The instructions are as many (FP64
// multiply-adds run at the rate of single FP32 ones).
template <int IT, int R>
struct TwProg {
  float2 ws[IT], wq[R];
  // from the three table values W^(m j0), W^(m DS), W^(m DQ)
  __host__ __device__ inline void set(double2 base, double2 A, double2 C) {
    ws[0] = make_float2((float)base.x, (float)base.y);
#pragma unroll
    for (int s = 1; s < IT; ++s) {
      base = cmul64(base, A);
      ws[s] = make_float2((float)base.x, (float)base.y);
    }
    double2 c[R];
    wq[0] = make_float2(1.0f, 0.0f);
#pragma unroll
    for (int q = 1; q < R; ++q) {
      c[q] = q == 1 ? C : cmul64(c[q / 2], c[q - q / 2]);
      wq[q] = make_float2((float)c[q].x, (float)c[q].y);
    }
  }
};
