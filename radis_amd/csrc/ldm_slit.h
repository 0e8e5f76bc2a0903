// Instrumental slit convolution on the device: RADIS convolves the
// *_noslit quantities with the slit function sampled on the spectrum grid
// (radis/tools/slit.py:477-757, scipy.signal.oaconvolve(I, slit, 'same') *
// wstep).  Here the sum is direct:
//   out[i] = scale * sum_j slit[j] * in[i + c - j],  c = (k - 1) / 2,
// with in[] outside [0, n) read as zero: k products and additions per point in
// FP64 (the product of two FP32 values is exact there), so every output is the
// exact sum rounded to FP32, whatever the slit length and the range of the
// spectrum, and a value that is not finite reaches the outputs within the
// slit's reach only.
//
// Bound by FP64 multiply-adds (about 56 TFLOP/s here; the FP64 matrix products
// of a Toeplitz form ran at 43).  With the taps reversed,
//   out[i] = sum_m h[m] x[i + m],  x[q] = in[q + c - k + 1],
// a lane takes R consecutive outputs and walks the taps in groups of R: 2 R
// inputs in registers give R^2 products, and the next group needs R new ones
// (an earlier form with a tap and an input read from LDS for every product
// spent more on the reads and conversions than on the sums).  The inputs lie
// transposed in LDS (element e at row e % R, column e / R), so the lanes'
// reads are consecutive; the taps are read as broadcasts.  The waves of a
// workgroup take the same 64 R outputs and a share of the taps each, and add
// their sums at the end.  (Few taps on a long grid: k_slit_short below.)
#pragma once

#define SLIT_KCH 2048  // slit taps per LDS chunk

template <int R, int NW>
struct SlitTile {
  static constexpr int T = 64 * NW, OUT = 64 * R;
  static constexpr int COLS = 64 + SLIT_KCH / R + 1;          // columns of the input window
  static constexpr int S = COLS + (COLS % 2 == 0 ? 5 : 4);     // odd row stride
  static constexpr int RED = NW * R * 65 * 8, STAGE = SLIT_KCH * 8 + R * S * 4;
  static constexpr int LDS = RED > STAGE ? RED : STAGE;
};

template <int R, int NW>
__global__ __launch_bounds__(64 * NW) void k_slit_conv(const float* __restrict__ in, long long n,
                                                       const float* __restrict__ slit, int k, double scale,
                                                       float* __restrict__ out) {
  using Tile = SlitTile<R, NW>;
  constexpr int S = Tile::S, T = Tile::T;
  __shared__ __align__(16) char lds[Tile::LDS];
  double* const s_h = reinterpret_cast<double*>(lds);               // [SLIT_KCH]
  float* const s_x = reinterpret_cast<float*>(lds + SLIT_KCH * 8);  // [R][S]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long o0 = (long long)blockIdx.x * Tile::OUT;
  const long long x0 = o0 + (k - 1) / 2 - (k - 1);  // in[] index of x[o0]
  double acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.0;
  for (int m0 = 0; m0 < k; m0 += SLIT_KCH) {
    const int kc = k - m0 < SLIT_KCH ? k - m0 : SLIT_KCH;
    if (m0) __syncthreads();  // the previous chunk has been consumed
    for (int m = threadIdx.x; m < kc; m += T) s_h[m] = (double)slit[k - 1 - (m0 + m)];
    for (int e = threadIdx.x; e < Tile::OUT + kc - 1; e += T) {
      const long long q = x0 + m0 + e;
      s_x[(e % R) * S + e / R] = (q >= 0 && q < n) ? in[q] : 0.0f;
    }
    __syncthreads();
    // whole groups of R taps, a contiguous share per wave
    const int groups = kc / R, per = (groups + NW - 1) / NW;
    const int g0 = wave * per, g1 = g0 + per < groups ? g0 + per : groups;
    auto column = [&](int g, double (&v)[R]) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = (double)s_x[r * S + lane + g];
    };
    // taps of group g over the columns lo (g) and hi (g + 1)
    auto products = [&](int g, const double (&lo)[R], const double (&hi)[R]) {
#pragma unroll
      for (int m = 0; m < R; m += 2) {
        const double2 h = *reinterpret_cast<const double2*>(s_h + g * R + m);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = __builtin_fma(h.x, r + m < R ? lo[r + m] : hi[r + m - R], acc[r]);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = __builtin_fma(h.y, r + m + 1 < R ? lo[r + m + 1] : hi[r + m + 1 - R], acc[r]);
      }
    };
    double a[R], b[R];
    if (g0 < g1) column(g0, a);
    for (int g = g0; g < g1; g += 2) {
      column(g + 1, b);
      products(g, a, b);
      if (g + 1 == g1) break;
      column(g + 2, a);
      products(g + 1, b, a);
    }
    // the remaining taps, one each for the last waves in turn
    for (int m = groups * R + (NW - 1 - wave); m < kc; m += NW) {
      const double h = s_h[m];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int e = r + m;
        acc[r] = __builtin_fma(h, (double)s_x[(e % R) * S + lane + e / R], acc[r]);
      }
    }
  }
  // the waves' sums: output lane * R + r of wave w at [w][r][lane], rows of 65
  __syncthreads();
  double* const red = reinterpret_cast<double*>(lds);
#pragma unroll
  for (int r = 0; r < R; ++r) red[(wave * R + r) * 65 + lane] = acc[r];
  __syncthreads();
  for (int e = threadIdx.x; e < Tile::OUT; e += T) {
    if (o0 + e >= n) break;
    const double* p = red + (e % R) * 65 + e / R;
    double s = p[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += p[w * R * 65];
    out[o0 + e] = (float)(s * scale);
  }
}

// Slits of up to SLIT_SHORT taps on long grids: bound by the bytes, which the
// tiles above pass through LDS twice more (the waves' sums).  A workgroup takes
// SLIT_SHORT_OUT consecutive outputs, a lane one of each quarter: consecutive
// inputs per read, the taps as broadcasts.  8 M points, 9 taps 35.1 (SlitTile<8, 4>)
// -> 17.4 us (the copy alone is 14), 21 taps 40.9 -> 23.2, 33 taps 40.4 -> 28.1.
#define SLIT_SHORT 48
#define SLIT_SHORT_OUT 1024

__global__ __launch_bounds__(256) void k_slit_short(const float* __restrict__ in, long long n,
                                                    const float* __restrict__ slit, int k, double scale,
                                                    float* __restrict__ out) {
  __shared__ float s_x[SLIT_SHORT_OUT + SLIT_SHORT];
  __shared__ double s_h[SLIT_SHORT];
  const long long o0 = (long long)blockIdx.x * SLIT_SHORT_OUT;
  const long long x0 = o0 + (k - 1) / 2 - (k - 1);  // in[] index of the first output's first input
  if ((int)threadIdx.x < k) s_h[threadIdx.x] = (double)slit[k - 1 - threadIdx.x];
  for (int e = threadIdx.x; e < SLIT_SHORT_OUT + k - 1; e += 256) {
    const long long q = x0 + e;
    s_x[e] = (q >= 0 && q < n) ? in[q] : 0.0f;
  }
  __syncthreads();
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int m = 0; m < k; ++m) {
    const double h = s_h[m];
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = __builtin_fma(h, (double)s_x[threadIdx.x + 256 * r + m], acc[r]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const long long o = o0 + threadIdx.x + 256 * r;
    if (o < n) out[o] = (float)(acc[r] * scale);
  }
}
