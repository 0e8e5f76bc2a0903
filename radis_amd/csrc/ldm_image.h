// Half-length transforms: RADIS's spectrum, the convolution at period 2 N_v
// (radis/lbl/broadening.py:1900-1902, 2340-2346), from passes that run at a
// period L' just above N_v.
//
// A kernel periodised at L' takes LDM column k' to output j through
// P_L'(j - k').  With N_v < L' < 2 N_v the wanted P_2Nv differs from it by
//   c(d) = P_2Nv(d) - P_L'(d),  |d| <= N_v,
// the images at +-L', +-2 N_v, ...: every one at least D = L' - N_v grid steps
// from any output, so c is smooth at the scale of D and the sum
//   y_j += (1 / wstep) sum_k' c(j - k') x_k'
// goes through a coarse description of both sides.  With gamma the HWHM of
// the row's L-axis node in grid steps, a = 2 pi gamma / L,
//   P_L(d) = (1/L) sinh(a) / (cosh(a) - cos(2 pi d / L))
// (the Fourier series of the periodised Lorentzian); the row's Gaussian enters
// through its variance, c -> c + (sigma^2 / 2) c''.  Rows of one L-axis node
// share c, so they are summed before it (each with its 1/F(0), as RADIS
// divides the folded template by its value at x = 0).
//
//   TileMoments   (fill launch, the tile still in LDS) four moments of every
//                 tile and L-axis node: the sums of x times 1, u,
//                 (u^2 + sigma^2) / 2 and (u^3 + 3 u sigma^2) / 6, u from the
//                 tile's centre (the Taylor terms of c at it)
//   image_item    (first workgroups of the pass B launch, one per cell of
//                 cell_tiles tiles) the cell's moments to IMG_NODES Chebyshev
//                 nodes, c between them and every cell's nodes, summed over the
//                 L-axis nodes, added to img_u
//   pass C        adds the cells' Chebyshev interpolants to the spectrum
//
// c is formed in FP64 from one fraction (the two periods agree to many digits
// near d = 0), and the cells' contributions to a node are summed in FP64 (in
// any order: the FP32 value they round to does not depend on it, as for the
// fill's sums); everything else is FP32: it is a small part of the spectrum.
#pragma once
#include "ldm_fft.h"

struct WrapNode {
  double omE, omE2, E;  // 1 - e^-a, 1 - e^-2a, e^-a for the period's a = 2 pi gamma / period
};

__device__ __forceinline__ WrapNode wrap_node(double gamma, double period) {
  const double a = 6.283185307179586 * gamma / period;
  WrapNode w;
  w.omE = -expm1(-a);
  w.omE2 = -expm1(-2.0 * a);
  w.E = exp(-a);
  return w;
}

// Barrier that orders LDS only: __syncthreads() would also wait for the
// global loads and stores in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The value of lane i ^ X of this lane's row of 16 (X = 7: the half-row mirror).
template <int X>
__device__ __forceinline__ float lane_xor(float v) {
  constexpr int ctrl = X == 1 ? 0xB1 : X == 2 ? 0x4E : X == 7 ? 0x141 : 0x128;  // quad_perm, row_half_mirror, row_ror:8
  static_assert(X == 1 || X == 2 || X == 7 || X == 8, "one DPP move");
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true));
}

// Sums of eight values over groups of n lanes (8, 16, 32 or 64): lane i ends
// with the sum of v[i & 7].  Halving the values at each of the first three
// steps takes 7 additions for them instead of 24.
__device__ __forceinline__ float lane_sums(const float (&v)[8], int n) {
  const int lane = threadIdx.x;
  float a[4], b[2], c;
#pragma unroll
  for (int i = 0; i < 4; ++i) a[i] = ((lane & 4) ? v[i + 4] : v[i]) + lane_xor<7>((lane & 4) ? v[i] : v[i + 4]);
#pragma unroll
  for (int i = 0; i < 2; ++i) b[i] = ((lane & 2) ? a[i + 2] : a[i]) + lane_xor<2>((lane & 2) ? a[i] : a[i + 2]);
  c = ((lane & 1) ? b[1] : b[0]) + lane_xor<1>((lane & 1) ? b[0] : b[1]);
  if (n > 8) c += lane_xor<8>(c);
  if (n > 16) c += __shfl_xor(c, 16);
  if (n > 32) c += __shfl_xor(c, 32);
  return c;
}

// A row's values for the moments: 1/F(0) and sigma^2.
__device__ __forceinline__ float2 tile_row(const LdmJob& J, int r) {
  // row_a = (pi FWHM_G)^2 / (4 ln 2) = 2 pi^2 sigma^2 (cm-2)
  const float s2 = (float)(1.0 / (19.739208802178716 * J.wstep * J.wstep));
  return make_float2(gld(J.row_inv_f0, 4u * (unsigned)r), s2 * gld(J.row_a, 4u * (unsigned)r));
}

// The moments of a fill tile.  The flush hands in what it writes: pair() takes
// two columns (c, c + 1) of the rows 2p and 2p + 1 and sums them over the
// lanes that hold the pair's columns; nodes(), behind a barrier, adds the rows
// of each L-axis node.
struct TileMoments {
  float2* rows;   // [M]
  float4* red;    // [parts][M + 1]
  int M, W;
  float mid;
  __device__ __forceinline__ TileMoments(double* behind, int M_, int W_) : M(M_), W(W_), mid(0.5f * (float)(W_ - 1)) {
    char* p = reinterpret_cast<char*>(behind);
    p += (16 - (reinterpret_cast<unsigned long long>(p) & 15)) & 15;
    rows = reinterpret_cast<float2*>(p);
    red = reinterpret_cast<float4*>(p + ((8 * M + 15) & ~15));
  }
  __device__ __forceinline__ void pair(int p, int c, float a0, float a1, float b0, float b1) {
    const float u = (float)c - mid, w = u + 1.0f;
    const float u2 = 0.5f * u * u, w2 = 0.5f * w * w, u3 = u * u2 * (1.0f / 3.0f), w3 = w * w2 * (1.0f / 3.0f);
    const float v[8] = {a0 + a1, u * a0 + w * a1, u2 * a0 + w2 * a1, u3 * a0 + w3 * a1,
                        b0 + b1, u * b0 + w * b1, u2 * b0 + w2 * b1, u3 * b0 + w3 * b1};
    const int n = W < 128 ? W >> 1 : 64;
    const float s = lane_sums(v, n);
    if ((threadIdx.x & (n - 1)) < 8) {
      float* dst = reinterpret_cast<float*>(red + (c >> 7) * (M + 1) + 2 * p);
      dst[threadIdx.x & 7] = s;
    }
  }
  // (the rows of G-axis nodes [l0, l1]: the others hold zeros)
  __device__ __forceinline__ void nodes(const LdmJob& J, int l0, int l1, int nl, int tile) {
    typedef float v4f __attribute__((ext_vector_type(4)));
    const int m = threadIdx.x, parts = tile_parts(W);
    if (m >= nl) return;  // N_L <= LDM_MAX_AX < LDM_FILL_T
    v4f v = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int part = 0; part < parts; ++part) {
      const float4* x = red + part * (M + 1) + m;
#pragma unroll 4
      for (int l = l0; l <= l1; ++l) {
        const float2 q = rows[l * nl + m];
        const float4 d = x[l * nl];
        const float hs = 0.5f * q.y;
        v += q.x * v4f{d.x, d.y, d.z + hs * d.x, d.w + hs * d.y};
      }
    }
    *(gptr<v4f>)((char*)J.mom + 16u * (unsigned)(tile * nl + m)) = v;
  }
};

// LDS bytes of one image item
constexpr int IMG_LDS = LDM_MAX_AX * 48 + FC_T_B * IMG_NODES * 4 + 2 * LDM_MAX_AX * IMG_NODES * 4;

// One cell's sources onto the nodes [IMG_TARGETS part, IMG_TARGETS (part + 1)),
// by FC_T_B threads.
__device__ __noinline__ void image_item(const LdmJob& J, const LdmAxes& A, int cell, int part, char* lds) {
  typedef float v4f __attribute__((ext_vector_type(4)));
  const int nl = A.nl, tid = threadIdx.x;
  if (J.status || nl == 0) return;
  double* cs = reinterpret_cast<double*>(lds);  // [nl][6]: per period (1 - E)^2, 4 E, (1 - E^2) / L
  float* qp = reinterpret_cast<float*>(lds + LDM_MAX_AX * 48);
  float* q = qp + FC_T_B * IMG_NODES;  // [nl][IMG_NODES] Chebyshev moments
  float* S = q + LDM_MAX_AX * IMG_NODES;  // [nl][IMG_NODES] node sources
  const int T = J.cell_tiles, W = J.tile_w, h = T * W;
  const int t0 = cell * T, t1 = t0 + T < J.n_tiles ? t0 + T : J.n_tiles;
  const double Ls = (double)J.wrap_ls, Lp = (double)J.tL;
  if (tid < nl) {
    const double gamma = exp(A.laL[tid]) * (0.5 / J.wstep);
    const WrapNode s = wrap_node(gamma, Ls), p = wrap_node(gamma, Lp);
    double* c = cs + 6 * tid;
    c[0] = s.omE * s.omE; c[1] = 4.0 * s.E; c[2] = s.omE2 / Ls;
    c[3] = p.omE * p.omE; c[4] = 4.0 * p.E; c[5] = p.omE2 / Lp;
  }
  // the tiles' moments in the cell's Chebyshev polynomials: with u the tile's
  // centre in [-1, 1], sum over q of mu_q T_k^(q)(u) / hw^q
  const int slices = FC_T_B / nl, m = tid % nl, sl = tid / nl;
  if (sl < slices) {
    float Q[IMG_NODES];
#pragma unroll
    for (int k = 0; k < IMG_NODES; ++k) Q[k] = 0.0f;
    const float ihw = 2.0f / (float)h;
#pragma unroll 2
    for (int t = t0 + sl; t < t1; t += slices) {
      const unsigned o = 16u * (unsigned)(t * nl + m);
      const v4f mu = *(gptr<const v4f>)((const char*)J.mom + o);
      const float m0 = mu.x, m1 = mu.y * ihw, m2 = mu.z * (ihw * ihw), m3 = mu.w * (ihw * ihw * ihw);
      const float u = (float)(2 * (t - t0) + 1 - T) / (float)T;
      float a0 = 1.0f, a1 = u, d0 = 0.0f, d1 = 1.0f, e0 = 0.0f, e1 = 0.0f, g0 = 0.0f,
            g1 = 0.0f;  // T and its derivatives of k - 1 and k
      Q[0] += m0;
      Q[1] += m0 * u + m1;
#pragma unroll
      for (int k = 2; k < IMG_NODES; ++k) {
        const float a2 = 2.0f * u * a1 - a0, d2 = 2.0f * a1 + 2.0f * u * d1 - d0, e2 = 4.0f * d1 + 2.0f * u * e1 - e0,
                    g2 = 6.0f * e1 + 2.0f * u * g1 - g0;
        a0 = a1; a1 = a2; d0 = d1; d1 = d2; e0 = e1; e1 = e2; g0 = g1; g1 = g2;
        Q[k] += m0 * a2 + m1 * d2 + m2 * e2 + m3 * g2;
      }
    }
#pragma unroll
    for (int k = 0; k < IMG_NODES; ++k) qp[(sl * nl + m) * IMG_NODES + k] = Q[k];
  }
  __syncthreads();
  for (int e = tid; e < nl * IMG_NODES; e += FC_T_B) {
    float v = 0.0f;
    for (int s = 0; s < slices; ++s) v += qp[s * nl * IMG_NODES + e];
    q[e] = v;
  }
  __syncthreads();
  // onto the nodes cos(pi (2 i + 1) / 16): the Lagrange basis' weights
  for (int e = tid; e < nl * IMG_NODES; e += FC_T_B) {
    const int i = e & (IMG_NODES - 1);
    const float* p = q + (e - i);
    float v = 0.5f * p[0];
#pragma unroll
    for (int k = 1; k < IMG_NODES; ++k) v += cospif((float)(k * (2 * i + 1)) * (0.5f / IMG_NODES)) * p[k];
    S[e] = v * (2.0f / IMG_NODES);
  }
  __syncthreads();
  // eight lanes (source nodes) per target, R targets per thread
  constexpr int STEP = FC_T_B / IMG_NODES, R = IMG_TARGETS / STEP;
  const int i = tid & (IMG_NODES - 1), a0 = part * IMG_TARGETS + tid / IMG_NODES, n_tgt = J.n_cell * IMG_NODES;
  const double hw = 0.5 * (double)h;
  auto node = [&](int c, int k) {
    return (double)(c * h) + 0.5 * (double)(h - 1) + hw * cospi((double)(2 * k + 1) * (0.5 / IMG_NODES));
  };
  const double xi = node(cell, i), xk = node(0, a0 & (IMG_NODES - 1));  // STEP is a multiple of IMG_NODES
  const double iLs = 1.0 / Ls, iLp = 1.0 / Lp;
  double s2s[R], s2p[R];
  float v[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const double d = xk + (double)(((a0 + j * STEP) / IMG_NODES) * h) - xi;
    const double ss = sinpi(d * iLs), sp = sinpi(d * iLp);
    s2s[j] = ss * ss;
    s2p[j] = sp * sp;
    v[j] = 0.0f;
  }
  for (int mm = 0; mm < nl; ++mm) {
    const double* c = cs + 6 * mm;
    const float w = S[mm * IMG_NODES + i];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const double ds = c[0] + c[1] * s2s[j], dp = c[3] + c[4] * s2p[j];
      const double den = ds * dp, num = c[2] * dp - c[5] * ds;
      double r = __builtin_amdgcn_rcp(den);
      r = r + r * (1.0 - den * r);
      v[j] += (float)(num * r) * w;
    }
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    float x = v[j];
    x += lane_xor<7>(x);
    x += lane_xor<2>(x);
    x += lane_xor<1>(x);
    const int at = a0 + j * STEP;
    if (i == 0 && at < n_tgt) unsafeAtomicAdd(J.img_u + at, (double)x);
  }
}

// Pass C: the cells' interpolants as Chebyshev coefficients (times 1 / wstep)
// in LDS, and their value at grid point n.
struct ImageEval {
  const float* cf;
  int h, n_cell;
  float inv_h;
  __device__ __forceinline__ void load(const LdmJob& J, float* s_cf, int threads) {
    cf = s_cf;
    h = J.cell_tiles * J.tile_w;
    n_cell = J.n_cell;
    inv_h = 1.0f / (float)h;
    const float sc = (float)(1.0 / J.wstep) * (2.0f / IMG_NODES);
    const int k = threadIdx.x & (IMG_NODES - 1);  // threads: a multiple of IMG_NODES
    float w[IMG_NODES];
#pragma unroll
    for (int i = 0; i < IMG_NODES; ++i) w[i] = cospif((float)(k * (2 * i + 1)) * (0.5f / IMG_NODES)) * (k ? sc : 0.5f * sc);
    for (int e = threadIdx.x; e < n_cell * IMG_NODES; e += threads) {
      float v = 0.0f;
#pragma unroll
      for (int i = 0; i < IMG_NODES; ++i) v += w[i] * (float)glb(J.img_u)[e - k + i];
      s_cf[e] = v;
    }
  }
  __device__ __forceinline__ float operator()(int n) const {
    int c = (int)(((float)n + 0.5f) * inv_h);
    c = c < n_cell - 1 ? c : n_cell - 1;
    const float u2 = 2.0f * ((float)(2 * (n - c * h) + 1 - h) * inv_h);
    const float* a = cf + c * IMG_NODES;
    float b1 = a[IMG_NODES - 1], b2 = 0.0f;  // Clenshaw
#pragma unroll
    for (int k = IMG_NODES - 2; k > 0; --k) {
      const float b = a[k] + u2 * b1 - b2;
      b2 = b1;
      b1 = b;
    }
    return a[0] + 0.5f * u2 * b1 - b2;
  }
};
