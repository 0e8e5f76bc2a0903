// Compile-time-sized LDS FFT and the four-step passes built on it (gfx950).
//
// The generic transform (ldm_fft.h) takes N and its radices at run time; here
// N is a template parameter, so the radix plan, every loop bound, every
// division and the LDS offsets of a butterfly's inputs and outputs are
// constants: an R-point butterfly reads and writes LDS through one base
// address plus immediate offsets.  Stage twiddles come from a table of
// W_N^e (e < N) staged in LDS once per workgroup.
//
// Plan for N = 2^a * f, f in {1, 3, 5}: the odd factor f first (no twiddles),
// then radix-16 stages, then one radix-2/4/8 stage for the remaining power
// (fc_plan: the sizes with another one).
// Columns: B = 2^bs independent columns of length N, element i of column b at
// LDS slot pad_idx(i*B + b) (the same layout as the generic transform).
#pragma once
#include <type_traits>

#include "ldm_fft.h"
#include "ldm_image.h"
#include "ldm_kernels.h"
#include "ldm_twiddle.h"

constexpr int fc_odd(int n) { return n % 3 == 0 ? 3 : (n % 5 == 0 ? 5 : 1); }
constexpr int fc_log2(int n) { return n <= 1 ? 0 : 1 + fc_log2(n >> 1); }
constexpr bool fc_pow2(int n) { return n > 0 && (n & (n - 1)) == 0; }
// Radices (hexadecimal digits, the first stage's lowest)
// of the sizes whose plan is not the general one; 0: general.  64 and 512 take
// radix-8 stages only: as many stages as 16 x 4 and 16 x 16 x 2, with every
// thread busy in each (a radix-16 stage of a 2048-element tile is 128
// butterflies on 256 threads).  Plan variant pv = 1 (pass B): it keeps its first
// and last stages' elements in registers (the next pair's prefetch; the
// accumulated spectrum and the lineshape FTs), so a radix-16 end stage over 8
// rows of 256 held 16 elements per thread on half the threads (187 VGPRs);
// radix-4 ends at 256 and radix-8 ends at 1024 hold 8 on all.
constexpr int fc_plan(int n, int pv) {
  return n == 64 ? 0x88 : n == 512 ? 0x888 : pv == 1 && n == 256 ? 0x4f4 : pv == 1 && n == 1024 ? 0x8f8 : 0;  // f: 16
}
// number of stages and radix of stage s
constexpr int fc_nstages(int n, int pv = 0) {
  if (fc_plan(n, pv)) return fc_plan(n, pv) >> 8 ? 3 : 2;
  const int f = fc_odd(n);
  const int a = fc_log2(n / f);
  return (f > 1 ? 1 : 0) + a / 4 + (a % 4 ? 1 : 0);
}
constexpr int fc_radix(int n, int s, int pv = 0) {
  if (fc_plan(n, pv)) {
    const int r = fc_plan(n, pv) >> (4 * s) & 15;
    return r == 15 ? 16 : r;
  }
  const int f = fc_odd(n);
  const int a = fc_log2(n / f);
  if (f > 1) {
    if (s == 0) return f;
    --s;
  }
  if (s < a / 4) return 16;
  return 1 << (a % 4);
}
// product of the radices before stage s
constexpr int fc_ns(int n, int s, int pv = 0) { return s == 0 ? 1 : fc_ns(n, s - 1, pv) * fc_radix(n, s - 1, pv); }
// the sizes with a compiled transform
constexpr bool fc_supported(int n) {
  const int f = fc_odd(n);
  return n % f == 0 && fc_pow2(n / f) && n / f >= 64;
}

// padded LDS offset of a constant element offset c (valid as an addition to
// pad_idx(e) when c is a multiple of 32, or when e mod 32 + c mod 32 < 32)
constexpr int pad_c(int c) { return c + ((c >> 5) << 1); }

// LDS paddings: PD = 5 is pad_idx (2 slots after every 32 elements); PD = 4
// puts 1 slot after every 16, which makes the stride-16 writes of a radix-16
// stage over one column (B = 1) conflict-free.  Both add N/16 slots.
template <int PD>
__device__ __forceinline__ int pad_e(int e) {
  return PD == 5 ? pad_idx(e) : e + (e >> 4);
}
template <int PD>
constexpr int pad_ce(int c) {
  return PD == 5 ? pad_c(c) : c + (c >> 4);
}

// Per-stage twiddle tables (fc_load_tw_stages): stage s >= 1 (radix R, NS)
// holds W^(q k), q in [1, R), k < NS, as (q-1)*NS + k; a stage with
// NS >= 64 holds only q = 1 (NS entries) and its butterflies form the
// powers W^(q k) = W^(a k) W^(b k), a + b = q, a = q/2 (products at most
// log2(R) deep).  fc_tw_off is a stage's offset in the concatenated table.
constexpr bool fc_tw_compact(int n, int s, int pv = 0) { return s > 0 && fc_ns(n, s, pv) >= 64; }
constexpr int fc_tw_size(int n, int s, int pv = 0) {
  return s == 0 ? 0 : (fc_tw_compact(n, s, pv) ? fc_ns(n, s, pv) : fc_ns(n, s, pv) * (fc_radix(n, s, pv) - 1));
}
constexpr int fc_tw_off(int n, int s, int pv = 0) {
  return s <= 1 ? 0 : fc_tw_off(n, s - 1, pv) + fc_tw_size(n, s - 1, pv);
}

// One Stockham DIT stage (see ldm_fft.h for the recursion) with compile-time
// N, radix R, Ns, B and T.  Element e = i*B + b is element i of column b.
// IN_REG: the stage's inputs come from ld(s, q, e) instead of LDS (the first
// stage, fed from registers or global memory; its LDS writes need the
// buffer free, which the caller guarantees).  OUT_REG: its outputs go to
// st(s, q, e, value) instead of LDS (the last stage; no trailing barrier).
// (s, q) = (thread pass, butterfly leg), the same for a given e in every
// call, so callers can keep per-element state in registers indexed by them.
// threadIdx.x behind an empty asm barrier: the stages' per-thread LDS and
// twiddle addresses are then computed where they are used, instead of being
// hoisted out of a caller's loop and held in registers across it
__device__ __forceinline__ int fc_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// PD: the LDS padding (pad_e).  TWO >= 0: stage twiddles from a per-stage
// table (fc_load_tw_stages) at tw[TWO + (q-1)*NS + k] (TWC: only q = 1,
// powers formed here), so lanes with consecutive k read consecutive slots;
// TWO < 0: from the W_N table at tw[q*k*N/(NS*R)], whose power-of-two
// strides put a wave's lanes on a few LDS banks when B is small.
// OOP: the stage writes obuf, a buffer other than the one it reads (buf),
// so no barrier is needed between its reads and its writes.
template <int N, int B, int T, int R, int NS, bool FWD, bool IN_REG, bool OUT_REG, bool OPQ, int PD, int TWO, bool TWC,
          bool OOP, class LD, class ST>
__device__ __forceinline__ void fc_stage_io(const float2* buf, float2* obuf, const float2* __restrict__ tw, LD& ld,
                                            ST& st) {
  const int tid = OPQ ? fc_tid() : (int)threadIdx.x;
  constexpr int NR = N / R;
  constexpr int ITEMS = NR * B;
  constexpr int IT = (ITEMS + T - 1) / T;
  constexpr int LB = fc_log2(B);
  constexpr int G = 1 << PD;  // padding group
  // read offsets q*NR*B pad linearly when NR*B is a multiple of G
  constexpr bool RD_LIN = (NR * B) % G == 0;
  // write offsets q*NS*B: linear when NS*B is a multiple of G, or when NS*B
  // divides G and the group base (j - k)*R*B is a multiple of G
  constexpr bool WR_LIN = (NS * B) % G == 0 || (G % (NS * B) == 0 && (NS * R * B) % G == 0);
  float2 v[IT][R];
#pragma unroll
  for (int s = 0; s < IT; ++s) {
    const int it = tid + s * T;
    if (ITEMS % T == 0 || it < ITEMS) {
      if constexpr (IN_REG) {
#pragma unroll
        for (int q = 0; q < R; ++q) v[s][q] = ld(s, q, it + q * NR * B);
      } else if constexpr (RD_LIN) {
        const float2* src = buf + pad_e<PD>(it);
#pragma unroll
        for (int q = 0; q < R; ++q) v[s][q] = src[pad_ce<PD>(q * NR * B)];
      } else {
#pragma unroll
        for (int q = 0; q < R; ++q) v[s][q] = buf[pad_e<PD>(it + q * NR * B)];
      }
      if constexpr (NS > 1) {
        const int j = it >> LB;
        const int k = j % NS;
        const int e = k * (N / (NS * R));
        if constexpr (TWO >= 0 && TWC) {
          float2 w[R];
          w[1] = tw[TWO + k];
#pragma unroll
          for (int q = 2; q < R; ++q) w[q] = cmul(w[q / 2], w[q - q / 2]);
#pragma unroll
          for (int q = 1; q < R; ++q) v[s][q] = FWD ? cmul(v[s][q], w[q]) : cmulc(v[s][q], w[q]);
        } else {
#pragma unroll
          for (int q = 1; q < R; ++q) {
            const float2 w = TWO >= 0 ? tw[TWO + (q - 1) * NS + k] : tw[q * e];
            v[s][q] = FWD ? cmul(v[s][q], w) : cmulc(v[s][q], w);
          }
        }
      }
      dft<R, FWD>(v[s]);
    }
  }
  // LDS inputs must all be read before any output overwrites them
  if constexpr (!IN_REG && !OUT_REG && !OOP) __syncthreads();
#pragma unroll
  for (int s = 0; s < IT; ++s) {
    const int it = tid + s * T;
    if (ITEMS % T == 0 || it < ITEMS) {
      const int j = it >> LB, b = it & (B - 1);
      const int k = j % NS;
      const int e0 = (((j - k) * R + k) << LB) + b;
      if constexpr (OUT_REG) {
#pragma unroll
        for (int q = 0; q < R; ++q) st(s, q, e0 + q * NS * B, v[s][q]);
      } else if constexpr (WR_LIN) {
        float2* dst = obuf + pad_e<PD>(e0);
#pragma unroll
        for (int q = 0; q < R; ++q) dst[pad_ce<PD>(q * NS * B)] = v[s][q];
      } else {
#pragma unroll
        for (int q = 0; q < R; ++q) obuf[pad_e<PD>(e0 + q * NS * B)] = v[s][q];
      }
    }
  }
  if constexpr (!OUT_REG) __syncthreads();
}

struct FcNone {
  __device__ float2 operator()(int, int, int) const { return make_float2(0.0f, 0.0f); }
  __device__ void operator()(int, int, int, float2) const {}
};

// Transform of the B columns in buf.  IN_REG: the first stage reads its
// inputs through ld (then calls after_first()); OUT_REG: the last stage
// hands its outputs to st (after before_last()).  A transform with both set
// touches LDS only between its stages.
// OPQ: the stages take the thread index through fc_tid() (for callers that
// run the transform inside a loop).
// PD: the LDS padding (pad_e).  TWS: tw is the per-stage twiddle table
// (fc_load_tw_stages) instead of W_N.  Ping-pong (b1 != b0): stage S writes
// b0 for even S and b1 for odd S and reads the other one, so no stage needs
// a barrier between its reads and its writes; b1 == b0: in place.
template <int N, int B, int T, bool FWD, bool IN_REG, bool OUT_REG, bool OPQ, int PD = 5, bool TWS = false,
          bool PP = false, int PV = 0, int S = 0, class LD, class ST, class AF, class BL>
__device__ __forceinline__ void fc_fft_pp(float2* b0, float2* b1, const float2* __restrict__ tw, LD& ld, ST& st,
                                          AF& after_first, BL& before_last) {
  constexpr int NST = fc_nstages(N, PV);
  if constexpr (S < NST) {
    if constexpr (S == NST - 1) before_last();
    constexpr int TWO = (TWS && S > 0) ? fc_tw_off(N, S, PV) : -1;
    float2* ib = (PP && (S & 1) == 0) ? b1 : b0;  // stage S reads what stage S-1 wrote
    float2* ob = (PP && (S & 1)) ? b1 : b0;
    fc_stage_io<N, B, T, fc_radix(N, S, PV), fc_ns(N, S, PV), FWD, IN_REG && S == 0, OUT_REG && S == NST - 1, OPQ, PD,
                TWO, fc_tw_compact(N, S, PV), PP>(ib, ob, tw, ld, st);
    if constexpr (S == 0) after_first();
    fc_fft_pp<N, B, T, FWD, IN_REG, OUT_REG, OPQ, PD, TWS, PP, PV, S + 1>(b0, b1, tw, ld, st, after_first,
                                                                          before_last);
  }
}
template <int N, int B, int T, bool FWD, bool IN_REG, bool OUT_REG, bool OPQ, int PD = 5, bool TWS = false, class LD,
          class ST, class AF, class BL>
__device__ __forceinline__ void fc_fft_io(float2* __restrict__ buf, const float2* __restrict__ tw, LD& ld, ST& st,
                                          AF& after_first, BL& before_last) {
  fc_fft_pp<N, B, T, FWD, IN_REG, OUT_REG, OPQ, PD, TWS, false>(buf, buf, tw, ld, st, after_first, before_last);
}
template <int N, int B, int T, bool FWD, bool IN_REG, bool OUT_REG, class LD, class ST, class AF>
__device__ __forceinline__ void fc_fft_io(float2* __restrict__ buf, const float2* __restrict__ tw, LD& ld, ST& st,
                                          AF& after_first) {
  auto nop = [] {};
  fc_fft_io<N, B, T, FWD, IN_REG, OUT_REG, false>(buf, tw, ld, st, after_first, nop);
}

template <int N, int B, int T, bool FWD>
__device__ __forceinline__ void fc_fft(float2* __restrict__ buf, const float2* __restrict__ tw) {
  FcNone none;
  auto nop = [] {};
  fc_fft_io<N, B, T, FWD, false, false>(buf, tw, none, none, nop);
}

// (thread pass, leg) extents of a transform's first and last stages, for
// callers that keep per-element values in registers
template <int N, int B, int T, int PV = 0>
struct FcShape {
  static constexpr int R0 = fc_radix(N, 0, PV), IT0 = (N / R0 * B + T - 1) / T;
  static constexpr int RL = fc_radix(N, fc_nstages(N, PV) - 1, PV), ITL = (N / RL * B + T - 1) / T;
  static constexpr int ITEMS0 = N / R0 * B, ITEMSL = N / RL * B;
};

// stage the forward twiddle table W_N^e, e < N, into LDS
template <int N, int T>
__device__ __forceinline__ void fc_load_tw(float2* __restrict__ s_tw, const float2* __restrict__ tw) {
#pragma unroll
  for (int e = threadIdx.x; e < N; e += T) s_tw[e] = gld(tw, 8u * (unsigned)e);
}

// Per-stage twiddle tables from the W_N table tw (global): stage
// S >= 1 (radix R, NS) holds W_N^(q k N/(NS R)) for k < NS and q in
// [1, R) (q = 1 only when fc_tw_compact) at fc_tw_off(N, S) + (q-1)*NS + k.
// The tables add up to fewer than N entries (fc_tw_off(N, fc_nstages(N))).
template <int N, int T, int PV = 0, int S = 1>
__device__ __forceinline__ void fc_load_tw_stages(float2* __restrict__ s_tw, const float2* __restrict__ tw) {
  if constexpr (S < fc_nstages(N, PV)) {
    constexpr int NS = fc_ns(N, S, PV), R = fc_radix(N, S, PV), LNS = fc_log2(NS);
    constexpr int O = fc_tw_off(N, S, PV), STEP = N / (NS * R), SZ = fc_tw_size(N, S, PV);
    static_assert(fc_pow2(NS), "stages after the first have power-of-two NS");
    for (int i = threadIdx.x; i < SZ; i += T) {
      const int q = (i >> LNS) + 1, k = i & (NS - 1);
      s_tw[O + i] = gld(tw, 8u * (unsigned)(q * k * STEP));
    }
    fc_load_tw_stages<N, T, PV, S + 1>(s_tw, tw);
  }
}

// the table halves of W_L^e (e < L) of the compiled passes
__device__ __forceinline__ void twiddle_halves(const LdmJob& J, unsigned e, double2 (&h)[2]) {
  h[0] = gld(J.twd_hi, 16u * (e >> LDM_TW_LO_BITS));
  h[1] = gld(J.twd_lo, 16u * (e & ((1u << LDM_TW_LO_BITS) - 1)));
}

// ---------------------------------------------------------------------------
// Pass A with N1 fixed (see k_fft_a): B = fc_cols_a(N1) columns per workgroup.
// ---------------------------------------------------------------------------
// Pass A reads B consecutive elements of each of a column block's N1 rows
// (stride N2); an element is the float2 of the pair's two interleaved LDM
// rows, so a row segment is 8 B bytes.  Segments of 128 B or more stream at
// close to the full HBM rate, 64 B ones at about 0.6 of it and 32 B ones at
// about 0.35, so pass A takes the widest tile that fits LDS (one
// 1024-thread workgroup per CU).
// (tile sizes FC_CAP_A, FC_CAP, FC_CAP_B and fc_cols_a / fc_cols_c /
// fc_rows_b are in ldm_job.h: the host planner sizes the work items with them)

template <int N1, int B, int T>
__global__ __launch_bounds__(T, T >= FC_T_A ? 4 : 2) void k_fft_a_c(const LdmJob* __restrict__ jobs, const LdmAxes* __restrict__ axes,
                                                   const int4* __restrict__ items, int n_items) {
  constexpr int LB = fc_log2(B), CAPE = N1 * B;
  static_assert(CAPE % T == 0 && T % B == 0, "tile is a whole number of thread passes");
  using SH = FcShape<N1, B, T>;
  constexpr int NR0 = N1 / SH::R0;
  constexpr int NSL = fc_ns(N1, fc_nstages(N1) - 1);
  __shared__ float2 buf[LdsSize<CAPE>::value];
  __shared__ float2 s_tw[N1];
  // Persistent: workgroup g takes the column blocks g', g' + G, g' + 2G, ...
  // (G = gridDim.x <= n_items).  Blocks of fewer than 32 columns take
  // g' = xcd_block(g, G): the workgroups of one XCD then take consecutive
  // blocks.  That was worth 339 -> 330 us at N1 = 640 when a 16-column
  // block read 64-B row segments; with the LDM's interleaved row pairs it
  // reads 128 B per row and the remap measures neutral.  32-column blocks
  // keep g' = g (the remap cost them 2.6 us at N1 = 512).  A block's first-stage inputs
  // sit in v; the next block's loads go into v right after the first stage
  // has consumed them, so they are in flight during the LDS stages and the
  // stores.
  float2 v[SH::IT0][SH::R0];
  // The twiddle progression's factors W^(m DS) and W^(m DQ) of the tile's B
  // columns, in LDS by the first 2 B threads: 144 rows of 600,001 points took 111
  // us with six 16-byte gathers per thread (107 from FP32 tables), so 104.
  // Not in narrow tiles, which take one block each, nor in transforms of two
  // stages, without a barrier between the write and the use.
  constexpr bool AC = T >= FC_T_A && fc_nstages(N1) > 2;
  static_assert(2 * B <= T, "a thread per column and factor");
  __shared__ double2 s_ac[AC ? 2 * B : 1];
  // issue the loads of block idx into v; false (for the whole workgroup)
  // when the block has no work
  auto fetch = [&](int idx) -> bool {
    if (idx >= n_items) return false;
    const int4 it = items[idx];
    const LdmJob& J = jobs[it.x];
    const int p = it.y;
    if (J.status || p >= axes[it.x].p) return false;
    const int N2 = J.tn2, n2_0 = it.z * B, V = (int)J.v;
    // pair p's rows, interleaved: z = (x_2p, x_2p+1) is one float2
    const float2* rz = reinterpret_cast<const float2*>(J.ldm) + (long long)p * J.ldm_stride;
    const bool has_b = (2 * p + 1) < axes[it.x].m;
    // L >= 2 N_v, so V = N_v + 1 <= L/2 unless L = 2 N_v exactly: then the
    // upper half of every column (n1 >= N1/2, n >= L/2) is zero and its
    // loads are skipped
    const bool upper_zero = (long long)V <= J.tL / 2;
    // the two LDM rows, zero beyond V and where the fill wrote none (and row b
    // zero when the pair is odd)
    const PairColumns written(J, axes[it.x], p);
    auto rows = [&](auto sparse) {
#pragma unroll
      for (int s = 0; s < SH::IT0; ++s) {
        const int it0 = threadIdx.x + s * T;
#pragma unroll
        for (int q = 0; q < SH::R0; ++q) {
          // s*(T/B) + q*NR0 is the smallest row n1 = e >> LB of this (s, q)
          if (upper_zero && s * (T >> LB) + q * NR0 >= N1 / 2) {
            v[s][q] = make_float2(0.0f, 0.0f);
            continue;
          }
          const int e = it0 + q * NR0 * B;
          const int n = n2_0 + (e & (B - 1)) + N2 * (e >> LB);
          const bool in = (SH::ITEMS0 % T == 0 || it0 < SH::ITEMS0) && n < V;
          if constexpr (decltype(sparse)::value) {
            // (lanes skipped: at one common address per pair they took longer)
            float2 z = make_float2(0.0f, 0.0f);
            if (in & written(n)) z = gld(rz, 8u * (unsigned)n);
            v[s][q] = make_float2(z.x, has_b ? z.y : 0.0f);
          } else {
            const unsigned o = in ? 8u * (unsigned)n : 0u;  // n < V < 2^28
            const float2 z = gld(rz, o);
            v[s][q] = make_float2(in ? z.x : 0.0f, (in && has_b) ? z.y : 0.0f);
          }
        }
      }
    };
    if (written.all) rows(std::false_type{});
    else rows(std::true_type{});
    return true;
  };
  // W_N1 table: the same for every request of this N1
  const int first = B < 32 ? xcd_block(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  fc_load_tw<N1, T>(s_tw, jobs[items[first].x].tw1);
  bool live = fetch(first);
  for (int idx = first; idx < n_items; idx += gridDim.x) {
    if (!live) {
      live = fetch(idx + gridDim.x);
      continue;
    }
    const int4 it = items[idx];
    const LdmJob& J = jobs[it.x];
    const int N2 = J.tn2, n2_0 = it.z * B;
    float2* Y = J.ybuf + (long long)it.y * J.tL;
    // output k1 of this thread's last-stage element (s, q): j0 + s*(T/B) + q*NS;
    // the table halves of its base (and factors) load now and are multiplied out
    // just before the last stage
    const int b = threadIdx.x & (B - 1);
    const unsigned m = n2_0 + b;
    double2 twr[AC ? 1 : 3][2], twc[2];
    twiddle_halves(J, m * (threadIdx.x >> LB), twr[0]);  // < L <= 2^21
    if constexpr (AC) {
      if (threadIdx.x < 2 * B) twiddle_halves(J, m * (threadIdx.x < B ? T >> LB : NSL), twc);
    } else {
      twiddle_halves(J, m * (T >> LB), twr[1]);
      twiddle_halves(J, m * NSL, twr[2]);
    }
    TwProg<SH::ITL, SH::RL> tw;
    auto before_last = [&] {
      if constexpr (AC) tw.set(cmul64(twr[0][0], twr[0][1]), s_ac[b], s_ac[B + b]);
      else tw.set(cmul64(twr[0][0], twr[0][1]), cmul64(twr[1][0], twr[1][1]), cmul64(twr[2][0], twr[2][1]));
    };
    auto ld = [&](int s, int q, int) -> float2 { return v[s][q]; };
    auto st = [&](int s, int q, int e, float2 z) {
      const unsigned k1 = (unsigned)e >> LB, n2 = n2_0 + (e & (B - 1));
      // byte offsets are below 8 L <= 2^24
      gst(Y, 8u * (k1 * (unsigned)N2 + n2), cmul(z, cmul(tw.ws[s], tw.wq[q])));
    };
    bool next = false;
    auto prefetch = [&] {
      if (AC && threadIdx.x < 2 * B) s_ac[threadIdx.x] = cmul64(twc[0], twc[1]);
      next = fetch(idx + gridDim.x);
    };
    // first stage from v, last stage straight to Y with the W_L twiddle
    fc_fft_io<N1, B, T, true, true, true, true>(buf, s_tw, ld, st, prefetch, before_last);
    live = next;
    // the last stage read LDS; the next block's first stage writes it
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Pass B with N2 fixed (see k_fft_b): B = FC_CAP_B / N2 rows k1 per workgroup.
// Per pair the forward transform's first stage reads the pair's block from
// registers (fetched during the previous pair) and its last stage multiplies
// by the lineshape FTs and accumulates in registers; only the accumulated
// spectrum goes through LDS into the inverse transform, whose last stage
// writes B with the W_L twiddle.  Item (job, y, z): number
// y * split_b + z, row block number / n_share, share number % n_share of its
// pairs, whose partial spectrum goes to bbuf + share_at[share] (pass C
// adds them).  The dynamic LDS (sized per
// launch) holds the rows' lineshape coefficients (n_rows_lds float4), then
// the image-correction values of the block's rows at its two corrected bins
// (2 x B x n_wh floats, n_wh >= N_L of every request with a correction).
// ---------------------------------------------------------------------------
template <int N2>
__global__ __launch_bounds__(FC_T_B, N2 >= 256 ? 4 : 2) void k_fft_b_c(const LdmJob* __restrict__ jobs,
                                                      const LdmAxes* __restrict__ axes,
                                                      const int4* __restrict__ items, int n_rows_lds, int n_wh,
                                                      const int4* __restrict__ img, int n_img) {
  constexpr int CAP = FC_CAP_B, T = FC_T_B;
  constexpr int B = fc_rows_b(N2), LB = fc_log2(B);
  static_assert(fc_pow2(N2), "pass B rows are powers of two");
  constexpr int PV = 1;  // plan variant (fc_plan)
  using SH = FcShape<N2, B, T, PV>;
  constexpr int NR0 = N2 / SH::R0;
  constexpr int NSL = fc_ns(N2, fc_nstages(N2, PV) - 1, PV);
  // Two transform buffers, used ping-pong (stage s writes one, stage s+1
  // reads it and writes the other): no stage needs a barrier between its
  // reads and its writes, and the next pair's first stage writes a buffer
  // whose last readers have passed a stage barrier.  With an even number of
  // stages the last stage reads the first stage's buffer, so the pairs
  // alternate the two roles.
  __shared__ float2 bufs[2][LdsSize<CAP>::value];
  constexpr bool SWAP = fc_nstages(N2, PV) % 2 == 0;
  __shared__ float2 s_tw[fc_tw_off(N2, fc_nstages(N2, PV), PV)];  // per-stage twiddle tables
  if ((int)blockIdx.x < n_img) {  // the cells' image corrections (half-length transforms)
    static_assert(sizeof(bufs) >= IMG_LDS, "an image item's LDS");
    const int4 c = img[blockIdx.x];
    image_item(jobs[c.x], axes[c.x], c.y, c.z, reinterpret_cast<char*>(bufs));
    return;
  }
  const int4 it = items[blockIdx.x - n_img];
  const LdmJob& J = jobs[it.x];
  if (J.status) return;
  const int N1 = J.tn1;
  const int share = it.w & 15, k1_0 = (it.w >> 4) * B;
  const int L = (int)J.tL;  // <= 2^21
  const int P = axes[it.x].p, M = axes[it.x].m;
  const int2 mine = share_pairs(J, P, share);  // this workgroup's pairs
  const int p0 = mine.x, p1 = mine.y;
  fc_load_tw_stages<N2, T, PV>(s_tw, J.tw2);
  // The rows' lineshape coefficients (a_l, b_m, 1/F(0), fold count) staged
  // in LDS.  Read from global memory they are scalar loads, and the LDS
  // waits of the transform stages then also wait for them.
  extern __shared__ float4 s_row[];
  const bool rows_lds = M <= n_rows_lds;
  if (rows_lds) {
    for (int r = threadIdx.x; r < M; r += T) {
      const unsigned o = 4u * (unsigned)r;
      s_row[r] = make_float4(gld(J.row_a, o), gld(J.row_b, o), gld(J.row_inv_f0, o), __int_as_float(gld(J.nfold, o)));
    }
  }
  __syncthreads();
  auto row_c = [&](int r) -> float4 {
    if (rows_lds) return s_row[r];
    const unsigned o = 4u * (unsigned)r;
    return make_float4(gld(J.row_a, o), gld(J.row_b, o), gld(J.row_inv_f0, o), __int_as_float(gld(J.nfold, o)));
  };
  float2 acc[SH::ITL][SH::RL];
#pragma unroll
  for (int s = 0; s < SH::ITL; ++s)
#pragma unroll
    for (int q = 0; q < SH::RL; ++q) acc[s][q] = make_float2(0.0f, 0.0f);
  // pair p's block: rows k1_0 .. k1_0+B-1 of Y_p, element e = n2*B + b
  const float2* Yb = J.ybuf + (long long)k1_0 * N2;
  float2 pre[SH::IT0][SH::R0];
  auto prefetch = [&](int p) {
    const float2* Yp = Yb + (long long)p * (long long)L;
#pragma unroll
    for (int s = 0; s < SH::IT0; ++s) {
      const int t = threadIdx.x + s * T;
      if (SH::ITEMS0 % T == 0 || t < SH::ITEMS0) {
#pragma unroll
        for (int q = 0; q < SH::R0; ++q) {
          const int e = t + q * NR0 * B;
          pre[s][q] = gld(Yp, 8u * (unsigned)((e & (B - 1)) * N2 + (e >> LB)));
        }
      }
    }
  };
  // frequencies of this thread's bins (forward last-stage element (s, q):
  // k2 = j + q*NS, j = (tid + s*T) >> LB), folded to [0, L/2]
  float xs[SH::ITL][SH::RL];
#pragma unroll
  for (int s = 0; s < SH::ITL; ++s) {
    const int t = threadIdx.x + s * T;
#pragma unroll
    for (int q = 0; q < SH::RL; ++q) {
      const int k = k1_0 + (t & (B - 1)) + N1 * (t >> LB) + q * (N1 * NSL);
      const int kk = min(k, L - k);
      xs[s][q] = (float)kk * J.inv_Lws;
    }
  }
  // Lineshape FTs of this thread's bins.  F_r(x) = exp(-a_l x^2) exp(-b_m x)
  // for row r = l*N_L + m (plus alias terms where the row folds).  The
  // Gaussian factor depends on l only and is kept per bin while consecutive
  // rows share l (refilled N_G times).  The Lorentzian factor is geometric
  // along a thread's bins: for fixed s the RL bins are kk = kk0 + i*L/RL in
  // two runs of RL/2 (below and above L/2, folded), so exp(-b x) takes one
  // exponential per run and a product per bin.  That is about 3 exponentials
  // per row and thread instead of RL*ITL.
  const int NLr = axes[it.x].nl;
  const float dlt = (float)(L / SH::RL) * J.inv_Lws;
  float u0[SH::ITL][2];
#pragma unroll
  for (int s = 0; s < SH::ITL; ++s) {
    const int t = threadIdx.x + s * T;
    const int ks = k1_0 + (t & (B - 1)) + N1 * (t >> LB);  // bin of q = 0
    u0[s][0] = (float)ks * J.inv_Lws;                    // q = 0, 1, ..., RL/2-1
    u0[s][1] = (float)(L / SH::RL - ks) * J.inv_Lws;     // q = RL-1, RL-2, ..., RL/2
  }
  // bins below the circular-image cutoff (kk < wrap_k <= N1, wrap_item): with
  // k = k1 + N1 k2 only k2 = 0 (kk = k1) and k2 = N2 - 1 (kk = N1 - k1)
  // qualify.  The first is slot (0, 0) of thread b < B (t >> LB == 0); the
  // second is slot (s, RL - 1) of the thread with t >> LB == NSL - 1.  The
  // workgroup's table values (both bins of its B rows, every L-axis node)
  // are staged in LDS here, so the pair loop reads no global memory for
  // them (a global load there would wait behind the next pair's prefetch).
  // w_lo / w_hi hold the row b of those bins (-1: none), w_s the second's s.
  float* const s_wh = reinterpret_cast<float*>(s_row + n_rows_lds);  // [2][B][n_wh]
  auto wh = [&](int c, int b, int m) -> float& { return s_wh[(c * B + b) * n_wh + m]; };
  const int WK = J.half ? 0 : J.wrap_k;
  int w_lo = -1, w_hi = -1, w_s = 0;
  if (WK) {
    const int NLw = axes[it.x].nl;
    for (int i = threadIdx.x; i < 2 * B * NLw; i += T) {
      const int c = i / (B * NLw), b = (i / NLw) % B, m = i % NLw;
      const int k1 = k1_0 + b, kk = c ? N1 - k1 : k1;
      wh(c, b, m) = kk < WK ? J.wrap_h[m * WK + kk] : 0.0f;
    }
    if ((int)threadIdx.x < B && k1_0 + (int)threadIdx.x < WK) w_lo = threadIdx.x;
#pragma unroll
    for (int s = 0; s < SH::ITL; ++s) {
      const int t = threadIdx.x + s * T;
      const int b = t & (B - 1);
      if ((t >> LB) == NSL - 1 && N1 - (k1_0 + b) < WK) { w_hi = b; w_s = s; }
    }
    __syncthreads();  // WK is the job's: uniform over the workgroup
  }
  float gcache[SH::ITL][SH::RL];
  // the L-axis node of the next row; the Gaussian factors are refilled when it
  // wraps (counted, as a division and a remainder per row are 100 instructions)
  int m_next = NLr > 0 ? (2 * p0) % NLr : 0;
  bool refill = true;
  auto gauss_fill = [&](int r) {
    const float a = row_c(r).x;
#pragma unroll
    for (int s = 0; s < SH::ITL; ++s)
#pragma unroll
      for (int q = 0; q < SH::RL; ++q) gcache[s][q] = __expf(-(a * xs[s][q] * xs[s][q]));
  };
  auto row_ft = [&](int r, float (&F)[SH::ITL][SH::RL]) {
    if (refill) gauss_fill(r);
    const int m = m_next;
    refill = ++m_next == NLr;
    if (refill) m_next = 0;
    const float4 c = row_c(r);
    const float bco = c.y;
    const float E = __expf(-bco * dlt);
#pragma unroll
    for (int s = 0; s < SH::ITL; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float H = __expf(-bco * u0[s][h]);
#pragma unroll
        for (int i = 0; i < SH::RL / 2; ++i) {
          const int q = h ? SH::RL - 1 - i : i;
          F[s][q] = gcache[s][q] * H;
          H *= E;
        }
      }
    const int nf = __float_as_int(c.w);
    if (nf > 0) {
      const float a = c.x;
#pragma unroll
      for (int s = 0; s < SH::ITL; ++s)
#pragma unroll
        for (int q = 0; q < SH::RL; ++q)
          for (int n = 1; n <= nf; ++n) {
            // the folded frequency's mirror L/2 - kk (alias terms are rare: recomputed)
            const float xr = (float)(L / 2) * J.inv_Lws - xs[s][q];
            const float xa = (n & 1) ? ((float)n * J.half_inv_ws + xr) : ((float)n * J.half_inv_ws + xs[s][q]);
            F[s][q] += __expf(-(a * xa * xa) - bco * xa);
          }
    }
    if (w_lo >= 0 || w_hi >= 0) {
      if (w_lo >= 0) F[0][0] += wh(0, w_lo, m);
      if (w_hi >= 0) {
        const float hv = wh(1, w_hi, m);
#pragma unroll
        for (int s = 0; s < SH::ITL; ++s)
          if (s == w_s) F[s][SH::RL - 1] += hv;
      }
    }
    const float f0 = c.z;
#pragma unroll
    for (int s = 0; s < SH::ITL; ++s)
#pragma unroll
      for (int q = 0; q < SH::RL; ++q) F[s][q] *= f0;
  };
  if (p1 > p0) prefetch(p0);
  for (int p = p0; p < p1; ++p) {
    const int ra = 2 * p, rb = 2 * p + 1;
    // the pair's lineshape FTs, evaluated just before the last stage that
    // uses them (they are then not live across the earlier stages)
    float fa[SH::ITL][SH::RL], fb[SH::ITL][SH::RL];
    auto lineshapes = [&] {
      row_ft(ra, fa);
      if (rb < M) {
        row_ft(rb, fb);
      } else {
#pragma unroll
        for (int s = 0; s < SH::ITL; ++s)
#pragma unroll
          for (int q = 0; q < SH::RL; ++q) fb[s][q] = 0.0f;
      }
    };
    auto ld = [&](int s, int q, int) -> float2 { return pre[s][q]; };
    auto st = [&](int s, int q, int, float2 z) {
      acc[s][q].x += z.x * fa[s][q] + z.y * fb[s][q];
      acc[s][q].y += z.y * fa[s][q] - z.x * fb[s][q];
    };
    auto next = [&] {
      if (p + 1 < p1) prefetch(p + 1);
    };
    float2* const x0 = bufs[SWAP ? (p & 1) : 0];
    float2* const x1 = bufs[SWAP ? 1 - (p & 1) : 1];
    fc_fft_pp<N2, B, T, true, true, true, false, 4, true, true, PV>(x0, x1, s_tw, ld, st, next, lineshapes);
  }
  __syncthreads();
  // the accumulated spectrum into LDS (bufs[1]), in the forward last stage's element order
#pragma unroll
  for (int s = 0; s < SH::ITL; ++s) {
    const int t = threadIdx.x + s * T;
    if (SH::ITEMSL % T == 0 || t < SH::ITEMSL) {
      const int j = t >> LB, b = t & (B - 1);
      const int k = j % NSL;
      const int e0 = (((j - k) * SH::RL + k) << LB) + b;
#pragma unroll
      for (int q = 0; q < SH::RL; ++q) bufs[1][pad_e<4>(e0 + q * NSL * B)] = acc[s][q];
    }
  }
  __syncthreads();
  float2* Bo = J.bbuf + J.share_at[share] + (long long)k1_0 * N2;
  // output n2 of this thread's last-stage element (s, q): j0 + s*(T/B) + q*NS, row k1 fixed
  TwProg<SH::ITL, SH::RL> tw;
  {
    const unsigned m = k1_0 + (threadIdx.x & (B - 1));
    double2 h[3][2];
    twiddle_halves(J, m * (threadIdx.x >> LB), h[0]);  // < L <= 2^21
    twiddle_halves(J, m * (T >> LB), h[1]);
    twiddle_halves(J, m * NSL, h[2]);
    tw.set(cmul64(h[0][0], h[0][1]), cmul64(h[1][0], h[1][1]), cmul64(h[2][0], h[2][1]));
  }
  auto st_out = [&](int s, int q, int e, float2 z) {
    const int b = e & (B - 1), n2 = e >> LB;
    gst(Bo, 8u * (unsigned)(b * N2 + n2), cmulc(z, cmul(tw.ws[s], tw.wq[q])));
  };
  FcNone none;
  auto nop = [] {};
  // first stage reads bufs[1] (ping-pong)
  fc_fft_pp<N2, B, T, false, false, true, false, 4, true, true, PV>(bufs[0], bufs[1], s_tw, none, st_out, nop, nop);
}

// ---------------------------------------------------------------------------
// Pass C with N1 fixed (see k_fft_c): first stage straight from B, last
// stage straight to the output.  SUM: B is the sum of pass B's shares.  After a
// half-length transform the image correction is added.
// ---------------------------------------------------------------------------
template <int N1, bool SUM, int B, int T>
__global__ __launch_bounds__(T, 4) void k_fft_c_c(const LdmJob* __restrict__ jobs, const int4* __restrict__ items,
                                                     int n_items) {
  constexpr int LB = fc_log2(B), CAPE = N1 * B;
  static_assert(CAPE % T == 0, "tile is a whole number of thread passes");
  __shared__ float2 buf[LdsSize<CAPE>::value];
  __shared__ float2 s_tw[N1];
  __shared__ float s_cf[IMG_MAX_CELLS * IMG_NODES];
  const int4 it = items[xcd_block(blockIdx.x, n_items)];
  const LdmJob& J = jobs[it.x];
  const int N2 = J.tn2;
  const int n2_0 = it.z * B;
  const int nv = (int)J.nv;
  if (J.status) {
#pragma unroll
    for (int s = 0; s < CAPE / T; ++s) {
      const int e = threadIdx.x + s * T;
      const int n = n2_0 + (e & (B - 1)) + N2 * (e >> LB);
      if (n < nv) gst(J.out, 4u * (unsigned)n, 0.0f);
    }
    return;
  }
  fc_load_tw<N1, T>(s_tw, J.tw1);
  const float sc = J.out_scale;
  auto nop = [] {};
  auto off = [&](int e) { return 8u * (unsigned)((e >> LB) * N2 + n2_0 + (e & (B - 1))); };  // < 8 L <= 2^24
  // the first stage's inputs, a share at a time (a share's loads in flight
  // together)
  using SH = FcShape<N1, B, T>;
  float2 v[SH::IT0][SH::R0];
  auto fetch = [&](const float2* b, bool add) {
#pragma unroll
    for (int s = 0; s < SH::IT0; ++s) {
      const int t = threadIdx.x + s * T;
      if (SH::ITEMS0 % T == 0 || t < SH::ITEMS0) {
#pragma unroll
        for (int q = 0; q < SH::R0; ++q) {
          const float2 z = gld(b, off(t + q * (N1 / SH::R0) * B));
          v[s][q] = add ? cadd(v[s][q], z) : z;
        }
      }
    }
  };
  fetch(SUM ? J.bbuf + J.share_at[0] : J.bbuf, false);
  if constexpr (SUM) {
    for (int s = 1; s < J.n_share; ++s) fetch(J.bbuf + J.share_at[s], true);
  }
  auto ld = [&](int s, int q, int) -> float2 { return v[s][q]; };
  ImageEval img{};
  const bool half = J.half != 0;
  if (half) img.load(J, s_cf, T);  // the transform's barriers lie between this and its use
  if (J.derived) {  // uniform per workgroup: the plain store path stays as lean as without the epilogue
    auto st = [&](int, int, int e, float2 z) {
      const int n = n2_0 + (e & (B - 1)) + N2 * (e >> LB);
      if (n < nv) store_derived(J, n, half ? z.x * sc + img(n) : z.x * sc);
    };
    fc_fft_io<N1, B, T, false, true, true>(buf, s_tw, ld, st, nop);
  } else {
    auto st = [&](int, int, int e, float2 z) {
      const int n = n2_0 + (e & (B - 1)) + N2 * (e >> LB);
      if (n < nv) gst(J.out, 4u * (unsigned)n, half ? z.x * sc + img(n) : z.x * sc);
    };
    fc_fft_io<N1, B, T, false, true, true>(buf, s_tw, ld, st, nop);
  }
}
