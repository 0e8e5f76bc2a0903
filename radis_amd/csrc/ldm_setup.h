// Set-up kernels: FFT twiddle tables, and for the no-allocation entry point
// the job table and work items of one request written into its scratch
// buffer (no host copies, so the sequence is also capturable).
#pragma once
#include "ldm_fft.h"
#include "ldm_plan.h"

// Element i of the twiddle tables of one size set: W_n1^e (e < n1), W_n2^e
// (e < n2) and the two-level W_L table: hi[q] = W_L^((q * 1024) mod L),
// q < ceil(L / 1024), then lo[e] = W_L^e, e < 1024.  W_N^e = exp(-2 pi i e / N),
// evaluated as sincospi(-2 e / N) in FP64 and rounded to FP32 (the W_L table of
// the compiled passes stays FP64: twl64).  Null tables are skipped.
struct LdmTwiddles {
  float2 *tw1, *tw2;
  void* twl;
  int n1, n2;
  long long L;
  bool twl64;
  __host__ __device__ long long nhi() const { return (L + (1 << LDM_TW_LO_BITS) - 1) >> LDM_TW_LO_BITS; }
  __host__ __device__ long long total() const {
    return (tw1 ? n1 : 0) + (tw2 ? n2 : 0) + (twl ? nhi() + (1 << LDM_TW_LO_BITS) : 0);
  }
  __device__ void put(long long k) const {
    float2* dst = nullptr;
    double e, N;
    if (tw1 && k < n1) {
      dst = tw1 + k; e = (double)k; N = (double)n1;
    } else {
      if (tw1) k -= n1;
      if (tw2 && k < n2) {
        dst = tw2 + k; e = (double)k; N = (double)n2;
      } else {
        if (tw2) k -= n2;
        if (!twl64) dst = (float2*)twl + k;
        N = (double)L;
        e = k < nhi() ? (double)((k << LDM_TW_LO_BITS) % L) : (double)(k - nhi());
      }
    }
    double sn, cs;
    sincospi(-2.0 * e / N, &sn, &cs);
    if (dst) *dst = make_float2((float)cs, (float)sn);
    else ((double2*)twl)[k] = make_double2(cs, sn);
  }
};

// The tables of a batch layout, a row of workgroups each (one launch: a launch
// per table, up to 13 of a few hundred elements, was 40 us of a served batch's
// set-up, which waits for them).
#define LDM_TW_TABLES 32
struct LdmTwiddleSet {
  LdmTwiddles t[LDM_TW_TABLES];
};
__global__ __launch_bounds__(256) void k_twiddles(LdmTwiddleSet set) {
  const LdmTwiddles& t = set.t[blockIdx.y];
  const long long total = t.total();
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x)
    t.put(i);
}

// Everything the no-allocation entry point writes into its scratch array before
// the pipeline: the job table (passed by value, a kernel argument, so a captured
// launch holds its own copy) by workgroup 0, then the request's work items, the
// image correction's W table and the passes' tables, one element per thread.
// One launch: as four, each a few hundred elements, they took 9 of 61 us of a
// 20,001-point request.
__global__ __launch_bounds__(256) void k_setup(LdmJob job, LdmJob* __restrict__ dst, LdmItemPlan P,
                                               int4* __restrict__ items, int n_items, LdmTwiddles wrap, LdmTwiddles t) {
  static_assert(sizeof(LdmJob) % 4 == 0, "job table copied as 32-bit words");
  if (blockIdx.x == 0) {
    const unsigned* s = (const unsigned*)&job;
    unsigned* d = (unsigned*)dst;
    for (int w = threadIdx.x; w < (int)(sizeof(LdmJob) / 4); w += blockDim.x) d[w] = s[w];
    return;
  }
  long long i = (blockIdx.x - 1) * 256ll + threadIdx.x;
  if (i < n_items) {
    items[i] = plan_item(P, (int)i);
    return;
  }
  if ((i -= n_items) < wrap.total()) wrap.put(i);
  else if ((i -= wrap.total()) < t.total()) t.put(i);
}

// The first `rows` LDM rows of a request de-interleaved into dst[rows][cols]
// (the LDM stores rows 2p and 2p+1 interleaved; a diagnostic copy; zeros where
// the fill wrote none).
__global__ __launch_bounds__(256) void k_copy_ldm(const LdmJob* __restrict__ job, const LdmAxes* __restrict__ axes,
                                                  int rows, long long cols, float* __restrict__ dst) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)rows * cols) return;
  const int r = (int)(i / cols);
  const long long n = i - (long long)r * cols;
  const PairColumns written(*job, *axes, r >> 1);
  dst[i] = written((int)n) ? job->ldm[(long long)(r >> 1) * 2 * job->ldm_stride + 2 * n + (r & 1)] : 0.0f;
}
