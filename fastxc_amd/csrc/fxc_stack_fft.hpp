// Length-n transforms of the stacks and the helpers their kernels share.
#pragma once

#include "fxc_plan_cache.hpp"
#include "fastxc_amd.h"

namespace fxc {

constexpr int kLdsReserve = 16;    // float2 slots left for static LDS
constexpr int kVoiceChunk = 32;    // TF-PWS voices per workgroup

// Length-n transform of the stacks: the direct mixed-radix plan when n
// factors into the implemented radices (rows of n values, digit-reversed
// output), else Bluestein's convolution of length m (rows of m values,
// natural-order output).
struct StackFftDev {
  FftPlanDev fwd;              // length ld, sign -1
  FftPlanDev inv;              // length ld, sign +1
  int n, ld, blue;
  const float2 *chirp;         // [n] exp(-i pi j^2 / n) (Bluestein only)
  const float2 *bhat_f;        // [m] forward-sign convolution kernel spectrum
  const float2 *bhat_i;        // [m] inverse-sign
  const float2 *hhat;          // [m] Hilbert-transform convolution spectrum
};

struct StackFft {
  StackFftDev dev{};
  const float2 *tw_f = nullptr, *tw_i = nullptr;
  int twc = 0;                 // LDS twiddle slots of both tables
};

__device__ __forceinline__ int stack_pos(const StackFftDev &F, int k) {
  return F.blue ? k : fft_pos(F.fwd, k);
}

// twl: [fwd table | inv table]
__device__ __forceinline__ void stage_stack_tw(float2 *twl, const StackFftDev &F,
                                               const float2 *__restrict__ tw_f,
                                               const float2 *__restrict__ tw_i) {
  const int cf = kTwFine + F.fwd.ncoarse, ci = kTwFine + F.inv.ncoarse;
  for (int i = threadIdx.x; i < cf + ci; i += blockDim.x) twl[i] = i < cf ? tw_f[i] : tw_i[i - cf];
}

// In-place transforms (sgn -1 forward, +1 inverse) of nt rows at stride
// F.ld whose input is natural order in [0, n).  The caller synchronises
// before the call; the call ends with a barrier.  Output position of bin k:
// stack_pos(F, k).
__device__ __forceinline__ void stack_fft(float2 *buf, int nt, const StackFftDev &F, const float2 *twl, float sgn) {
  const float2 *twf = twl;
  const float2 *twi = twl + kTwFine + F.fwd.ncoarse;
  if (!F.blue) {
    if (sgn < 0.f)
      lds_fft<kRadixAll>(buf, nt, F.fwd, twf, -1.f);
    else
      lds_fft<kRadixAll>(buf, nt, F.inv, twi, 1.f);
    return;
  }
  const int n = F.n, m = F.ld, total = nt * m;
  const float cs = sgn < 0.f ? 1.f : -1.f;  // c_s = c_{-1} or its conjugate
  const float2 *bh = sgn < 0.f ? F.bhat_f : F.bhat_i;
  for (int i = threadIdx.x; i < total; i += blockDim.x) {
    const int j = i % m;
    float2 v = make_float2(0.f, 0.f);
    if (j < n) {
      const float2 c = F.chirp[j];
      v = cmul(buf[i], make_float2(c.x, cs * c.y));
    }
    buf[i] = v;
  }
  __syncthreads();
  lds_fft<kRadixAll>(buf, nt, F.fwd, twf, -1.f);
  for (int i = threadIdx.x; i < total; i += blockDim.x) buf[i] = cmul(buf[i], bh[i % m]);
  __syncthreads();
  lds_fft_dit<kRadixAll>(buf, nt, F.inv, twi, 1.f);
  for (int i = threadIdx.x; i < total; i += blockDim.x) {
    const int j = i % m;
    if (j < n) {
      const float2 c = F.chirp[j];
      buf[i] = cmul(buf[i], make_float2(c.x, cs * c.y));
    }
  }
  __syncthreads();
}

// stack_fft with the direction and the Bluestein choice fixed at compile
// time.  In a kernel that inlines both directions of the runtime form the
// compiler copies the plan structure into scratch memory (976 B per lane at
// the plan sizes here); with both choices fixed, the plan is indexed in the
// kernel arguments.
template <int kSgn, bool kBlue>
__device__ __forceinline__ void stack_fft_dir(float2 *buf, int nt, const StackFftDev &F,
                                              const float2 *twl) {
  if constexpr (kBlue)
    stack_fft(buf, nt, F, twl, (float)kSgn);
  else if constexpr (kSgn < 0)
    lds_fft<kRadixAll>(buf, nt, F.fwd, twl, -1.f);
  else
    lds_fft<kRadixAll>(buf, nt, F.inv, twl + kTwFine + F.fwd.ncoarse, 1.f);
}

// Row t[u] and column j[u] of flat index i0 + u step in rows of n, u < kB,
// from one division (a division per element costs a kernel that issues VALU
// most of its time several percent).
template <int kB>
__device__ __forceinline__ void flat_rows(int i0, int step, int n, int (&t)[kB], int (&j)[kB]) {
  int tt = i0 / n, jj = i0 - tt * n;
#pragma unroll
  for (int u = 0; u < kB; ++u) {
    t[u] = tt;
    j[u] = jj;
    jj += step;
    while (jj >= n) {
      jj -= n;
      ++tt;
    }
  }
}

// Scale of a row whose largest |x| is mx: a power of two that brings it into
// [1/2, 1), so that rows which share one complex transform carry its rounding
// relative to their own size and the unscaling is exact; 1 for an all-zero row
// (or a non-finite maximum).  The exponent stays within 126, where the scale and
// its reciprocal are both normal: rows beyond are brought as near as that.
__device__ __forceinline__ float pow2_scale(float mx) {
  const unsigned e = __float_as_uint(mx) >> 23;  // mx >= 0: the exponent field
  return mx == 0.f || e == 255 ? 1.f : __uint_as_float((253 - min(e, 252u)) << 23);
}
// Its inverse; 0 for an all-zero row, which then stays zero: what the transform
// leaves in its part is the rounding of the row beside it, and a phase of that is
// as large as any other.
__device__ __forceinline__ float pow2_unscale(float mx) {
  const unsigned e = __float_as_uint(mx) >> 23;
  return mx == 0.f ? 0.f : e == 255 ? 1.f : __uint_as_float((min(e, 252u) + 1) << 23);
}

// Loads of rows a kernel reads exactly once: nontemporal, so the twiddles
// and tables every workgroup reads stay in L2.
__device__ __forceinline__ float stream_load(const float *p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ float2 stream_load(const float2 *p) {
  return __builtin_bit_cast(float2, __builtin_nontemporal_load((const unsigned long long *)p));
}

// |W|^power from |W|^2: power 1 (the reference) is the square root, power 2
// the square itself, other powers powf (spec mode).
__device__ __forceinline__ float mag_pow(float mag2, float power) {
  if (power == 1.f) return sqrtf(mag2);
  if (power == 2.f) return mag2;
  return mag2 > 0.f ? powf(mag2, 0.5f * power) : 0.f;
}

// Direct plan when n factors, else the Bluestein plan.  create = false
// only looks the plans up (no device allocation).
int stack_fft_plan(int n, StackFft *S, bool create = true);

// Argument error for lengths the PWS kernels do not serve.
int pws_check(const StackFft &S);
// PWS of every pair (offsets: device copy of h_off).  scratch_bytes from
// pws_scratch_bytes; the caller synchronises.  create = false: no device
// allocation (pws_prepare ran for the length).
int pws_prepare(int n);
size_t pws_scratch_bytes(const long long *h_off, int npairs, int n);
int pws_run(const StackFft &S, const float *d_pre, const float *d_weights, const long long *h_off,
            const long long *d_off, const float *d_linear, int npairs, int n, float power,
            float2 *d_scratch, float *d_out, hipStream_t st, bool create = true);

// TF-PWS voices of lengths that are products of coprime prime powers (fxc_tfpws.hip);
// the arguments are those of the general voice kernel's launch.
bool tfpws_pfa_length(const StackFft &S);
int tfpws_pfa_run(const StackFft &S, const float2 *Ag, const float2 *Alin, const float *weights,
                  const long long *h_off, const long long *d_off, int npairs, int nrows,
                  int nbatch, int nfreq, float power, const unsigned char *active,
                  const float *gtab, float2 *spec, hipStream_t st);

}  // namespace fxc
