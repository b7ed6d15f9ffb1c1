// Real transforms whose complex half fits one workgroup's LDS in two parts.
#pragma once

#include "fxc_fft_large.hpp"
#include "fxc_plan_cache.hpp"

#include <algorithm>
#include <cstdlib>

namespace fxc {

// ---------------------------------------------------------------------------
// Real transforms of n = 2M = 4Q samples whose M complex values exceed the LDS
// but whose Q do not (one-hour windows at 20 Hz: Q = 18000 .. 18522): a
// workgroup runs the two Q-point transforms of a row one after the other in its
// LDS and combines them, instead of four passes over HBM (pack, columns, rows,
// unfold).  The first half's result waits in natural order in a scratch row of
// the workgroup (Q complex, L2).  Bound: the LDS transforms, as for the lengths
// that fit.  1440 rows of 72000: 0.50 ms forward and 0.46 ms inverse against
// 1.55 ms each in four passes.
//
// What a caller does to every sample or bin next to a transform goes into its
// loads and stores (SampleOp, BinOp: value of element i of row `row` from the
// stored one) instead of a pass over HBM of its own.
// ---------------------------------------------------------------------------
constexpr int kHalfThreads = 1024;

// [data: Q][twiddles]
inline size_t half_lds_bytes(int Q) { return ((size_t)Q + tw_lds_count(Q)) * sizeof(float2); }

struct PlainSample {
  __device__ __forceinline__ float operator()(long long, int, float v) const { return v; }
};
struct PlainBin {
  __device__ __forceinline__ float2 operator()(long long, int, float2 v) const { return v; }
};
struct ScaledBin {
  float scale;
  __device__ __forceinline__ float2 operator()(long long, int, float2 v) const {
    return make_float2(v.x * scale, v.y * scale);
  }
};

// Forward: z[j] = x[2j] + i x[2j+1] (zero past in_len) splits into its even and
// odd elements, Z[k] = E[k] + w^k O[k] and Z[k + Q] = E[k] - w^k O[k], w =
// exp(-2 pi i / M).  Bins k and Q - k of both halves give Z at k, Q - k, Q + k
// and M - k, two mirror pairs of the unfold.
template <unsigned kMask, class SampleOp, class BinOp>
__global__ void __launch_bounds__(kHalfThreads)
half_r2c_kernel(const float *__restrict__ in, long long in_dist, int in_len, long long rows,
                float2 *__restrict__ out, long long out_dist, FftPlanDev plan,
                const float2 *__restrict__ tw, const float2 *__restrict__ twM,
                const float2 *__restrict__ half, float2 *__restrict__ scratch, SampleOp sample,
                BinOp bin) {
  extern __shared__ float2 lds[];
  const int Q = plan.n, M = 2 * Q, tid = threadIdx.x;
  float2 *twl = lds + Q;
  for (int i = tid; i < kTwFine + plan.ncoarse; i += kHalfThreads) twl[i] = tw[i];
  float2 *E = scratch + (size_t)blockIdx.x * Q;
  for (long long row = blockIdx.x; row < rows; row += gridDim.x) {
    const float *x = in + row * in_dist;
    float2 *X = out + row * out_dist;
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
      __syncthreads();  // the previous half is read
#pragma unroll 8
      for (int j = tid; j < Q; j += kHalfThreads) {
        const int a = 4 * j + 2 * part;
        lds[j] = make_float2(a < in_len ? sample(row, a, x[a]) : 0.f,
                             a + 1 < in_len ? sample(row, a + 1, x[a + 1]) : 0.f);
      }
      __syncthreads();
      lds_fft<kMask, true>(lds, 1, plan, twl, -1.f);
      if (part == 0)
        for (int k = tid; k < Q; k += kHalfThreads) E[k] = lds[fft_pos(plan, k)];
    }
    // X[k] = (a + conj b)/2 - (i/2) h_k (a - conj b) of a = Z[k], b = Z[M-k], and
    // its mirror X[M-k] = conj((a + conj b)/2) - (i/2) conj(h_k (a - conj b))
    auto unfold = [&](int k, float2 a, float2 b) {
      const float2 e = make_float2(0.5f * (a.x + b.x), 0.5f * (a.y - b.y));
      const float2 d = cmul(half[k], make_float2(0.5f * (a.x - b.x), 0.5f * (a.y + b.y)));
      X[k] = bin(row, k, make_float2(e.x + d.y, e.y - d.x));
      X[M - k] = bin(row, M - k, make_float2(e.x - d.y, -e.y - d.x));
    };
    for (int k = tid; 2 * k <= Q; k += kHalfThreads) {
      const float2 e0 = E[k], o0 = lds[fft_pos(plan, k)];
      const float2 p0 = cmul(twM[k], o0);  // w^k O[k]
      const float2 zk = cadd(e0, p0), zkq = csub(e0, p0);
      if (k == 0) {
        // Z[0] is its own mirror: X[0] and X[M] are real; so is Z[Q]
        X[0] = bin(row, 0, make_float2(zk.x + zk.y, 0.f));
        X[M] = bin(row, M, make_float2(zk.x - zk.y, 0.f));
        const float2 d = cmul(half[Q], make_float2(0.f, zkq.y));
        X[Q] = bin(row, Q, make_float2(zkq.x + d.y, -d.x));
        continue;
      }
      const float2 e1 = E[Q - k], o1 = lds[fft_pos(plan, Q - k)];
      const float2 p1 = cmul(twM[Q - k], o1);
      const float2 zq = cadd(e1, p1), zm = csub(e1, p1);  // Z[Q-k], Z[M-k]
      unfold(k, zk, zm);
      if (2 * k != Q) unfold(Q - k, zq, zkq);
    }
  }
}

// Inverse: the folded spectrum Z splits into its even and odd bins, each closed
// under the fold's mirror (2i with 2(Q-i), 2i+1 with 2(Q-1-i)+1), and
// z[n] = F_0[n] + w^n F_1[n], z[n + Q] = F_0[n] - w^n F_1[n], w = exp(2 pi i / M).
template <unsigned kMask, class BinOp>
__global__ void __launch_bounds__(kHalfThreads)
half_c2r_kernel(const float2 *__restrict__ in, long long in_dist, long long rows,
                float *__restrict__ out, long long out_dist, int out_len, double scale,
                FftPlanDev plan, const float2 *__restrict__ tw, const float2 *__restrict__ twM,
                const float2 *__restrict__ half, float2 *__restrict__ scratch, BinOp bin) {
  extern __shared__ float2 lds[];
  const int Q = plan.n, M = 2 * Q, tid = threadIdx.x;
  float2 *twl = lds + Q;
  for (int i = tid; i < kTwFine + plan.ncoarse; i += kHalfThreads) twl[i] = tw[i];
  float2 *F = scratch + (size_t)blockIdx.x * Q;
  for (long long row = blockIdx.x; row < rows; row += gridDim.x) {
    const float2 *X = in + row * in_dist;
    float *y = out + row * out_dist;
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
      __syncthreads();  // the previous half is read
      const int mir = Q - part;
#pragma unroll 4
      for (int i = tid; 2 * i <= mir; i += kHalfThreads) {
        const int k = 2 * i + part;
        const float2 a = bin(row, k, X[k]), b = bin(row, M - k, X[M - k]);
        if (k == 0) {
          lds[0] = make_float2(a.x + b.x, a.x - b.x);  // imaginary parts ignored
        } else {
          const float2 s = make_float2(a.x + b.x, a.y - b.y);
          const float2 d = cmul(half[k], make_float2(a.x - b.x, a.y + b.y));
          if (2 * i != mir) lds[mir - i] = make_float2(s.x + d.y, d.x - s.y);
          lds[i] = make_float2(s.x - d.y, s.y + d.x);
        }
      }
      __syncthreads();
      lds_fft<kMask, true>(lds, 1, plan, twl, 1.f);
      if (part == 0)
        for (int n = tid; n < Q; n += kHalfThreads) F[n] = lds[fft_pos(plan, n)];
    }
    auto put = [&](int n, float2 v) {
      if (2 * n < out_len) y[2 * n] = (float)((double)v.x * scale);
      if (2 * n + 1 < out_len) y[2 * n + 1] = (float)((double)v.y * scale);
    };
    for (int n = tid; n < Q; n += kHalfThreads) {
      const float2 f0 = F[n], p = cmul(twM[n], lds[fft_pos(plan, n)]);
      put(n, cadd(f0, p));
      put(n + Q, csub(f0, p));
    }
  }
}

// Whether a call of `rows` rows takes the halves.  A row is one workgroup's, so
// few rows leave the chip to the serial chain of two transforms, where the four
// passes spread over it.  Measured over 21 lengths from 40960 to 80640 (times of
// the halves over those of the passes, r2c / c2r):
//   Q <= 12000            1 row 0.94 / 0.91, 16 rows 0.93 / 0.92;
//   Q > 12000             1 row 1.03-1.10 / 0.98-1.04, 8 rows 1.00-1.05 / 0.96-1.02,
//                         24 rows 0.92-0.97 / 0.88-0.93;
//   Q > 17000, radix 21   (few butterflies of many registers) 1 row 1.10-1.23 /
//                         1.04-1.15, 16 rows 1.01-1.06 / 0.96-1.01, 32 rows
//                         0.92-0.99 / 0.90-0.95.
// fused: with a call's steps inside the halves and passes of their own beside the
// four (sac2spec of one channel at 20 Hz, 72000 samples): 1 row 382 against 317
// us, 12 rows 412 against 379, 16 rows 411 against 396, 24 rows 415 against 415,
// and with the multi-band running mean 16 rows 745 against 757.
// FXC_FFT_HALVES=0 or 1 overrides (tests).
inline bool half_pays(const LargeFft *p, long long rows, bool fused) {
  if (!p->pq || rows < 1) return false;
  if (const char *env = getenv("FXC_FFT_HALVES")) return atoi(env) != 0;
  if (p->pq->dev.n <= 12000) return true;
  if (fused) return rows >= 16;
  const bool r21 = p->pq->dev.n > 17000 && p->pq->dev.radix[0] == 21;
  if (p->sign > 0) return rows >= (r21 ? 16 : 1);
  return rows >= (r21 ? 24 : 12);
}

inline int half_grid(long long rows, unsigned *grid) {
  int dev = 0, ncu = 0;
  FXC_HIP(hipGetDevice(&dev));
  FXC_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  *grid = (unsigned)std::min<long long>(rows, std::max(ncu, 1));
  return FXC_OK;
}

// Launches over rows 0 .. rows-1 (rows >= 1) of plans with pq; scratch: min(rows,
// compute units) x M/2 complex.
template <class SampleOp, class BinOp>
int half_r2c(const LargeFft *p, const float *in, long long in_dist, int in_len, float2 *out,
             long long out_dist, long long rows, float2 *scratch, const SampleOp &sample,
             const BinOp &bin, hipStream_t st) {
  unsigned grid = 0;
  FXC_TRY(half_grid(rows, &grid));
  const size_t lds = half_lds_bytes(p->M / 2);
  auto k = half_r2c_kernel<kRadixSmooth, SampleOp, BinOp>;
  FXC_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds));
  hipLaunchKernelGGL(k, dim3(grid), dim3(kHalfThreads), lds, st, in, in_dist, in_len, rows, out,
                     out_dist, p->pq->dev, p->pq->d_tw, p->d_tw, p->d_half, scratch, sample, bin);
  FXC_HIP(hipGetLastError());
  return FXC_OK;
}

template <class BinOp>
int half_c2r(const LargeFft *p, const float2 *in, long long in_dist, float *out,
             long long out_dist, int out_len, long long rows, float2 *scratch, double scale,
             const BinOp &bin, hipStream_t st) {
  unsigned grid = 0;
  FXC_TRY(half_grid(rows, &grid));
  const size_t lds = half_lds_bytes(p->M / 2);
  auto k = half_c2r_kernel<kRadixSmooth, BinOp>;
  FXC_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds));
  hipLaunchKernelGGL(k, dim3(grid), dim3(kHalfThreads), lds, st, in, in_dist, rows, out, out_dist,
                     out_len, scale, p->pq->dev, p->pq->d_tw, p->d_tw, p->d_half, scratch, bin);
  FXC_HIP(hipGetLastError());
  return FXC_OK;
}

}  // namespace fxc
