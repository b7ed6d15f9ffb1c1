// Phase-weighted stack (ncf_pws hot path): replaces compute_pws_host_batch
// (native/pws/worker/gpu.cu:87-282).  Per pair, with group means x_g [n]:
//   a_g = analytic signal of x_g (bins 1 .. ceil(n/2)-1 doubled, the rest 0),
//   phi_g = a_g / max(|a_g|, 1e-7),  W = sum_g w_g phi_g,  out = lin |W|^power.
//
// MI355X design.  The real part of a_g is x_g without its bin 0 (and, for even
// n, bin n/2); only its imaginary part, the Hilbert transform, needs transforms,
// and that is a real-to-real map.  Two rows therefore share one complex row,
// z = s0 x_0 + i s1 x_1, whose spectrum is multiplied by -i sgn(k) in place, in
// the forward transform's digit-reversed order, and transformed back by the
// pass order that consumes it (s0, s1: pow2_scale): one forward and one inverse transform per two
// rows, in one LDS row, with no spectrum in HBM.  Lengths of coprime axes
// (2001 = 3 x 23 x 29) take both transforms without twiddles and their large
// primes on the matrix instructions (fxc_pfa.hpp).  Rows of other lengths
// (Bluestein plans) are convolved with the Hilbert kernel directly: also two
// transforms, of the convolution length, where a Bluestein transform each way
// takes four.
//
// Bound: VALU and LDS latency of the transforms (2 x n points per two rows);
// rows are read once.  The form it replaced transformed one and a half complex
// rows per row, through an HBM workspace of 8 n bytes per row that each call
// allocated: 6000 pairs of up to 30 rows of 2001 (145 000 rows) 3.5 ms of
// kernels and about 50 ms of allocation.
#include "fxc_pfa.hpp"
#include "fxc_stack_fft.hpp"

#include <algorithm>

namespace fxc {

constexpr int kPwsMaxLen = 8192;
constexpr float kSumScale = 0x1p-14f;  // of a row's sums (exact)

// How a length's Hilbert transforms run: mixed-radix passes, convolution
// (Bluestein lengths), or axes of coprime radices without twiddles.
enum PwsForm { kPwsMixed, kPwsConv, kPwsAxes };

constexpr int pws_waves(int form, int per) { return per > 8 ? 2 : form == kPwsAxes ? 4 : 3; }

// One workgroup per pair and split: split s of nsplit takes the pair's row
// pairs [s T / nsplit, (s+1) T / nsplit), kBatch at a time.  Thread t owns the
// samples t + k kThreads of every row, so rows stay in registers from their
// load to their phase and W needs no exchange.  A batch with a non-finite value
// transforms its rows one by one, so such a value stays in its own row.
// Mixed radix: three waves per SIMD (168 registers), 2.38 ms for the call of
// 6000 pairs against 2.61 at two waves and 3.45 at four, whose 128 registers
// spill; reading the rows again instead of holding them took 4.06.  Axes: 1.64.
// nsplit 1 writes the stack, otherwise the partial W to part [pair][split][n].
template <int kThreads, int kPer, int kBatch, int kForm>
__global__ void __launch_bounds__(kThreads, pws_waves(kForm, kPer))
pws_kernel(const float *__restrict__ x, const float *__restrict__ weights,
           const long long *__restrict__ offsets, const float *__restrict__ lin, StackFftDev F,
           const float2 *__restrict__ tw_f, const float2 *__restrict__ tw_i,
           const unsigned *__restrict__ map, const unsigned *__restrict__ tpos, int nsplit,
           float power, float2 *__restrict__ part, float *__restrict__ out) {
  extern __shared__ float2 lds[];
  constexpr bool kBlue = kForm == kPwsConv, kAxes = kForm == kPwsAxes;
  constexpr int kWaves = kThreads / 64;
  __shared__ float red[2][2 * kBatch][kWaves];   // per row and wave: max |x|; sums (Bluestein)
  __shared__ float alt[2 * kBatch][kWaves];      // alternating sums (Bluestein, even n)
  __shared__ float2 dc[kBatch], ny[kBatch];      // bins 0 and n/2 of the complex rows
  __shared__ int bad;
  const int n = F.n, ld = F.ld, tid = threadIdx.x;
  float2 *buf = lds;                             // [kBatch][ld]
  float2 *twl = buf + (size_t)kBatch * ld;
  if constexpr (!kAxes) stage_stack_tw(twl, F, tw_f, tw_i);
  const int pair = blockIdx.x / nsplit, split = blockIdx.x - pair * nsplit;
  const long long g0 = offsets[pair], g1 = offsets[pair + 1];
  const long long T = (g1 - g0 + 1) / 2;         // row pairs
  const long long t_end = (split + 1) * T / nsplit;
  const int half = (n + 1) / 2;
  const bool even = (n & 1) == 0;
  const float invn = 1.f / (float)n;
  float2 W[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) W[k] = make_float2(0.f, 0.f);
  // mixed radix: the digit-reversed positions of the bins this thread
  // multiplies; axes: the positions of its samples, and the signs of the bins
  // at its positions (bit k of neg: negative frequency, of off: bin 0 or n/2)
  int pos[kPer];
  unsigned neg = 0, off = 0;
  PfaLanes lanes;
  if constexpr (kAxes) lanes = pfa_lanes(F.fwd);
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int f = tid + k * kThreads;
    pos[k] = 0;
    if constexpr (kForm == kPwsMixed)
      if (f < n) pos[k] = fft_pos(F.fwd, f);
    if constexpr (kAxes)
      if (f < n) {
        pos[k] = (int)tpos[f];
        const int q = (int)(map[f] & 0xffffu);
        if (q >= half) neg |= 1u << k;
        if (q == 0 || (even && q == n / 2)) off |= 1u << k;
      }
  }
  if (tid == 0) bad = 0;
  for (long long t0 = split * T / nsplit; t0 < t_end; t0 += kBatch) {
    const int nt = (int)min((long long)kBatch, t_end - t0);
    float2 xs[kBatch][kPer];
#pragma unroll
    for (int t = 0; t < kBatch; ++t) {
      const long long r = g0 + 2 * (t0 + t);
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int j = tid + k * kThreads;
        xs[t][k] = make_float2(0.f, 0.f);
        if (t < nt && j < n) {
          xs[t][k].x = stream_load(x + r * n + j);
          if (r + 1 < g1) xs[t][k].y = stream_load(x + (r + 1) * n + j);
        }
      }
    }
    __syncthreads();  // the previous batch is done with the reductions and bad
    bool nonfinite = false;
#pragma unroll
    for (int t = 0; t < kBatch; ++t) {
      float2 mx = make_float2(0.f, 0.f), sm = mx, sa = mx;
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const float2 v = xs[t][k];
        mx.x = fmaxf(mx.x, fabsf(v.x));
        mx.y = fmaxf(mx.y, fabsf(v.y));
        nonfinite |= !isfinite(v.x) || !isfinite(v.y);
        if constexpr (kBlue) {
          // (kPwsMaxLen times any finite value stays finite)
          const float s = (tid + k * kThreads) & 1 ? -kSumScale : kSumScale;
          sm.x += v.x * kSumScale;
          sm.y += v.y * kSumScale;
          sa.x += s * v.x;
          sa.y += s * v.y;
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        mx.x = fmaxf(mx.x, __shfl_down(mx.x, off));
        mx.y = fmaxf(mx.y, __shfl_down(mx.y, off));
        if constexpr (kBlue) {
          sm.x += __shfl_down(sm.x, off);
          sm.y += __shfl_down(sm.y, off);
          sa.x += __shfl_down(sa.x, off);
          sa.y += __shfl_down(sa.y, off);
        }
      }
      if ((tid & 63) == 0) {
        red[0][2 * t][tid >> 6] = mx.x;
        red[0][2 * t + 1][tid >> 6] = mx.y;
        if constexpr (kBlue) {
          red[1][2 * t][tid >> 6] = sm.x;
          red[1][2 * t + 1][tid >> 6] = sm.y;
          alt[2 * t][tid >> 6] = sa.x;
          alt[2 * t + 1][tid >> 6] = sa.y;
        }
      }
    }
    if (nonfinite) bad = 1;
    __syncthreads();
    const bool alone = bad != 0;
    for (int h = 0; h < (alone ? 2 : 1); ++h) {
      const bool use0 = !alone || h == 0, use1 = !alone || h == 1;
#pragma unroll
      for (int t = 0; t < kBatch; ++t) {
        if (t >= nt) break;
        float m0 = 0.f, m1 = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          m0 = fmaxf(m0, red[0][2 * t][w]);
          m1 = fmaxf(m1, red[0][2 * t + 1][w]);
        }
        const float s0 = pow2_scale(m0), s1 = pow2_scale(m1);
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          const int j = tid + k * kThreads;
          if (j < n)
            buf[t * ld + (kAxes ? pos[k] : j)] = make_float2(use0 ? xs[t][k].x * s0 : 0.f, use1 ? xs[t][k].y * s1 : 0.f);
        }
        if constexpr (kBlue)
          for (int j = n + tid; j < ld; j += kThreads) buf[t * ld + j] = make_float2(0.f, 0.f);
      }
      __syncthreads();
      const float2 *twi = twl + kTwFine + F.fwd.ncoarse;
      if constexpr (kAxes)
        lds_pfa(buf, nt, F.fwd, -1.f, lanes);
      else
        lds_fft<kRadixAll>(buf, nt, F.fwd, twl, -1.f);
      if constexpr (kAxes) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          const int i = tid + k * kThreads;
          if (i >= n) continue;
          const float s = (neg >> k) & 1 ? -1.f : 1.f;
          const bool zero = (off >> k) & 1;
          for (int t = 0; t < nt; ++t) {
            const float2 z = buf[t * ld + i];
            if (zero) (i == 0 ? dc : ny)[t] = z;  // bin 0 sits at position 0
            // -i s z
            buf[t * ld + i] = zero ? make_float2(0.f, 0.f) : make_float2(s * z.y, -s * z.x);
          }
        }
      } else if constexpr (kBlue) {
        for (int i = tid; i < ld; i += kThreads) {
          const float2 c = F.hhat[i];
          for (int t = 0; t < nt; ++t) buf[t * ld + i] = cmul(buf[t * ld + i], c);
        }
      } else {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          const int f = tid + k * kThreads;
          if (f >= n) continue;
          const bool zero = f == 0 || (even && f == n / 2);
          const float s = f < half ? 1.f : -1.f;
          for (int t = 0; t < nt; ++t) {
            const float2 z = buf[t * ld + pos[k]];
            if (f == 0) dc[t] = z;
            if (even && f == n / 2) ny[t] = z;
            // -i s z
            buf[t * ld + pos[k]] = zero ? make_float2(0.f, 0.f) : make_float2(s * z.y, -s * z.x);
          }
        }
      }
      __syncthreads();
      if constexpr (kAxes)
        lds_pfa(buf, nt, F.fwd, 1.f, lanes);
      else
        lds_fft_dit<kRadixAll>(buf, nt, F.inv, twi, 1.f);
#pragma unroll
      for (int t = 0; t < kBatch; ++t) {
        if (t >= nt) break;
        float m0 = 0.f, m1 = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          m0 = fmaxf(m0, red[0][2 * t][w]);
          m1 = fmaxf(m1, red[0][2 * t + 1][w]);
        }
        const float u0 = pow2_unscale(m0), u1 = pow2_unscale(m1);
        // mean and n/2 component of both rows
        float2 mean, nyq = make_float2(0.f, 0.f);
        if constexpr (kBlue) {
          float2 a = make_float2(0.f, 0.f), b = a;
#pragma unroll
          for (int w = 0; w < kWaves; ++w) {
            a.x += red[1][2 * t][w];
            a.y += red[1][2 * t + 1][w];
            b.x += alt[2 * t][w];
            b.y += alt[2 * t + 1][w];
          }
          constexpr float up = 1.f / kSumScale;
          mean = make_float2(a.x * invn * up, a.y * invn * up);
          if (even) nyq = make_float2(b.x * invn * up, b.y * invn * up);
        } else {
          mean = make_float2(dc[t].x * (u0 * invn), dc[t].y * (u1 * invn));
          if (even) nyq = make_float2(ny[t].x * (u0 * invn), ny[t].y * (u1 * invn));
        }
        // the convolution kernel carries 1/n already
        const float v0 = kBlue ? u0 : u0 * invn, v1 = kBlue ? u1 : u1 * invn;
        const long long r = g0 + 2 * (t0 + t);
        const float w0 = use0 ? weights[r] : 0.f;
        const float w1 = use1 && r + 1 < g1 ? weights[r + 1] : 0.f;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          const int j = tid + k * kThreads;
          if (j >= n) continue;
          const float2 z = buf[t * ld + (kAxes ? pos[k] : j)];
          const float s = even && (j & 1) ? -1.f : 1.f;
          float2 acc = W[k];
          auto add = [&](float re, float im, float w) {
            // w a / max(|a|, 1e-7): the reciprocal root is correct to an ulp;
            // |a| <= 1e-7 divides by 1e-7
            const float m2 = re * re + im * im;
            const float q = m2 > 1e-14f ? w * __builtin_amdgcn_rsqf(m2) : w * 1e7f;
            acc.x += re * q;
            acc.y += im * q;
          };
          if (use0) add(xs[t][k].x - mean.x - s * nyq.x, z.x * v0, w0);
          if (use1 && r + 1 < g1) add(xs[t][k].y - mean.y - s * nyq.y, z.y * v1, w1);
          W[k] = acc;
        }
      }
      __syncthreads();
    }
    if (tid == 0) bad = 0;
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int j = tid + k * kThreads;
    if (j >= n) continue;
    if (nsplit == 1) {
      const size_t o = (size_t)pair * n + j;
      out[o] = lin[o] * mag_pow(W[k].x * W[k].x + W[k].y * W[k].y, power);
    } else {
      part[(size_t)blockIdx.x * n + j] = W[k];
    }
  }
}

// Sums the splits' W in split order and forms the stack.
__global__ void __launch_bounds__(256)
pws_join_kernel(const float2 *__restrict__ part, const float *__restrict__ lin, int n, int nsplit,
                float power, float *__restrict__ out) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= n) return;
  const size_t pair = blockIdx.y;
  float2 w = make_float2(0.f, 0.f);
  for (int s = 0; s < nsplit; ++s) w = cadd(w, part[(pair * nsplit + s) * n + j]);
  const size_t o = pair * n + j;
  out[o] = lin[o] * mag_pow(w.x * w.x + w.y * w.y, power);
}

// Workgroups per pair: with fewer pairs than the device holds workgroups (four
// per CU) the rows of each pair are split, into at most the pairs' mean row
// count, so that the partial sums never exceed n complex values per row.
static int pws_splits(const long long *off, int npairs) {
  return (int)std::max(1ll, std::min(1024ll / npairs, off[npairs] / npairs));
}

size_t pws_scratch_bytes(const long long *h_off, int npairs, int n) {
  const int s = pws_splits(h_off, npairs);
  return s > 1 ? (size_t)npairs * s * n * sizeof(float2) : 0;
}

int pws_prepare(int n) {
  PfaTables t;
  return pfa_length(n) ? pfa_tables(n, &t) : FXC_OK;
}

int pws_check(const StackFft &S) {
  FXC_CHECK_ARG((size_t)S.dev.ld + S.twc + kLdsReserve <= (size_t)kLdsComplexCapacity,
                "fxc_pws: length %d too long for the LDS transforms", S.dev.n);
  FXC_CHECK_ARG(S.dev.n <= kPwsMaxLen, "fxc_pws: length %d too long", S.dev.n);
  return FXC_OK;
}

namespace {
struct PwsArgs {
  StackFftDev F;
  const float2 *tw_f, *tw_i;
  int form, twc;
  PfaTables axes;
  const float *pre, *weights;
  const long long *off;
  const float *lin;
  int npairs, nsplit;
  float power;
  float2 *part;
  float *out;
};

template <int kThreads, int kPer, int kBatch, bool kAxes = false>
int pws_launch(const PwsArgs &a, hipStream_t st) {
  auto *k = pws_kernel<kThreads, kPer, kBatch, kAxes ? kPwsAxes : kPwsMixed>;
  if constexpr (!kAxes)
    if (a.form == kPwsConv) k = pws_kernel<kThreads, kPer, kBatch, kPwsConv>;
  const size_t lds = ((size_t)kBatch * a.F.ld + a.twc) * sizeof(float2);
  FXC_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds));
  hipLaunchKernelGGL(k, dim3((unsigned)a.npairs * (unsigned)a.nsplit), dim3(kThreads), lds, st,
                     a.pre, a.weights, a.off, a.lin, a.F, a.tw_f, a.tw_i, a.axes.d_map,
                     a.axes.d_tpos, a.nsplit, a.power, a.part, a.out);
  FXC_HIP(hipGetLastError());
  return FXC_OK;
}
}  // namespace

int pws_run(const StackFft &S, const float *d_pre, const float *d_weights, const long long *h_off,
            const long long *d_off, const float *d_linear, int npairs, int n, float power,
            float2 *d_scratch, float *d_out, hipStream_t st, bool create) {
  FXC_TRY(pws_check(S));
  PwsArgs a{S.dev, S.tw_f, S.tw_i, S.dev.blue ? kPwsConv : kPwsMixed, S.twc, {}, d_pre, d_weights,
            d_off, d_linear, npairs, pws_splits(h_off, npairs), power, d_scratch, d_out};
  if (pfa_length(n)) {
    FXC_TRY(pfa_tables(n, &a.axes, create));
    a.form = kPwsAxes;
    a.F.fwd = a.axes.plan;
    a.twc = 0;
  }
  // Row pairs per batch: as many as keep a thread's rows within 32 registers,
  // so that the large-radix passes (n / 29 butterflies per row) have work for
  // the workgroup's waves; one in the axes form, whose matrix passes need only
  // 16 butterflies per wave and which four waves per SIMD serve better (2001:
  // 1.41 ms of 6000 pairs against 1.46 at two row pairs and three waves).
  const bool two = 2 * (size_t)S.dev.ld + S.twc + kLdsReserve <= (size_t)kLdsComplexCapacity;
  if (a.form == kPwsAxes) {
    if (n <= 512)
      FXC_TRY((pws_launch<256, 2, 4, true>(a, st)));
    else if (n <= 2048)
      FXC_TRY((pws_launch<256, 8, 1, true>(a, st)));
    else if (n <= 4096)
      FXC_TRY((pws_launch<512, 8, 1, true>(a, st)));
    else
      FXC_TRY((pws_launch<512, 16, 1, true>(a, st)));
  } else if (n <= 512) {
    FXC_TRY((pws_launch<256, 2, 4>(a, st)));
  } else if (n <= 2048) {
    FXC_TRY((pws_launch<256, 8, 2>(a, st)));
  } else if (n <= 4096 && two) {
    FXC_TRY((pws_launch<512, 8, 2>(a, st)));
  } else {
    FXC_TRY((pws_launch<512, 16, 1>(a, st)));
  }
  if (a.nsplit > 1) {
    hipLaunchKernelGGL(pws_join_kernel, dim3((unsigned)ceil_div((size_t)n, 256), (unsigned)npairs),
                       dim3(256), 0, st, d_scratch, d_linear, n, a.nsplit, power, d_out);
    FXC_HIP(hipGetLastError());
  }
  return FXC_OK;
}

}  // namespace fxc
