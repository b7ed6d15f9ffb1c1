// TF-PWS voices of lengths that are products of coprime prime powers (the usual
// 2001 = 3 x 23 x 29 among them); fxc_stack.hip has the other lengths.
//
// Per pair and voice f (tfpws_compute.cu:224, cuda.stransform.cu:59-198):
//   S_g(tau) = sum_c A_g[f + c] G_f(c) exp(2 pi i c tau / n),
//   out[f] = sum_tau S_lin(tau) |sum_g w_g S_g / (|S_g| n)|^power.
//
// Two identities shape the kernel.
//   * With k = f + c, S_g(tau) = exp(-2 pi i f tau / n) Y_g(tau), Y_g the
//     inverse transform of A_g[k] G_f(k - f).  The factor is common to all
//     groups, so |W| needs only the Y_g; the linear stack's voice takes the
//     factor in its sum over tau.  A_g[k] then stands still while f moves: a
//     thread keeps its bins of every row in registers for a whole chunk of
//     voices and per voice only multiplies them by the window.
//   * The transform has no twiddles (fxc_pfa.hpp), and the sum over tau takes
//     the positions in any order, so neither index map costs a reordering.
// A thread owns the same positions before and after the transform, so a voice
// takes one barrier for the rows and one per axis.
//
// Bound: latency between LDS, VALU and matrix work at four waves per SIMD.  400
// pairs x 3 groups x 1001 voices of 2001: 10.4 ms, 58 VALU operations per
// transformed point (VALU busy 46 %, matrix pipe 32 %, LDS 35 %), against 15.5
// ms and 187 for the general kernel.  With the 23- and 29-point butterflies on
// the vector ALU: 12.0 ms at four waves per SIMD (128 registers, spilling),
// 15.0 at three, where two workgroups no longer share a CU.
#include "fxc_pfa.hpp"
#include "fxc_stack_fft.hpp"

#include <algorithm>

namespace fxc {

// Voices [f0, f0 + chunk) of one pair.  rows: LDS rows; the groups go through
// them nbatch at a time, the linear stack in a row of the last batch (or alone
// after it).  kRows > 0: one batch of up to kRows rows holds every group and
// the linear stack, so their bins stay in registers; 0: they are read again
// per voice.
// map[i] = k | tau << 16 of position i.  gtab: the windows of
// tfpws_gauss_kernel, [voice][half + 1].  phase[q] = exp(-2 pi i q / n).
constexpr int kPfaMaxRows = 5;
constexpr int pfa_waves(int per) { return per > 4 ? 2 : 4; }

template <int kThreads, int kPer, int kRows>
__global__ void __launch_bounds__(kThreads, pfa_waves(kPer))
tfpws_pfa_kernel(const float2 *__restrict__ Ag, const float2 *__restrict__ Alin,
                 const float *__restrict__ weights, const long long *__restrict__ offsets,
                 FftPlanDev plan, const unsigned *__restrict__ map,
                 const float2 *__restrict__ phase, int nbatch, int nrows, int nfreq, float power,
                 const unsigned char *__restrict__ chunk_active, const float *__restrict__ gtab,
                 float2 *__restrict__ out_spec) {
  extern __shared__ float2 lds[];  // [nrows][n]
  constexpr int kWaves = kThreads / 64;
  __shared__ float2 red[2][kWaves];
  const int pair = blockIdx.y, chunk = blockIdx.x;
  if (chunk_active && !chunk_active[chunk]) return;  // uniform per workgroup
  const int n = plan.n, half = (n + 1) / 2, tid = threadIdx.x;
  const long long g0 = offsets[pair];
  const int G = (int)(offsets[pair + 1] - g0);
  const float2 *Al = Alin + (size_t)pair * n;
  const int nbat = (G + nbatch - 1) / nbatch;
  const bool lin_joins = G - (nbat - 1) * nbatch < nrows;
  const int total = nbat + (lin_joins ? 0 : 1);
  const float invn = 1.f / (float)n;
  constexpr bool kHeld = kRows > 0;
  const PfaLanes lanes = pfa_lanes(plan);
  unsigned own[kPer];  // map of the thread's positions
  int ph[kPer];        // f tau mod n
  const int f0 = chunk * kVoiceChunk, f1 = min(nfreq, f0 + kVoiceChunk);
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = tid + j * kThreads;
    own[j] = i < n ? map[i] : 0u;  // k = 0 holds no energy
    ph[j] = (int)((long long)(own[j] >> 16) * f0 % n);
  }
  auto bin = [&](int j) { return (int)(own[j] & 0xffffu); };
  auto live = [&](int j) { return bin(j) > 0 && bin(j) < half; };  // bins an analytic row holds
  float2 a[kHeld ? kRows : 1][kPer];
  if constexpr (kHeld) {  // rows 0 .. G-1: groups, row G: linear stack
#pragma unroll
    for (int row = 0; row < kRows; ++row)
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        a[row][j] = make_float2(0.f, 0.f);
        if (row <= G && live(j)) a[row][j] = (row < G ? Ag + (g0 + row) * n : Al)[bin(j)];
      }
  }
  float gw[kPer];
  auto window = [&](int f) {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int d = bin(j) - f;
      gw[j] = live(j) ? gtab[(size_t)f * (half + 1) + (d < 0 ? -d : d)] : 0.f;
    }
  };
  window(f0);
  for (int f = f0; f < f1; ++f) {
    float2 W[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) W[j] = make_float2(0.f, 0.f);
    for (int bi = 0; bi < (kHeld ? 1 : total); ++bi) {
      const int gb = bi * nbatch;
      const int nb = kHeld ? G : bi < nbat ? min(nbatch, G - gb) : 0;
      const int rows = nb + (bi == total - 1 ? 1 : 0);
      // own positions: nobody else reads them before the barrier
      if constexpr (kHeld) {
#pragma unroll
        for (int row = 0; row < kRows; ++row) {
          if (row >= rows) break;
#pragma unroll
          for (int j = 0; j < kPer; ++j) {
            const int i = tid + j * kThreads;
            if (i < n) lds[row * n + i] = cscale(a[row][j], gw[j]);
          }
        }
      } else {
        for (int row = 0; row < rows; ++row) {
          const float2 *src = row == nb ? Al : Ag + (g0 + gb + row) * n;
#pragma unroll
          for (int j = 0; j < kPer; ++j) {
            const int i = tid + j * kThreads;
            const float2 v = gw[j] != 0.f ? src[bin(j)] : make_float2(0.f, 0.f);
            if (i < n) lds[row * n + i] = cscale(v, gw[j]);
          }
        }
      }
      if (bi == total - 1 && f + 1 < f1) window(f + 1);  // in flight behind the transform
      __syncthreads();
      if (tid == 0 && bi == 0 && f > f0) {  // the previous voice's partial sums are in
        float2 s = make_float2(0.f, 0.f);
        for (int w = 0; w < kWaves; ++w) s = cadd(s, red[(f - 1) & 1][w]);
        out_spec[(size_t)pair * n + f - 1] = s;
      }
      lds_pfa(lds, rows, plan, 1.f, lanes);
      float2 rot[kPer];  // exp(-2 pi i f tau / n)
      if (bi == total - 1) {
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          rot[j] = phase[ph[j]];
          ph[j] += (int)(own[j] >> 16);
          ph[j] = ph[j] >= n ? ph[j] - n : ph[j];
        }
      }
      for (int b = 0; b < nb; ++b) {
        const float wn = weights[g0 + gb + b] * invn;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          const int i = tid + j * kThreads;
          if (i >= n) continue;
          const float2 z = lds[b * n + i];
          // w z / (|z| n), |z| <= 1e-7 divided by 1 (the bound is the largest
          // float whose root is at most 1e-7f); the reciprocal root is correct
          // to an ulp
          const float m2 = z.x * z.x + z.y * z.y;
          const float q = m2 <= 0x1.6849ba0000000p-47f ? wn : wn * __builtin_amdgcn_rsqf(m2);
          W[j].x += z.x * q;
          W[j].y += z.y * q;
        }
      }
      if (bi == total - 1) {
        float sx = 0.f, sy = 0.f;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          const int i = tid + j * kThreads;
          if (i >= n) continue;
          const float mag = mag_pow(W[j].x * W[j].x + W[j].y * W[j].y, power);
          const float2 y = cmul(lds[nb * n + i], rot[j]);
          sx += y.x * mag;
          sy += y.y * mag;
        }
        for (int off = 32; off > 0; off >>= 1) {
          sx += __shfl_down(sx, off);
          sy += __shfl_down(sy, off);
        }
        if ((tid & 63) == 0) red[f & 1][tid >> 6] = make_float2(sx, sy);
      }
    }
  }
  __syncthreads();
  if (tid == 0) {
    float2 s = make_float2(0.f, 0.f);
    for (int w = 0; w < kWaves; ++w) s = cadd(s, red[(f1 - 1) & 1][w]);
    out_spec[(size_t)pair * n + f1 - 1] = s;
  }
}

bool tfpws_pfa_length(const StackFft &S) { return pfa_length(S.dev.n); }

namespace {
struct PfaArgs {
  const float2 *Ag, *Alin;
  const float *weights;
  const long long *off;
  int npairs, nchunks, nbatch, nrows, nfreq;
  float power;
  const unsigned char *active;
  const float *gtab;
  float2 *spec;
  PfaTables t;
};

template <int kThreads, int kPer>
int pfa_launch(const StackFft &S, const PfaArgs &a, bool held, hipStream_t st) {
  auto *k = tfpws_pfa_kernel<kThreads, kPer, 0>;
  if constexpr (kPer <= 4) {
    if (held && a.nrows == 2) k = tfpws_pfa_kernel<kThreads, kPer, 2>;
    if (held && a.nrows == 3) k = tfpws_pfa_kernel<kThreads, kPer, 3>;
    if (held && a.nrows == 4) k = tfpws_pfa_kernel<kThreads, kPer, 4>;
    if (held && a.nrows == 5) k = tfpws_pfa_kernel<kThreads, kPer, 5>;
  }
  const size_t lds = (size_t)a.nrows * S.dev.n * sizeof(float2);
  FXC_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds));
  hipLaunchKernelGGL(k, dim3((unsigned)a.nchunks, (unsigned)a.npairs), dim3(kThreads), lds, st,
                     a.Ag, a.Alin, a.weights, a.off, a.t.plan, a.t.d_map, a.t.d_phase, a.nbatch,
                     a.nrows, a.nfreq, a.power, a.active, a.gtab, a.spec);
  FXC_HIP(hipGetLastError());
  return FXC_OK;
}
}  // namespace

int tfpws_pfa_run(const StackFft &S, const float2 *Ag, const float2 *Alin, const float *weights,
                  const long long *h_off, const long long *d_off, int npairs, int nrows,
                  int nbatch, int nfreq, float power, const unsigned char *active,
                  const float *gtab, float2 *spec, hipStream_t st) {
  const int n = S.dev.n;
  PfaArgs a{Ag, Alin, weights, d_off, npairs, (nfreq + kVoiceChunk - 1) / kVoiceChunk, nbatch, nrows,
            nfreq, power, active, gtab, spec, {}};
  FXC_TRY(pfa_tables(n, &a.t));
  long long most = 0;
  for (int i = 0; i < npairs; ++i) most = std::max(most, h_off[i + 1] - h_off[i]);
  // a pair's groups and linear stack in one batch: up to 5 rows of 4 bins per
  // thread (40 registers) stay held; longer lengths read the rows again per voice
  const bool held = most < nrows && most <= nbatch && nrows <= kPfaMaxRows;
  if (n <= 1024) return pfa_launch<256, 4>(S, a, held, st);
  if (n <= 2048) return pfa_launch<512, 4>(S, a, held, st);
  if (n <= 4096) return pfa_launch<512, 8>(S, a, held, st);
  return pfa_launch<512, 12>(S, a, held, st);
}

}  // namespace fxc
