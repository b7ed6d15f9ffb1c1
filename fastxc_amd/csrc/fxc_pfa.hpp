// Prime-factor (Good-Thomas) transforms of n = product of pairwise coprime
// radices, in LDS (device code).
//
// With index k placed at (k mod R_p)_p on the axes of the mixed-radix layout
// and t at the digits b_p of t = sum_p (n / R_p) b_p mod n, exp(+-2 pi i k t/n)
// is the product over the axes of exp(+-2 pi i (k mod R_p) b_p / R_p): the
// transform is one R_p-point DFT per axis, without twiddles, from either
// placement to the other.
//
// The 23- and 29-point DFTs run on the fp32 matrix instructions.  Folding legs
// m and R - m into t_m = a_m + a_{R-m} and u_m = a_m - a_{R-m} leaves two real
// products, cos [q][m] t_m and sin [q][m] u_m with q, m <= (R-1)/2 < 16, for
// the real and the imaginary part: four 16 x 16 x 16 products per 16
// butterflies.  On the vector ALU the same butterflies take about 28 and 33
// operations per point and hold 2 R registers, which left one or two waves per
// SIMD; here they hold 24, and their multiply-adds run beside the vector work
// of other waves.
#pragma once

#include "fxc_fft_device.hpp"

namespace fxc {

typedef float pfa_f32x4 __attribute__((ext_vector_type(4)));

template <int R>
__device__ const RootTable<R> kPfaRoots{};

// A lane's share of the cos and sin matrices of one radix: entry [lane mod 16]
// [4 s + lane / 16], zero outside q, m <= (R-1)/2.
struct PfaLane {
  float c[4], s[4];
};
template <int R>
__device__ __forceinline__ PfaLane pfa_lane() {
  constexpr int H = (R - 1) / 2;
  const int lane = threadIdx.x & 63, q = lane & 15;
  PfaLane l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = 4 * i + (lane >> 4);
    const bool in = q <= H && m <= H;
    l.c[i] = in ? kPfaRoots<R>.c[m * q % R] : 0.f;
    l.s[i] = in ? kPfaRoots<R>.s[m * q % R] : 0.f;
  }
  return l;
}
struct PfaLanes {
  PfaLane r23, r29;
};
__device__ __forceinline__ PfaLanes pfa_lanes(const FftPlanDev &plan) {
  PfaLanes l{};
  for (int p = 0; p < plan.npass; ++p) {
    if (plan.radix[p] == 23) l.r23 = pfa_lane<23>();
    if (plan.radix[p] == 29) l.r29 = pfa_lane<29>();
  }
  return l;
}

// Offset of butterfly b of axis p (of ntrans transforms of plan.n values).
template <int R, bool kLast>
__device__ __forceinline__ int pfa_offset(int b, int ntrans, const FftPlanDev &plan, int p) {
  if constexpr (kLast) return b * R;  // stride 1, and rows are whole multiples of R
  const int nbt = plan.n / R, stride = plan.stride[p];
  const int t = ntrans > 1 ? (int)udiv_magic((unsigned)b, (unsigned)nbt, plan.bmagic[p]) : 0;
  const int r = b - t * nbt;
  const int blk = (int)udiv_magic((unsigned)r, (unsigned)stride, plan.smagic[p]);
  return t * plan.n + blk * plan.span[p] + (r - blk * stride);
}

// DFTs along one axis.  kLast: the last axis, whose values are adjacent, so
// the legs' offsets are constants.
template <int R, bool kLast>
__device__ __forceinline__ void pfa_pass(float2 *buf, int ntrans, const FftPlanDev &plan, int p,
                                         float sgn) {
  const int stride = kLast ? 1 : plan.stride[p];
  const int total = ntrans * (plan.n / R);
  for (int b = threadIdx.x; b < total; b += blockDim.x) {
    float2 *base = buf + pfa_offset<R, kLast>(b, ntrans, plan, p);
    float2 v[R];
#pragma unroll
    for (int m = 0; m < R; ++m) v[m] = base[m * stride];
    dft<R>(v, sgn);
#pragma unroll
    for (int q = 0; q < R; ++q) base[q * stride] = v[q];
  }
  __syncthreads();
}

// The same for R = 23 and 29 on the matrix instructions: a wave takes 16
// butterflies at a time, lane l legs 4 s + l / 16 (and their mirrors) of
// butterfly l mod 16, and holds outputs 4 (l / 16) + r (and their mirrors).
template <int R, bool kLast>
__device__ __forceinline__ void pfa_pass_mfma(float2 *buf, int ntrans, const FftPlanDev &plan,
                                              int p, float sgn, const PfaLane &w) {
  constexpr int H = (R - 1) / 2;
  static_assert((R & 1) == 1 && H < 16, "one 16 x 16 tile holds the folded DFT");
  const int stride = kLast ? 1 : plan.stride[p];
  const int total = ntrans * (plan.n / R);
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwaves = blockDim.x >> 6;
  for (int b0 = wave * 16; b0 < total; b0 += nwaves * 16) {
    const int b = b0 + (lane & 15);
    // past the last butterfly: the last one again, not stored
    float2 *base = buf + pfa_offset<R, kLast>(b < total ? b : total - 1, ntrans, plan, p);
    float2 t[4], u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = 4 * i + g;
      // legs past H stay inside the butterfly; their matrix entries are zero,
      // and so must they be (a non-finite value would not vanish)
      const float2 x = base[m * stride];
      const float2 y = base[(m ? R - m : 0) * stride];
      t[i] = m == 0 ? x : cadd(x, y);
      u[i] = csub(x, y);
      if (4 * i + 3 > H && m > H) t[i] = u[i] = make_float2(0.f, 0.f);
    }
    pfa_f32x4 cr = {0.f, 0.f, 0.f, 0.f}, ci = cr, sr = cr, si = cr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      cr = __builtin_amdgcn_mfma_f32_16x16x4f32(w.c[i], t[i].x, cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f32_16x16x4f32(w.c[i], t[i].y, ci, 0, 0, 0);
      sr = __builtin_amdgcn_mfma_f32_16x16x4f32(w.s[i], u[i].x, sr, 0, 0, 0);
      si = __builtin_amdgcn_mfma_f32_16x16x4f32(w.s[i], u[i].y, si, 0, 0, 0);
    }
    if (b < total) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int q = 4 * g + r;
        if (q > H) continue;
        base[q * stride] = make_float2(cr[r] - sgn * si[r], ci[r] + sgn * sr[r]);
        if (q > 0) base[(R - q) * stride] = make_float2(cr[r] + sgn * si[r], ci[r] - sgn * sr[r]);
      }
    }
  }
  __syncthreads();
}

// Every axis of ntrans transforms; the caller synchronises before, the call
// ends with a barrier.
__device__ __forceinline__ void lds_pfa(float2 *buf, int ntrans, const FftPlanDev &plan, float sgn,
                                        const PfaLanes &w) {
  for (int p = 0; p < plan.npass; ++p) {
    const bool last = p == plan.npass - 1;
    switch (plan.radix[p]) {
#define FXC_PFA(R)                                    \
  case R:                                             \
    if (last)                                         \
      pfa_pass<R, true>(buf, ntrans, plan, p, sgn);   \
    else                                              \
      pfa_pass<R, false>(buf, ntrans, plan, p, sgn);  \
    break;
#define FXC_PFA_MFMA(R)                                          \
  case R:                                                        \
    if (last)                                                    \
      pfa_pass_mfma<R, true>(buf, ntrans, plan, p, sgn, w.r##R);  \
    else                                                         \
      pfa_pass_mfma<R, false>(buf, ntrans, plan, p, sgn, w.r##R); \
    break;
      FXC_PFA(2) FXC_PFA(3) FXC_PFA(4) FXC_PFA(5) FXC_PFA(7) FXC_PFA_MFMA(23) FXC_PFA_MFMA(29)
#undef FXC_PFA
#undef FXC_PFA_MFMA
      default: break;
    }
  }
}

// Plan and device tables of a length (cached per device, freed by
// fxc_release_plans): map[i] = k | t << 16 of position i, tpos[t] = i, phase[q]
// = exp(-2 pi i q / n).
struct PfaTables {
  FftPlanDev plan{};
  unsigned *d_map = nullptr;
  unsigned *d_tpos = nullptr;
  float2 *d_phase = nullptr;
};
// Whether n is a product of distinct radices among 2 or 4, 3, 5, 7, 23 and 29
// (one axis each, small butterflies first): few lengths, of the odd ones from 201
// to 4001 these 12: 203, 345, 435, 483, 609, 667, 805, 1015, 2001, 2415, 3045,
// 3335.  Axes of 8, 9, 16 and 25, and the primes 11 to 19 and 31, whose folded
// form fits the matrix pass, are not tried; other lengths keep the kernels of
// fxc_stack_fft.hpp's transforms.
bool pfa_length(int n);
int pfa_tables(int n, PfaTables *out, bool create = true);
void pfa_release();

}  // namespace fxc
