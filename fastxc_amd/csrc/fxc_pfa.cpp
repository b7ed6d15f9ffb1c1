#include "fxc_pfa.hpp"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <vector>

namespace fxc {

namespace {
std::mutex g_mu;
std::map<std::pair<int, int>, PfaTables> g_tables;  // (device, n)

int upload(void **dst, const void *src, size_t bytes) {
  FXC_TRY(dmalloc(dst, bytes));
  FXC_HIP(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
  return FXC_OK;
}

void free_tables(PfaTables &t) {
  dfree(t.d_map);
  dfree(t.d_tpos);
  dfree(t.d_phase);
}
}  // namespace

static bool pfa_plan(int n, FftPlanDev *plan) {
  FftPlanDev d{};
  if (n < 2 || n >= (1 << 16)) return false;
  d.n = n;
  int m = n;
  const int prime[] = {2, 3, 5, 7, 23, 29}, most[] = {4, 3, 5, 7, 23, 29};
  for (int i = 0; i < 6; ++i) {
    int r = 1;
    while (m % prime[i] == 0) {
      r *= prime[i];
      m /= prime[i];
    }
    if (r > most[i]) return false;
    if (r > 1) d.radix[d.npass++] = r;
  }
  if (m != 1) return false;
  std::sort(d.radix, d.radix + d.npass);
  auto magic = [](int v) -> unsigned {
    return v <= 1 ? 0u : (unsigned)(((1ull << 32) + (unsigned long long)v - 1) / (unsigned long long)v);
  };
  int span = n;
  for (int p = 0; p < d.npass; ++p) {
    d.span[p] = span;
    d.stride[p] = span / d.radix[p];
    d.smagic[p] = magic(d.stride[p]);
    d.bmagic[p] = magic(n / d.radix[p]);
    span = d.stride[p];
  }
  *plan = d;
  return true;
}

bool pfa_length(int n) {
  FftPlanDev d;
  return pfa_plan(n, &d);
}

int pfa_tables(int n, PfaTables *out, bool create) {
  FftPlanDev p;
  FXC_CHECK_ARG(pfa_plan(n, &p), "length %d is not a product of coprime axes", n);
  int dev = 0;
  FXC_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_mu);
  auto it = g_tables.find({dev, n});
  if (it != g_tables.end()) {
    *out = it->second;
    return FXC_OK;
  }
  FXC_CHECK_ARG(create, "index tables of length %d are not prepared on device %d", n, dev);
  std::vector<unsigned> map((size_t)n, 0u), tpos((size_t)n, 0u);
  std::vector<float2> phase((size_t)n);
  for (int k = 0; k < n; ++k) {  // k at (k mod R_p)_p
    int i = 0;
    for (int a = 0; a < p.npass; ++a) i += (k % p.radix[a]) * p.stride[a];
    map[(size_t)i] |= (unsigned)k;
    const double w = -2.0 * M_PI * (double)k / (double)n;
    phase[(size_t)k] = make_float2((float)std::cos(w), (float)std::sin(w));
  }
  for (int i = 0; i < n; ++i) {  // t = sum (n / R_p) b_p, b_p the digits of i
    long long t = 0;
    int r = i;
    for (int a = 0; a < p.npass; ++a) {
      const int b = r / p.stride[a];
      r -= b * p.stride[a];
      t += (long long)(n / p.radix[a]) * b;
    }
    map[(size_t)i] |= (unsigned)(t % n) << 16;
    tpos[(size_t)(t % n)] = (unsigned)i;
  }
  PfaTables t;
  t.plan = p;
  int rc = upload((void **)&t.d_map, map.data(), map.size() * sizeof(unsigned));
  if (rc == FXC_OK) rc = upload((void **)&t.d_tpos, tpos.data(), tpos.size() * sizeof(unsigned));
  if (rc == FXC_OK) rc = upload((void **)&t.d_phase, phase.data(), phase.size() * sizeof(float2));
  if (rc != FXC_OK) {
    free_tables(t);
    return rc;
  }
  g_tables[{dev, n}] = t;
  *out = t;
  return FXC_OK;
}

void pfa_release() {
  std::lock_guard<std::mutex> lk(g_mu);
  for (auto &kv : g_tables) free_tables(kv.second);
  g_tables.clear();
}

}  // namespace fxc
