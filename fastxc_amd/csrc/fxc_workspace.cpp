#include "fxc_workspace.hpp"

#include <algorithm>
#include <mutex>
#include <vector>

namespace fxc {

namespace {
struct Block {
  unsigned char *ptr;
  size_t bytes;
  int dev;
};
std::mutex g_mu;
std::vector<Block> g_idle;
}  // namespace

int Workspace::acquire(size_t bytes) {
  FXC_HIP(hipGetDevice(&dev_));
  // powers of two from 64 KiB, so calls of nearby sizes reuse one block
  size_t want = (size_t)64 << 10;
  while (want < bytes && want < kWsBlock) want *= 2;
  want = std::max(want, bytes);
  {
    std::lock_guard<std::mutex> lk(g_mu);
    auto best = g_idle.end();
    for (auto it = g_idle.begin(); it != g_idle.end(); ++it)
      if (it->dev == dev_ && it->bytes >= bytes && (best == g_idle.end() || it->bytes < best->bytes))
        best = it;
    if (best != g_idle.end()) {
      ptr_ = best->ptr;
      bytes_ = best->bytes;
      g_idle.erase(best);
      return FXC_OK;
    }
  }
  int rc = dmalloc((void **)&ptr_, want);
  if (rc != FXC_OK) {  // the device may be full of idle blocks
    (void)hipGetLastError();
    workspace_release();
    want = bytes;
    rc = dmalloc((void **)&ptr_, want);
  }
  if (rc == FXC_OK) bytes_ = want;
  return rc;
}

Workspace::~Workspace() {
  if (!ptr_) return;
  if (idle_ && bytes_ <= kWsBlock) {
    std::lock_guard<std::mutex> lk(g_mu);
    size_t held = bytes_;
    for (const Block &b : g_idle)
      if (b.dev == dev_) held += b.bytes;
    if (held <= kWsIdle) {
      g_idle.push_back({ptr_, bytes_, dev_});
      return;
    }
  }
  dfree(ptr_);
}

void workspace_release() {
  std::vector<Block> all;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    all.swap(g_idle);
  }
  for (const Block &b : all) dfree(b.ptr);
}

}  // namespace fxc
