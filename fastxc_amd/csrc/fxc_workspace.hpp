// Device workspaces of the synchronous stack calls, kept between calls.
//
// A call that returns with its stream synchronised takes its workspace here
// instead of from hipMalloc, whose cost grows with the size (a 2.6 GB
// workspace cost 50 ms of a 4 ms call).  Idle blocks of up to kWsBlock bytes
// are kept, at most kWsIdle bytes per device; larger ones are freed at the end
// of their call.  fxc_release_plans() frees the idle ones.  Every call holds
// a block of its own, so calls from several threads and on several streams
// never share one.
#pragma once

#include "fxc_common.hpp"

namespace fxc {

constexpr size_t kWsBlock = (size_t)64 << 20;
constexpr size_t kWsIdle = (size_t)128 << 20;

inline size_t align256(size_t n) { return (n + 255) / 256 * 256; }

class Workspace {
 public:
  Workspace() = default;
  Workspace(const Workspace &) = delete;
  Workspace &operator=(const Workspace &) = delete;
  ~Workspace();
  // A block of at least `bytes` on the current device.
  int acquire(size_t bytes);
  unsigned char *data() const { return ptr_; }
  // The work on the block is complete (its stream was synchronised): it may
  // be given to another call.  Without this the destructor frees it, which
  // waits for the device.
  void idle() { idle_ = true; }

 private:
  unsigned char *ptr_ = nullptr;
  size_t bytes_ = 0;
  int dev_ = 0;
  bool idle_ = false;
};

void workspace_release();

}  // namespace fxc
