// Device workspaces that stay with their owner between calls: no HIP in here, so it also
// builds for the host alone.
#pragma once
#include <algorithm>
#include <cstddef>
#include <mutex>
#include <vector>

namespace og {

// One owner's workspace (a handle's or a batch's).  Its contents last for one call.
struct Workspace {
  void* p = nullptr;
  size_t bytes = 0;
  bool busy = false;  // a call of the owner is using it
  bool kept = false;  // in the pool's list
};

// The idle workspaces of all owners, so that none of them costs another allocation its
// memory: an allocation that fails gives back every idle one and is tried again, and no
// more than `each` bytes of one owner and `total` of all are kept at any time.  Dev has
// static bool alloc(void**, size_t) and static void free(void*), the latter waiting for
// the device.  One lock; a busy workspace is touched by its owner's call alone.
template <typename Dev>
class WorkspacePool {
 public:
  WorkspacePool(size_t each, size_t total) : each_(each), total_(total) {}

  // plain allocation
  bool alloc(void** p, size_t bytes) {
    if (Dev::alloc(p, bytes)) return true;
    return release_idle() && Dev::alloc(p, bytes);
  }

  // at least `bytes` for a call of w's owner, given back with give()
  bool take(Workspace& w, size_t bytes) {
    {
      std::lock_guard<std::mutex> g(m_);
      unlist(w);
      w.busy = true;
    }
    if (w.bytes >= bytes) return true;
    clear(w);
    if (alloc(&w.p, bytes)) {
      w.bytes = bytes;
      return true;
    }
    w.p = nullptr;
    w.busy = false;
    return false;
  }

  void give(Workspace& w) {
    std::lock_guard<std::mutex> g(m_);
    w.busy = false;
    if (w.bytes == 0) return;
    bool keep = w.bytes <= each_ && held_ + w.bytes <= total_;
    if (keep) {
      try {
        idle_.push_back(&w);
        w.kept = true;
        held_ += w.bytes;
      } catch (...) {  // no host memory for the list
        keep = false;
      }
    }
    if (!keep) clear(w);
  }

  // the owner goes away
  void drop(Workspace& w) {
    std::lock_guard<std::mutex> g(m_);
    unlist(w);
    clear(w);
  }

  size_t held() {
    std::lock_guard<std::mutex> g(m_);
    return held_;
  }

 private:
  static void clear(Workspace& w) {
    if (w.p) Dev::free(w.p);
    w.p = nullptr;
    w.bytes = 0;
  }
  void unlist(Workspace& w) {
    if (!w.kept) return;
    idle_.erase(std::find(idle_.begin(), idle_.end(), &w));
    w.kept = false;
    held_ -= w.bytes;
  }
  bool release_idle() {
    std::lock_guard<std::mutex> g(m_);
    const bool any = !idle_.empty();
    for (Workspace* w : idle_) {
      w->kept = false;
      clear(*w);
    }
    idle_.clear();
    held_ = 0;
    return any;
  }

  const size_t each_, total_;
  std::mutex m_;
  std::vector<Workspace*> idle_;
  size_t held_ = 0;
};

}  // namespace og
