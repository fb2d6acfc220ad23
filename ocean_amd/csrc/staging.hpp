// Host side of a vector's upload: no HIP in here, so it also builds for the host alone.
#pragma once
#include <cstddef>
#include <thread>

namespace og {

// fill(a, b) over [0, n) in `parts` equal parts (at most kStageParts), each on a thread of
// its own but the first, and send(a, b) -> 0 or an error code in order as each is filled.
// No exception leaves: a part whose thread cannot be had is filled here.  Returns the
// first error; parts past it are filled but not sent.
constexpr int kStageParts = 4;

template <typename Fill, typename Send, typename Wait>
int stage(size_t n, int parts, Fill fill, Send send, Wait wait) {
  std::thread th[kStageParts];
  auto at = [&](int t) { return n * t / parts; };
  for (int t = 1; t < parts; ++t) {
    try {
      th[t] = std::thread(fill, at(t), at(t + 1));
    } catch (...) {  // std::system_error without a thread, std::bad_alloc without its state
    }
  }
  int rc = 0;
  for (int t = 0; t < parts; ++t) {
    if (th[t].joinable()) th[t].join();
    else fill(at(t), at(t + 1));
    if (rc == 0) rc = send(at(t), at(t + 1));
  }
  const int rw = wait();
  return rc ? rc : rw;
}

}  // namespace og
