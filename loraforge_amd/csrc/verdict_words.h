// Which words of a fixed set are in use: a call takes one for as long as a
// kernel may write it or the host read it, so calls in flight at the same time
// (threads, streams) never share one. Host code only.
#pragma once

#include <cstdint>
#include <mutex>

namespace lf {

class VerdictWords {
 public:
  static constexpr int kWords = 256;

  // A free word's index, or -1 when all are taken.
  int take() {
    std::lock_guard<std::mutex> guard(lock_);
    for (int i = 0; i < kWords / 64; ++i)
      if (free_[i]) {
        const int bit = __builtin_ctzll(free_[i]);
        free_[i] &= free_[i] - 1;
        return 64 * i + bit;
      }
    return -1;
  }

  void give(int word) {
    std::lock_guard<std::mutex> guard(lock_);
    free_[word / 64] |= uint64_t(1) << (word % 64);
  }

 private:
  std::mutex lock_;
  uint64_t free_[kWords / 64] = {~uint64_t(0), ~uint64_t(0), ~uint64_t(0), ~uint64_t(0)};
};

}  // namespace lf
