// Host memory that copies in flight still write.
#pragma once

#include <cstddef>
#include <utility>
#include <vector>

namespace mcnla {

// `count` host ints as targets of device-to-host copies, and the wait for those copies: unless
// they are known to have landed, the destructor waits, and only then the memory goes.  (One object
// for both, so that no order of declarations can let a copy land in freed memory.)
template <class Wait>
class PendingInts {
 public:
  PendingInts(size_t count, Wait wait) : value_(count, 0), wait_(std::move(wait)) {}
  PendingInts(const PendingInts&) = delete;
  PendingInts& operator=(const PendingInts&) = delete;
  ~PendingInts() {
    if (!landed_) wait_();
  }
  int* at(size_t i) { return &value_[i]; }
  int operator[](size_t i) const { return value_[i]; }
  void landed() { landed_ = true; }

 private:
  std::vector<int> value_;
  Wait wait_;
  bool landed_ = false;
};

}  // namespace mcnla
