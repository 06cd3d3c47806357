// scratch.hpp — device scratch that makes a call faster and that it can do without.
//
// Host-only policy (the device calls are the caller's functions). The block grows to what
// was asked for, up to a limit; a replaced block is freed only once its successor exists; and
// a size that could not be allocated is not asked for again, so that calls which cannot have
// the scratch go on without it at no cost.
#pragma once
#include <stddef.h>

namespace vgi {

class OptionalScratch {
 public:
  explicit OptionalScratch(size_t limit) : limit_(limit) {}

  void* data() const { return data_; }
  size_t bytes() const { return bytes_; }

  // True if data() holds `need` bytes. allocate(bytes) gives a block or null; drain() waits
  // for the work queued on the old block and returns false if that failed (the block is then
  // kept, and the new one freed); release(block) frees it.
  template <class Allocate, class Drain, class Release>
  bool reserve(size_t need, Allocate&& allocate, Drain&& drain, Release&& release) {
    if (need <= bytes_) return true;
    if (need > limit_ || need >= refused_) return false;
    void* p = allocate(need);
    if (!p) {
      refused_ = need;
      return false;
    }
    if (data_) {
      if (!drain()) {
        release(p);
        return false;
      }
      release(data_);
    }
    data_ = p;
    bytes_ = need;
    return true;
  }

 private:
  size_t limit_;
  void* data_ = nullptr;
  size_t bytes_ = 0;
  size_t refused_ = ~(size_t)0;  // the least size that could not be allocated
};

}  // namespace vgi
