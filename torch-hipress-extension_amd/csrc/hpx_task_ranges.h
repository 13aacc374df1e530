// The memory that tasks of the scheduler name, as address ranges.  Tasks may be queued side by side only if they share no
// byte: a caller's tensors may be views into one bucket, and a host buffer C may be one slot of a gathered buffer that
// another task names as a whole, so equal base addresses are not what decides.  Host code only.
#ifndef HPX_TASK_RANGES_H_
#define HPX_TASK_RANGES_H_

#include <algorithm>
#include <cstdint>
#include <vector>

#include "hpx_sched.h"

namespace hpx {

class Ranges {
 public:
  void clear() { r_.clear(); }
  void swap(Ranges& o) { r_.swap(o.r_); }
  void add(const void* p, int64_t bytes) {
    if (p && bytes > 0) r_.push_back({reinterpret_cast<uintptr_t>(p), reinterpret_cast<uintptr_t>(p) + uint64_t(bytes)});
  }
  // Every byte that task `t` may read or write: the buffers as the caller declared them.  (A residual holds at least as
  // many elements as its tensor, also where the caller left its length out.)
  void add(const hpx_task_t& t) {
    add(t.tensor, t.tensor_numel * 4);
    add(t.residual, std::max(t.residual_numel, t.tensor_numel) * 4);
    add(t.B, t.B_bytes);
    add(t.C, t.C_bytes);
    add(t.M, int64_t(t.n) * t.m * 4);
    add(t.P, int64_t(t.n) * t.r * 4);
    add(t.Q, int64_t(t.m) * t.r * 4);
  }
  // Sorts what was added and joins what overlaps; whether anything did.  Before meets().
  bool close() {
    std::sort(r_.begin(), r_.end(), [](const R& a, const R& b) { return a.lo < b.lo; });
    bool shared = false;
    size_t n = 0;
    for (const R& x : r_) {
      if (n > 0 && x.lo < r_[n - 1].hi) {
        shared = true;
        r_[n - 1].hi = std::max(r_[n - 1].hi, x.hi);
      } else {
        r_[n++] = x;
      }
    }
    r_.resize(n);
    return shared;
  }
  // Whether the two share a byte.
  bool meets(const Ranges& o) const {
    auto a = r_.begin(), b = o.r_.begin();
    while (a != r_.end() && b != o.r_.end()) {
      if (a->lo < b->hi && b->lo < a->hi) return true;
      if (a->hi <= b->hi) ++a; else ++b;
    }
    return false;
  }

 private:
  struct R { uintptr_t lo, hi; };
  std::vector<R> r_;
};

}  // namespace hpx
#endif  // HPX_TASK_RANGES_H_
