// The staging memory of ray queries that no query uses at the moment.
#pragma once
#include <cstddef>
#include <utility>

namespace ttgpu {

// Up to kMax idle stages (T: int device, int slots (0: none), size_t slot_rays).  Storage is fixed, so that
// nothing here can throw: a stage comes back while a query's error may be under way.
template <class T, int kMax>
class IdleStages {
 public:
  // The smallest idle stage for a query that asked for `want`: of its device and number of slots (a query of
  // one slot runs on its handle's stream and has no use for the streams of several), each large enough.
  // Without one, a stage with slots = 0.
  T Take(const T &want) noexcept {
    int best = -1;
    for (int k = 0; k < count_; ++k)
      if (idle_[k].device == want.device && idle_[k].slots == want.slots && idle_[k].slot_rays >= want.slot_rays &&
          (best < 0 || idle_[k].slot_rays < idle_[best].slot_rays))
        best = k;
    return best < 0 ? T{} : Remove(best);
  }
  // Keeps `s`.  When that makes too many, the smallest leaves: it is returned, to be freed.
  T Put(T s) noexcept {
    if (count_ < kMax) {
      idle_[count_++] = s;
      return T{};
    }
    for (int k = 0; k < kMax; ++k)
      if (Rays(idle_[k]) < Rays(s)) std::swap(idle_[k], s);
    return s;
  }
  // Any idle stage, or one with slots = 0 when there is none left.
  T Drop() noexcept { return count_ > 0 ? Remove(count_ - 1) : T{}; }

 private:
  static std::size_t Rays(const T &s) { return s.slots * s.slot_rays; }
  T Remove(int k) noexcept {
    const T s = idle_[k];
    idle_[k] = idle_[--count_];
    return s;
  }
  T idle_[kMax];
  int count_ = 0;
};

}  // namespace ttgpu
