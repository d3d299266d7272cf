// A table of plans by the sizes they were made for.
#pragma once

#include <cstdint>
#include <cstring>
#include <memory>

namespace mellin {

// `Places` sizes of `Words` words each, the first of them never 0.  A size takes the first free place from its hash on, so that
// it is found again as long as the table has not met more sizes than it has places; from then on a new size takes the place its
// hash names.  (With one place for each hash two layers of a stack could throw each other's plans out at every look-up: the
// half-precision ten-layer linear stack of 32 to 256 channels did, 9.4 us to look its layers up instead of 4.8.)
template <typename Value, int Places, int Words>
class PlanTable {
 public:
  // The value of a size.  A new one is value-initialised.
  Value &at(const int64_t (&key)[Words]) {
    if (!places_) places_.reset(new Place[Places]());
    uint64_t h = 0;
    for (int64_t k : key) h = (h ^ (uint64_t)k) * 0x9E3779B97F4A7C15ull, h ^= h >> 29;
    Place *free = &places_[h % Places];
    for (int i = 0; i < Places; ++i) {
      Place &p = places_[(h + i) % Places];
      if (p.key[0] == 0) { free = &p; break; }
      if (memcmp(p.key, key, sizeof key) == 0) return p.value;
    }
    memcpy(free->key, key, sizeof key);
    free->value = Value();
    return free->value;
  }

 private:
  struct Place { int64_t key[Words]; Value value; };
  std::unique_ptr<Place[]> places_;
};

}  // namespace mellin
