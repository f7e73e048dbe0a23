// Which pair of work counters a launch uses (host only).
//
// A launch's pair is zero before it and zero after it, so two launches may share one unless they run
// at the same time.  Eager launches take the pairs of a ring in turn: two share one only if the later
// runs while kEagerSlots launches issued since the earlier have come and it has not ended.  A captured
// launch keeps its pair for as long as its graph may be replayed, beside whatever runs then: it takes
// one of kCapturedSlots that no other launch ever uses, and none (-1) once those are gone.
#pragma once
#include <atomic>
#include <cstdint>

namespace dr {

constexpr int kEagerSlots = 16384;
constexpr int kCapturedSlots = 1024;
constexpr int kWorkSlots = kEagerSlots + kCapturedSlots;

struct WorkSlots {
  std::atomic<uint32_t> next_eager{0}, next_captured{0};
  int eager() { return (int)(next_eager.fetch_add(1) % kEagerSlots); }
  int captured() {
    uint32_t k = next_captured.load();
    while (k < (uint32_t)kCapturedSlots && !next_captured.compare_exchange_weak(k, k + 1)) {}
    return k < (uint32_t)kCapturedSlots ? kEagerSlots + (int)k : -1;
  }
};

}  // namespace dr
