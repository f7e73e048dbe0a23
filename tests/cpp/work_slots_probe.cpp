// Captured launches never share their work counters with any other launch (dr_work_slots.h).
#include <cstdio>
#include <set>
#include <thread>
#include <vector>
#include "dr_work_slots.h"

int main() {
  dr::WorkSlots w;
  std::vector<int> eager, got[4];
  for (int k = 0; k < 3 * dr::kEagerSlots; k++) eager.push_back(w.eager());
  std::vector<std::thread> threads;
  for (auto &g : got)
    threads.emplace_back([&g, &w] { for (int k = 0; k < dr::kCapturedSlots / 3; k++) g.push_back(w.captured()); });
  for (auto &t : threads) t.join();
  std::set<int> seen;
  int none = 0;
  for (auto &g : got)
    for (int s : g) {
      if (s < 0) { none++; continue; }
      if (s < dr::kEagerSlots || s >= dr::kWorkSlots || !seen.insert(s).second) return 1;
    }
  if ((int)seen.size() != dr::kCapturedSlots || none != 4 * (dr::kCapturedSlots / 3) - dr::kCapturedSlots) return 2;
  if (w.captured() != -1) return 3;
  for (int k = 0; k < (int)eager.size(); k++) if (eager[k] != k % dr::kEagerSlots) return 4;
  std::puts("ok");
  return 0;
}
