// flow_budget.hpp -- how many waves that wait for each other may be on a device.
//
// A data-flow kernel (kernels.hip) ends only if all its waves run together.
// Alone on a device it has room; beside the kernels of other solvers each may
// get in part of its waves and wait for the rest.  So every solver takes its
// need out of its device's budget for the length of a call, and uses launches
// that wait for nothing when the budget has too little left.
//
// A kernel of which `fit` one-wave workgroups fit a CU takes 1/fit of a CU a
// wave and 4/fit of a SIMD.  Every wave finds room, in whatever order they come
// and on whatever SIMDs the others are, while one of these holds:
// - all waves together are at most SIMDs * the fit of the largest: a SIMD with
//   fewer waves than that has room for any;
// - the sum of the needs is at most CUs * (1 - the largest share of a SIMD): a
//   SIMD turns a wave away only when more than 1 - its share is taken.
// (Half of the device each is not enough: kernels of three and of two waves a
// SIMD can fill 1,000 SIMDs in pairs and 24 in threes, with both short of waves.)
#pragma once

#include <algorithm>
#include <map>
#include <mutex>
#include <vector>

namespace spg {

// what one solver's data-flow kernels take at most at any time (its stream runs
// one of them after the other)
struct FlowNeed {
  long waves = 0;
  int fit = 8;        // waves of the largest that fit a SIMD
  double cus = 0.0;   // of the device
  double simd = 0.0;  // largest share of a SIMD one wave takes
  void add(long n, int per_cu) {
    if (n <= 0) return;
    const int f = std::max(per_cu, 1);
    waves = std::max(waves, n);
    fit = std::min(fit, std::max(f / 4, 1));
    cus = std::max(cus, (double)n / f);
    simd = std::max(simd, std::min(1.0, 4.0 / f));
  }
  bool operator==(const FlowNeed& o) const {
    return waves == o.waves && fit == o.fit && cus == o.cus && simd == o.simd;
  }
};

class FlowBudget {
 public:
  // false: not now
  bool take(int dev, int cus, const FlowNeed& need) {
    std::lock_guard<std::mutex> lock(mu_);
    std::vector<FlowNeed>& held = held_[dev];
    FlowNeed all = need;
    for (const FlowNeed& h : held) {
      all.waves += h.waves;
      all.fit = std::min(all.fit, h.fit);
      all.cus += h.cus;
      all.simd = std::max(all.simd, h.simd);
    }
    // alone, its kernels run one after the other and each packs without loss
    const bool ok = held.empty() ? all.cus <= cus
                                 : all.waves <= 4L * cus * all.fit || all.cus <= cus * (1.0 - all.simd);
    if (!ok) return false;
    held.push_back(need);
    return true;
  }
  void give(int dev, const FlowNeed& need) {
    std::lock_guard<std::mutex> lock(mu_);
    std::vector<FlowNeed>& held = held_[dev];
    for (size_t i = 0; i < held.size(); ++i)
      if (held[i] == need) {
        held.erase(held.begin() + (long)i);
        return;
      }
  }

 private:
  std::mutex mu_;
  std::map<int, std::vector<FlowNeed>> held_;
};

}  // namespace spg
