// flow_budget.hpp -- how many waves that wait for each other may be on a device.
//
// A data-flow kernel (kernels.hip) ends only if all its waves run together.
// Alone on a device it has room; beside the kernels of other solvers each may
// get in part of its waves and wait for the rest.  So every solver takes its
// need out of its device's budget for the length of a call, and uses launches
// that wait for nothing when the budget has too little left.
//
// A kernel of which `fit` one-wave workgroups fit a CU takes 1/fit of a CU a
// wave and 4/fit of a SIMD.  A SIMD turns a wave away only when more than 1 -
// 4/fit of it is taken, so while the sum of all needs is at most CUs * (1 - the
// largest share of a SIMD), there is a SIMD with room for every wave, in
// whatever order they come and on whatever SIMDs the others are.  (Half of the
// device each is not enough: kernels of three and of two waves a SIMD can fill
// 1,000 SIMDs in pairs and 24 in threes, with both short of waves.)
#pragma once

#include <algorithm>
#include <map>
#include <mutex>
#include <vector>

namespace spg {

// what one solver's data-flow kernels take at most at any time (its stream runs
// one of them after the other)
struct FlowNeed {
  double cus = 0.0;   // of the device
  double simd = 0.0;  // largest share of a SIMD one wave takes
  void add(long waves, int fit) {
    if (waves <= 0) return;
    const int f = std::max(fit, 1);
    cus = std::max(cus, (double)waves / f);
    simd = std::max(simd, std::min(1.0, 4.0 / f));
  }
};

class FlowBudget {
 public:
  // false: not now
  bool take(int dev, int cus, const FlowNeed& need) {
    std::lock_guard<std::mutex> lock(mu_);
    std::vector<FlowNeed>& held = held_[dev];
    double sum = need.cus, simd = need.simd;
    for (const FlowNeed& h : held) {
      sum += h.cus;
      simd = std::max(simd, h.simd);
    }
    // alone, its kernels of one size pack without loss
    if (sum > (held.empty() ? (double)cus : cus * (1.0 - simd))) return false;
    held.push_back(need);
    return true;
  }
  void give(int dev, const FlowNeed& need) {
    std::lock_guard<std::mutex> lock(mu_);
    std::vector<FlowNeed>& held = held_[dev];
    for (size_t i = 0; i < held.size(); ++i)
      if (held[i].cus == need.cus && held[i].simd == need.simd) {
        held.erase(held.begin() + (long)i);
        return;
      }
  }

 private:
  std::mutex mu_;
  std::map<int, std::vector<FlowNeed>> held_;
};

}  // namespace spg
