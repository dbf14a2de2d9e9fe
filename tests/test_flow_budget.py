"""The budget of waves that wait for each other (csrc/flow_budget.hpp), compiled
on its own: what it accepts can always be placed, whatever the order in which
the waves of several solvers come and the SIMDs they go to."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spgrid_topo_opt_amd", "csrc")

PROGRAM = r"""
#include "flow_budget.hpp"
#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
using namespace spg;
#define CHECK(x) do { if (!(x)) { std::printf("failed: %s (line %d)\n", #x, __LINE__); std::exit(1); } } while (0)
static FlowNeed need(long waves, int fit) { FlowNeed n; n.add(waves, fit); return n; }

// waves of several kernels, each of a number of registers a lane, on SIMDs of
// 512: placed in random order on random SIMDs with room.  A kernel of which some
// waves find no room while all others wait too never ends.
static bool all_placed(std::mt19937& g, const std::vector<std::pair<long, int>>& k, int simds) {
  std::vector<int> left(simds, 512), slots(simds, 8), todo;
  for (size_t i = 0; i < k.size(); ++i) todo.insert(todo.end(), (size_t)k[i].first, (int)i);
  std::shuffle(todo.begin(), todo.end(), g);
  for (int i : todo) {
    const int r = k[(size_t)i].second, s0 = (int)(g() % (unsigned)simds);
    int s = 0;
    while (s < simds && (left[(s0 + s) % simds] < r || slots[(s0 + s) % simds] == 0)) ++s;
    if (s == simds) return false;
    left[(s0 + s) % simds] -= r;
    slots[(s0 + s) % simds]--;
  }
  return true;
}
static int fit(int regs) { return 4 * std::min(8, 512 / regs); }

int main() {
  {  // alone: the whole device, and no more
    FlowBudget b;
    CHECK(b.take(0, 256, need(4096, 32)));
    b.give(0, need(4096, 32));
    CHECK(b.take(0, 256, need(256 * 12, 12)));
    b.give(0, need(256 * 12, 12));
    CHECK(!b.take(0, 256, need(256 * 12 + 1, 12)));
  }
  {  // two halves that need not fit beside each other; another device; give back
    FlowBudget b;
    CHECK(b.take(0, 256, need(1536, 12)));
    CHECK(!b.take(0, 256, need(1024, 8)));
    CHECK(b.take(1, 256, need(1024, 8)));
    b.give(0, need(1536, 12));
    CHECK(b.take(0, 256, need(1024, 8)));
  }
  {  // two halves of waves of one size fit exactly
    FlowBudget b;
    CHECK(b.take(0, 256, need(1536, 12)));
    CHECK(b.take(0, 256, need(1536, 12)));
    CHECK(!b.take(0, 256, need(1, 12)));
  }
  {  // many small solvers run beside each other, also with waves of a whole SIMD
    FlowBudget b;
    for (int i = 0; i < 4; ++i) CHECK(b.take(0, 256, need(360, 12)));
    for (int i = 0; i < 16; ++i) CHECK(b.take(1, 256, need(64, 4)));
    CHECK(!b.take(1, 256, need(64, 4)));
  }
  std::mt19937 g(1);
  const int regs[] = {64, 80, 96, 128, 144, 168, 248, 256, 280};
  int accepted = 0, tight = 0;
  for (int t = 0; t < 2000; ++t) {
    const int cus = 8;
    FlowBudget b;
    std::vector<std::pair<long, int>> k;
    for (int i = 0; i < 8; ++i) {
      const int r = regs[g() % 9];
      const long waves = 1 + (long)(g() % (unsigned)(cus * fit(r) / 2));
      if (b.take(0, cus, need(waves, fit(r)))) k.emplace_back(waves, r);
    }
    accepted += (int)k.size();
    tight += k.size() > 1;
    CHECK(all_placed(g, k, 4 * cus));
  }
  CHECK(tight > 500);
  {  // from several threads: never more than the limit at a time
    FlowBudget b;
    std::mutex m;
    double held = 0.0, most = 0.0;
    std::vector<std::thread> th;
    for (int t = 0; t < 8; ++t)
      th.emplace_back([&] {
        for (int i = 0; i < 2000; ++i) {
          const FlowNeed n = need(600, 16);
          if (!b.take(0, 256, n)) continue;
          {
            std::lock_guard<std::mutex> l(m);
            held += n.cus;
            most = std::max(most, held);
          }
          std::this_thread::yield();
          {
            std::lock_guard<std::mutex> l(m);
            held -= n.cus;
          }
          b.give(0, n);
        }
      });
    for (auto& t : th) t.join();
    CHECK(most > 0 && most <= 256);
    CHECK(b.take(0, 256, need(4096, 16)));  // all given back
  }
  std::printf("ok %d\n", accepted);
}
"""


def test_accepted_needs_can_always_be_placed(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    src = tmp_path / "budget.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "budget"
    subprocess.run([cxx, "-std=c++17", "-O2", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
