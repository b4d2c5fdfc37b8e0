"""The level schedule (ccq_amd/csrc/levels.h) keeps every buffer unwritten while it
is read, on the CPU: a product split along K reads its folded addend on its
second level too."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "levels.h"
#include <cstdio>
#include <cstdlib>
#include <random>
using namespace ccqlv;
int main(int, char** argv) {
  std::mt19937_64 rng(atoi(argv[1]));
  auto rnd = [&](int n) { return (int)(rng() % n); };
  for (int prog = 0; prog < 300; ++prog) {
    const int nb = 3 + rnd(10), nu = 1 + rnd(60);
    std::vector<Unit> us;
    for (int i = 0; i < nu; ++i) {
      Unit u;
      for (int k = rnd(3); k >= 0; --k) u.reads.push_back(1 + rnd(nb));
      u.writes.push_back(1 + rnd(nb));
      u.term = rnd(6) > 0;
      u.assign = u.term && rnd(4) == 0;
      u.full = rnd(3) > 0;
      u.size = 1ll << rnd(25);
      u.lat = u.term ? 1 + rnd(2) : 1;
      us.push_back(u);
    }
    Scheduler s;
    s.run(us);
    // writers of each buffer's own storage (slot 0), by level: unit, or -1 for a sum
    std::map<std::pair<Key, int>, std::vector<int>> wr;
    for (int i = 0; i < nu; ++i)
      if (!us[i].term || us[i].slot == 0) wr[{us[i].writes[0], us[i].level + us[i].lat - 1}].push_back(i);
    for (auto& m : s.sums) wr[{m.out, m.level}].push_back(-1);
    for (int i = 0; i < nu; ++i)
      for (size_t r = 0; r < us[i].reads.size(); ++r) {
        // the last read of a split unit is its addend
        const int end = us[i].level + (r + 1 == us[i].reads.size() ? us[i].lat - 1 : 0);
        for (int l = us[i].level; l <= end; ++l) {
          auto it = wr.find({us[i].reads[r], l});
          if (it == wr.end()) continue;
          for (int w : it->second)
            if (w != i) { printf("program %d: unit %d reads %ld on level %d, written by %d\n", prog, i, (long)us[i].reads[r], l, w); return 1; }
        }
      }
  }
  printf("ok\n");
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("addend")
    (d / "t.cpp").write_text(SRC)
    exe = str(d / "t")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-I", os.path.join(ROOT, "ccq_amd", "csrc"),
                    str(d / "t.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("seed", [1, 2, 3, 4])
def test_no_write_while_read(program, seed):
    r = subprocess.run([program, str(seed)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    assert r.stdout.strip() == "ok"
