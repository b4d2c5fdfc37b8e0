"""The level schedule (ccq_amd/csrc/levels.h) against program order, on the
CPU: random programs of reads, assignments and accumulations are placed on
levels and run level by level, each level in a shuffled order, with the slots,
zeros and sums the schedule asks for; every buffer ends with the value program
order gives (integer arithmetic, exact).  No read may share a level with a
write of its buffer."""

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
typedef long long ll;
int main(int argc, char** argv) {
  std::mt19937_64 rng(atoi(argv[1]));
  auto rnd = [&](int n) { return (int)(rng() % n); };
  for (int prog = 0; prog < 300; ++prog) {
    const int nb = 3 + rnd(10), nu = 1 + rnd(60);
    // a buffer holds two halves; a term that is not full writes the first only
    struct B { ll v[2]; };
    std::vector<B> seq(nb + 1), par;
    for (auto& b : seq) b = {{rnd(9), rnd(9)}};
    par = seq;
    std::vector<Unit> us;
    std::vector<ll> coef;
    for (int i = 0; i < nu; ++i) {
      Unit u;
      const int r = rnd(20);
      if (r == 0) { u.barrier = true; }
      else {
        for (int k = rnd(3); k >= 0; --k) u.reads.push_back(1 + rnd(nb));
        u.writes.push_back(1 + rnd(nb));
        u.term = r > 3;
        u.assign = u.term && rnd(4) == 0;
        u.full = rnd(3) > 0;
        u.size = 1ll << rnd(25);
        u.lat = u.term ? 1 + rnd(2) : 1;
      }
      us.push_back(u);
      coef.push_back(1 + rnd(5));
    }
    auto value = [&](const std::vector<B>& b, const Unit& u, ll c, int h) {
      ll s = c;
      for (Key k : u.reads) s += c * b[k].v[h] % 1009;
      return s % 1009;
    };
    for (int i = 0; i < nu; ++i) {
      const Unit& u = us[i];
      if (u.barrier) continue;
      for (int h = 0; h < 2; ++h) {
        if (u.term && !u.full && h) continue;
        const ll x = value(seq, u, coef[i], h);
        B next = seq[u.writes[0]];
        next.v[h] = (!u.term || u.assign) ? x : next.v[h] + x;
        if (std::find(u.reads.begin(), u.reads.end(), u.writes[0]) == u.reads.end() || u.term) seq[u.writes[0]] = next;
        else seq[u.writes[0]].v[h] = x;
      }
    }
    Scheduler s;
    s.run(us);
    std::map<std::pair<Key, int>, B> slot;   // garbage until zeroed or overwritten
    auto at = [&](Key k, int sl) -> B& {
      if (!sl) return par[k];
      auto it = slot.find({k, sl});
      if (it == slot.end()) it = slot.emplace(std::make_pair(k, sl), B{{777777, 777777}}).first;
      return it->second;
    };
    struct Late { Key k; int slot; B x; bool over, full; };
    std::vector<std::vector<Late>> late(s.levels + 2);
    for (int l = 0; l < s.levels; ++l) {
      // reads and writes of the level must not meet
      std::vector<int> here;
      for (int i = 0; i < nu; ++i) if (!us[i].barrier && us[i].level == l) here.push_back(i);
      std::shuffle(here.begin(), here.end(), rng);
      std::map<std::pair<Key, int>, int> writers;
      for (int i : here) if (us[i].lat == 1) ++writers[{us[i].writes[0], us[i].slot}];
      for (auto& x : late[l]) ++writers[{x.k, x.slot}];
      for (auto& z : s.zeros) if (z.level == l) ++writers[{z.out, z.slot}];
      for (auto& m : s.sums) if (m.level == l) {
        ++writers[{m.out, 0}];
        for (int k = 1; k < m.nslots; ++k) if (writers.count({m.out, k})) { printf("sum reads a written slot\n"); return 1; }
      }
      for (auto& w : writers) if (w.second > 1) { printf("two writers in a level\n"); return 1; }
      for (int i : here) for (Key k : us[i].reads)
        if (writers.count({k, 0}) && !(us[i].writes[0] == k && writers[{k, 0}] == 1 && us[i].lat == 1 && us[i].slot == 0)) {
          printf("read and write of a buffer in one level\n"); return 1; }
      for (auto& z : s.zeros) if (z.level == l) at(z.out, z.slot) = B{{0, 0}};
      for (auto& x : late[l]) for (int h = 0; h < (x.full ? 2 : 1); ++h) {
        ll& d = at(x.k, x.slot).v[h];
        d = x.over ? x.x.v[h] : d + x.x.v[h];
      }
      for (int i : here) {
        const Unit& u = us[i];
        B x;
        for (int h = 0; h < 2; ++h) x.v[h] = value(par, u, coef[i], h);
        const bool over = u.term ? u.overwrite : true, full = u.term ? u.full : true;
        if (u.lat == 2) { late[l + 1].push_back({u.writes[0], u.slot, x, over, full}); continue; }
        for (int h = 0; h < (full ? 2 : 1); ++h) {
          ll& d = at(u.writes[0], u.slot).v[h];
          d = over ? x.v[h] : d + x.v[h];
        }
      }
      for (auto& m : s.sums) if (m.level == l)
        for (int k = 1; k < m.nslots; ++k) for (int h = 0; h < 2; ++h) par[m.out].v[h] += at(m.out, k).v[h];
    }
    for (int b = 1; b <= nb; ++b) for (int h = 0; h < 2; ++h)
      if (par[b].v[h] != seq[b].v[h]) { printf("program %d buffer %d: %lld, program order %lld\n", prog, b, par[b].v[h], seq[b].v[h]); return 1; }
  }
  printf("ok\n");
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("levels")
    (d / "t.cpp").write_text(SRC)
    exe = str(d / "t")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-I", os.path.join(ROOT, "ccq_amd", "csrc"),
                    str(d / "t.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("seed", [1, 2, 3, 4])
def test_levels_equal_program_order(program, seed):
    r = subprocess.run([program, str(seed)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    assert r.stdout.strip() == "ok"
