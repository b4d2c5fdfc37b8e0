// Dependency levels of a program's operations (host code, no GPU types).
//
// Every operation reads some buffers and writes one.  An operation runs one
// level after everything it depends on: reads wait for the buffer's last
// write, writes for its last write and last read.  Operations of one level
// are independent and run as one launch.
//
// Accumulations C += ... would be serial under that rule: a residual takes 5
// to 120 of them, one level each, while the products behind them need 5 to 8
// levels (CCSD, 24 orbitals: 61 levels; CCSDTQ, 14: 365).  They commute, so a
// term that would wait for its turn goes to a partial accumulator of its own
// (slot) instead, and one sum adds the slots to C before C is next read.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <map>
#include <vector>

namespace ccqlv {

using Key = uintptr_t;   // identity of a buffer

struct Unit {
  std::vector<Key> reads;
  std::vector<Key> writes;
  // a term writes one accumulator (writes[0]); assign: it overwrites it;
  // full: it writes every element (else its slot has to start from zeros)
  bool term = false, assign = false, full = true;
  int64_t size = 0;        // elements of the accumulator
  int lat = 1;             // levels it takes (2: split along K, reduced in the second)
  bool barrier = false;    // after everything before it, before everything after it
  // results
  int level = 0;
  int slot = 0;            // 0: the accumulator itself
  bool overwrite = false;  // the first term of its slot: stores instead of adding
};

struct Sum {
  Key out;
  int nslots;   // slots 1 .. nslots - 1 are added to the accumulator
  int level;
};
struct Zero {
  Key out;
  int slot, level;
};

// Most slots of an accumulator.  A slot costs one more write and read of the
// accumulator's size per epoch and saves levels of about 6 us: worth it while
// that traffic stays below a few levels; an accumulator of 64 MB is written
// by products that fill the chip one at a time.
inline int max_slots(int64_t size) { return size <= (1 << 19) ? 8 : size <= (1 << 21) ? 6 : size <= (1 << 23) ? 2 : 1; }
constexpr int kMaxSlots = 8;

class Scheduler {
 public:
  std::vector<Sum> sums;
  std::vector<Zero> zeros;
  int levels = 0;
  int slot_cap = kMaxSlots;   // 1: no partial accumulators

  void run(std::vector<Unit>& units) {
    for (Unit& u : units) place(u);
    close_all();
  }

 private:
  struct Track {
    int wr = -1, rd = -1;   // levels of the last write and read
  };
  struct Epoch {
    bool open = false;
    std::vector<int> free;   // per slot: first level its next term can run on
  };
  std::map<Key, Track> track_;
  std::map<std::pair<Key, int>, Track> slot_track_;
  std::map<Key, Epoch> epoch_;
  std::vector<Key> order_;   // accumulators in the order of their first term
  int floor_ = 0;

  void use(int level) { levels = std::max(levels, level + 1); }

  void close(Key out) {
    auto it = epoch_.find(out);
    if (it == epoch_.end() || !it->second.open) return;
    Epoch& e = it->second;
    e.open = false;
    Track& t = track_[out];
    int last = floor_;
    for (int f : e.free) last = std::max(last, f);
    if (e.free.size() == 1) {
      t.wr = std::max(t.wr, last - 1);
      return;
    }
    sums.push_back({out, (int)e.free.size(), last});
    for (int s = 1; s < (int)e.free.size(); ++s) {
      Track& st = slot_track_[{out, s}];
      st.rd = std::max(st.rd, last);
      st.wr = std::max(st.wr, e.free[s] - 1);
    }
    t.wr = std::max(t.wr, last);
    use(last);
  }
  void close_all() {
    for (Key k : order_) close(k);
  }

  int ready(const Unit& u) {
    int l = floor_;
    for (Key r : u.reads) {
      close(r);
      l = std::max(l, track_[r].wr + 1);
    }
    return l;
  }

  void place(Unit& u) {
    if (u.barrier) {
      close_all();
      u.level = levels;
      floor_ = u.level + 1;
      use(u.level);
      return;
    }
    int l = ready(u);
    if (!u.term) {
      for (Key w : u.writes) {
        close(w);
        l = std::max({l, track_[w].wr + 1, track_[w].rd + 1});
      }
      u.level = l;
      for (Key w : u.writes) track_[w].wr = l + u.lat - 1;
    } else {
      const Key out = u.writes[0];
      if (std::find(u.reads.begin(), u.reads.end(), out) != u.reads.end() || u.assign) close(out);
      Epoch& e = epoch_[out];
      if (!e.open) {
        if (std::find(order_.begin(), order_.end(), out) == order_.end()) order_.push_back(out);
        e.open = true;
        e.free.assign(1, std::max({floor_, track_[out].wr + 1, track_[out].rd + 1}));
        u.slot = 0;
        u.overwrite = u.assign;
        u.level = std::max(l, e.free[0]);
      } else {
        int best = 0, at = std::max(l, e.free[0]);
        for (int s = 1; s < (int)e.free.size(); ++s)
          if (std::max(l, e.free[s]) < at) at = std::max(l, e.free[s]), best = s;
        const int fresh = (int)e.free.size();
        u.overwrite = false;
        if (fresh < std::min(max_slots(u.size), slot_cap)) {
          const Track& st = slot_track_[{out, fresh}];
          const int from = std::max({floor_, st.wr + 1, st.rd + 1});
          const int fl = std::max(l, from + (u.full ? 0 : 1));
          if (fl < at) {
            best = fresh;
            at = fl;
            e.free.push_back(0);
            u.overwrite = u.full;
            if (!u.full) {
              zeros.push_back({out, fresh, from});
              use(from);
            }
          }
        }
        u.slot = best;
        u.level = at;
      }
      e.free[u.slot] = u.level + u.lat;
    }
    // (the second level of a split still reads a folded addend)
    for (Key r : u.reads) track_[r].rd = std::max(track_[r].rd, u.level + u.lat - 1);
    use(u.level + u.lat - 1);
  }
};

}  // namespace ccqlv
