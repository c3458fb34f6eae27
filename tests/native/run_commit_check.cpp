// Every order of the accesses of a few tiles that agree on a run of steps (sem2d::run_commit):
// all of them decide alike, they keep the run only if every tile is through, and a run that is
// through is kept where every wait is long enough.  A tile's code is run again from its start
// with the answers it has had so far, up to its next access; states already seen are not
// followed again.  Prints one line: "<states> <wrong>".
#include <stdio.h>

#include <set>
#include <string>
#include <vector>

#include "sem2d_commit.hpp"

struct Pending {
  int kind;  // 0 add, 1 load, 2 compare-and-exchange
  unsigned a, b;
};
struct Replay {
  const std::vector<unsigned>* had;
  size_t at = 0;
  unsigned next(int kind, unsigned a, unsigned b) {
    if (at == had->size()) throw Pending{kind, a, b};
    return (*had)[at++];
  }
  unsigned add(unsigned x) { return next(0, x, 0); }
  unsigned load() { return next(1, 0, 0); }
  bool cas(unsigned& e, unsigned d) {
    const unsigned seen = next(2, e, d);
    const bool ok = seen == e;
    e = seen;
    return ok;
  }
};

struct Tile {
  bool through;
  int spins;
  std::vector<unsigned> had;
  int kept = -1;  // -1: not decided yet
};
struct Check {
  std::set<std::string> seen;
  long wrong = 0;
  void go(std::vector<Tile> t, unsigned word) {
    std::string key((const char*)&word, sizeof word);
    for (const Tile& x : t) {
      key.append((const char*)x.had.data(), x.had.size() * sizeof(unsigned));
      key += (char)('a' + x.kept);
      key += '|';
    }
    if (!seen.insert(key).second) return;
    bool all = true, through = true;
    for (size_t i = 0; i < t.size(); ++i) {
      through = through && t[i].through;
      if (t[i].kept >= 0) continue;
      all = false;
      if (t[i].had.size() > 64) {  // an end in sight for every tile
        ++wrong;
        return;
      }
      std::vector<Tile> u = t;
      unsigned w = word;
      Replay r{&u[i].had};
      try {
        u[i].kept = sem2d::run_commit(r, u[i].through, (unsigned)t.size(), u[i].spins);
      } catch (const Pending& p) {
        u[i].had.push_back(w);
        if (p.kind == 0) w += p.a;
        if (p.kind == 2 && w == p.a) w = p.b;
      }
      go(u, w);
    }
    if (!all) return;
    for (const Tile& x : t)
      if (x.kept != t[0].kept || (x.kept && !through)) {
        ++wrong;
        return;
      }
  }
};

int main() {
  long states = 0, wrong = 0;
  for (int n = 1; n <= 4; ++n)
    for (int spins = 0; spins <= (n <= 3 ? 2 : 1); ++spins)
      for (int stopped = 0; stopped <= (n < 2 ? n : 2); ++stopped) {  // tiles that gave up in their steps
        Check c;
        std::vector<Tile> t;
        for (int i = 0; i < n; ++i) t.push_back({i >= stopped, spins, {}});
        c.go(t, 0);
        states += (long)c.seen.size();
        wrong += c.wrong;
      }
  // one after the other, the last finds the count full; the others' waits see it too
  for (int n = 1; n <= 4; ++n) {
    std::vector<Tile> t(n, {true, 8, {}});
    unsigned w = 0;
    for (int round = 0; round < 16; ++round)
      for (Tile& x : t) {
        if (x.kept >= 0) continue;
        Replay r{&x.had};
        try {
          x.kept = sem2d::run_commit(r, true, (unsigned)n, 8);
        } catch (const Pending& p) {
          x.had.push_back(w);
          if (p.kind == 0) w += p.a;
          if (p.kind == 2 && w == p.a) w = p.b;
        }
      }
    for (const Tile& x : t) wrong += x.kept != 1;
  }
  printf("%ld %ld\n", states, wrong);
  return wrong != 0;
}
