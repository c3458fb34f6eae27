// How the tiles of k_run_steps agree on whether a run of steps is kept.
//
// One 32-bit word holds the number of tiles that are through with the steps and, once a tile
// has given up, the bit RUN_GAVE_UP.  The bit is only set by a compare-and-exchange from a
// value below `want`, so of "every tile is through" and "a tile has given up" the one that
// comes first stands: a word that has reached `want` never gets the bit, and one with the bit
// never equals `want`.  Every tile decides by the word, and so all of them alike.
//
// Host and device, so that a host build can try every order of the tiles' accesses.
#pragma once
#include <hip/hip_runtime.h>

namespace sem2d {

constexpr unsigned RUN_GAVE_UP = 1u << 31;  // tiles are counted below it

// through: this tile has taken every step; spins: polls of its wait for the others.  True:
// every tile is through, and stores its state.  M: add (returns the old value), load, cas (as
// compare_exchange_strong).  At most `want` exchanges fail before one succeeds or the word has
// reached a value that stays.
template <typename M>
__host__ __device__ inline bool run_commit(M& m, bool through, unsigned want, int spins) {
  unsigned at;
  if (through) {
    at = m.add(1u) + 1u;
    for (int left = spins; at < want && left > 0; --left) at = m.load();
  } else {
    at = m.load();
  }
  while (at < want)
    if (m.cas(at, at | RUN_GAVE_UP)) return false;
  return at == want;
}

}  // namespace sem2d
