// tree_hints.h -- what a tree build takes from the last tree of its context: the
// grids of its levels, and how many leading key bits to sort the bodies by.
#pragma once
#include <algorithm>
#include <cstdint>
#include <vector>

namespace tfmm {

constexpr int KEY_LEVELS = 19;  // levels of a Morton key
constexpr int WHOLE_KEY = 3 * KEY_LEVELS;

inline int bits_for(int64_t v) {
  int b = 1;
  while (b < 62 && (((int64_t)1 << b) <= v)) b++;
  return b;
}

// Grids of the levels, an eighth more cells than the last tree had (hint).  fits:
// the build that leaves all sizes on the device can run with them (words: of the
// read-back of its level table, two a level).
struct LevelGrids {
  std::vector<int32_t> grid;
  int64_t cells = 0, largest = 0;
  bool fits = false;
};

inline LevelGrids level_grids(const std::vector<int32_t> &hint, int32_t nroots, int words) {
  LevelGrids g;
  if (hint.empty()) return g;
  for (size_t d = 0; d < hint.size(); d++) {
    const int64_t h = hint[d];
    int32_t cells = (int32_t)std::min<int64_t>(INT32_MAX / 16, h + h / 8 + 256);
    if (d == 0) cells = std::max(cells, nroots);
    g.grid.push_back(cells);
    g.cells += cells;
    g.largest = std::max<int64_t>(g.largest, cells);
  }
  g.fits = 2 * ((int)hint.size() + 1) + 1 <= words && g.cells + 4096 <= INT32_MAX / 2;
  return g;
}

// Leading key bits to sort the n bodies by before the runs that agree on them are
// sorted, WHOLE_KEY for all of them.  Only a build on the device sees that a run was
// too long.  levels: of the last tree, where a cell holds at most ncrit bodies, and
// what experience adds; bodies spread evenly agree in a few at n's bits.  Whole
// passes of 9 bits; with six or more the runs would save nothing.
inline int key_prefix_bits(bool on_device, int levels, int64_t n, int64_t ncrit) {
  if (!on_device) return WHOLE_KEY;
  for (int64_t m = ncrit; m > 128; m /= 4) levels++;
  const int bits = std::max({3 * levels, bits_for(n) - 4, 1});
  const int passes = (bits + 8) / 9;
  return passes >= 6 ? WHOLE_KEY : 9 * passes;
}

// Levels to sort by beyond the last tree's: two more for every build that met a run
// too long, and two fewer again, on trial, after `patience` builds that met none (the
// context may hold other bodies by then).  A trial that fails costs one sort, and
// doubles the patience.
struct SortDepth {
  static constexpr int STEP = 2, CALM = 16, MOST = 1024;
  int extra = 0, calm = 0, patience = CALM;
  bool trial = false;

  void long_run() {
    extra += STEP;
    calm = 0;
    if (trial) patience = std::min(2 * patience, MOST);
    trial = false;
  }
  void sorted() {
    if (extra == 0 || ++calm < patience) return;
    extra -= STEP;
    calm = 0;
    trial = true;
  }
};

}  // namespace tfmm
