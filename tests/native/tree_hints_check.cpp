// CPU check of what a tree build takes from the last tree
// (tapas-reduce_amd/csrc/tree_hints.h).  Prints the name of the first part that
// fails, or "ok".
#include <cstdio>

#include "../../tapas-reduce_amd/csrc/tree_hints.h"

using namespace tfmm;

// Bodies sorted by fewer bits than their keys have are only told apart from sorted
// ones by the build on the device, so a build that cannot run there sorts them whole.
static bool whole_keys_without_the_device_build() {
  struct {
    std::vector<int32_t> hint;
    int32_t roots;
    int words;
    bool fits;
  } cases[] = {
      {{}, 1, 256, false},                                 // the first tree
      {{1, 8, 64}, 1, 256, true},                          //
      {{1, 8, 64}, 1, 9, true},                            // 2 (3 + 1) + 1 words
      {{1, 8, 64}, 1, 8, false},                           //
      {{1, 1 << 27, 1 << 27, 1 << 27, 1 << 27, 1 << 27, 1 << 27, 1 << 27, 1 << 27}, 1, 256, false},
      {std::vector<int32_t>(9, INT32_MAX), 1, 256, false}, // more cells than an index holds
  };
  for (const auto &k : cases) {
    const LevelGrids g = level_grids(k.hint, k.roots, k.words);
    if (g.fits != k.fits) return false;
    for (int64_t n : {1, 4096, 1 << 20, 1 << 23})
      for (int ncrit : {1, 64, 128, 512, 1 << 20}) {
        const int bits = key_prefix_bits(g.fits, (int)k.hint.size() - 1, n, ncrit);
        if (!g.fits ? bits != WHOLE_KEY : bits % 9 != 0 && bits != WHOLE_KEY) return false;
      }
    for (size_t d = 0; d < k.hint.size(); d++)
      if (g.grid[d] < std::min(k.hint[d], INT32_MAX / 16) || g.largest < g.grid[d]) return false;
  }
  // a forest's roots are more than the last tree's
  return level_grids({1, 8}, 5000, 256).grid[0] == 5000;
}

// evaluations of bodies that need `need` levels more than the tree has; the long
// runs among them
static int evaluate(SortDepth &d, int need, int times) {
  int longs = 0;
  for (int i = 0; i < times; i++) {
    if (d.extra < need) {
      d.long_run();
      longs++;
    } else {
      d.sorted();
    }
  }
  return longs;
}

// A context that saw clustered bodies sorts even ones by few bits again; one that
// keeps its clustered bodies seldom sorts twice.
static bool depth_comes_back() {
  SortDepth d;
  if (evaluate(d, 0, 100) != 0 || d.extra != 0) return false;
  if (evaluate(d, 8, 10) != 4 || d.extra != 8) return false;
  evaluate(d, 0, 200);
  if (d.extra != 0) return false;
  evaluate(d, 8, 10);
  if (evaluate(d, 8, 10000) > 20) return false;
  evaluate(d, 0, 5000);
  return d.extra == 0;
}

int main() {
  if (!depth_comes_back()) return printf("depth\n"), 1;
  if (!whole_keys_without_the_device_build()) return printf("whole keys\n"), 1;
  printf("ok\n");
  return 0;
}
