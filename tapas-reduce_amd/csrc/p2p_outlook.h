// p2p_outlook.h -- whether an evaluation's P2P will outweigh its M2L, as the last one
// of a problem like it did: what the start of the upward pass is chosen by, before
// the traversal has counted the pairs.  No result depends on it.
#pragma once
#include <cstdint>

namespace tfmm {

// A problem, as far as the work of its kernels goes.
struct P2pProblem {
  int64_t n;
  double theta;
  int32_t nprob, ncrit, precision, mutual, basis, images;

  // the same settings, and bodies that may have become an eighth more or fewer
  bool like(const P2pProblem &o) const {
    const int64_t d = n < o.n ? o.n - n : n - o.n;
    return theta == o.theta && nprob == o.nprob && ncrit == o.ncrit &&
           precision == o.precision && mutual == o.mutual && basis == o.basis &&
           images == o.images && d <= o.n / 8;
  }
};

// The last few problems that a context evaluated.
class P2pOutlook {
  static constexpr int KEPT = 4;
  struct Seen {
    P2pProblem p;
    bool heavy;
  } seen[KEPT];
  int used = 0, next = 0;

  int find(const P2pProblem &p) const {
    for (int i = 0; i < used; i++)
      if (p.like(seen[i].p)) return i;
    return -1;
  }

 public:
  // (a problem not seen yet: no)
  bool heavy(const P2pProblem &p) const {
    const int i = find(p);
    return i >= 0 && seen[i].heavy;
  }
  void saw(const P2pProblem &p, bool heavy) {
    int i = find(p);
    if (i < 0) {
      i = next;
      next = (next + 1) % KEPT;
      if (used < KEPT) used++;
    }
    seen[i] = {p, heavy};
  }
};

}  // namespace tfmm
