// CPU check of the P2P's outlook (tapas-reduce_amd/csrc/p2p_outlook.h).  Prints
// the name of the first part that fails, or "ok".
#include <cstdio>
#include <initializer_list>

#include "../../tapas-reduce_amd/csrc/p2p_outlook.h"

using namespace tfmm;

static P2pProblem problem(int64_t n, int ncrit) { return {n, 0.4, 1, ncrit, 0, 0, 0, 0}; }

int main() {
  const P2pProblem heavy = problem(4000000, 128), light = problem(250000, 64);
  P2pOutlook o;
  if (o.heavy(heavy) || o.heavy(light)) return printf("unseen\n"), 1;
  // alternating problems: each by its own last evaluation
  for (int i = 0; i < 5; i++) {
    if (o.heavy(light) || o.heavy(heavy) != (i > 0)) return printf("alternating\n"), 2;
    o.saw(heavy, true);
    o.saw(light, false);
  }
  // bodies come and go
  P2pProblem p = heavy;
  for (int i = 0; i < 20; i++) {
    p.n += p.n / 20;
    if (!o.heavy(p)) return printf("growing\n"), 3;
    o.saw(p, true);
  }
  o.saw(p, false);
  if (o.heavy(p)) return printf("changed\n"), 4;
  // a bounded memory: the oldest goes
  P2pOutlook b;
  for (int c = 1; c <= 6; c++) b.saw(problem(1000, c), true);
  if (b.heavy(problem(1000, 1)) || !b.heavy(problem(1000, 6)) || !b.heavy(problem(1000, 3)))
    return printf("bounded\n"), 5;
  // every setting counts
  P2pProblem q = light;
  P2pOutlook s;
  s.saw(q, true);
  for (int32_t P2pProblem::*f : {&P2pProblem::nprob, &P2pProblem::ncrit, &P2pProblem::precision,
                                 &P2pProblem::mutual, &P2pProblem::basis, &P2pProblem::images}) {
    P2pProblem r = q;
    r.*f += 1;
    if (s.heavy(r)) return printf("setting\n"), 6;
  }
  q.theta = 0.5;
  if (s.heavy(q)) return printf("theta\n"), 7;
  printf("ok\n");
  return 0;
}
