// CPU check of the FP64 P2P's scale (tapas-reduce_amd/csrc/p2p_range.h): for
// bodies of many magnitudes, with and without periodic images, that whenever
// p2p_frame finds a scale, no two bodies that do not coincide come closer than 2,
// and the smallest charge's 8 q / r^3 at the farthest pair is a normal number.
// Prints "scaled <number> wide <number>".
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../../tapas-reduce_amd/csrc/p2p_range.h"

using namespace tfmm;

static uint32_t exponent(double v) {
  uint64_t b;
  memcpy(&b, &v, 8);
  return (uint32_t)(b >> 52) & 0x7ffu;
}

int main() {
  std::mt19937_64 r(7);
  std::uniform_real_distribution<double> u(-1, 1);
  long scaled = 0, wide = 0;
  for (int trial = 0; trial < 20000; trial++) {
    const int centre = (int)(r() % 1200) - 600, spread = 1 << r() % 11;
    const double cycle = trial % 3 ? 0 : std::ldexp(1.5, centre + (int)(r() % 3));
    const int qc = (int)(r() % 1400) - 700;
    std::vector<double> c, q;
    for (int i = 0; i < 12; i++) {
      const int e = std::max(-1080, std::min(1000, centre - (int)(r() % spread)));
      c.push_back(r() % 8 ? std::ldexp(u(r), e) : 0.0);
      // neighbours in the last place, and opposite sides of the period
      if (r() % 4 == 0) c.push_back(std::nextafter(c.back(), 1.0));
      if (cycle > 0 && r() % 4 == 0) c.push_back(c.back() + cycle);
      q.push_back(std::ldexp(u(r), std::max(-1000, std::min(1000, qc - (int)(r() % spread)))));
    }
    BodyRange b{BodyRange::NONE, 0, BodyRange::NONE, 0};
    for (double v : c) {
      if (v != 0) b.lo = std::min(b.lo, exponent(v));
      b.hi = std::max(b.hi, exponent(v));
    }
    double qmin = INFINITY, qmax = 0;
    for (double v : q) {
      if (v != 0) b.qlo = std::min(b.qlo, exponent(v)), qmin = std::min(qmin, std::fabs(v));
      b.qhi = std::max(b.qhi, exponent(v));
      qmax = std::max(qmax, std::fabs(v));
    }
    const P2pFrame f = p2p_frame(b, cycle);
    if (f.wide) {
      wide++;
      continue;
    }
    scaled++;
    const double up = std::ldexp(1.0, f.scale);
    double far = 0;
    for (double x : c)
      for (double y : c)
        for (int i = cycle > 0 ? -1 : 0; i <= (cycle > 0 ? 1 : 0); i++) {
          const double d = std::fabs(x * up - (y + i * cycle) * up);
          if (d != 0 && !(d >= 2)) return printf("close %a %a %a\n", x, y, d), 1;
          far = std::max(far, d);
        }
    const double rinv = 2 / (far * std::sqrt(3.0));
    if (far > 0 && !(qmin * rinv * (rinv * rinv) >= 0x1p-1022)) return printf("far\n"), 2;
    if (!(std::isfinite(far * far * 3) && qmax < 0x1p902)) return printf("large\n"), 3;
  }
  // what programs use has a scale: a unit box and charges near 1, down to 2^-250 apart
  for (uint32_t lo : {1013u, 963u, 823u})
    if (p2p_frame({lo, 1023, 900, 1040}, 0.0).wide || p2p_frame({lo, 1023, 900, 1040}, 1.0).wide)
      return printf("ordinary\n"), 4;
  printf("scaled %ld wide %ld\n", scaled, wide);
  return 0;
}
