// p2p_range.h -- when the FP64 P2P may work on scaled coordinates with its clamp
// (p2p.hip), from the exponents of the bodies' coordinates and charges.
#pragma once
#include <cstdint>
#include <cstring>

namespace tfmm {

// Biased exponents (0 ... 2046, 0 also for denormal numbers) of the smallest and
// largest non-zero coordinate and of the smallest and largest non-zero charge;
// NONE in lo and qlo, 0 in hi and qhi where there is none.
struct BodyRange {
  static constexpr uint32_t NONE = 2047;
  uint32_t lo, hi, qlo, qhi;
};

struct P2pFrame {
  int scale;  // the coordinates are taken times 2^scale
  bool wide;  // no scale: the guard has to take any distance
};

// Every coordinate is a multiple of the last place of the smallest one, 2^g, and so
// is every difference (a displacement by the period c, 0 without images, included:
// its own last place counts as well).  Two bodies that do not coincide are therefore
// at least 2^g apart, whatever the cells' widths, and the scale makes that 2: twice
// the inverse distance never exceeds 1.  The farthest pair, at less than 2^D after
// scaling, must leave 8 q / r^3 a normal number.
#ifdef __HIPCC__
__host__ __device__
#endif
inline P2pFrame p2p_frame(BodyRange b, double c) {
  constexpr int BIAS = 1023, LAST = 52, MOST = 1000;
  int lo = (int)b.lo, hi = (int)b.hi;
  if (c > 0) {
    uint64_t bits;
    memcpy(&bits, &c, 8);
    const int e = (int)(bits >> 52);  // 0 if denormal
    lo = lo < e ? lo : e;
    hi = (hi > e ? hi : e) + 1;  // a body and its displacement
  }
  lo = lo > 1 ? lo : 1;
  const int scale = 1 - (lo - BIAS - LAST);
  const int D = hi - BIAS + 1 + 2 + scale;  // differences of two, three axes
  const bool fits = b.lo <= b.hi && scale >= -400 && scale <= 400 && 3 * D <= MOST &&
                    (int)b.qlo - BIAS - 3 * D >= -MOST && (int)b.qhi - BIAS <= 900;
  return {fits ? scale : 0, !fits};
}

}  // namespace tfmm
