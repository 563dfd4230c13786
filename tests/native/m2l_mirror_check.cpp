// CPU check of the mirrored M2L groups (tapas-reduce_amd/csrc/m2l_groups.h):
// every slot decodes to the offset that made it, and for offsets in all eight
// octants, on the axes and on the planes, the operator of the offset is the
// operator of its mirror image in the non-negative octant between the sign
// changes of mirror_sign, against the oracle's per-pair M2L
// (orc_m2l, LaplaceSphericalCPU_tapas.h:208-273).
// Prints "slots <number> max_rel <value>".
#define __host__
#define __device__
#include <cmath>
#include <cstdio>
#include <random>

#include "../../tapas-reduce_amd/csrc/m2l_groups.h"

extern "C" void orc_m2l(double *Li, const double *Mj, const double *dX);

using namespace tfmm::m2lg;

int main() {
  int seen = 0;
  for (int dl = -DL_MAX - 1; dl <= DL_MAX + 1; dl++)
    for (int x = -26; x <= 26; x++)
      for (int y = -26; y <= 26; y++)
        for (int z = -26; z <= 26; z++) {
          const int o[3] = {x, y, z};
          const int32_t slot = group_slot(4, 4 + dl, o);
          const bool same = dl == 0;
          bool inside = std::abs(dl) <= DL_MAX;
          for (int d = 0; d < 3; d++)
            inside = inside && (o[d] & 1) == (same ? 0 : 1) &&
                     std::abs(o[d]) <= (same ? 2 * SAME_N - 2 : 2 * CROSS_N - 1);
          if ((slot >= 0) != inside || slot >= SLOTS << MIRROR_BITS) return 1;
          if (!inside) continue;
          int sl, r[3];
          slot_decode(slot >> MIRROR_BITS, sl, r);
          for (int d = 0; d < 3; d++)
            if ((slot >> d & 1 ? -r[d] : r[d]) != o[d]) return 2;
          if (sl != dl) return 3;
          seen++;
        }
  std::mt19937_64 rng(11);
  std::uniform_real_distribution<double> u(-1, 1);
  double worst = 0;
  for (int t = 0; t < 400; t++) {
    double o[3], dx[3];
    for (int d = 0; d < 3; d++) o[d] = (double)((int)(rng() % 8));
    if (t % 5 == 0) o[t % 3] = 0;
    if (t % 7 == 0) o[0] = o[1] = 0;  // on the z axis
    if (o[0] + o[1] + o[2] < 3) o[2] += 3;
    const unsigned mirror = (unsigned)(rng() % 8);
    for (int d = 0; d < 3; d++) dx[d] = (mirror >> d & 1) ? -o[d] : o[d];
    double M[110], S[110], L[110] = {0}, Lo[110] = {0};
    for (int r = 0; r < 110; r++) M[r] = u(rng);
    for (int n = 0, r = 0; n < 10; r += 2 * (++n)) M[r + 1] = 0;  // m = 0 is real
    for (int r = 0; r < 110; r++) {
      int s = 0;
      for (int d = 0; d < 3; d++) s ^= (mirror >> d & 1) ? mirror_sign(d, r) : 0;
      S[r] = s ? -1 : 1;
    }
    orc_m2l(L, M, dx);
    for (int r = 0; r < 110; r++) M[r] *= S[r];
    orc_m2l(Lo, M, o);
    double num = 0, den = 0;
    for (int r = 0; r < 110; r++) {
      num += (L[r] - S[r] * Lo[r]) * (L[r] - S[r] * Lo[r]);
      den += L[r] * L[r];
    }
    worst = std::fmax(worst, std::sqrt(num / den));
  }
  printf("slots %d max_rel %.3e\n", seen, worst);
  return 0;
}
