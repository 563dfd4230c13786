// m2l_groups.h -- the direct-mapped table of M2L offset groups, shared by
// the traversal (which gives every M2L pair its slot as it emits the pair)
// and the batched M2L (which turns the used slots into groups).
#pragma once
#include <cmath>
#include <cstdint>

namespace tfmm {
namespace m2lg {

// Slot of a (level difference, offset) in the direct-mapped table, and the
// mirror bits of the offset: offsets are in units of half the finer width;
// same-level offsets are even with |o| <= 22, offsets across levels odd with
// |o| <= 23.  An M2L pair's parents were not well separated, so a same-level
// or adjacent-level offset is at most about 2 (2 / theta + 1) half widths (the
// table covers theta >= 0.2 there); pairs 2 or 3 levels apart, which a leaf
// next to a much finer region makes, reach |o| = 15 and 23 at theta = 0.4.
//
// In units of the cells' widths the operator of an offset does not depend on
// the level.  The operators of mirrored offsets differ by signs only: for the
// reflection R of any of the axes, T(R o) = S T(o) S with S = diag(+-1) over
// the coefficients (mirror_sign).  So one group holds the offsets of the
// non-negative octant, of every level; the pair keeps which axes to mirror.
constexpr int SAME_N = 12;   // |o| / 2 in [0, 11]
constexpr int CROSS_N = 12;  // (|o| - 1) / 2 in [0, 11]
constexpr int DL_MAX = 3;    // level differences -3 .. 3
constexpr int SLOTS_SAME = SAME_N * SAME_N * SAME_N;
constexpr int SLOTS_CROSS = CROSS_N * CROSS_N * CROSS_N;
constexpr int SLOTS = SLOTS_SAME + 2 * DL_MAX * SLOTS_CROSS;
constexpr int MIRROR_BITS = 3;  // bit d: axis d mirrored
// slot << MIRROR_BITS | mirror bits, or -1 outside the table
__host__ __device__ inline int32_t group_slot(int lt, int ls, const int o[3]) {
  const int dl = ls - lt;
  if (dl < -DL_MAX || dl > DL_MAX) return -1;
  const int parity = dl == 0 ? 0 : 1, n = dl == 0 ? SAME_N : CROSS_N;
  int idx = 0, mirror = 0;
  for (int d = 0; d < 3; d++) {
    if ((o[d] & 1) != parity) return -1;
    const int m = o[d] < 0 ? -o[d] : o[d];
    if (m / 2 >= n) return -1;
    idx = idx * n + m / 2;
    mirror |= o[d] < 0 ? 1 << d : 0;
  }
  if (dl != 0) idx += SLOTS_SAME + (2 * ((dl > 0 ? dl : -dl) - 1) + (dl < 0 ? 1 : 0)) * SLOTS_CROSS;
  return idx << MIRROR_BITS | mirror;
}
// level difference (source less target) and offset of a slot
__host__ __device__ inline void slot_decode(int32_t idx, int &dl, int o[3]) {
  const bool same = idx < SLOTS_SAME;
  const int blk = same ? 0 : (idx - SLOTS_SAME) / SLOTS_CROSS;
  dl = same ? 0 : (blk & 1) ? -(blk / 2 + 1) : blk / 2 + 1;
  int r = same ? idx : (idx - SLOTS_SAME) % SLOTS_CROSS;
  const int n = same ? SAME_N : CROSS_N;
  for (int d = 2; d >= 0; d--) {
    o[d] = 2 * (r % n) + (same ? 0 : 1);
    r /= n;
  }
}
// 1 if mirroring axis d changes the sign of coefficient row r = 2 tri(n, m) +
// (0 re | 1 im): Y_n^m(x, y, -z) = (-1)^(n+m) Y_n^m, Y_n^m(x, -y, z) is the
// conjugate, and -x is the conjugate times (-1)^m.  Rows past the 110
// coefficients never change.
__host__ __device__ constexpr int mirror_sign(int d, int r) {
  if (r >= 110) return 0;
  int n = 0;
  while ((n + 1) * (n + 2) / 2 <= r / 2) n++;
  const int m = r / 2 - n * (n + 1) / 2;
  return d == 2 ? (n + m) & 1 : d == 1 ? r & 1 : (m + r) & 1;
}

// slot of an M2L pair from the cells' depths and the offset of target less source
// in half widths of the finer cell, up to rounding; -1 outside the table
__device__ inline int32_t offset_slot(int lt, int ls, const double *v) {
  int o[3];
  for (int d = 0; d < 3; d++) {
    if (!(fabs(v[d]) < 64.0)) return -1;
    o[d] = (int)rint(v[d]);
  }
  return group_slot(lt, ls, o);
}

// the same from the cells' depths, widths (max over the dimensions) and centres
__device__ inline int32_t pair_slot(int lt, int ls, double wt, double ws, const double *ct,
                                    const double *cs) {
  const double half = 0.5 * fmin(wt, ws);
  const double v[3] = {(ct[0] - cs[0]) / half, (ct[1] - cs[1]) / half, (ct[2] - cs[2]) / half};
  return offset_slot(lt, ls, v);
}

}  // namespace m2lg
}  // namespace tfmm
