// m2l_batched.hip -- M2L regrouped by relative cell offset and run as
// block-sparse batched contractions on the gfx950 matrix cores (MFMA).
//
// Math (reference: LaplaceSphericalCPU_tapas.h:208-273, evalLocal :102-135):
// the M2L of one pair is a linear map of the source's 55 complex multipole
// coefficients onto the target's 55 local coefficients, whose entries are the
// singular harmonics Y_{j+n}^{m-k}(dX) with signs.  Written on real and
// imaginary parts it is a 112 x 112 real matrix T(dX) (110 + 2 padding rows
// and columns), non-zero only where j + n <= P - 1; in 16 x 16 blocks only 18
// of the 49 blocks are non-zero.
//
// Cells of one level sit on a lattice, so dX of a pair is an integer
// multiple of half the finer cell's width: pairs are grouped by
// (level difference, offset), offsets that mirror each other in one group
// (their operators differ by signs, which the kernel applies to the operands
// as it takes a group's mirror).  Every pair of a group shares T, so a group's pairs
// become the columns of a matrix product T * [M_s1 ... M_s16].  The harmonics
// of each group are formed once, in FP64.
//
// Scaling: with sigma the width of each cell, the kernel works on
//   M~_n = M_n / sigma_s^n,  L~_j = L_j sigma_t^(j+1),  Y~_p = Y_p sigma_t^(p+1)
// so that L~_j = sum_n 2^(n (l_t - l_s)) Y~_(j+n) M~_n with all quantities
// O(1): FP32 neither under- nor overflows at P = 10 on deep trees, and the
// power-of-two factors are exact.  Y~ depends only on the offset in units of
// the cells' widths, so one group serves every tree of a batch.
//
// Work decomposition: targets are taken in sets of 16 consecutive cells (breadth
// first, so one set is two families of siblings), and the 16 cells are the 16
// columns of every product of the set: a column never changes its target, so
// the 110 x 16 local expansions of a set stay in one wave's MFMA accumulators
// over all its work, and nothing is read, added and written back per item.  The
// pairs of a set are sorted by group; a work item is one group and, for each
// target, one of the target's pairs in that group (in different mirrors, since
// a target meets each offset once), or none.  That the mirrors of an offset
// share a group is what fills the columns: siblings see the same offsets
// mirrored, and a target at the edge of a region lacks some mirrors of many
// offsets rather than whole offsets.  An item is 61 MFMA 16x16x4 steps.  A
// set's items are cut into work units, one wave each, so that few or uneven
// sets still fill the chip; the first unit writes the set's local expansions,
// the others leave FP64 slabs that a second kernel adds in unit order.  Pairs
// whose offset falls outside the group table (level difference above 3, or an
// offset beyond the table's range) go to the per-pair kernel of m2l.hip.
//
// Per-group factors: the level factor 2^(n dl), n the source degree and
// dl = l_t - l_s, is split as 2^(p dl) 2^(-j dl) with p = j + n, the first
// folded into the group's harmonics (index p) and the second into the rows
// (degree j) of the group's A operands, which are formed once per group
// before the set kernel; both are exact powers of two.
#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

#include "m2l_codes.h"
#include "m2l_groups.h"
#include "tfmm_device.h"
#include "tfmm_kernels.h"
#include "tfmm_internal.h"

namespace tfmm {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d4 __attribute__((ext_vector_type(4)));

using m2lc::BLK_CB;
using m2lc::BLK_RB;
using m2lc::NBLK;
using m2lc::NR;
constexpr int NCODE = NBLK * 4 * 64;
constexpr int SRC_BITS = 25;  // source cell bits of a grouped pair's value
constexpr int TILE = 16;      // cells of a target set
constexpr int SET_BITS = 4;

// ---------------------------------------------------------------------------
// group table
// ---------------------------------------------------------------------------
using m2lg::MIRROR_BITS;
// A grouped pair's value and an item's column word: source cell (SRC_BITS) |
// in a value the target's place in its set << SRC_BITS | mirror bits << MIR_AT.
constexpr int MIR_AT = SRC_BITS + SET_BITS;
static_assert(MIR_AT + MIRROR_BITS == 32, "a value is one word");

// Split the executed M2L pairs into grouped ones (sort key: set << gbits |
// group) and the rest (key: target | source).  Among the pairs of one key,
// target and mirror name the pair (a target has one level, so they fix the
// source): k_items places each by them alone, whatever order the traversal's
// atomics left.
// Grouped keys stay at the pair's index; a pair outside the groups leaves
// the key NO_GROUP there, which sorts after every grouped key (the set
// field of a key is at most 2^tbits - 2), so a sort of all n keys puts the
// grouped pairs first.  The pairs outside the groups are appended compactly
// (counters[1], one atomic per block that has any); k_grouped_count then
// sets counters[0] to the grouped count.
// With dn the pair count is *dn (n its capacity), and group indices are
// clamped below gcap (a capacity the caller checks after the launch).
constexpr uint32_t NO_GROUP = 0xffffffffu;

__device__ inline uint32_t pair_value(int2 p, uint32_t slot) {
  return ((uint32_t)p.y & CELL_MASK) | ((uint32_t)p.x % TILE) << SRC_BITS |
         (slot & ((1u << MIRROR_BITS) - 1u)) << MIR_AT;
}

__global__ __launch_bounds__(1024) void k_classify(const int2 *pairs, const int32_t *slot_of,
                                                  uint32_t n, const uint32_t *gid_of_slot, int gbits,
                                                  int sbits, uint32_t *gkeys, uint32_t *gvals,
                                                  uint64_t *fkeys, uint32_t *fvals,
                                                  uint32_t *counters, const uint32_t *dn,
                                                  uint32_t gcap) {
  critical_path_priority();
  __shared__ uint32_t scratch[17];
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) counters[2] = 0;  // no repeats (k_items)
  if (dn) n = min(n, *dn);
  const bool valid = i < n;
  int2 p = make_int2(0, 0);
  int32_t slot = -1;
  if (valid) {
    p = pairs[i];
    slot = slot_of[i];
  }
  const bool grouped = valid && slot >= 0;
  const bool fallback = valid && slot < 0;
  if (valid) {
    gkeys[i] = grouped ? ((uint32_t)p.x / TILE) << gbits | min(gid_of_slot[slot >> MIRROR_BITS], gcap - 1u)
                       : NO_GROUP;
    gvals[i] = grouped ? pair_value(p, (uint32_t)slot) : 0u;
  }
  if (!__syncthreads_or(fallback)) return;  // the usual block: nothing outside the groups
  const uint32_t af = block_append<16>(&counters[1], fallback, 1, scratch);
  if (fallback) {
    fkeys[af] = ((uint64_t)(uint32_t)p.x << sbits) | (uint64_t)(uint32_t)p.y;
    fvals[af] = 0;
  }
}

// counters[0] = the grouped pairs: the pair count less those outside
__global__ void k_grouped_count(uint32_t n, const uint32_t *dn, uint32_t *counters) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  if (dn) n = min(n, *dn);
  counters[0] = n - min(n, counters[1]);
}

// k_classify when every pair is in the table: keys and values in pair order
__global__ void k_classify_all(const int2 *pairs, const int32_t *slot_of, uint32_t n,
                               const uint32_t *gid_of_slot, int gbits, uint32_t *gkeys,
                               uint32_t *gvals, uint32_t *counters) {
  critical_path_priority();
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) counters[2] = 0;  // no repeats (k_items)
  if (i >= n) return;
  const int2 p = pairs[i];
  const uint32_t slot = (uint32_t)slot_of[i];
  gkeys[i] = ((uint32_t)p.x / TILE) << gbits | gid_of_slot[slot >> MIRROR_BITS];
  gvals[i] = pair_value(p, slot);
}

// Harmonics of every used group, FP64, scaled: Y~_p^q = Y_p^q sigma_t^(p+1)
// 2^(p dl), dl = l_t - l_s, i.e. the harmonics of the offset measured in
// target widths.  Stored as NR reals (re/im interleaved, index 2 tri(p, q)),
// in FP64 and FP32.
constexpr int HARM_BITS = 4;
__global__ void k_group_harmonics(const uint32_t *used, const uint32_t *gid_of_slot, double *Y64,
                                  float *Y32, int8_t *gdl, uint32_t gcap) {
  critical_path_priority();
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t slot = t >> HARM_BITS;
  const int m = t & ((1 << HARM_BITS) - 1);  // one column of one slot per thread
  if (m >= P || slot >= m2lg::SLOTS || !used[slot]) return;
  const uint32_t g = gid_of_slot[slot];
  if (g >= gcap) return;  // more groups than the buffers hold (checked by the caller)
  int sl, o[3];  // source level less target level
  m2lg::slot_decode(slot, sl, o);
  const double half = ldexp(0.5, -max(sl, 0));  // half the finer width, target width = 1
  const double dx = o[0] * half, dy = o[1] * half, dz = o[2] * half;
  double rho, x, y;
  cd ei;
  sph_frame(dx, dy, dz, rho, x, y, ei);
  double *yo = Y64 + (int64_t)g * NR;
  float *yf = Y32 + (int64_t)g * NR;
  local_column(m, rho, x, y, ei, [&](int n, int mm, cd v) {
    const double sc = ldexp(1.0, -n * sl);  // 2^(n dl)
    const int t = tri(n, mm);
    yo[2 * t] = v.re * sc;
    yo[2 * t + 1] = v.im * sc;
    yf[2 * t] = (float)(v.re * sc);
    yf[2 * t + 1] = (float)(v.im * sc);
  });
  if (m > 0) return;
  yo[110] = yo[111] = 0;
  yf[110] = yf[111] = 0;
  gdl[g] = (int8_t)-sl;
}

// M~ of every cell, in the order the MFMA B operands are read: row r = 4 t + q
// (r = 2 tri(n, m) + (0 re | 1 im)) at 16 (t / 4) + 4 q + t % 4, so that the
// four lanes (q) that read a column vector (four k-steps) of one source read
// 64 contiguous bytes in FP32 (128 in FP64).  With each lane's 28 values
// contiguous instead, every lane of a load would touch a cache line of its own,
// 64 lines an instruction instead of 16.
// Cell ncells is the source of empty columns: zeros.
template <class T>
__global__ void k_scale_m(Cells c, int32_t ncells, const double *M, T *Mq) {
  critical_path_priority();
  const int32_t ci = blockIdx.x;
  if (ci > ncells) return;
  const int r = threadIdx.x;  // 0..111
  if (r >= NR) return;
  const int q = r & 3, t = r >> 2;
  double v = 0;
  if (r < 110 && ci < ncells) {
    const int tt = r >> 1;
    int n = 0;
    while (tri(n + 1, 0) <= tt) n++;
    const double w = c.width[ci];
    const double isig = w > 0 ? 1.0 / w : 0.0;  // zero width: only degree 0 is non-zero
    double sc = 1;
    for (int i = 0; i < n; i++) sc *= isig;
    v = M[2 * ((int64_t)ci * NTERM + tt) + (r & 1)] * sc;
  }
  Mq[(int64_t)ci * NR + 16 * (t >> 2) + 4 * q + (t & 3)] = (T)v;
}

// ---------------------------------------------------------------------------
// work items
// ---------------------------------------------------------------------------
// The items of the sorted pairs.  The pairs of one key (a segment: one set and
// group) have at most 16 targets x 8 mirrors, each combination once, so a
// segment is a 128-bit presence mask, and everything follows from it: the
// segment needs as many items as its fullest target has pairs, and a pair goes
// to the item given by its rank among its target's mirrors.  A block handles
// the segments that start among its 1024 keys and reads 128 keys more for the
// end of the last one.  The first pass (WRITE false) counts the block's items;
// the second, with the exclusive prefix of the blocks' counts in bstart,
// writes every item's key and 16 column words (empty: empty).  With dn the
// pair count is *dn (n its capacity); items at or past items_cap are not
// written (a capacity the caller checks).  A target's place in a group may
// repeat: in lists that the caller of the library gives, and in the library's own
// where cells are as narrow as the last place of their coordinates, so that centres
// round together.  The counting pass then sets *repeats.  (A segment longer than
// the block can see has a repeat among the 129 keys that it does see.)
constexpr int IT_THREADS = 1024;
constexpr int IT_ROWS = IT_THREADS / 64 + 2;  // 2 rows after the block's own
constexpr int SEG_WORDS = TILE * 8 / 32;      // words of a segment's mask

template <bool WRITE>
__global__ __launch_bounds__(IT_THREADS) void k_items(const uint32_t *keys, const uint32_t *vals,
                                                      uint32_t n, uint32_t *bcount,
                                                      const uint32_t *bstart, uint32_t empty,
                                                      uint32_t *ikey, uint32_t *cols,
                                                      const uint32_t *dn, uint32_t items_cap,
                                                      uint32_t *repeats) {
  critical_path_priority();
  __shared__ uint32_t sk[IT_ROWS * 64];        // keys of the window
  __shared__ uint32_t rowstart[IT_ROWS + 1];   // segments that start before a row
  __shared__ uint64_t mark[IT_ROWS];           // segment starts of a row
  __shared__ uint32_t mask[IT_THREADS * SEG_WORDS];
  __shared__ uint32_t first[IT_THREADS];       // a segment's first item, in the block
  __shared__ uint32_t segkey[IT_THREADS];
  __shared__ uint32_t wsum[IT_THREADS / 64];
  if (dn) n = min(n, *dn);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t w0 = (int64_t)blockIdx.x * IT_THREADS;
  const uint32_t before = w0 > 0 && w0 - 1 < (int64_t)n ? keys[w0 - 1] : NO_GROUP;
  for (int t = threadIdx.x; t < IT_ROWS * 64; t += IT_THREADS)
    sk[t] = w0 + t < (int64_t)n ? keys[w0 + t] : NO_GROUP;
  for (int t = threadIdx.x; t < IT_THREADS * SEG_WORDS; t += IT_THREADS) mask[t] = 0;
  __syncthreads();
  for (int r = wid; r < IT_ROWS; r += IT_THREADS / 64) {
    const int t = 64 * r + lane;
    const uint64_t m = __ballot(sk[t] != NO_GROUP && sk[t] != (t ? sk[t - 1] : before));
    if (lane == 0) mark[r] = m;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t run = 0;
    for (int r = 0; r < IT_ROWS; r++) {
      rowstart[r] = run;
      run += (uint32_t)__popcll(mark[r]);
    }
    rowstart[IT_ROWS] = run;
  }
  __syncthreads();
  const uint32_t nseg = rowstart[IT_THREADS / 64];  // segments that start in the block's own keys
  const uint64_t upto = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);  // bits <= lane
  // segment of window key t, or -1: it starts before the block or after its keys
  auto segment = [&](int t) -> int {
    if (sk[t] == NO_GROUP) return -1;
    const int s = (int)(rowstart[t >> 6] + (uint32_t)__popcll(mark[t >> 6] & upto)) - 1;
    return s < (int)nseg ? s : -1;
  };
  for (int t = threadIdx.x; t < IT_ROWS * 64; t += IT_THREADS) {
    const int s = segment(t);
    if (s < 0) continue;
    const uint32_t v = vals[w0 + t];
    const uint32_t sl = (v >> SRC_BITS) & (TILE - 1), mi = v >> MIR_AT;
    const uint32_t bit = 1u << (8 * (sl & 3) + mi);
    if ((atomicOr(&mask[s * SEG_WORDS + (sl >> 2)], bit) & bit) && !WRITE) *repeats = 1;
    segkey[s] = sk[t];
  }
  __syncthreads();
  // items of segment threadIdx.x, and their exclusive prefix in the block
  uint32_t cnt = 0;
  if (threadIdx.x < nseg) {
    for (int w = 0; w < SEG_WORDS; w++) {
      const uint32_t m = mask[threadIdx.x * SEG_WORDS + w];
      for (int b = 0; b < 4; b++) cnt = max(cnt, (uint32_t)__popc((m >> (8 * b)) & 0xffu));
    }
  }
  uint32_t inc = cnt;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  if (lane == 63) wsum[wid] = inc;
  __syncthreads();
  uint32_t pre = 0, tot = 0;
#pragma unroll 4
  for (int w = 0; w < IT_THREADS / 64; w++) {
    pre += w < wid ? wsum[w] : 0u;
    tot += wsum[w];
  }
  if (!WRITE) {
    if (threadIdx.x == 0) bcount[blockIdx.x] = tot;
    return;
  }
  const uint32_t base = bstart[blockIdx.x];
  first[threadIdx.x] = pre + inc - cnt;
  if (threadIdx.x < nseg)
    for (uint32_t k = 0; k < cnt; k++) {
      const uint32_t it = base + first[threadIdx.x] + k;
      if (it < items_cap) ikey[it] = segkey[threadIdx.x];
    }
  __syncthreads();
  // the pairs' columns
  for (int t = threadIdx.x; t < IT_ROWS * 64; t += IT_THREADS) {
    const int s = segment(t);
    if (s < 0) continue;
    const uint32_t v = vals[w0 + t];
    const uint32_t sl = (v >> SRC_BITS) & (TILE - 1), mi = v >> MIR_AT;
    const uint32_t m = (mask[s * SEG_WORDS + (sl >> 2)] >> (8 * (sl & 3))) & 0xffu;
    const uint32_t it = base + first[s] + (uint32_t)__popc(m & ((1u << mi) - 1u));
    if (it < items_cap)
      cols[(int64_t)it * TILE + sl] = (v & ((1u << SRC_BITS) - 1u)) | mi << MIR_AT;
  }
  // the empty columns
  for (uint32_t e = threadIdx.x; e < nseg * TILE; e += IT_THREADS) {
    const uint32_t s = e / TILE, sl = e % TILE;
    const uint32_t end = s + 1 < nseg ? first[s + 1] : tot;
    const uint32_t m = (mask[s * SEG_WORDS + (sl >> 2)] >> (8 * (sl & 3))) & 0xffu;
    for (uint32_t it = first[s] + (uint32_t)__popc(m); it < end; it++)
      if (base + it < items_cap) cols[(int64_t)(base + it) * TILE + sl] = empty;
  }
}

// first item of every set, and the set's work units (of chunk items, *dchunk
// with dchunk; at least one)
__global__ void k_set_offsets(const uint32_t *ikey, uint32_t nitems, int gbits, int32_t nsets,
                              int32_t *off, int32_t chunk, uint32_t *ucnt,
                              const uint32_t *dnitems, const int32_t *dchunk) {
  critical_path_priority();
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > nsets) return;
  if (dnitems) nitems = min(nitems, *dnitems);
  if (dchunk) chunk = *dchunk;
  // the first items of sets t and t + 1, their searches in step
  uint32_t lo = 0, hi = nitems, lo1 = 0, hi1 = nitems;
  while (lo < hi || lo1 < hi1) {
    const uint32_t mid = lo + ((hi - lo) >> 1), mid1 = lo1 + ((hi1 - lo1) >> 1);
    const uint32_t k = lo < hi ? ikey[mid] : 0u, k1 = lo1 < hi1 ? ikey[mid1] : 0u;
    if (lo < hi) {
      if ((k >> gbits) < (uint32_t)t) lo = mid + 1;
      else hi = mid;
    }
    if (lo1 < hi1) {
      if ((k1 >> gbits) <= (uint32_t)t) lo1 = mid1 + 1;
      else hi1 = mid1;
    }
  }
  off[t] = (int32_t)lo;
  if (t < nsets) {
    const int32_t n = (int32_t)(lo1 - lo);
    ucnt[t] = n > chunk ? (uint32_t)((n + chunk - 1) / chunk) : 1u;
  }
}

// ---------------------------------------------------------------------------
// the set kernel
// ---------------------------------------------------------------------------
template <class T>
struct Mfma;
// Operands (both types): lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16].  Result i of lane l is D[row(l / 16, i)][l % 16], with
// the row order differing between the two instructions (checked on gfx950).
template <>
struct Mfma<float> {
  typedef f4 V;
  static __device__ inline V step(float a, float b, V c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ constexpr int row(int q, int i) { return 4 * q + i; }
};
template <>
struct Mfma<double> {
  typedef d4 V;
  static __device__ inline V step(double a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ constexpr int row(int q, int i) { return q + 4 * i; }
};

// The steps of one item.  T has 7 row blocks of 16 rows and 28 k-steps of 4
// columns; the step (row block, k-step) is non-zero only while the smallest
// degrees of its rows and columns add up to at most P - 1, which leaves 61 of
// the 196 (18 whole 16 x 16 blocks would be 72): the first RB_STEPS[rb] k-steps
// of row block rb.  The last three row blocks (6 steps) are taken in turn, then
// the others upwards, the first, which needs every k-step, last: a B vector then
// has its last use early enough to be loaded over itself for the next item at
// least 24 steps before that item's first use of it.
constexpr int NRB = 7;
constexpr int RB_STEPS[NRB] = {28, 14, 8, 5, 3, 2, 1};
constexpr int NST = 61;
constexpr int NAV = (NST + 3) / 4;  // A operand vectors of an item (four steps each)
constexpr int NBV = NR / 16;        // B operand vectors (four k-steps each)

__host__ __device__ constexpr int coef_degree(int r) {
  int n = 0;
  while ((n + 1) * (n + 2) / 2 <= r / 2) n++;
  return n;
}
constexpr bool steps_cover() {
  int n = 0;
  for (int rb = 0; rb < NRB; rb++)
    for (int t = 0; t < 28; t++) {
      const bool need = coef_degree(16 * rb) + coef_degree(4 * t) <= P - 1;
      if (need != (t < RB_STEPS[rb])) return false;
      n += need;
    }
  return n == NST;
}
static_assert(steps_cover(), "every non-zero k-step of the operator once");
// row block, k-step and MFMA block (m2l_codes.h; block * 4 + k-step in it) of
// every step, -1 for the padding of the last vector
struct StepTab {
  int16_t rb[NAV * 4], t[NAV * 4], code[NAV * 4];
};
constexpr StepTab make_steps() {
  StepTab s{};
  int n = 0;
  for (int t = 0; t < 3; t++)
    for (int rb = 4; rb < NRB; rb++)
      if (t < RB_STEPS[rb]) {
        s.rb[n] = (int16_t)rb;
        s.t[n++] = (int16_t)t;
      }
  for (int rb = 3; rb >= 0; rb--)
    for (int t = 0; t < RB_STEPS[rb]; t++, n++) {
      s.rb[n] = (int16_t)rb;
      s.t[n] = (int16_t)t;
    }
  for (int i = 0; i < n; i++)
    for (int b = 0; b < NBLK; b++)
      if (BLK_RB[b] == s.rb[i] && BLK_CB[b] == s.t[i] / 4) s.code[i] = (int16_t)(4 * b + s.t[i] % 4);
  for (; n < NAV * 4; n++) s.rb[n] = s.t[n] = s.code[n] = -1;
  return s;
}
constexpr StepTab STEP = make_steps();
__constant__ StepTab c_steps = make_steps();
// first step of k-step t, last step that uses B vector v, and the last step of row
// block rb
constexpr int first_use(int t) {
  int i = 0;
  while (STEP.t[i] != t) i++;
  return i;
}
constexpr int last_use(int v) {
  int i = NST - 1;
  while (STEP.t[i] / 4 != v) i--;
  return i;
}
constexpr int last_step(int rb) {
  int i = NST - 1;
  while (STEP.rb[i] != rb) i--;
  return i;
}

__device__ inline int row_degree(int r) {
  if (r >= 110) return 0;
  const int t = r >> 1;
  int n = 0;
  while (tri(n + 1, 0) <= t) n++;
  return n;
}

// A operands of every group, in the order the set kernel's lanes read them:
// Af[g][s / 4][lane][s % 4] is what lane supplies at step s (four steps are a
// 16-byte vector per lane in FP32, 32 in FP64).
constexpr int AF_PER_GROUP = NAV * 4 * 64;  // elements per group

template <class T>
struct Vec4;
template <>
struct Vec4<float> {
  typedef f4 V;
};
template <>
struct Vec4<double> {
  typedef d4 V;
};

// Signs of a mirrored offset (m2l_groups.h): T(R o) = S T(o) S.  The operator
// stays that of the unmirrored offset; a column's source and its products are
// multiplied by S.  Bit t of b[d][q]: mirroring axis d changes the sign of row
// 4 t + q (a lane's B operands).
// p[FP64][d][q]: the same for bit 4 rb + i, result i of row block rb.
struct MirrorTab {
  uint32_t b[3][4], p[2][3][4];
};
constexpr MirrorTab make_mirror() {
  MirrorTab t{};
  for (int d = 0; d < 3; d++) {
    for (int r = 0; r < NR; r++) t.b[d][r & 3] |= (uint32_t)m2lg::mirror_sign(d, r) << (r >> 2);
    for (int q = 0; q < 4; q++)
      for (int rb = 0; rb < NRB; rb++)
        for (int i = 0; i < 4; i++) {
          const int bit = 4 * rb + i;
          t.p[0][d][q] |= (uint32_t)m2lg::mirror_sign(d, 16 * rb + Mfma<float>::row(q, i)) << bit;
          t.p[1][d][q] |= (uint32_t)m2lg::mirror_sign(d, 16 * rb + Mfma<double>::row(q, i)) << bit;
        }
  }
  return t;
}
__constant__ MirrorTab c_mirror = make_mirror();

// a lane's sign masks for the three axes: its B operands and its products
struct LaneSigns {
  uint32_t b[3], p[3];
  __device__ static uint32_t of(const uint32_t (&m)[3], uint32_t mirror) {
    return ((mirror & 1u) ? m[0] : 0u) ^ ((mirror & 2u) ? m[1] : 0u) ^ ((mirror & 4u) ? m[2] : 0u);
  }
};
template <class T>
__device__ inline LaneSigns lane_signs(int q) {
  LaneSigns s;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    s.b[d] = c_mirror.b[d][q];
    s.p[d] = c_mirror.p[sizeof(T) == 8][d][q];
  }
  return s;
}

// x with its sign changed where bit `at` of mask is set
__device__ inline float flip(float x, uint32_t mask, int at) {
  return __uint_as_float(__float_as_uint(x) ^ ((mask << (31 - at)) & 0x80000000u));
}
__device__ inline double flip(double x, uint32_t mask, int at) {
  return __hiloint2double(__double2hiint(x) ^ (int)((mask << (31 - at)) & 0x80000000u),
                          __double2loint(x));
}

// sums of row block rb += products, with their signs: result i
template <class T>
__device__ inline void add_product(typename Mfma<T>::V (&sum)[NRB], int rb,
                                   const typename Mfma<T>::V &v, uint32_t signs, int i) {
  sum[rb][i] += flip(v[i], signs, 4 * rb + i);
  asm volatile("" : "+v"(sum[rb][i]));  // added here, not when the sum is next needed
}

// One wave's registers: the A operands of the next steps, the B operands, the
// sums, and the products of the item before's last row block (with their signs),
// which are added during this one.
constexpr int RING = 4;  // A vectors held: 16 steps ahead
static_assert(NAV % RING == 0, "an A vector's place is the same in every item");
template <class T>
struct SetRegs {
  typename Vec4<T>::V a[RING], b[NBV];
  typename Mfma<T>::V sum[NRB], late;
  uint32_t late_signs;
};

// One item: 61 MFMAs, and between them the loads of what comes next, every vector
// over itself once its last step is issued: the A operands RING vectors ahead
// (af, then the next item's afn), the next item's B operands from next.  A wave
// issues in order and waits at an MFMA until the matrix unit is free, so what is
// written between two MFMAs costs little as long as it is short.  The steps are
// kept in this order (sched_barrier): the compiler would lift the loads above the
// vectors' last uses, into registers of their own, and move the values back at
// the end, waiting for them.  The A operands are read again for an item of the
// same group: holding all 61 for as long as a group lasts took 225 registers (446
// in FP64) instead of 128 (217), two waves a SIMD instead of four (one instead of
// two).  Alone, us, then and now (the shortest units last, see k_unit_map,
// included): 4M Plummer 2,830 and 2,610, 256 problems 3,020 and 2,820, 1M cube FP64
// 1,420 and 1,255, 500K ellipsoid FP64 1,770 and 1,700.
// Every row block's products are summed from zero over the item and then added
// to the target's sums: long chains into the sums themselves would lose more to
// rounding in FP32 (relative 1.2e-6 between two groupings of one problem's
// pairs, against 6e-7).  They are added four steps after their last one (an
// MFMA's results take a while to arrive), one result a step.  bs, ss: signs of b and
// of the products.
template <class T, int S>
__device__ inline void set_step(SetRegs<T> &r, typename Mfma<T>::V (&p)[NRB], uint32_t bs,
                                uint32_t ss, const T *next, const T *af, const T *afn) {
  typedef typename Vec4<T>::V V;
  constexpr int rb = STEP.rb[S], t = STEP.t[S], v = t / 4, k = S / 4;
  if constexpr (S == first_use(t)) r.b[v][t % 4] = flip(r.b[v][t % 4], bs, t);
  if constexpr (t == 0) p[rb] = (typename Mfma<T>::V){0, 0, 0, 0};
  p[rb] = Mfma<T>::step(r.a[k % RING][S % 4], r.b[v][t % 4], p[rb]);
  if constexpr (S >= 4 && S < 8) add_product<T>(r.sum, 0, r.late, r.late_signs, S - 4);
#pragma unroll
  for (int i = 1; i < NRB; i++)
    if (S >= last_step(i) + 4 && S < last_step(i) + 8)
      add_product<T>(r.sum, i, p[i], ss, S - last_step(i) - 4);
  if constexpr (S == last_use(v)) r.b[v] = *reinterpret_cast<const V *>(next + 16 * v);
  if constexpr (S % 4 == 3 || S == NST - 1)
    r.a[k % RING] = *reinterpret_cast<const V *>(
        k + RING < NAV ? af + (k + RING) * 256 : afn + (k + RING - NAV) * 256);
  __builtin_amdgcn_sched_barrier(0);
}

template <class T, int... S>
__device__ inline void set_steps(std::integer_sequence<int, S...>, SetRegs<T> &r, uint32_t bs,
                                 uint32_t ss, const T *next, const T *af, const T *afn) {
  typename Mfma<T>::V p[NRB];
  (set_step<T, S>(r, p, bs, ss, next, af, afn), ...);
  r.late = p[0];
  r.late_signs = ss;
}

// Workgroups are dispatched to the 8 XCDs round robin (workgroup b to XCD
// b % 8) and every XCD has its own L2.  Consecutive sets are neighbouring
// target ranges of one level and share most of their source cells, so units
// are dealt out in runs of RUN_UNITS x run consecutive units, one run per XCD
// in turn: the units an XCD runs at the same time read the same sources from
// its L2.  The last partial round keeps the identity order (a bijection).
// The run length is a tuning knob (32 by default).
constexpr int RUN_UNITS = 8;
constexpr int NXCD = 8;
__device__ inline int unit_of_block(int b, int nunits, int run) {
  run *= RUN_UNITS;
  const int S = NXCD * run;
  if (b >= (nunits / S) * S) return b;
  const int local = b % S;
  return (b - local) + (local % NXCD) * run + local / NXCD;
}

// Work units: unit k of a set is its items [k chunk, (k + 1) chunk).  The first
// unit writes the set's L, the others leave theirs in part[] (one 16 x 110 slab
// per extra unit, FP64), which k_unit_combine adds in unit order after the
// launch, so the sums do not depend on timing.
// (set, number) of every unit, 16 threads a set: all whole units first, then every
// set's last one, which is the shortest: the launch ends on short units.
__global__ void k_unit_map(const uint32_t *ucnt, const uint32_t *uoff, int32_t ntiles,
                           int2 *units, uint32_t units_cap) {
  critical_path_priority();
  const int32_t t = (blockIdx.x * blockDim.x + threadIdx.x) >> 4;
  if (t >= ntiles) return;
  const uint32_t n = ucnt[t], o = uoff[t] - (uint32_t)t;
  const uint32_t total = uoff[ntiles - 1] + ucnt[ntiles - 1];
  for (uint32_t k = threadIdx.x & 15; k < n; k += 16) {
    const uint32_t at = k + 1 < n ? o + k : total - (uint32_t)(ntiles - t);
    if (at < units_cap) units[at] = make_int2(t, (int)k);
  }
}

// slab of extra unit k >= 1 of tile t: every tile has at least one unit
__device__ inline int64_t extra_slab(const uint32_t *uoff, int32_t t, int k) {
  return (int64_t)uoff[t] - t + k - 1;
}

// nslab: slabs the part buffer holds (units past them were not run; the
// caller checks the unit count against its capacity)
__global__ void k_unit_combine(const uint32_t *ucnt, const uint32_t *uoff, int32_t ntiles,
                               const double *part, int32_t ncells, double *L, int64_t nslab) {
  critical_path_priority();
  const int32_t t = blockIdx.x;
  int n = (int)ucnt[t];
  while (n > 1 && extra_slab(uoff, t, n - 1) >= nslab) n--;
  if (n <= 1) return;
  const int32_t first = t * TILE;
  const int e = blockIdx.y * blockDim.x + threadIdx.x;
  if (e >= TILE * 110) return;
  const int sl = e / 110, row = e - sl * 110;
  const int32_t ci = first + sl;
  if (ci >= ncells) return;
  double *dst = &L[2 * ((int64_t)ci * NTERM + (row >> 1)) + (row & 1)];
  const double *p = part + extra_slab(uoff, t, 1) * (TILE * 110) + e;
  double v = *dst;
  int k = 1;
  for (; k + 8 <= n; k += 8) {  // eight loads in flight, added in order
    double x[8];
#pragma unroll
    for (int i = 0; i < 8; i++) x[i] = p[(int64_t)(k - 1 + i) * (TILE * 110)];
#pragma unroll
    for (int i = 0; i < 8; i++) v += x[i];
  }
  for (; k < n; k++) v += p[(int64_t)(k - 1) * (TILE * 110)];
  *dst = v;
}

// A fragments of every group from its harmonics: the entry that lane
// supplies at (block, k-step) is the sum of two table elements addressed by
// the operand code (byte offsets into the harmonics at multiples +1, -1, +2,
// -2); the multiples are exact, so each entry is formed with one rounding.
template <class T>
__device__ inline T table_elem(const T *y, uint32_t byte_off) {
  const uint32_t i = byte_off / (uint32_t)sizeof(T);
  const uint32_t m = i / NR;
  const T v = y[i - m * NR];
  return m == 0 ? v : m == 1 ? -v : m == 2 ? v + v : -(v + v);
}

template <class T>
__global__ void k_group_afrag(const T *Yg, uint32_t ng, const uint32_t *codes, const int8_t *gdl,
                              T *Af, const uint32_t *dng) {
  critical_path_priority();
  constexpr int VPG = AF_PER_GROUP / 4;  // vectors per group
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (dng) ng = min(ng, *dng);
  if (t >= (int64_t)ng * VPG) return;
  const int64_t g = t / VPG;
  const int r = (int)(t - g * VPG);
  const int slot = r >> 6, lane = r & 63;
  const T *y = Yg + g * NR;
  typename Vec4<T>::V out;
#pragma unroll
  for (int kk = 0; kk < 4; kk++) {
    const int at = c_steps.code[slot * 4 + kk];
    if (at < 0) {
      out[kk] = 0;
      continue;
    }
    // row factor 2^(-j dl) of the entry's row (degree j)
    const int rexp = -row_degree(BLK_RB[at >> 2] * 16 + (lane & 15)) * (int)gdl[g];
    const uint32_t cw = codes[at * 64 + lane];
    out[kk] = ldexp(table_elem(y, cw & 0xffffu) + table_elem(y, cw >> 16), rexp);
  }
  *reinterpret_cast<typename Vec4<T>::V *>(Af + t * 4) = out;
}

// degree of result i of row block rb: a constant per lane quarter q
template <class T>
__device__ inline int result_degree(int rb, int i, int q) {
  uint32_t d = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int row = 16 * rb + Mfma<T>::row(k, i);
    d |= (uint32_t)(row < 110 ? coef_degree(row) : 0) << (8 * k);
  }
  return (int)((d >> (8 * q)) & 0xffu);
}

// One work unit per wave.
template <class T>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2)))
void k_m2l_sets(
    const int32_t *set_off, const int2 *units, const uint32_t *ucnt, const uint32_t *uoff,
    int32_t nsets, int32_t chunk, int xcd_run, const uint32_t *ikey, int gbits,
    const uint32_t *cols, const T *Af, const T *Mq, Cells c, int32_t ncells, double *L,
    double *part, const int32_t *dchunk, int64_t nslab) {
  critical_path_priority();
  typedef typename Vec4<T>::V V;
  const int lane = threadIdx.x & 63;
  const int q = lane >> 4, j = lane & 15;
  const int u = unit_of_block(blockIdx.x, gridDim.x, xcd_run);
  if ((uint32_t)u >= uoff[nsets - 1] + ucnt[nsets - 1]) return;  // grid is an upper bound
  const int2 su = units[u];
  const int set = su.x, k = su.y;
  if (k > 0 && extra_slab(uoff, set, k) >= nslab) return;  // no slab (capacity exceeded)
  if (dchunk) chunk = *dchunk;
  const int32_t sb = set_off[set], se = set_off[set + 1];
  const int32_t ib = (int32_t)min((int64_t)sb + (int64_t)k * chunk, (int64_t)se);
  const int32_t ie = (int32_t)min((int64_t)ib + chunk, (int64_t)se);
  SetRegs<T> r;
#pragma unroll
  for (int rb = 0; rb < NRB; rb++) r.sum[rb] = (typename Mfma<T>::V){0, 0, 0, 0};
  if (ib < ie) {
    const int32_t last = ie - 1;
    const uint32_t gmask = (1u << gbits) - 1u;
    auto word = [&](int32_t it) { return cols[(int64_t)min(it, last) * TILE + j]; };
    auto key = [&](int32_t it) { return ikey[min(it, last)]; };
    auto group = [&](uint32_t k) {
      return (uint32_t)__builtin_amdgcn_readfirstlane((int)(k & gmask));
    };
    auto source = [&](uint32_t w) {
      return Mq + (int64_t)(w & ((1u << SRC_BITS) - 1u)) * NR + 4 * q;
    };
    auto operands = [&](uint32_t g) { return Af + (int64_t)g * AF_PER_GROUP + lane * 4; };
    const LaneSigns signs = lane_signs<T>(q);
    // keys and column words are loaded two items ahead of their use
    uint32_t w0 = word(ib), w1 = word(ib + 1), k1 = key(ib + 1);
    const T *af = operands(group(key(ib)));
    {
      const T *m = source(w0);
#pragma unroll
      for (int v = 0; v < NBV; v++) r.b[v] = *reinterpret_cast<const V *>(m + 16 * v);
#pragma unroll
      for (int v = 0; v < RING; v++) r.a[v] = *reinterpret_cast<const V *>(af + v * 256);
    }
    r.late = (typename Mfma<T>::V){0, 0, 0, 0};
    r.late_signs = 0;
    for (int32_t it = ib; it < ie; it++) {
      const uint32_t m = w0 >> MIR_AT;
      const T *afn = operands(group(k1)), *next = source(w1);
      w0 = w1;
      w1 = word(it + 2);
      k1 = key(it + 2);
      set_steps<T>(std::make_integer_sequence<int, NST>{}, r, LaneSigns::of(signs.b, m),
                   LaneSigns::of(signs.p, m), next, af, afn);
      af = afn;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) add_product<T>(r.sum, 0, r.late, r.late_signs, i);
  }
  // L_j = L~_j / sigma_t^(j+1)
  const int32_t ci = set * TILE + j;
  if (ci >= ncells) return;
  const double w = c.width[ci];
  double *dst = k ? part + extra_slab(uoff, set, k) * (TILE * 110) + j * 110
                  : L + 2 * (int64_t)ci * NTERM;
  const double p1 = 1.0 / w, p2 = p1 * p1, p4 = p2 * p2, p8 = p4 * p4;
#pragma unroll
  for (int rb = 0; rb < NRB; rb++) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int row = 16 * rb + Mfma<T>::row(q, i);
      const double v = (double)r.sum[rb][i];
      const int n = result_degree<T>(rb, i, q);
      double out = 0;
      if (v != 0) {  // (nothing arrived; a zero-width tree must not form 0 * inf)
        double sc = p1;
        if (n & 1) sc *= p1;
        if (n & 2) sc *= p2;
        if (n & 4) sc *= p4;
        if (n & 8) sc *= p8;
        out = v * sc;
      }
      if (row < 110) dst[row] = out;
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

// Operand codes of both element types, FP32 first (NCODE words each).
hipError_t m2l_upload_codes(uint32_t *dev_codes, hipStream_t s) {
  std::vector<uint32_t> c32, c64;
  if (!m2lc::build_codes(c32, 4) || !m2lc::build_codes(c64, 8)) return hipErrorInvalidValue;
  if (c32.size() != (size_t)NCODE || c64.size() != (size_t)NCODE) return hipErrorInvalidValue;
  c32.insert(c32.end(), c64.begin(), c64.end());
  hipError_t e = hipMemcpyAsync(dev_codes, c32.data(), c32.size() * 4, hipMemcpyHostToDevice, s);
  if (e != hipSuccess) return e;
  return hipStreamSynchronize(s);
}

size_t m2l_codes_bytes() { return (size_t)2 * NCODE * 4; }

int32_t m2l_group_slots() { return m2lg::SLOTS; }

hipError_t launch_m2l_classify_all(const int2 *pairs, const int32_t *slot_of, uint32_t n,
                                   const uint32_t *gid_of_slot, int gbits, uint32_t *gkeys,
                                   uint32_t *gvals, uint32_t *counters, hipStream_t s) {
  if (n == 0) return hipSuccess;
  k_classify_all<<<(n + 255) / 256, 256, 0, s>>>(pairs, slot_of, n, gid_of_slot, gbits, gkeys,
                                                 gvals, counters);
  return hipGetLastError();
}

hipError_t launch_m2l_classify(const int2 *pairs, const int32_t *slot_of, uint32_t n,
                               const uint32_t *gid_of_slot, int gbits, int sbits,
                               uint32_t *gkeys, uint32_t *gvals, uint64_t *fkeys,
                               uint32_t *fvals, uint32_t *counters, hipStream_t s,
                               const uint32_t *dn, uint32_t gcap) {
  if (n == 0) return hipSuccess;
  k_classify<<<(n + 1023) / 1024, 1024, 0, s>>>(pairs, slot_of, n, gid_of_slot, gbits, sbits,
                                                  gkeys, gvals, fkeys, fvals, counters, dn,
                                                  gcap);
  k_grouped_count<<<1, 64, 0, s>>>(n, dn, counters);
  return hipGetLastError();
}

hipError_t launch_m2l_group_harmonics(const uint32_t *used, const uint32_t *gid_of_slot,
                                      double *Y64, float *Y32, int8_t *gdl, hipStream_t s,
                                      uint32_t gcap) {
  k_group_harmonics<<<((m2lg::SLOTS << HARM_BITS) + 255) / 256, 256, 0, s>>>(used, gid_of_slot, Y64, Y32, gdl, gcap);
  return hipGetLastError();
}

hipError_t launch_m2l_scale_m(Cells c, int32_t ncells, const double *M, void *Mq, bool fp32,
                              hipStream_t s) {
  if (ncells <= 0) return hipSuccess;
  if (fp32) k_scale_m<float><<<ncells + 1, NR, 0, s>>>(c, ncells, M, (float *)Mq);
  else k_scale_m<double><<<ncells + 1, NR, 0, s>>>(c, ncells, M, (double *)Mq);
  return hipGetLastError();
}

size_t m2l_mq_bytes(int64_t ncells, bool fp32) {
  return (size_t)(ncells + 1) * NR * (fp32 ? 4 : 8);
}

uint32_t m2l_item_blocks(uint32_t n) {
  return std::max<uint32_t>(1, (n + IT_THREADS - 1) / IT_THREADS);
}

// the item count on the device: the block counts summed
__global__ void k_items_total(const uint32_t *bcount, const uint32_t *bstart, uint32_t nb,
                              uint32_t *nitems) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *nitems = bstart[nb - 1] + bcount[nb - 1];
}

hipError_t launch_m2l_count_items_dev(const uint32_t *keys, const uint32_t *vals, uint32_t n,
                                      const uint32_t *dn, uint32_t *bcount, uint32_t *bstart,
                                      void *scan_tmp, uint32_t *counters, uint32_t *nitems,
                                      hipStream_t s) {
  const unsigned nb = m2l_item_blocks(n);
  k_items<false><<<nb, IT_THREADS, 0, s>>>(keys, vals, n, bcount, nullptr, 0, nullptr, nullptr, dn,
                                           0, counters + 2);
  hipError_t e = scan_exclusive_u32(bcount, bstart, nb, scan_tmp, s);
  if (e != hipSuccess) return e;
  k_items_total<<<1, 64, 0, s>>>(bcount, bstart, nb, nitems);
  return hipGetLastError();
}

hipError_t launch_m2l_count_items(const uint32_t *keys, const uint32_t *vals, uint32_t n,
                                  uint32_t *bcount, uint32_t *bstart, void *scan_tmp,
                                  uint32_t *counters, uint32_t *h_pinned, hipStream_t s) {
  h_pinned[0] = h_pinned[1] = 0;
  if (n == 0) return hipSuccess;
  hipError_t e = launch_m2l_count_items_dev(keys, vals, n, nullptr, bcount, bstart, scan_tmp,
                                            counters, counters + 3, s);
  if (e != hipSuccess) return e;
  e = hipMemcpyAsync(h_pinned, counters + 2, 8, hipMemcpyDeviceToHost, s);
  if (e != hipSuccess) return e;
  return hipStreamSynchronize(s);
}

hipError_t launch_m2l_write_items(const uint32_t *keys, const uint32_t *vals, uint32_t n,
                                  const uint32_t *bstart, int32_t ncells, uint32_t *ikey,
                                  uint32_t *cols, hipStream_t s, const uint32_t *dn,
                                  uint32_t items_cap) {
  if (n == 0) return hipSuccess;
  k_items<true><<<m2l_item_blocks(n), IT_THREADS, 0, s>>>(keys, vals, n, nullptr, bstart,
                                                          (uint32_t)ncells, ikey, cols, dn,
                                                          items_cap, nullptr);
  return hipGetLastError();
}

hipError_t launch_m2l_set_offsets(const uint32_t *ikey, uint32_t nitems, int gbits, int32_t nsets,
                                  int32_t *off, int32_t chunk, uint32_t *ucnt, hipStream_t s,
                                  const uint32_t *dnitems, const int32_t *dchunk) {
  k_set_offsets<<<(nsets + 1 + 255) / 256, 256, 0, s>>>(ikey, nitems, gbits, nsets, off, chunk,
                                                        ucnt, dnitems, dchunk);
  return hipGetLastError();
}

// Items of a work unit.  With a factor, factor x the mean items per set.
// Without, enough units for several turns of the chip's 2,048 wave slots
// (UNITS), but a unit of at least UNIT_MIN items (its start and end, about
// UNIT_MIN items' time, must not outweigh it) and at most UNIT_MAX (the last
// units to start leave the rest of the chip idle).
constexpr int UNITS = 8192, UNIT_MIN = 8, UNIT_MAX = 128;
__host__ __device__ inline int32_t unit_chunk(uint32_t nitems, int32_t nsets, double factor) {
  if (factor <= 0) {
    const uint32_t want = (nitems + UNITS - 1) / UNITS;
    return (int32_t)(want < UNIT_MIN ? UNIT_MIN : want > UNIT_MAX ? UNIT_MAX : want);
  }
  const double mean = nsets > 0 ? (double)nitems / (double)nsets : 1.0;
  return (int32_t)fmin((double)(INT32_MAX / 2), fmax((double)UNIT_MIN, ceil(mean * factor)));
}

// m2l_unit_chunk on the device, from the item and set counts there
__global__ void k_unit_chunk(const uint32_t *nitems, const uint32_t *nsets, double factor,
                             int32_t *chunk) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  *chunk = unit_chunk(*nitems, (int32_t)*nsets, factor);
}

hipError_t launch_m2l_unit_chunk(const uint32_t *nitems, const uint32_t *ntiles, double factor,
                                 int32_t *chunk, hipStream_t s) {
  k_unit_chunk<<<1, 64, 0, s>>>(nitems, ntiles, factor, chunk);
  return hipGetLastError();
}

int32_t m2l_unit_chunk(uint32_t nitems, int32_t nsets, double factor) {
  return unit_chunk(nitems, nsets, factor);
}

uint32_t m2l_units_bound(uint32_t nitems, int32_t ntiles, int32_t chunk) {
  return (uint32_t)ntiles + nitems / (uint32_t)chunk;
}

// the same for a chunk chosen on the device from at most nitems items and
// nsets sets
uint32_t m2l_units_cap(uint32_t nitems, int32_t nsets, double factor) {
  const double extra = factor > 0 ? std::ceil(nsets / factor) + 1
                                  : std::max<double>(UNITS, nitems / (double)UNIT_MAX) + 1;
  return (uint32_t)std::min<double>(UINT32_MAX / 4, nsets + extra);
}

size_t m2l_unit_part_bytes(uint32_t units_bound, int32_t ntiles) {
  const size_t extra = units_bound > (uint32_t)ntiles ? units_bound - (uint32_t)ntiles : 0;
  return std::max<size_t>(extra, 1) * TILE * 110 * 8;
}

hipError_t launch_m2l_units(int32_t ntiles, const uint32_t *ucnt, uint32_t *uoff, int2 *units,
                            void *scan_tmp, hipStream_t s, uint32_t units_cap) {
  if (ntiles <= 0) return hipSuccess;
  hipError_t e = scan_exclusive_u32(ucnt, uoff, ntiles, scan_tmp, s);
  if (e != hipSuccess) return e;
  k_unit_map<<<(ntiles + 15) / 16, 256, 0, s>>>(ucnt, uoff, ntiles, units, units_cap);
  return hipGetLastError();
}

size_t m2l_afrag_bytes(uint32_t ngroups, bool fp32) {
  return (size_t)std::max<uint32_t>(ngroups, 1) * AF_PER_GROUP * (fp32 ? 4 : 8);
}

hipError_t launch_m2l_group_afrag(const void *Yg, uint32_t ngroups, const uint32_t *codes,
                                  const int8_t *gdl, void *Af, bool fp32, hipStream_t s,
                                  const uint32_t *dng) {
  if (ngroups == 0) return hipSuccess;
  const int64_t n = (int64_t)ngroups * (AF_PER_GROUP / 4);
  const unsigned nb = (unsigned)((n + 255) / 256);
  if (fp32)
    k_group_afrag<float><<<nb, 256, 0, s>>>((const float *)Yg, ngroups, codes, gdl, (float *)Af,
                                            dng);
  else
    k_group_afrag<double><<<nb, 256, 0, s>>>((const double *)Yg, ngroups, codes + NCODE, gdl,
                                             (double *)Af, dng);
  return hipGetLastError();
}

hipError_t launch_m2l_sets(const int32_t *set_off, const int2 *units, const uint32_t *ucnt,
                           const uint32_t *uoff, int32_t nsets, int32_t chunk, int xcd_run,
                           uint32_t units_bound, const uint32_t *ikey, int gbits,
                           const uint32_t *cols, const void *Af, const void *Mq, Cells c,
                           int32_t ncells, double *L, double *part, bool fp32, hipStream_t s,
                           const int32_t *dchunk) {
  if (nsets <= 0) return hipSuccess;
  // slabs of the part buffer (m2l_unit_part_bytes)
  const int64_t nslab = units_bound > (uint32_t)nsets ? (int64_t)units_bound - nsets : 0;
  if (fp32)
    k_m2l_sets<float><<<units_bound, 64, 0, s>>>(set_off, units, ucnt, uoff, nsets, chunk, xcd_run,
                                                 ikey, gbits, cols, (const float *)Af,
                                                 (const float *)Mq, c, ncells, L, part, dchunk,
                                                 nslab);
  else
    k_m2l_sets<double><<<units_bound, 64, 0, s>>>(set_off, units, ucnt, uoff, nsets, chunk,
                                                  xcd_run, ikey, gbits, cols, (const double *)Af,
                                                  (const double *)Mq, c, ncells, L, part, dchunk,
                                                  nslab);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  k_unit_combine<<<dim3(nsets, (TILE * 110 + 255) / 256), 256, 0, s>>>(ucnt, uoff, nsets, part,
                                                                      ncells, L, nslab);
  return hipGetLastError();
}

int m2l_tile_size() { return TILE; }
int m2l_src_bits() { return SRC_BITS; }

}  // namespace tfmm
