// tree.hip -- octree construction on the GPU: scalar-cube bounding box,
// Morton keys, body permutation and the level-synchronous cell build.
//
// Reference semantics (cpp/include/tapas/):
//   bounding box    hot/buildtree.h:72-87 (a Vec assigned from a scalar inside a
//                   per-dimension loop: min/max over every coordinate of every
//                   body except body 0's x and y) and vec.h:39-43
//   keys            hot/buildtree.h:504-539, sfc_morton.h:387-402
//   cells           hot/buildtree.h:388-459: a cell is a leaf iff nb <= ncrit;
//                   every internal cell gets all 8 children, empty ones too;
//                   region by halving (sfc_morton.h:536-557), centre (max+min)/2
//                   (hot.h:232-238)
// The cell set is built breadth first: level d+1 is produced from level d by
// one scan over the "split" flags, so cells of one level are contiguous and
// the 8 children of a cell are adjacent, which the level-synchronous upward
// and downward passes rely on.
#include <algorithm>

#include "tfmm_device.h"
#include "tfmm_kernels.h"

namespace tfmm {
namespace {

constexpr int BB_THREADS = 256;
constexpr int BB_WAVES = BB_THREADS / 64;

// What one pass over the bodies finds: the box (lo, hi), which leaves out the first
// body's x and y, and the exponents of all coordinates and charges.
struct BoxRange {
  double lo, hi;
  BodyRange r;

  static __device__ inline BoxRange none() {
    return {INFINITY, -INFINITY, {BodyRange::NONE, 0, BodyRange::NONE, 0}};
  }
  static __device__ inline void widen(uint32_t &a, uint32_t &b, double v) {
    const uint32_t e = (uint32_t)__double2hiint(v) >> 20 & 0x7ffu;
    a = v != 0 ? min(a, e) : a;
    b = max(b, e);
  }
  __device__ inline void box(double v) {
    lo = fmin(lo, v);
    hi = fmax(hi, v);
  }
  __device__ inline void body(double x, double y, double z, double q, bool first) {
    box(z);
    if (!first) {
      box(x);
      box(y);
    }
    widen(r.lo, r.hi, x);
    widen(r.lo, r.hi, y);
    widen(r.lo, r.hi, z);
    widen(r.qlo, r.qhi, q);
  }
  __device__ inline void merge(const BoxRange &o) {
    lo = fmin(lo, o.lo);
    hi = fmax(hi, o.hi);
    merge(o.r);
  }
  __device__ inline void merge(const BodyRange &o) {
    r.lo = min(r.lo, o.lo);
    r.hi = max(r.hi, o.hi);
    r.qlo = min(r.qlo, o.qlo);
    r.qhi = max(r.qhi, o.qhi);
  }
  // over the workgroup: whole in thread 0
  __device__ inline void merge_block() {
    __shared__ BoxRange part[BB_WAVES];
    for (int o = 32; o > 0; o >>= 1) {
      BoxRange b;
      b.lo = __shfl_xor(lo, o, 64);
      b.hi = __shfl_xor(hi, o, 64);
      b.r = {__shfl_xor(r.lo, o, 64), __shfl_xor(r.hi, o, 64), __shfl_xor(r.qlo, o, 64),
             __shfl_xor(r.qhi, o, 64)};
      merge(b);
    }
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = *this;
    __syncthreads();
    if (threadIdx.x == 0)
      for (int w = 1; w < BB_WAVES; w++) merge(part[w]);
  }
  __device__ inline void write_region(double *region) const {
    for (int d = 0; d < 3; d++) {
      region[d] = lo;
      region[3 + d] = hi;
    }
  }
};

__global__ __launch_bounds__(BB_THREADS) void k_bbox_partial(const double *x, const double *y,
                                                             const double *z, const double *q,
                                                             int64_t n, BoxRange *part) {
  BoxRange b = BoxRange::none();
  for (int64_t i = (int64_t)blockIdx.x * BB_THREADS + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * BB_THREADS)
    b.body(x[i], y[i], z[i], q[i], i == 0);
  b.merge_block();
  if (threadIdx.x == 0) part[blockIdx.x] = b;
}

__global__ __launch_bounds__(BB_THREADS) void k_bbox_final(const BoxRange *part, int nparts,
                                                           double *region, BodyRange *range) {
  BoxRange b = BoxRange::none();
  for (int i = threadIdx.x; i < nparts; i += BB_THREADS) b.merge(part[i]);
  b.merge_block();
  if (threadIdx.x > 0) return;
  b.write_region(region);
  *range = b.r;
}

// Problem of body i of a forest: the last p with off[p] <= i.
__device__ inline int problem_of(const int64_t *off, int nprob, int64_t i) {
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= i) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Keys against the region of the body's own problem (off == nullptr: one
// problem); the problem index is kept per body for the forest sort.
// Also packs each body into one 32-byte record (x, y, z, q): the permutation
// gathers in random order, and one record per body is one cache line where
// four arrays are four.
__global__ void k_keys(const double *x, const double *y, const double *z, const double *q,
                       int64_t n, const double *regions, const int64_t *off, int nprob,
                       uint64_t *keys, uint32_t *idx, uint32_t *bprob, double4 *rec,
                       uint32_t *long_run) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) *long_run = 0;
  if (i >= n) return;
  const int pb = off ? problem_of(off, nprob, i) : 0;
  if (bprob) bprob[i] = (uint32_t)pb;
  const double *region = regions + 6 * pb;
  const int nfin = 1 << MAXDEPTH;
  const double p[3] = {x[i], y[i], z[i]};
  int a[3];
  for (int d = 0; d < 3; d++) {
    const double pitch = (region[3 + d] - region[d]) / (double)nfin;
    double o = p[d] - region[d];
    o = o / pitch;
    int v = (int)o;
    if (v == nfin) v--;
    a[d] = v;
  }
  keys[i] = finest_key(a[0], a[1], a[2]);
  idx[i] = (uint32_t)i;
  rec[i] = make_double4(p[0], p[1], p[2], q[i]);
}

// Bounding box of every problem of a forest, one block per problem, with
// the same scalar-cube rule as the single-problem box: problem p is its own
// Partition, so its first body's x and y are the ones left out.
__global__ __launch_bounds__(BB_THREADS) void k_bbox_forest(const double *x, const double *y,
                                                            const double *z, const double *q,
                                                            const int64_t *off, double *regions,
                                                            BodyRange *ranges) {
  const int pb = blockIdx.x;
  const int64_t first = off[pb], e = off[pb + 1];
  BoxRange b = BoxRange::none();
  for (int64_t i = first + threadIdx.x; i < e; i += BB_THREADS)
    b.body(x[i], y[i], z[i], q[i], i == first);
  b.merge_block();
  if (threadIdx.x > 0) return;
  b.write_region(regions + 6 * pb);
  ranges[pb] = b.r;
}

// the forest's range from its problems'
__global__ __launch_bounds__(BB_THREADS) void k_range_forest(const BodyRange *ranges, int nprob,
                                                             BodyRange *range) {
  BoxRange b = BoxRange::none();
  for (int i = threadIdx.x; i < nprob; i += BB_THREADS) b.merge(ranges[i]);
  b.merge_block();
  if (threadIdx.x == 0) *range = b.r;
}

// Forest order, step 1: after the bodies are sorted by key, the problem of
// each sorted body becomes the key of a second, stable sort.
__global__ void k_problem_keys(const uint32_t *order, const uint32_t *bprob, int64_t n,
                               uint32_t *pkey, uint32_t *pos) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  pkey[i] = bprob[order[i]];
  pos[i] = (uint32_t)i;
}

// Forest order, step 2: keys and body order by (problem, key).
__global__ void k_problem_gather(const uint32_t *pos, const uint64_t *keys1,
                                 const uint32_t *order1, int64_t n, uint64_t *keys,
                                 uint32_t *order) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t j = pos[i];
  keys[i] = keys1[j];
  order[i] = order1[j];
}

// The bodies are sorted by the leading bits of their keys, down to about the level
// where the tree ends, and only then, run by run, by the rest: of the seven radix
// passes over 63 bits a 1M-body cube (level 5) needs two, and this kernel costs
// less than one.  A run is the bodies of one problem (sprob, in a forest) that
// agree on the bits above shift; a body's place in it is the number of smaller
// keys, ties by position (the sort is stable).  A run longer than RUN_MAX stays as
// it is and sets *long_run: the caller sorts again by the whole key.
// Evaluations, us: 4,096-body cube 520 to 465, 16K cube as one graph 680 to 610, 100K
// periodic 1,100 to 985, 256K Plummer 2,130 to 2,060, 1M cube 5,210 to 5,095.
constexpr int RUN_TILE = 1024;  // bodies per workgroup, one per thread
constexpr int RUN_MAX = 512;
constexpr int RUN_WIN = RUN_TILE + 2 * RUN_MAX;  // a run of any of them lies in the window

__global__ __launch_bounds__(RUN_TILE) void k_sort_runs(const uint64_t *keys, const uint32_t *idx,
                                                        const uint32_t *sprob, int64_t n,
                                                        int shift, uint64_t *keys_out,
                                                        uint32_t *idx_out, uint32_t *long_run) {
  __shared__ uint64_t sk[RUN_WIN + 1];         // from one body before the window
  __shared__ uint64_t head[RUN_WIN / 64 + 1];  // bit: a run starts here (or the bodies end)
  const int lane = threadIdx.x & 63;
  const int64_t w0 = (int64_t)blockIdx.x * RUN_TILE - RUN_MAX;  // body of window place 0
  for (int t = threadIdx.x; t < RUN_WIN + 1; t += RUN_TILE) {
    const int64_t i = w0 + t - 1;
    sk[t] = i >= 0 && i < n ? keys[i] : 0;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < RUN_WIN; t += RUN_TILE) {
    const int64_t i = w0 + t;
    bool h = i == 0 || i == n;
    if (i > 0 && i < n)
      h = (sk[t + 1] >> shift) != (sk[t] >> shift) || (sprob && sprob[i] != sprob[i - 1]);
    const uint64_t m = __ballot(h);
    if (lane == 0) head[t >> 6] = m;
  }
  if (threadIdx.x == 0) head[RUN_WIN / 64] = w0 + RUN_WIN == n ? 1u : 0u;
  __syncthreads();
  const int t = RUN_MAX + threadIdx.x;
  const int64_t i = w0 + t;
  if (i >= n) return;
  // the run's first place, at most RUN_MAX before, and its end, at most RUN_MAX after
  int beg = -1, end = -1;
  uint64_t m = head[t >> 6] & (~0ull >> (63 - (t & 63)));
  for (int w = t >> 6;; m = head[--w]) {
    if (m) {
      beg = 64 * w + 63 - __clzll((long long)m);
      break;
    }
    if (w == 0 || 64 * w <= t - RUN_MAX) break;
  }
  m = (t & 63) == 63 ? 0 : head[t >> 6] & (~0ull << ((t & 63) + 1));
  for (int w = t >> 6;; m = head[++w]) {
    if (m) {
      end = 64 * w + __ffsll((unsigned long long)m) - 1;
      break;
    }
    if (w == RUN_WIN / 64) break;
  }
  int64_t to = i;
  if (beg < 0 || end < 0 || end - beg > RUN_MAX) {
    *long_run = 1;
  } else {
    const uint64_t k = sk[t + 1];
    int r = 0;
    for (int u = beg; u < t; u++) r += sk[u + 1] <= k ? 1 : 0;
    for (int u = t + 1; u < end; u++) r += sk[u + 1] < k ? 1 : 0;
    to = w0 + beg + r;
  }
  keys_out[to] = sk[t + 1];
  idx_out[to] = idx[i];
}

// Gather the caller's bodies into sorted order (SoA FP64) and keep the
// permutation.  perm[sorted] = original index.
__global__ void k_permute(const uint32_t *order, const double4 *rec, int64_t n, double *sx,
                          double *sy, double *sz, double *sq, int32_t *perm) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t o = order[i];
  const double4 r = rec[o];
  sx[i] = r.x;
  sy[i] = r.y;
  sz[i] = r.z;
  sq[i] = r.w;
  perm[i] = (int32_t)o;
}

// Root cell of problem pb (off == nullptr: the single root 0 of n bodies).
__device__ inline void make_root(const Cells &c, int pb, int64_t n, const int64_t *off,
                                 const double *regions) {
  const int64_t b = off ? off[pb] : 0, e = off ? off[pb + 1] : n;
  c.key[pb] = 0;
  c.beg[pb] = (int32_t)b;
  c.nb[pb] = (int32_t)(e - b);
  c.parent[pb] = -1;
  c.child[pb] = -1;
  c.depth[pb] = 0;
  const double *region = regions + 6 * pb;
  double w = 0;
  for (int d = 0; d < 3; d++) {
    c.center[3 * (int64_t)pb + d] = (region[3 + d] + region[d]) / 2;
    const double wd = region[3 + d] - region[d];
    w = (w < wd) ? wd : w;
  }
  c.width[pb] = w;
}

__global__ void k_roots(Cells c, int64_t n, const int64_t *off, int nprob,
                        const double *regions) {
  const int pb = blockIdx.x * blockDim.x + threadIdx.x;
  if (pb < nprob) make_root(c, pb, n, off, regions);
}

__global__ void k_split_flags(Cells c, int32_t lbeg, int32_t lcnt, int ncrit, uint32_t *flag) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= lcnt) return;
  const int32_t ci = lbeg + i;
  const bool split = c.nb[ci] > ncrit && c.depth[ci] < MAXDEPTH;
  flag[i] = split ? 1u : 0u;
  if (!split) c.child[ci] = -1;
}

__device__ inline int32_t lower_bound_keys(const uint64_t *k, int32_t lo, int32_t hi,
                                           uint64_t v) {
  while (lo < hi) {
    const int32_t mid = lo + ((hi - lo) >> 1);
    if (k[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// child ch of split parent p, at cell index first + ch
__device__ inline void make_child(Cells c, int32_t p, int ch, int32_t first, const uint64_t *keys,
                                  const double *regions, const uint32_t *sprob) {
  const int32_t ci = first + ch;
  const uint64_t pk = c.key[p];
  const uint64_t ck = key_child(pk, ch);
  const int32_t pb = c.beg[p], pe = c.beg[p] + c.nb[p];
  const int32_t b = lower_bound_keys(keys, pb, pe, ck);
  const int32_t e = (ch == 7) ? pe : lower_bound_keys(keys, pb, pe, key_child(pk, ch + 1));
  c.key[ci] = ck;
  c.beg[ci] = b;
  c.nb[ci] = e - b;
  c.parent[ci] = p;
  c.child[ci] = -1;
  c.depth[ci] = c.depth[p] + 1;
  // a split cell holds bodies, so its first body names its problem
  const double *region = regions + (sprob ? 6 * (int64_t)sprob[pb] : 0);
  double rmin[3] = {region[0], region[1], region[2]};
  double rmax[3] = {region[3], region[4], region[5]};
  double mn[3], mx[3];
  cell_region(ck, rmin, rmax, mn, mx);
  double w = 0;
  for (int d = 0; d < 3; d++) {
    c.center[3 * (int64_t)ci + d] = (mx[d] + mn[d]) / 2;
    const double wd = mx[d] - mn[d];
    w = (w < wd) ? wd : w;
  }
  c.width[ci] = w;
  if (ch == 0) c.child[p] = first;
}

__global__ void k_children(Cells c, int32_t lbeg, int32_t lcnt, const uint32_t *flag,
                           const uint32_t *slot, int32_t next_beg, const uint64_t *keys,
                           const double *regions, const uint32_t *sprob) {
  // one thread per (parent, child) -> 8 threads per parent
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)lcnt * 8) return;
  const int32_t i = (int32_t)(t >> 3);
  const int ch = (int)(t & 7);
  if (!flag[i]) return;
  make_child(c, lbeg + i, ch, next_beg + 8 * (int32_t)slot[i], keys, regions, sprob);
}

// ---------------------------------------------------------------------------
// The same level step with every size on the device (no host round trip per
// level): lev[2 d], lev[2 d + 1] = first cell and cell count of level d.  The
// grids come from the sizes of an earlier tree; the host checks afterwards
// that every level fitted its grid and the cell capacity (status bits), and
// builds again the synchronous way if not.
constexpr int LV_BLOCK = 256;

// split flags, the exclusive prefix of the flags inside each 256-cell block,
// and the block totals
__global__ __launch_bounds__(LV_BLOCK) void k_level_flags(Cells c, const int32_t *lev, int d,
                                                          int ncrit, uint32_t *flag,
                                                          uint32_t *loc, uint32_t *bsum) {
  const int32_t lbeg = lev[2 * d], lcnt = lev[2 * d + 1];
  const int32_t i = blockIdx.x * LV_BLOCK + threadIdx.x;
  bool split = false;
  if (i < lcnt) {
    const int32_t ci = lbeg + i;
    split = c.nb[ci] > ncrit && c.depth[ci] < MAXDEPTH;
    if (!split) c.child[ci] = -1;
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const uint64_t m = __ballot(split);
  __shared__ uint32_t wsum[LV_BLOCK / 64];
  if (lane == 0) wsum[wid] = (uint32_t)__popcll(m);
  __syncthreads();
  uint32_t pre = 0, tot = 0;
  for (int w = 0; w < LV_BLOCK / 64; w++) {
    pre += w < wid ? wsum[w] : 0u;
    tot += wsum[w];
  }
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  if (i < lcnt) {
    flag[i] = split ? 1u : 0u;
    loc[i] = pre + (uint32_t)__popcll(m & lt);
  }
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// one block: exclusive scan of the block totals, the next level's extent;
// status bit 1: cell capacity exceeded, bit 2: level larger than its grid,
// bit 4: splits on the last planned level
__global__ __launch_bounds__(1024) void k_level_scan(int32_t *lev, int d, uint32_t *bsum,
                                                     int32_t nblk, int32_t cap,
                                                     uint32_t *status, int last) {
  const int32_t lbeg = lev[2 * d], lcnt = lev[2 * d + 1];
  const int32_t nb = min(nblk, (lcnt + LV_BLOCK - 1) / LV_BLOCK);
  __shared__ uint32_t part[1024];
  // each thread scans a contiguous run of the block totals
  const int per = (nb + 1023) / 1024;
  const int b0 = threadIdx.x * per, b1 = min(nb, b0 + per);
  uint32_t s = 0;
  for (int b = b0; b < b1; b++) s += bsum[b];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const uint32_t v = threadIdx.x >= (unsigned)o ? part[threadIdx.x - o] : 0u;
    __syncthreads();
    part[threadIdx.x] += v;
    __syncthreads();
  }
  uint32_t run = part[threadIdx.x] - s;
  for (int b = b0; b < b1; b++) {
    const uint32_t v = bsum[b];
    bsum[b] = run;
    run += v;
  }
  if (threadIdx.x == 0) {
    const uint32_t total = part[1023];
    const int64_t next_beg = (int64_t)lbeg + lcnt;
    int64_t next_cnt = 8 * (int64_t)total;
    uint32_t st = 0;
    if (lcnt > nblk * LV_BLOCK) st |= 2u;
    if (next_beg + next_cnt > cap) st |= 1u;
    if (last && next_cnt > 0) st |= 4u;
    if (st) {
      atomicOr(status, st);
      next_cnt = 0;  // stop: this tree is built again on the host's path
    }
    lev[2 * (d + 1)] = (int32_t)next_beg;
    lev[2 * (d + 1) + 1] = (int32_t)next_cnt;
  }
}

__global__ void k_level_children(Cells c, const int32_t *lev, int d, const uint32_t *flag,
                                 const uint32_t *loc, const uint32_t *bsum,
                                 const uint64_t *keys, const double *regions,
                                 const uint32_t *sprob) {
  const int32_t lbeg = lev[2 * d], lcnt = lev[2 * d + 1];
  const int32_t next_beg = lev[2 * (d + 1)], next_cnt = lev[2 * (d + 1) + 1];
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (next_cnt == 0 || t >= (int64_t)lcnt * 8) return;
  const int32_t i = (int32_t)(t >> 3);
  const int ch = (int)(t & 7);
  if (!flag[i]) return;
  const uint32_t slot = bsum[i / LV_BLOCK] + loc[i];
  make_child(c, lbeg + i, ch, next_beg + 8 * (int32_t)slot, keys, regions, sprob);
}

// The roots and the first `levels` level steps in one workgroup: levels of a few
// hundred cells are three launches of a few microseconds each otherwise, most of it
// the gaps between them.  lev and *status are initialised here.  A level may hold
// any number of cells (each takes its turn); status as k_level_scan, bit 2 for a
// level larger than most.cells (what later launches over that level cover).
// With the other launches taken out beside it, a 4,096-body cube 650 to 565 us an
// evaluation, a 64K ellipsoid 1,760 to 1,680.
constexpr int TOP_THREADS = 1024;

struct LevelSizes {
  int32_t cells[MAXDEPTH + 2];
};

__global__ __launch_bounds__(TOP_THREADS) void k_tree_top(Cells c, int64_t n, const int64_t *off,
                                                          int nprob, int32_t *lev, int L,
                                                          int levels, int ncrit, int32_t cap,
                                                          uint32_t *status, const uint64_t *keys,
                                                          const double *regions,
                                                          const uint32_t *sprob, int last,
                                                          LevelSizes most,
                                                          const uint32_t *long_run) {
  __shared__ int32_t parent[TOP_THREADS];  // the split cells of a turn
  __shared__ uint32_t wsum[TOP_THREADS / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < 2 * (L + 1); i += TOP_THREADS)
    lev[i] = i == 1 ? nprob : 0;
  for (int pb = threadIdx.x; pb < nprob; pb += TOP_THREADS) make_root(c, pb, n, off, regions);
  int32_t lbeg = 0, lcnt = nprob;
  uint32_t st = *long_run ? (uint32_t)ST_SORT : 0u;  // keys out of order: no tree
  for (int d = 0; d < levels; d++) {
    if (lcnt > most.cells[d]) st |= 2u;
    const int32_t next_beg = lbeg + lcnt;
    int64_t total = 0;  // split cells so far
    for (int32_t base = 0; base < lcnt; base += TOP_THREADS) {
      __syncthreads();  // the cells of this level are written; the last turn is over
      const int32_t i = base + threadIdx.x, ci = lbeg + i;
      bool split = false;
      if (i < lcnt) {
        split = c.nb[ci] > ncrit && c.depth[ci] < MAXDEPTH;
        if (!split) c.child[ci] = -1;
      }
      const uint64_t m = __ballot(split);
      if (lane == 0) wsum[wid] = (uint32_t)__popcll(m);
      __syncthreads();
      uint32_t pre = 0, tot = 0;
      for (int w = 0; w < TOP_THREADS / 64; w++) {
        pre += w < wid ? wsum[w] : 0u;
        tot += wsum[w];
      }
      if (split) parent[pre + (uint32_t)__popcll(m & (lane == 0 ? 0ull : ~0ull >> (64 - lane)))] = ci;
      __syncthreads();
      if (next_beg + 8 * (total + tot) > cap) st |= 1u;
      if (!st)
        for (uint32_t t = threadIdx.x; t < tot * 8; t += TOP_THREADS)
          make_child(c, parent[t >> 3], (int)(t & 7),
                     next_beg + 8 * (int32_t)(total + (t >> 3)), keys, regions, sprob);
      total += tot;
    }
    if (last && d == L - 1 && total > 0) st |= 4u;
    lbeg = next_beg;
    lcnt = st ? 0 : (int32_t)(8 * total);
    if (threadIdx.x == 0) {
      lev[2 * (d + 1)] = lbeg;
      lev[2 * (d + 1) + 1] = lcnt;
    }
  }
  if (threadIdx.x == 0) *status = st;
}

// flag = 1 when a coordinate or charge of the n bodies is not finite (the
// host path rejects such bodies while unpacking them; device arrays are
// checked here)
__global__ void k_check_finite(const double *x, const double *y, const double *z,
                               const double *q, int64_t n, uint32_t *flag) {
  bool bad = false;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    bad |= !(isfinite(x[i]) && isfinite(y[i]) && isfinite(z[i]) && isfinite(q[i]));
  if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(flag, 1u);
}

// Periodic images: the root cell is the periodic cell, a cube of side cycle
// centred on the bodies' scalar bounding cube (region: min x, y, z, max x, y,
// z); flag = 1 when the bodies span more than one period.
__global__ void k_periodic_region(double *region, double cycle, uint32_t *flag) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const double lo = region[0], hi = region[3];
  if (!(hi - lo <= cycle)) *flag = 1u;
  const double c = 0.5 * (lo + hi), h = 0.5 * cycle;
  for (int d = 0; d < 3; d++) {
    region[d] = c - h;
    region[3 + d] = c + h;
  }
}

}  // namespace

hipError_t launch_periodic_region(double *region, double cycle, uint32_t *flag, hipStream_t s) {
  k_periodic_region<<<1, 64, 0, s>>>(region, cycle, flag);
  return hipGetLastError();
}

hipError_t launch_check_finite(const double *x, const double *y, const double *z,
                               const double *q, int64_t n, uint32_t *flag, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int64_t blocks = std::min<int64_t>(2048, (n + 255) / 256);
  k_check_finite<<<(unsigned)blocks, 256, 0, s>>>(x, y, z, q, n, flag);
  return hipGetLastError();
}

size_t bbox_part_bytes(int nparts) { return (size_t)nparts * sizeof(BoxRange); }

hipError_t launch_bbox(const double *x, const double *y, const double *z, const double *q,
                       int64_t n, void *part, int nparts, double *region, BodyRange *range,
                       hipStream_t s) {
  BoxRange *p = static_cast<BoxRange *>(part);
  k_bbox_partial<<<nparts, BB_THREADS, 0, s>>>(x, y, z, q, n, p);
  k_bbox_final<<<1, BB_THREADS, 0, s>>>(p, nparts, region, range);
  return hipGetLastError();
}

hipError_t launch_keys(const double *x, const double *y, const double *z, const double *q,
                       int64_t n, const double *regions, const int64_t *off, int nprob,
                       uint64_t *keys, uint32_t *idx, uint32_t *bprob, double4 *rec,
                       uint32_t *long_run, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  k_keys<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(x, y, z, q, n, regions, off, nprob, keys,
                                                      idx, bprob, rec, long_run);
  return hipGetLastError();
}

hipError_t launch_bbox_forest(const double *x, const double *y, const double *z, const double *q,
                              const int64_t *off, int nprob, double *regions, BodyRange *range,
                              hipStream_t s) {
  if (nprob <= 0) return hipSuccess;
  k_bbox_forest<<<nprob, BB_THREADS, 0, s>>>(x, y, z, q, off, regions, range + 1);
  k_range_forest<<<1, BB_THREADS, 0, s>>>(range + 1, nprob, range);
  return hipGetLastError();
}

hipError_t launch_problem_keys(const uint32_t *order, const uint32_t *bprob, int64_t n,
                               uint32_t *pkey, uint32_t *pos, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  k_problem_keys<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(order, bprob, n, pkey, pos);
  return hipGetLastError();
}

hipError_t launch_problem_gather(const uint32_t *pos, const uint64_t *keys1,
                                 const uint32_t *order1, int64_t n, uint64_t *keys,
                                 uint32_t *order, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  k_problem_gather<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(pos, keys1, order1, n, keys,
                                                                order);
  return hipGetLastError();
}

hipError_t launch_sort_runs(const uint64_t *keys, const uint32_t *idx, const uint32_t *sprob,
                            int64_t n, int shift, uint64_t *keys_out, uint32_t *idx_out,
                            uint32_t *long_run, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  k_sort_runs<<<(unsigned)((n + RUN_TILE - 1) / RUN_TILE), RUN_TILE, 0, s>>>(
      keys, idx, sprob, n, shift, keys_out, idx_out, long_run);
  return hipGetLastError();
}

hipError_t launch_permute(const uint32_t *order, const double4 *rec, int64_t n, double *sx,
                          double *sy, double *sz, double *sq, int32_t *perm, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  k_permute<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(order, rec, n, sx, sy, sz, sq, perm);
  return hipGetLastError();
}

hipError_t launch_roots(Cells c, int64_t n, const int64_t *off, int nprob,
                        const double *regions, hipStream_t s) {
  k_roots<<<(nprob + 255) / 256, 256, 0, s>>>(c, n, off, nprob, regions);
  return hipGetLastError();
}

// the leading levels that launch_tree_top takes, from the L level sizes of an earlier
// tree: those whose cells and children are one turn of its workgroup (a child costs a
// chain of keys read at random, which more workgroups hide better)
int tree_top_levels(const int32_t *sizes, int L) {
  auto one_turn = [&](int d) { return d >= L || sizes[d] <= TOP_THREADS; };
  int t = 0;
  while (t < L && t < MAXDEPTH + 2 && one_turn(t) && one_turn(t + 1)) t++;
  return t;
}

hipError_t launch_tree_top(Cells c, int64_t n, const int64_t *off, int nprob, int32_t *lev, int L,
                           int levels, int ncrit, int32_t cap, uint32_t *status,
                           const uint64_t *keys, const double *regions, const uint32_t *sprob,
                           const uint32_t *long_run, hipStream_t s, bool last,
                           const int32_t *most) {
  LevelSizes m;
  for (int d = 0; d < MAXDEPTH + 2; d++) m.cells[d] = most && d < levels ? most[d] : INT32_MAX;
  k_tree_top<<<1, TOP_THREADS, 0, s>>>(c, n, off, nprob, lev, L, levels, ncrit, cap, status, keys,
                                       regions, sprob, last ? 1 : 0, m, long_run);
  return hipGetLastError();
}

int32_t level_blocks(int32_t cells) { return (cells + LV_BLOCK - 1) / LV_BLOCK; }

hipError_t launch_level_step(Cells c, int32_t *lev, int d, int32_t grid_cells, int ncrit,
                             int32_t cap, uint32_t *flag, uint32_t *loc, uint32_t *bsum,
                             uint32_t *status, const uint64_t *keys, const double *regions,
                             const uint32_t *sprob, hipStream_t s, bool last) {
  const int32_t nblk = level_blocks(grid_cells);
  if (nblk <= 0) return hipSuccess;
  k_level_flags<<<nblk, LV_BLOCK, 0, s>>>(c, lev, d, ncrit, flag, loc, bsum);
  k_level_scan<<<1, 1024, 0, s>>>(lev, d, bsum, nblk, cap, status, last ? 1 : 0);
  const int64_t nt = (int64_t)nblk * LV_BLOCK * 8;
  k_level_children<<<(unsigned)((nt + 255) / 256), 256, 0, s>>>(c, lev, d, flag, loc, bsum, keys,
                                                                 regions, sprob);
  return hipGetLastError();
}

hipError_t launch_split_flags(Cells c, int32_t lbeg, int32_t lcnt, int ncrit, uint32_t *flag,
                              hipStream_t s) {
  if (lcnt <= 0) return hipSuccess;
  k_split_flags<<<(lcnt + 255) / 256, 256, 0, s>>>(c, lbeg, lcnt, ncrit, flag);
  return hipGetLastError();
}

hipError_t launch_children(Cells c, int32_t lbeg, int32_t lcnt, const uint32_t *flag,
                           const uint32_t *slot, int32_t next_beg, const uint64_t *keys,
                           const double *regions, const uint32_t *sprob, hipStream_t s) {
  if (lcnt <= 0) return hipSuccess;
  const int64_t nt = (int64_t)lcnt * 8;
  k_children<<<(unsigned)((nt + 255) / 256), 256, 0, s>>>(c, lbeg, lcnt, flag, slot, next_beg,
                                                           keys, regions, sprob);
  return hipGetLastError();
}

}  // namespace tfmm
