// expansions.hip -- FP64 upward (P2M, M2M) and downward (L2L, L2P) kernels.
//
// Reference (sample/exafmm-dev-13274dd4ac68/examples/):
//   FMM_Upward / FMM_Downward   tapas_exafmm.cxx:87-140
//   P2M  LaplaceSphericalCPU_tapas.h:138-163     L2P  :275-307
// (M2M and L2L are in translate.hip.)
#include "tfmm_device.h"
#include "tfmm_kernels.h"

namespace tfmm {
namespace {

__device__ inline int sgn(int n) { return (n & 1) ? -1 : 1; }
__device__ inline int ipow2n(int n) { return (n >= 0) ? 1 : sgn(n); }

// (j, k) of coefficient index t = tri(j, k)
__device__ inline void untri(int t, int &j, int &k) {
  j = 0;
  while (tri(j + 1, 0) <= t) j++;
  k = t - tri(j, 0);
}

// P2M: M[n,m] += q * conj(Y_n^m(body - centre)), summed over the leaf's
// bodies.  One wave per leaf, one body per lane (chunks of 64 bodies).  The 110
// real values come out of the recurrence in a fixed visit order and are summed over
// the lanes by halving: two values become one register, in which half the lanes hold
// the pairwise sums of the one and half those of the other, and two such registers
// become one as soon as both are there (six levels, at most seven registers
// waiting).  Value v ends in the lane of v's six bits reversed.  The sums' order is
// fixed.  (Through LDS, 16 values at a time, each summed by 16 serial reads: 4M
// Plummer 789 us beside the P2P against 343, 500K ellipsoid 131 against 89.)  Bound
// by FP64 issue: some 500 instructions of harmonics and 440 of sums per 64 bodies.
constexpr int P2M_WAVES = 4;
constexpr int NVAL = 2 * NTERM;  // 110 real values per cell

// lanes with bit 5 - LEVEL of their number clear: a summed over the two lanes that
// differ there (below bit 4: in the lower bits too); the others: b
template <int LEVEL>
__device__ inline double halve(double a, double b, int lane) {
  union {
    double d;
    uint32_t u[2];
  } p, q;
  if constexpr (LEVEL < 2) {
    p.d = a;
    q.d = b;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const auto r = LEVEL == 0 ? __builtin_amdgcn_permlane32_swap(p.u[h], q.u[h], false, false)
                                : __builtin_amdgcn_permlane16_swap(p.u[h], q.u[h], false, false);
      p.u[h] = r[0];
      q.u[h] = r[1];
    }
    return p.d + q.d;
  } else {
    // lane ^ 15, 7, 3, 1
    constexpr int CTRL = LEVEL == 2 ? 0x140 : LEVEL == 3 ? 0x141 : LEVEL == 4 ? 0x1b : 0xb1;
    const bool other = lane >> (5 - LEVEL) & 1;
    p.d = other ? a : b;
#pragma unroll
    for (int h = 0; h < 2; h++)
      q.u[h] = (uint32_t)__builtin_amdgcn_mov_dpp((int)p.u[h], CTRL, 0xf, 0xf, true);
    return (other ? b : a) + q.d;
  }
}

// The waiting registers: value v of 64 (a constant) goes in; at the last one, or with
// flush at the end of fewer, out holds a value per lane.
struct LaneSums {
  double wait[6];
  template <int LEVEL>
  __device__ inline void carry(int v, double x, int lane, double &out) {
    if constexpr (LEVEL == 6) out = x;
    else if (v >> LEVEL & 1) carry<LEVEL + 1>(v, halve<LEVEL>(wait[LEVEL], x, lane), lane, out);
    else wait[LEVEL] = x;
  }
  template <int LEVEL>
  __device__ inline void flush(int n, double x, bool have, int lane, double &out) {
    if constexpr (LEVEL == 6) out = x;
    else if (n >> LEVEL & 1)
      flush<LEVEL + 1>(n, halve<LEVEL>(wait[LEVEL], x, lane), true, lane, out);
    else if (have) flush<LEVEL + 1>(n, halve<LEVEL>(x, 0.0, lane), true, lane, out);
    else flush<LEVEL + 1>(n, 0.0, false, lane, out);
  }
};

// (n, m) of the v-th term of multipole_all's visit order (m outer, n inner)
__device__ inline int visit_term(int v) {
  int m = 0;
  while (v >= P - m) {
    v -= P - m;
    m++;
  }
  return tri(m + v, m);
}

__global__ __launch_bounds__(64 * P2M_WAVES) void k_p2m(Cells c, int32_t ncells, Bodies b,
                                                        double *M) {
  critical_path_priority();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int32_t ci = blockIdx.x * P2M_WAVES + w;
  if (ci >= ncells || c.child[ci] >= 0 || c.nb[ci] == 0) return;
  const double cx = c.center[3 * (int64_t)ci], cy = c.center[3 * (int64_t)ci + 1],
               cz = c.center[3 * (int64_t)ci + 2];
  const int32_t beg = c.beg[ci], end = beg + c.nb[ci];
  double own[2] = {0, 0};  // this lane's values of the first 64 and of the others
  for (int32_t base = beg; base < end; base += 64) {
    const int32_t i = base + lane;
    double dx = 1, dy = 0, dz = 0, q = 0;
    if (i < end) {
      dx = b.x[i] - cx;
      dy = b.y[i] - cy;
      dz = b.z[i] - cz;
      q = b.q[i];
    }
    double rho, ca, sa;
    cd ei;
    sph_frame(dx, dy, dz, rho, ca, sa, ei);
    LaneSums sums;
    double got[2];
    int v = 0;  // visit counter (a constant after unrolling)
    multipole_all<false>(rho, ca, sa, ei, [&](int, int, cd Y, cd) {
      sums.carry<0>(v & 63, Y.re, lane, got[v >> 6]);
      sums.carry<0>((v + 1) & 63, -Y.im, lane, got[(v + 1) >> 6]);
      v += 2;
    }, 0.0, q);
    sums.flush<0>(NVAL & 63, 0.0, false, lane, got[1]);
    own[0] += got[0];
    own[1] += got[1];
  }
  double *Mc = M + 2 * (int64_t)NTERM * ci;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int f = 64 * h + (int)(__brev((uint32_t)lane) >> 26);  // value, in visit order
    if (f < NVAL) Mc[2 * visit_term(f >> 1) + (f & 1)] += own[h];
  }
}

// leaf of every (sorted) body
__global__ void k_body_leaf(Cells c, int32_t ncells, int32_t *leaf_of) {
  const int32_t ci = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (ci >= ncells || c.child[ci] >= 0) return;
  const int32_t beg = c.beg[ci], end = beg + c.nb[ci];
  for (int32_t i = beg + (threadIdx.x & 63); i < end; i += 64) leaf_of[i] = ci;
}

// L2P: trg = p2p / q + local field of the leaf's expansion; one thread per
// body, written in sorted order (trg) and in input order (out[perm]).
// The block's bodies are consecutive in sorted order, so they belong to a few
// runs of one leaf each: the expansions of the first L2P_RUNS runs are
// staged in LDS and read from there (bodies of later runs read global
// memory).
constexpr int L2P_RUNS = 16;

__global__ __launch_bounds__(256) void k_l2p(Cells c, Bodies b, const int32_t *leaf_of,
                                             const double *L, const double *p2p,
                                             const int32_t *perm, double *trg, double *out) {
  __shared__ cd Lrun[L2P_RUNS][NTERM];
  __shared__ int32_t run_leaf[L2P_RUNS];
  __shared__ uint32_t wave_runs[4];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x;
  const bool valid = i < b.n;
  const int32_t ci = valid ? leaf_of[i] : -1;
  // run index of this body: run starts before it in the block
  const bool start = valid && (i == i0 || leaf_of[i - 1] != ci);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const uint64_t m = __ballot(start);
  if (lane == 0) wave_runs[wid] = (uint32_t)__popcll(m);
  __syncthreads();
  uint32_t before = 0;
  for (int w = 0; w < wid; w++) before += wave_runs[w];
  const uint64_t upto = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
  const int run = (int)(before + (uint32_t)__popcll(m & upto)) - 1;
  if (start && run < L2P_RUNS) run_leaf[run] = ci;
  __syncthreads();
  const int nruns = (int)(wave_runs[0] + wave_runs[1] + wave_runs[2] + wave_runs[3]);
  const int staged = nruns < L2P_RUNS ? nruns : L2P_RUNS;
  for (int e = threadIdx.x; e < staged * NTERM; e += blockDim.x) {
    const int r = e / NTERM, t = e - r * NTERM;
    Lrun[r][t] = reinterpret_cast<const cd *>(L)[(int64_t)run_leaf[r] * NTERM + t];
  }
  __syncthreads();
  if (!valid) return;
  const cd *Ls = run < L2P_RUNS ? Lrun[run] : reinterpret_cast<const cd *>(L) + (int64_t)ci * NTERM;
  const double dx = b.x[i] - c.center[3 * (int64_t)ci], dy = b.y[i] - c.center[3 * (int64_t)ci + 1],
               dz = b.z[i] - c.center[3 * (int64_t)ci + 2];
  const double q = b.q[i];
  double r, ct, st;
  cd ei;
  sph_frame(dx, dy, dz, r, ct, st, ei);
  const double iq = 1.0 / q, ir = 1.0 / r;
  double t0 = p2p[4 * i] * iq, t1 = p2p[4 * i + 1] * iq, t2 = p2p[4 * i + 2] * iq,
         t3 = p2p[4 * i + 3] * iq;
  double s0 = 0, s1 = 0, s2 = 0;
  multipole_all<true>(
      r, ct, st, ei,
      [&](int n, int m, cd Y, cd YT) {
        const cd l = Ls[tri(n, m)];
        const cd ly = cmul(l, Y);
        const double lyt = cmul(l, YT).re;
        if (m == 0) {
          t0 += ly.re;
          s0 += ly.re * ir * n;
          s1 += lyt;
        } else {
          t0 += 2 * ly.re;
          s0 += 2 * ly.re * ir * n;
          s1 += 2 * lyt;
          s2 += 2 * (-ly.im) * m;
        }
      },
      1.0 / st);
  const double sp = ei.im, cp = ei.re;
  t1 += st * cp * s0 + ct * cp * ir * s1 - sp * ir / st * s2;
  t2 += st * sp * s0 + ct * sp * ir * s1 + cp * ir / st * s2;
  t3 += ct * s0 - st * ir * s1;
  trg[4 * i] = t0;
  trg[4 * i + 1] = t1;
  trg[4 * i + 2] = t2;
  trg[4 * i + 3] = t3;
  const int64_t o = perm[i];
  out[4 * o] = t0;
  out[4 * o + 1] = t1;
  out[4 * o + 2] = t2;
  out[4 * o + 3] = t3;
}

// Zero fill (in place of hipMemsetAsync, which must not be recorded into a
// captured graph): 16-byte stores, the tail by single bytes.
__global__ void k_fill_zero(uint4 *p, size_t n16, unsigned char *tail, int ntail) {
  critical_path_priority();
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n16) p[i] = make_uint4(0, 0, 0, 0);
  if (i < (size_t)ntail) tail[i] = 0;
}

}  // namespace

hipError_t launch_fill_zero(void *ptr, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  const size_t n16 = bytes / 16;
  const int ntail = (int)(bytes - n16 * 16);
  const size_t nt = n16 > (size_t)ntail ? n16 : (size_t)ntail;
  k_fill_zero<<<(unsigned)((nt + 255) / 256), 256, 0, s>>>(
      static_cast<uint4 *>(ptr), n16, static_cast<unsigned char *>(ptr) + n16 * 16, ntail);
  return hipGetLastError();
}

hipError_t launch_p2m(Cells c, int32_t ncells, Bodies b, double *M, hipStream_t s) {
  if (ncells <= 0) return hipSuccess;
  k_p2m<<<(ncells + P2M_WAVES - 1) / P2M_WAVES, 64 * P2M_WAVES, 0, s>>>(c, ncells, b, M);
  return hipGetLastError();
}

hipError_t launch_body_leaf(Cells c, int32_t ncells, int32_t *leaf_of, hipStream_t s) {
  if (ncells <= 0) return hipSuccess;
  k_body_leaf<<<(ncells + 3) / 4, 256, 0, s>>>(c, ncells, leaf_of);
  return hipGetLastError();
}

// leaf_of: the leaf of every sorted body (launch_body_leaf)
hipError_t launch_l2p(Cells c, int32_t ncells, Bodies b, const double *L, const double *p2p,
                      const int32_t *perm, const int32_t *leaf_of, double *trg, double *out,
                      hipStream_t s) {
  if (ncells <= 0 || b.n <= 0) return hipSuccess;
  k_l2p<<<(unsigned)((b.n + 255) / 256), 256, 0, s>>>(c, b, leaf_of, L, p2p, perm, trg, out);
  return hipGetLastError();
}

}  // namespace tfmm
