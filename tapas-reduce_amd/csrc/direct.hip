// direct.hip -- FP64 O(N * targets) direct sum, the error judge of the FMM.
//
// Same interaction as the P2P functor and the same normalisation as the
// reference's CheckResult (sample/exafmm-dev-13274dd4ac68/examples/
// tapas_exafmm.cxx:338-367): each target accumulates q_i q_j / r and
// -q_i q_j dX / r^3 over all bodies j (r = 0 skipped), then divides by q_i.
// With periodic images (prange > 0) every body j is also seen at
// x_j + (ix, iy, iz) cycle for |ix|, |iy|, |iz| <= prange, dX = x_i - x_j -
// Xperiodic, in the reference's loop order (tapas_exafmm.cxx:328-345).
#include "tfmm_device.h"
#include "tfmm_kernels.h"

namespace tfmm {
namespace {

// Bound by FP64 VALU issue: 18 FP64 operations and one v_rsq_f64 a pair.  The
// bodies are what there is a lot of, the targets often are few (an error check
// takes a few thousand), so a workgroup's DT threads split the bodies and share
// T targets, whose coordinates are uniform (scalar registers); each body read
// serves T pairs.  Every target's sum has one order, whatever T and the other
// targets are: thread l takes bodies l, l + DT, ..., and the threads' partial
// sums are added in a fixed tree.  So the results of a call do not depend on how
// the targets are dealt to launches.
// 4096 targets of 1,000,003 bodies: 3.9 ms with T = 4 (4.0 with 8, whose 234
// registers leave two waves a SIMD, 4.6 with 2), 136 cycles a pair and SIMD; with
// one target a thread, which put 16 workgroups on the chip, 205 ms.
constexpr int DT = 512;
constexpr int DW = DT / 64;

// 1 / sqrt(x) for finite x > 0 to the last place or so, 0 for x = 0 and infinite
// x (a body at the target, and one beyond the range of the squares); NaN stays.
// v_rsq_f64 and one third-order step; one operation tells the excluded values.
__device__ inline double rsqrt_pair(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  y = fma(y * e, fma(e, 0.375, 0.5), y);
  constexpr int KEEP = 0x003 | 0x180;  // NaNs, positive denormal and normal numbers
  return __builtin_amdgcn_class(x, KEEP) ? y : 0.0;
}

template <int T>
__global__ __launch_bounds__(DT) void k_direct(const double *x, const double *y,
                                               const double *z, const double *q, int64_t n,
                                               const int64_t *targets, int64_t tbase,
                                               int64_t nt, double *out, int prange,
                                               double cycle) {
  __shared__ double part[DW][4 * T];
  const int64_t t0 = (int64_t)blockIdx.x * T;
  double xi[T], yi[T], zi[T], a[T][4];
#pragma unroll
  for (int u = 0; u < T; u++) {
    const int64_t i = targets[min(t0 + u, nt - 1)] - tbase;  // past the end: the last one again
    xi[u] = x[i];
    yi[u] = y[i];
    zi[u] = z[i];
#pragma unroll
    for (int e = 0; e < 4; e++) a[u][e] = 0;
  }
  for (int ix = -prange; ix <= prange; ix++)
    for (int iy = -prange; iy <= prange; iy++)
      for (int iz = -prange; iz <= prange; iz++) {
        const double px = ix * cycle, py = iy * cycle, pz = iz * cycle;
        double sx[T], sy[T], sz[T];
#pragma unroll
        for (int u = 0; u < T; u++) {
          sx[u] = xi[u] - px;
          sy[u] = yi[u] - py;
          sz[u] = zi[u] - pz;
        }
        for (int64_t j = threadIdx.x; j < n; j += DT) {
          const double xj = x[j], yj = y[j], zj = z[j], qj = q[j];
#pragma unroll
          for (int u = 0; u < T; u++) {
            const double dx = sx[u] - xj, dy = sy[u] - yj, dz = sz[u] - zj;
            const double invr = rsqrt_pair(dx * dx + dy * dy + dz * dz);
            const double v = qj * invr, f = invr * invr * v;
            a[u][0] += v;
            a[u][1] -= dx * f;
            a[u][2] -= dy * f;
            a[u][3] -= dz * f;
          }
        }
      }
#pragma unroll
  for (int u = 0; u < T; u++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      double v = a[u][e];
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
      if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6][4 * u + e] = v;
    }
  __syncthreads();
  const int o = threadIdx.x;
  if (o >= 4 * T || t0 + o / 4 >= nt) return;
  double v = part[0][o];
  for (int w = 1; w < DW; w++) v += part[w][o];
  const double qi = q[targets[t0 + o / 4] - tbase];
  out[4 * t0 + o] = v * qi / qi;  // the functor's q_i q_j, then divided by q_i
}

}  // namespace

hipError_t launch_direct_fp64(const double *x, const double *y, const double *z,
                              const double *q, int64_t n, const int64_t *targets, int64_t tbase,
                              int64_t nt, double *out, hipStream_t s, int prange, double cycle) {
  if (nt <= 0) return hipSuccess;
  // As many targets a workgroup as still leave two workgroups a CU: four take
  // a quarter of the reads, but below 2048 targets would leave CUs idle.
  auto go = [&](auto kernel, int per) {
    kernel<<<(unsigned)((nt + per - 1) / per), DT, 0, s>>>(x, y, z, q, n, targets, tbase, nt, out,
                                                           prange, cycle);
    return hipGetLastError();
  };
  if (nt >= 4 * 512) return go(k_direct<4>, 4);
  if (nt >= 2 * 512) return go(k_direct<2>, 2);
  return go(k_direct<1>, 1);
}

}  // namespace tfmm
