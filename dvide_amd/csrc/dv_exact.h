// D^T x body by body in the exact order: the terms of a body's three sums are
// those of its rows of D^T, bilateral rows ascending, then contacts ascending
// with the n, u, v rows in turn, added one by one from 0.0 without fused
// multiply-adds, so they round like a row-sorted COO SpMV.  Shared by the
// products of dv_assemble.hip and the passes of dv_apgd_plain.hip.
#pragma once

#include "dv_internal.h"

namespace dv {

struct GatherArgs {
  int nb, nbil, cap;
  const double* frame;
  const int* iStart;
  const int* inc;
  const int* bilIncStart;
  const int* bilInc;
  const double* minv;
  const int* heavy;     // ascending
  const int* counters;  // [2]: how many
};

// The gathering kernels run workgroups of one wavefront: blocks [0,
// gatherBlocks) take 64 bodies each, and kHeavyBlocks more take the bodies of
// the heavy list (more than kHeavyDegree contacts), one at a time.  (In
// workgroups of 256, a few thousand bodies crowded a few CUs; and a wavefront
// that summed the heavy bodies it met, the container's five in turn, took
// 0.29 ms at 112,000 spheres.)
constexpr int kGatherT = 64;
constexpr int kHeavyBlocks = 64;
inline int gatherBlocks(const GatherArgs& a) { return blocksFor(a.nb, kGatherT); }

template <class X>
__device__ __forceinline__ void gatherLoad(const GatherArgs& a, int e, X& x, double (&xr)[3], double (&f)[9]) {
  const int c = e >> 1;
  const long base = a.nbil + 3L * c, S = a.cap;
#pragma unroll
  for (int rr = 0; rr < 3; ++rr) xr[rr] = x(base + rr);
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const double v = a.frame[q * S + c];
    f[q] = (e & 1) ? -v : v;
  }
}

template <class X>
__device__ __forceinline__ void gatherBilateral(const GatherArgs& a, int g, X& x, double& s0, double& s1, double& s2) {
  s0 = s1 = s2 = 0.0;
  for (int k = a.bilIncStart[g]; k < a.bilIncStart[g + 1]; ++k) {
    const int e = a.bilInc[k];
    const int row = e >> 3, comp = (e >> 1) & 3;
    const double val = (e & 1) ? -1.0 : 1.0;
    const double t = val * x(row);
    if (comp == 0) s0 = s0 + t;
    else if (comp == 1) s1 = s1 + t;
    else s2 = s2 + t;
  }
}

// The sums of a light body g, x given by row.  The list entries of eight
// contacts and then the loads of kAhead contacts are issued together (one
// contact after another waited for its entry, then its row, each time).
template <class X>
__device__ __forceinline__ void gatherSums(const GatherArgs& a, int g, X x, double& s0, double& s1, double& s2) {
  constexpr int kAhead = 4, kIds = 8;
  const int k0 = a.iStart[g], k1 = a.iStart[g + 1];
  int id[kIds];
#pragma unroll
  for (int u = 0; u < kIds; ++u) id[u] = k0 + u < k1 ? a.inc[k0 + u] : 0;
  gatherBilateral(a, g, x, s0, s1, s2);
  for (int kb = k0; kb < k1;) {
#pragma unroll
    for (int h = 0; h < kIds; h += kAhead) {
      if (kb + h >= k1) break;
      double xr[kAhead][3], f[kAhead][9];
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (kb + h + u < k1) gatherLoad(a, id[h + u], x, xr[u], f[u]);
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        if (kb + h + u >= k1) continue;
#pragma unroll
        for (int rr = 0; rr < 3; ++rr) {
          s0 = s0 + f[u][3 * rr] * xr[u][rr];
          s1 = s1 + f[u][3 * rr + 1] * xr[u][rr];
          s2 = s2 + f[u][3 * rr + 2] * xr[u][rr];
        }
      }
    }
    kb += kIds;
    if (kb >= k1) break;
#pragma unroll
    for (int u = 0; u < kIds; ++u) id[u] = kb + u < k1 ? a.inc[kb + u] : 0;
  }
}

// The sums of a body of the heavy list by a wavefront: the lanes form the
// products of 64 contacts (the next 64's loads in flight meanwhile), and
// lanes 0 to 2 add one component each, in order.  Lane q < 3 returns
// component q.
template <class X>
__device__ __forceinline__ double gatherHeavy(const GatherArgs& a, int g, X x, double (&sh)[64][9]) {
  const int lane = threadIdx.x & 63;
  const int k0 = a.iStart[g], k1 = a.iStart[g + 1];
  double s0, s1, s2;
  gatherBilateral(a, g, x, s0, s1, s2);
  double s = lane == 0 ? s0 : lane == 1 ? s1 : s2;
  double xr[3], f[9];
  gatherLoad(a, a.inc[k0 + lane < k1 ? k0 + lane : k0], x, xr, f);
  for (int kb = k0; kb < k1; kb += 64) {
    const int n = min(64, k1 - kb);
#pragma unroll
    for (int rr = 0; rr < 3; ++rr)
#pragma unroll
      for (int q = 0; q < 3; ++q) sh[lane][3 * rr + q] = f[3 * rr + q] * xr[rr];
    if (kb + 64 < k1) gatherLoad(a, a.inc[kb + 64 + lane < k1 ? kb + 64 + lane : k0], x, xr, f);
    __syncthreads();
    if (lane < 3) {
#pragma unroll 4
      for (int e = 0; e < n; ++e) {
        s = s + sh[e][lane];
        s = s + sh[e][3 + lane];
        s = s + sh[e][6 + lane];
      }
    }
    __syncthreads();
  }
  return s;
}

inline GatherArgs gatherArgs(Scene& s) {
  GatherArgs a;
  a.nb = s.nb; a.nbil = s.nbil; a.cap = s.ncCap;
  a.frame = s.frame.p; a.iStart = s.iStart.p; a.inc = s.inc.p;
  a.bilIncStart = s.bilIncStart.p; a.bilInc = s.bilInc.p; a.minv = s.minv.p;
  a.heavy = s.heavy.p; a.counters = s.counters.p;
  return a;
}

}  // namespace dv
