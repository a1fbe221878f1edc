// Assembly and update kernels of the time step, and the exact-order D / D^T
// products.
//
// D is never materialised as COO: a contact row block is the 3x3 frame
// [n; u; v] (+ for body A, - for body B; System.cu:753-762, 904-909,
// 963-967, 1023-1027) and a bilateral row has +1 / -1 at its DOFs
// (System.cu:622-638).  The products below visit the terms in the order in
// which a row-sorted COO SpMV visits them (D's rows: A's three columns then
// B's; D^T's rows: bilateral rows ascending, then contacts ascending with the
// n, u, v rows in turn), and add them one by one from 0.0 without fused
// multiply-adds, so they round exactly like the oracle's COO SpMV.
#include "dv_exact.h"

namespace dv {
namespace {

constexpr int kT = 256;

// k = M v + h f - h f_elastic  (System.cu:1411-1417, 1502-1514; f_elastic = 0 for bodies)
// and y = M^-1 k (diagonal COO: 0.0 + minv * k)
__global__ __launch_bounds__(kT) void kBuildK(int nb, const double* __restrict__ minv,
                                              const double* __restrict__ v, const double* __restrict__ f,
                                              double* __restrict__ k, double* __restrict__ y, double h) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 3 * nb) return;
  const double mi = minv[i / 3];
  const double m = mi != 0 ? 1.0 / mi : mi;
  double kk = m * v[i];
  const double fEl = 0.0;
  kk = (h * f[i] + (-h) * fEl) + 1.0 * kk;
  k[i] = kk;
  double s = 0.0;
  s = s + mi * kk;
  y[i] = s;
}

struct RowArgs {
  int nc, nbil, cap;
  const double* frame;
  const int* cA;
  const int* cB;
  const int* bilA;
  const int* bilB;
};

// row q of D x, one thread per contact / bilateral row; put(row, value) takes
// its values
template <class Put>
__device__ __forceinline__ void rowOfD(const RowArgs& a, int q, const double* __restrict__ x, const Put& put) {
  if (q < a.nbil) {
    double s = 0.0;
    s = s + 1.0 * x[a.bilA[q]];
    if (a.bilB[q] >= 0) s = s + (-1.0) * x[a.bilB[q]];
    put(q, 0, s);
    return;
  }
  const int c = q - a.nbil;
  const long S = a.cap;
  const int A = a.cA[c], B = a.cB[c];
  const double xa0 = x[3 * A], xa1 = x[3 * A + 1], xa2 = x[3 * A + 2];
  const double xb0 = x[3 * B], xb1 = x[3 * B + 1], xb2 = x[3 * B + 2];
#pragma unroll
  for (int rr = 0; rr < 3; ++rr) {
    const double f0 = a.frame[(3 * rr + 0) * S + c];
    const double f1 = a.frame[(3 * rr + 1) * S + c];
    const double f2 = a.frame[(3 * rr + 2) * S + c];
    double s = 0.0;
    s = s + f0 * xa0;
    s = s + f1 * xa1;
    s = s + f2 * xa2;
    s = s + (-f0) * xb0;
    s = s + (-f1) * xb1;
    s = s + (-f2) * xb2;
    put(a.nbil + 3 * c + rr, rr, s);
  }
}

// y = D x  (+ optional b: y = 1.0*b + D x)
__global__ __launch_bounds__(kT) void kRowsD(RowArgs a, const double* __restrict__ x,
                                             const double* __restrict__ badd, double* __restrict__ y) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= a.nc + a.nbil) return;
  rowOfD(a, q, x, [&](int row, int, double s) { y[row] = badd ? 1.0 * badd[row] + s : s; });
}

// f = D^T x and tmp = M^-1 f per body, terms in D^T row order.  With
// skipFixed, bodies with M^-1 = 0 get tmp = +0 without the sum (0.0 + 0*f).
__global__ __launch_bounds__(kGatherT) void kGatherDT(GatherArgs a, const double* __restrict__ x,
                                                      double* __restrict__ fOut, double* __restrict__ tmpOut,
                                                      int skipFixed, int lightBlocks) {
  __shared__ double sh[64][9];
  auto row = [&](long r) { return x[r]; };
  if ((int)blockIdx.x >= lightBlocks) {
    for (int h = blockIdx.x - lightBlocks; h < a.counters[2]; h += kHeavyBlocks) {
      const int g = a.heavy[h], q = threadIdx.x;
      const double mi = a.minv[g];
      const bool fixed = skipFixed && mi == 0;
      const double s = fixed ? 0.0 : gatherHeavy(a, g, row, sh);
      if (q >= 3) continue;
      if (fOut && !fixed) fOut[3 * g + q] = s;
      if (tmpOut) {
        double t = 0.0;
        if (!fixed) t = t + mi * s;
        tmpOut[3 * g + q] = t;
      }
    }
    return;
  }
  const int g = blockIdx.x * kGatherT + threadIdx.x;
  if (g >= a.nb || a.iStart[g + 1] - a.iStart[g] > kHeavyDegree) return;
  const double mi = a.minv[g];
  if (skipFixed && mi == 0) {
    tmpOut[3 * g] = 0.0; tmpOut[3 * g + 1] = 0.0; tmpOut[3 * g + 2] = 0.0;
    return;
  }
  double s0, s1, s2;
  gatherSums(a, g, row, s0, s1, s2);
  if (fOut) { fOut[3 * g] = s0; fOut[3 * g + 1] = s1; fOut[3 * g + 2] = s2; }
  if (tmpOut) {
    double t0 = 0.0, t1 = 0.0, t2 = 0.0;
    t0 = t0 + mi * s0; t1 = t1 + mi * s1; t2 = t2 + mi * s2;
    tmpOut[3 * g] = t0; tmpOut[3 * g + 1] = t1; tmpOut[3 * g + 2] = t2;
  }
}

// b: bilateral rows violation / h (System.cu:1526-1544), contact rows
// (gap/h, 0, 0) (System.cu:1516-1524); and r = D M^-1 k + b.  Launches bound
// the assembly of small scenes: k, M^-1 k, b and r in four took 25 us of one
// sphere's step, in two 12.
__global__ __launch_bounds__(kT) void kBuildR(RowArgs a, const double* __restrict__ gap, const double* bilVel,
                                              const double* bilT0, const double* bilP0,
                                              const double* __restrict__ p, const double* __restrict__ x, double h,
                                              double time, double* __restrict__ b, double* __restrict__ r) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= a.nc + a.nbil) return;
  double first;
  if (q < a.nbil) {
    double vel = bilVel[q], t0 = bilT0[q];
    if (time < t0) vel = 0;
    double viol = a.bilB[q] < 0 ? p[a.bilA[q]] - bilP0[q] - vel * (time - t0)
                                : p[a.bilA[q]] - p[a.bilB[q]] - vel * (time - t0);
    first = viol / h;
  } else {
    first = gap[q - a.nbil] / h;
  }
  rowOfD(a, q, x, [&](int row, int rr, double s) {
    const double bb = rr ? 0.0 : first;
    b[row] = bb;
    r[row] = 1.0 * bb + s;
  });
}

// v = M^-1 (k + f_c), f_c /= h, p += h v  (System.cu:570-581)
struct UpdateArgs {
  int nb;
  const double* minv;
  const double* k;
  double* fc;
  double* v;
  double* p;
  double h;
};
// DOF i, whose contact impulse is f
__device__ __forceinline__ void updateDof(const UpdateArgs& u, int i, double mi, double f) {
  const double t = 1.0 * u.k[i] + 1.0 * f;
  double vv = 0.0;
  vv = vv + mi * t;
  u.fc[i] = (1.0 / u.h) * f;
  u.v[i] = vv;
  u.p[i] = u.h * vv + u.p[i];
}
__global__ __launch_bounds__(kT) void kUpdate(UpdateArgs u, int haveRows) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 3 * u.nb) return;
  const double mi = u.minv[i / 3];
  if (haveRows) {
    updateDof(u, i, mi, u.fc[i]);
    return;
  }
  double vv = 0.0;
  vv = vv + mi * u.k[i];
  u.fc[i] = 0.0;
  u.v[i] = vv;
  u.p[i] = u.h * vv + u.p[i];
}

// The update with f_c = D^T gamma formed as it is used: the bodies' sums in
// D^T row order (by one wavefront of a workgroup: 64 bodies each spread a small
// scene over more CUs), and in the first kHeavyBlocks workgroups those of the heavy
// list (more than kHeavyDegree incidences), one workgroup each, FP64 sums in
// a fixed tree order.  In one launch: gather, heavy bodies and update in three
// took 10 us of one sphere's step and 30 of 1,000 spheres'.
__global__ __launch_bounds__(kT) void kGatherUpdate(GatherArgs a, const double* __restrict__ x, UpdateArgs u) {
  if (blockIdx.x >= kHeavyBlocks) {
    const int g = ((int)blockIdx.x - kHeavyBlocks) * kGatherT + threadIdx.x;
    if (threadIdx.x >= kGatherT || g >= a.nb || a.iStart[g + 1] - a.iStart[g] > kHeavyDegree) return;
    const double mi = u.minv[g];
    double s0, s1, s2;
    gatherSums(a, g, [&](long r) { return x[r]; }, s0, s1, s2);
    updateDof(u, 3 * g, mi, s0);
    updateDof(u, 3 * g + 1, mi, s1);
    updateDof(u, 3 * g + 2, mi, s2);
    return;
  }
  const int nHeavy = a.counters[2];
  __shared__ double red[kT / 64][3];
  const long S = a.cap;
  for (int hq = blockIdx.x; hq < nHeavy; hq += kHeavyBlocks) {
    const int g = a.heavy[hq];
    double s0 = 0, s1 = 0, s2 = 0;
    for (int k = a.iStart[g] + threadIdx.x; k < a.iStart[g + 1]; k += kT) {
      const int e = a.inc[k];
      const int c = e >> 1;
      const double sg = (e & 1) ? -1.0 : 1.0;
      const long base = a.nbil + 3L * c;
#pragma unroll
      for (int rr = 0; rr < 3; ++rr) {
        const double xr = sg * x[base + rr];
        s0 += a.frame[(3 * rr + 0) * S + c] * xr;
        s1 += a.frame[(3 * rr + 1) * S + c] * xr;
        s2 += a.frame[(3 * rr + 2) * S + c] * xr;
      }
    }
    if (threadIdx.x == 0) {
      for (int k = a.bilIncStart[g]; k < a.bilIncStart[g + 1]; ++k) {
        const int e = a.bilInc[k];
        const double t = ((e & 1) ? -1.0 : 1.0) * x[e >> 3];
        const int comp = (e >> 1) & 3;
        if (comp == 0) s0 += t; else if (comp == 1) s1 += t; else s2 += t;
      }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
      s0 += __shfl_xor(s0, d, 64);
      s1 += __shfl_xor(s1, d, 64);
      s2 += __shfl_xor(s2, d, 64);
    }
    if ((threadIdx.x & 63) == 0) {
      red[threadIdx.x >> 6][0] = s0; red[threadIdx.x >> 6][1] = s1; red[threadIdx.x >> 6][2] = s2;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
      double v = 0;
      for (int w = 0; w < kT / 64; ++w) v += red[w][threadIdx.x];
      updateDof(u, 3 * g + threadIdx.x, u.minv[g], v);
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(kT) void kFillD(double* x, long n, double val) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = val;
}

RowArgs rowArgs(Scene& s) {
  RowArgs a;
  a.nc = s.nc; a.nbil = s.nbil; a.cap = s.ncCap;
  a.frame = s.frame.p; a.cA = s.cA.p; a.cB = s.cB.p;
  a.bilA = s.bilA.p; a.bilB = s.bilB.p;
  return a;
}

}  // namespace

void fillDevice(Scene& s, double* x, long n, double v) {
  if (n > 0) hipLaunchKernelGGL(kFillD, dim3(blocksFor(n, kT)), dim3(kT), 0, s.stream, x, n, v);
}

void buildK(Scene& s) {
  hipLaunchKernelGGL(kBuildK, dim3(blocksFor(3L * s.nb, kT)), dim3(kT), 0, s.stream, s.nb, s.minv.p, s.v.p,
                     s.f.p, s.k.p, s.tmp.p, s.h);
}

void ensureRowBuffers(Scene& s) {
  const int R = s.nbil + 3 * s.nc;
  s.R = R;
  s.r.reserve(std::max(R, 1));
  s.b.reserve(std::max(R, 1));
  // gamma keeps its leading values across steps and zero-fills growth, as
  // thrust::device_vector::resize does (APGD.cu:166)
  s.gamma.reserveKeep(std::max(R, 1), (size_t)s.gammaLen, s.stream);
  if (R > s.gammaLen) fillDevice(s, s.gamma.p + s.gammaLen, R - s.gammaLen, 0.0);
  s.gammaLen = R;
}

// r = D M^-1 k + b  (System.cu:1561-1580), from the M^-1 k that buildK left in
// tmp
void buildR(Scene& s) {
  ensureRowBuffers(s);
  const int items = s.nc + s.nbil;
  if (items == 0) return;
  hipLaunchKernelGGL(kBuildR, dim3(blocksFor(items, kT)), dim3(kT), 0, s.stream, rowArgs(s), s.gap.p, s.bilVel.p,
                     s.bilT0.p, s.bilP0.p, s.p.p, (const double*)s.tmp.p, s.h, s.time, s.b.p, s.r.p);
}

static void gatherExact(Scene& s, const double* x, double* fOut, double* tmpOut, bool skipFixed) {
  const GatherArgs a = gatherArgs(s);
  hipLaunchKernelGGL(kGatherDT, dim3(gatherBlocks(a) + kHeavyBlocks), dim3(kGatherT), 0, s.stream, a, x, fOut, tmpOut,
                     skipFixed ? 1 : 0, gatherBlocks(a));
}

// y = D (M^-1 (D^T x))  (APGD.cu:81-87)
void schurExact(Scene& s, const double* x, double* y) {
  gatherExact(s, x, nullptr, s.tmp.p, true);
  const int items = s.nc + s.nbil;
  if (items)
    hipLaunchKernelGGL(kRowsD, dim3(blocksFor(items, kT)), dim3(kT), 0, s.stream, rowArgs(s), (const double*)s.tmp.p,
                       (const double*)nullptr, y);
  else  // (the vectors keep the last step's length, whose rows are gone)
    fillDevice(s, y, s.R, 0.0);
}

void rowsD(Scene& s, const double* x, const double* badd, double* y) {
  const int items = s.nc + s.nbil;
  if (items)
    hipLaunchKernelGGL(kRowsD, dim3(blocksFor(items, kT)), dim3(kT), 0, s.stream, rowArgs(s), x, badd, y);
}

void updateState(Scene& s, bool haveRows, bool exactOrder) {
  const UpdateArgs u{s.nb, s.minv.p, s.k.p, s.fContact.p, s.v.p, s.p.p, s.h};
  if (haveRows && !exactOrder) {
    const GatherArgs a = gatherArgs(s);
    hipLaunchKernelGGL(kGatherUpdate, dim3(kHeavyBlocks + gatherBlocks(a)), dim3(kT), 0, s.stream, a,
                       (const double*)s.gamma.p, u);
    return;
  }
  if (haveRows) gatherExact(s, s.gamma.p, s.fContact.p, nullptr, false);
  hipLaunchKernelGGL(kUpdate, dim3(blocksFor(3L * s.nb, kT)), dim3(kT), 0, s.stream, u, haveRows ? 1 : 0);
}

}  // namespace dv
