// The plain FP64 APGD path: APGD::solve (APGD.cu:164-361) with every vector
// operation, dot product and norm rounded as the reference's CUSP calls
// round it.  Its products use the exact-order D / D^T sums and its reductions
// the fixed CR256 tree (blocks of 256 consecutive terms reduced with strides
// 128..1, block results added left to right), so every scalar it computes is
// the oracle's.
//
// The reference makes four Schur products a pass (N y before the step and
// again for the objective, N gamma_new for the objective and again for the
// residual), one launch per operation, and reads every scalar back.  Equal
// operands give equal products, so two are made here, and a pass is six
// launches over vectors that are read once:
//   gather   tmp = M^-1 D^T y, y = (1 + beta) gamma_k - beta gamma_{k-1}
//            formed as it is read                    (not after a backtrack)
//   step     N y, g = N y + r, gamma_new = Pi(y - t g)
//   gather   tmp = M^-1 D^T gamma_new
//   product  N gamma_new and the largest entry of getResidual
//   dots     CR256 block sums of the seven dot products
//   decide   the blocks' sums in order, then the Lipschitz test and the
//            acceptance, into the state that the next pass reads
// The state stays on the device: chunks of passes are a captured graph, and
// the host reads the state once per chunk.  Driven from the host, with nine
// read-backs an iteration, it took 250 us an iteration at 9,300 contacts and
// 450 at 256,000; so, 38 and 176 (gathers 12 + 8 us and 48 + 33, step 4 and 27,
// product 4 and 13, dots 3 and 11, decide 4 and 26: the small size bound by
// the launches' latency, the large one by the gathers' scattered reads and
// the serial sum).
#include "dv_exact.h"
#include "dv_geom.h"
#include "dv_internal.h"

#include <cmath>
#include <cstdio>

namespace dv {

struct PlainState {
  double L, t, theta, beta, best, objective;
  int it, bt, backtracks, restart, backtracked;
  int cur, prev, nxt;  // ring slots of gamma_k, gamma_{k-1} and gamma_new
  int hatSrc;          // and of gammaHat (-1: ones)
  int done, accepted;  // accepted: the last pass's step was taken (anti-relaxation follows it)
};

namespace {

constexpr int kT = 256;   // rows of a CR256 block
constexpr int kTR = 64;   // contacts: one wavefront to a workgroup, to reach more CUs
constexpr int kDots = 7;
constexpr int kBacktrackCap = 1100;  // L doubles past 1e308 long before this
constexpr int kPassesPerChunk = 8;

struct PlainArgs {
  GatherArgs ga;
  int nc, nbil, nblk, nMax, maxIt, antiRelax;
  long R;
  double mu, tol, gdiff;
  const int *cA, *cB, *bilA, *bilB;
  double* r;
  double* ring[4];
  double *Ny, *g, *Ng, *y, *ar;
  double *tmp, *fc, *v;
  const double* k;
  double* part;  // kDots runs of nblk, then nMax maxima
};

// y = D x of contact or bilateral row block q, terms in D's row order
template <class F>
__device__ __forceinline__ void rowsOf(const PlainArgs& a, int q, const double* __restrict__ x, F&& out) {
  if (q < a.nbil) {
    double s = 0.0;
    s = s + 1.0 * x[a.bilA[q]];
    if (a.bilB[q] >= 0) s = s + (-1.0) * x[a.bilB[q]];
    out(q, s);
    return;
  }
  const int c = q - a.nbil;
  const long S = a.ga.cap;
  const int A = a.cA[c], B = a.cB[c];
  const double xa0 = x[3 * A], xa1 = x[3 * A + 1], xa2 = x[3 * A + 2];
  const double xb0 = x[3 * B], xb1 = x[3 * B + 1], xb2 = x[3 * B + 2];
#pragma unroll
  for (int rr = 0; rr < 3; ++rr) {
    const double f0 = a.ga.frame[(3 * rr + 0) * S + c];
    const double f1 = a.ga.frame[(3 * rr + 1) * S + c];
    const double f2 = a.ga.frame[(3 * rr + 2) * S + c];
    double s = 0.0;
    s = s + f0 * xa0;
    s = s + f1 * xa1;
    s = s + f2 * xa2;
    s = s + (-f0) * xb0;
    s = s + (-f1) * xb1;
    s = s + (-f2) * xb2;
    out(a.nbil + 3 * c + rr, s);
  }
}

// y of a row: gamma_k, with the momentum term after an accepted step without restart
__device__ __forceinline__ double momentum(const PlainArgs& a, const PlainState& S, long row) {
  const double c = a.ring[S.cur][row];
  return S.restart ? c : (1.0 + S.beta) * c + (-S.beta) * a.ring[S.prev][row];
}

// tmp = M^-1 D^T x for x = y (which 0), gamma_new (1), d = gamma_0 - ones (2)
// or gammaHat (3); bodies without inverse mass get zero.  which 4, after an
// accepted step of anti-relaxation: f_contact = D^T gamma_k and v = M^-1 (k +
// f_contact) of every body.
template <int which>
__global__ __launch_bounds__(kGatherT) void kGather(const PlainArgs* __restrict__ ap, const PlainState* __restrict__ sp,
                                                    int lightBlocks) {
  __shared__ double sh[64][9];
  const PlainArgs& a = *ap;
  const PlainState S = *sp;
  if (which < 2 && S.done) return;
  if (which == 0 && S.backtracked) return;  // y and N y stand
  if (which == 4 && !S.accepted) return;
  const double* x = which == 1 ? a.ring[S.nxt] : which == 4 ? a.ring[S.cur] : S.hatSrc >= 0 ? a.ring[S.hatSrc] : nullptr;
  auto row = [&](long r) {
    if (which == 0) return momentum(a, S, r);
    if (which == 2) return 1.0 * a.ring[0][r] + (-1.0) * 1.0;
    return which != 3 || x ? x[r] : 1.0;
  };
  auto put = [&](int g, int q, double mi, double s) {
    const long i = 3L * g + q;
    double t = 0.0;
    if (which == 4) {
      a.fc[i] = s;
      t = t + mi * (1.0 * a.k[i] + 1.0 * s);
      a.v[i] = t;
    } else {
      if (mi != 0) t = t + mi * s;
      a.tmp[i] = t;
    }
  };
  if ((int)blockIdx.x >= lightBlocks) {
    for (int h = blockIdx.x - lightBlocks; h < a.ga.counters[2]; h += kHeavyBlocks) {
      const int g = a.ga.heavy[h];
      const double mi = a.ga.minv[g];
      const double s = which != 4 && mi == 0 ? 0.0 : gatherHeavy(a.ga, g, row, sh);
      if (threadIdx.x < 3) put(g, threadIdx.x, mi, s);
    }
    return;
  }
  const int g = blockIdx.x * kGatherT + threadIdx.x;
  if (g >= a.ga.nb || a.ga.iStart[g + 1] - a.ga.iStart[g] > kHeavyDegree) return;
  const double mi = a.ga.minv[g];
  double s[3] = {0, 0, 0};
  if (which == 4 || mi != 0) gatherSums(a.ga, g, row, s[0], s[1], s[2]);
  for (int q = 0; q < 3; ++q) put(g, q, mi, s[q]);
}

__global__ __launch_bounds__(kTR) void kStep(const PlainArgs* __restrict__ ap, const PlainState* __restrict__ sp) {
  const PlainArgs& a = *ap;
  const PlainState S = *sp;
  if (S.done) return;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= a.nc + a.nbil) return;
  const bool bil = q < a.nbil;
  const long row = bil ? q : a.nbil + 3L * (q - a.nbil);
  double x[3] = {0, 0, 0};
  if (!S.backtracked) {
    rowsOf(a, q, a.tmp, [&](long i, double ny) {
      const double y = momentum(a, S, i);
      const double g = 1.0 * ny + 1.0 * a.r[i];
      a.Ny[i] = ny;
      a.y[i] = y;
      a.g[i] = g;
      x[i - row] = 1.0 * y + (-S.t) * g;
    });
  } else {
    for (int rr = 0; rr < (bil ? 1 : 3); ++rr) x[rr] = 1.0 * a.y[row + rr] + (-S.t) * a.g[row + rr];
  }
  double* gn = a.ring[S.nxt];
  if (!bil) projectCone<double>(x[0], x[1], x[2], a.mu);
  for (int rr = 0; rr < (bil ? 1 : 3); ++rr) gn[row + rr] = x[rr];
}

// workgroup (one wavefront's) maximum into part
__device__ __forceinline__ void storeMax(double v, double* part) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmax(v, __shfl_xor(v, d, 64));
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

// N x of the vector gathered last; residual: of gamma_new, with getResidual
// (APGD.cu:90-102)
template <bool residual>
__global__ __launch_bounds__(kTR) void kProduct(const PlainArgs* __restrict__ ap, const PlainState* __restrict__ sp) {
  const PlainArgs& a = *ap;
  const PlainState S = *sp;
  if (residual && S.done) return;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  double worst = 0.0;
  if (q < a.nc + a.nbil) {
    const bool bil = q < a.nbil;
    const long row = bil ? q : a.nbil + 3L * (q - a.nbil);
    double t[3] = {0, 0, 0}, x[3] = {0, 0, 0};
    rowsOf(a, q, a.tmp, [&](long i, double n) {
      a.Ng[i] = n;
      if (!residual) return;
      x[i - row] = a.ring[S.nxt][i];
      t[i - row] = 1.0 * a.r[i] + 1.0 * n;
    });
    if (residual) {
      if (a.nc) {
        const double ig = 1.0 / a.gdiff, nig = -1.0 / a.gdiff;
        for (int rr = 0; rr < 3; ++rr) t[rr] = 1.0 * x[rr] + (-a.gdiff) * t[rr];
        if (!bil) projectCone<double>(t[0], t[1], t[2], a.mu);
        for (int rr = 0; rr < 3; ++rr) t[rr] = ig * x[rr] + nig * t[rr];
      }
      for (int rr = 0; rr < (bil ? 1 : 3); ++rr) {
        const double e = fabs(t[rr]);
        worst = fmax(worst, e == e ? e : INFINITY);  // fmax drops NaN; +inf is kept
      }
    }
  }
  if (residual) storeMax(worst, a.part + (long)kDots * a.nblk);
}

// CR256 of N values at once over a block of kT threads: t[i] += t[i + st],
// st = 128..1; the results in thread 0
template <int N>
__device__ __forceinline__ void cr256(double (&v)[N]) {
  __shared__ double sh[2][64][N];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave >= 2)
    for (int k = 0; k < N; ++k) sh[wave - 2][lane][k] = v[k];
  __syncthreads();
  if (wave < 2)
    for (int k = 0; k < N; ++k) v[k] = v[k] + sh[wave][lane][k];  // stride 128
  __syncthreads();
  if (wave == 1)
    for (int k = 0; k < N; ++k) sh[0][lane][k] = v[k];
  __syncthreads();
  if (wave == 0) {
    for (int k = 0; k < N; ++k) v[k] = v[k] + sh[0][lane][k];  // stride 64
#pragma unroll
    for (int st = 32; st >= 1; st >>= 1)
      for (int k = 0; k < N; ++k) v[k] = v[k] + __shfl_down(v[k], st, 64);
  }
}

// the pass's seven dot products: gamma_new.Ng, gamma_new.r, y.Ny, y.r, t.t,
// g.t (t = gamma_new - y) and g.(gamma_new - gamma_k)
__global__ __launch_bounds__(kT) void kDots7(const PlainArgs* __restrict__ ap, const PlainState* __restrict__ sp) {
  const PlainArgs& a = *ap;
  const PlainState S = *sp;
  if (S.done) return;
  const long i = (long)blockIdx.x * kT + threadIdx.x;
  if ((long)blockIdx.x * kT >= a.R) return;
  double v[kDots] = {0, 0, 0, 0, 0, 0, 0};
  if (i < a.R) {
    const double gn = a.ring[S.nxt][i], y = a.y[i], r = a.r[i], g = a.g[i];
    const double t = 1.0 * gn + (-1.0) * y, d = 1.0 * gn + (-1.0) * a.ring[S.cur][i];
    v[0] = gn * a.Ng[i];
    v[1] = gn * r;
    v[2] = y * a.Ny[i];
    v[3] = y * r;
    v[4] = t * t;
    v[5] = g * t;
    v[6] = g * d;
  }
  cr256(v);
  if (threadIdx.x == 0)
    for (int k = 0; k < kDots; ++k) a.part[(long)k * a.nblk + blockIdx.x] = v[k];
}

// setup (first): gamma_0 into ring slot 0 (APGD.cu:116-122, 195-201) and
// |gamma_0 - ones|^2; second: |N d|^2; last: gammaHat.N gammaHat, gammaHat.r
// with gamma := gammaHat
template <int which>
__global__ __launch_bounds__(kT) void kDotsEnds(const PlainArgs* __restrict__ ap, const PlainState* __restrict__ sp,
                                                double* gamma, int warm) {
  const PlainArgs& a = *ap;
  const long i = (long)blockIdx.x * kT + threadIdx.x;
  if ((long)blockIdx.x * kT >= a.R) return;
  double v[2] = {0, 0};
  if (i < a.R) {
    if (which == 0) {
      const double g = !warm && i < 3L * a.nc ? (i % 3 == 0 ? 1.0 : 0.0) : gamma[i];
      a.ring[0][i] = g;
      a.ar[i] = 0.0;  // APGD.cu:189
      const double t = 1.0 * g + (-1.0) * 1.0;
      v[0] = t * t;
    } else if (which == 1) {
      v[1] = a.Ng[i] * a.Ng[i];
    } else {
      const int h = sp->hatSrc;
      const double x = h >= 0 ? a.ring[h][i] : 1.0;
      v[0] = x * a.Ng[i];
      v[1] = x * a.r[i];
      gamma[i] = x;
    }
  }
  cr256(v);
  if (threadIdx.x == 0) {
    if (which != 1) a.part[blockIdx.x] = v[0];
    if (which != 0) a.part[(long)a.nblk + blockIdx.x] = v[1];
  }
}

// Block sums added left to right, and the maximum by the last wavefront.
// Wavefront k stages run k through LDS and lane k of the first wavefront adds
// it, so that one add serves all runs: a run to each wavefront, its blocks
// handed to the add from lane to lane, was bound by the issue of two
// wavefronts per SIMD (44 us for the 3,003 blocks of 256,000 contacts,
// against 26).
// out[k] valid in every thread.
constexpr int kStage = 512;
__device__ void serialSums(const PlainArgs& a, int runs, bool withMax, double* out) {
  constexpr int kPer = kStage / 64, kAdd = 16;
  __shared__ double st[2][kDots][kStage + 2];  // (padded: the lanes' reads fall in different banks)
  __shared__ double res[kDots + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int last = a.nblk - 1;
  double next[kPer];
  auto fetch = [&](int b) {
    const double* run = a.part + (long)(wave < runs ? wave : 0) * a.nblk;
#pragma unroll
    for (int i = 0; i < kPer; ++i) next[i] = run[min(b + 64 * i + lane, last)];
  };
  fetch(0);
  double acc = 0;
  int buf = 0;
  for (int b = 0; b < a.nblk; b += kStage, buf ^= 1) {
    if (wave < runs)
#pragma unroll
      for (int i = 0; i < kPer; ++i)  // (past the end: zeros, which change no sum that began at +0)
        st[buf][wave][64 * i + lane] = b + 64 * i + lane <= last ? next[i] : 0.0;
    __syncthreads();
    if (b + kStage < a.nblk) fetch(b + kStage);
    if (wave == 0 && lane < runs) {
      const double* mine = st[buf][lane];
      const int n = min(kStage, a.nblk - b);
      for (int i = 0; i < n; i += kAdd) {
        double x[kAdd];
#pragma unroll
        for (int k = 0; k < kAdd; ++k) x[k] = mine[i + k];
#pragma unroll
        for (int k = 0; k < kAdd; ++k) acc += x[k];
      }
    }
  }
  if (wave == 0 && lane < runs) res[lane] = acc;
  if (withMax && wave == kDots) {
    double m = 0;
    const double* run = a.part + (long)kDots * a.nblk;
    for (int b = 0; b < a.nMax; b += 512) {
      double x[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) x[k] = run[min(b + 64 * k + lane, a.nMax - 1)];
#pragma unroll
      for (int k = 0; k < 8; ++k) m = fmax(m, x[k]);
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) m = fmax(m, __shfl_xor(m, d, 64));
    if (lane == 0) res[kDots] = m;
  }
  __syncthreads();
  for (int k = 0; k <= kDots; ++k) out[k] = res[k];
}

__global__ __launch_bounds__(64 * (kDots + 1)) void kPlainSetup(const PlainArgs* __restrict__ ap, PlainState* sp) {
  double d[kDots + 1];
  serialSums(*ap, 2, false, d);
  if (threadIdx.x) return;
  PlainState S;
  double L = sqrt(d[0]);
  L = sqrt(d[1]) / L;
  S.L = L;
  S.t = 1.0 / L;
  S.theta = 1.0;
  S.beta = 0.0;
  S.best = 10e30;
  S.objective = 0;
  S.it = S.bt = S.backtracks = S.backtracked = S.accepted = 0;
  S.restart = 1;
  S.cur = S.prev = 0;
  S.nxt = 1;
  S.hatSrc = -1;
  S.done = ap->maxIt <= 0 ? 1 : 0;
  *sp = S;
}

__global__ __launch_bounds__(64 * (kDots + 1)) void kPlainDecide(const PlainArgs* __restrict__ ap, PlainState* sp) {
  const PlainArgs& a = *ap;
  if (sp->done) {  // (the passes queued after the last one: no step was taken)
    __syncthreads();
    if (threadIdx.x == 0) sp->accepted = 0;
    return;
  }
  double d[kDots + 1];
  serialSums(a, kDots, true, d);
  if (threadIdx.x) return;
  PlainState S = *sp;
  S.accepted = 0;
  const double obj1 = 0.5 * d[0] + d[1];
  double obj2 = 0.5 * d[2] + d[3];
  const double nr = sqrt(d[4]);
  obj2 += d[5] + 0.5 * S.L * (nr * nr);
  if (obj1 >= obj2 && S.bt < kBacktrackCap) {
    ++S.bt;
    ++S.backtracks;
    S.backtracked = 1;
    S.L = 2.0 * S.L;
    S.t = 1.0 / S.L;
    *sp = S;
    return;
  }
  S.bt = S.backtracked = 0;
  const double theta = S.theta;
  double thetaNew = (-(theta * theta) + theta * sqrt(theta * theta + 4.0)) / 2.0;
  S.beta = theta * (1.0 - theta) / (theta * theta + thetaNew);
  const double res = d[kDots];
  if (!(res < INFINITY)) {  // non-finite data: the solve ends as diverged
    S.best = res;
    S.done = 1;
    *sp = S;
    return;
  }
  if (res < S.best) {
    S.best = res;
    S.hatSrc = S.nxt;
  }
  if (S.best < a.tol) {
    S.done = 1;
    *sp = S;
    return;
  }
  S.restart = 0;
  if (d[6] > 0) {
    S.restart = 1;
    thetaNew = 1.0;
  }
  S.L = 0.9 * S.L;
  S.t = 1.0 / S.L;
  S.theta = thetaNew;
  S.prev = S.cur;
  S.cur = S.nxt;
  for (int k = 0; k < 4; ++k)  // a slot that holds none of gamma_k, gamma_{k-1} and gammaHat
    if (k != S.cur && k != S.prev && k != S.hatSrc) {
      S.nxt = k;
      break;
    }
  S.accepted = 1;
  if (++S.it >= a.maxIt) S.done = 1;
  *sp = S;
}

__global__ __launch_bounds__(64 * (kDots + 1)) void kPlainEnd(const PlainArgs* __restrict__ ap, PlainState* sp) {
  double d[kDots + 1];
  serialSums(*ap, 2, false, d);
  if (threadIdx.x == 0) sp->objective = 0.5 * d[0] + d[1];
}

// Anti-relaxation after an accepted step (APGD.cu:104-114, 335-345): r -= ar;
// f_contact = D^T gamma; v = M^-1 (k + f_contact) (kGather<4>); ar[3c] = mu |(s_u, s_v)| of
// s = D v, indexed from 0 without the bilateral offset as the reference
// indexes it; r += ar.  Like the reference it leaves v and f_contact
// overwritten (the update after the solve recomputes both) and r holding the
// last term.
__global__ __launch_bounds__(kTR) void kRelaxRows(const PlainArgs* __restrict__ ap, const PlainState* __restrict__ sp) {
  const PlainArgs& a = *ap;
  if (!sp->accepted) return;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= a.nc + a.nbil) return;
  rowsOf(a, q, a.v, [&](long i, double s) { a.Ng[i] = s; });
}
__global__ __launch_bounds__(kT) void kRelaxR(const PlainArgs* __restrict__ ap, const PlainState* __restrict__ sp) {
  const PlainArgs& a = *ap;
  if (!sp->accepted) return;
  const long i = (long)blockIdx.x * kT + threadIdx.x;
  if (i >= a.R) return;
  const double r = -1.0 * a.ar[i] + 1.0 * a.r[i];
  double n = a.ar[i];  // (rows past the contacts' keep theirs)
  if (i < 3L * a.nc) {
    if (i % 3 == 0) {
      const double u = a.Ng[i + 1], v = a.Ng[i + 2];
      n = sqrt(u * u + v * v) * a.mu;
    } else {
      n = 0.0;
    }
  }
  a.ar[i] = n;
  a.r[i] = 1.0 * n + 1.0 * r;
}

// grids by capacity, so that a captured chunk outlives changes of the counts
struct PlainGrid {
  const PlainArgs* a;
  PlainState* s;
  int bodies, items, rows, antiRelax;
};

void enqueuePass(const PlainGrid& P, hipStream_t st) {
  hipLaunchKernelGGL(kGather<0>, dim3(P.bodies + kHeavyBlocks), dim3(kGatherT), 0, st, P.a, (const PlainState*)P.s, P.bodies);
  hipLaunchKernelGGL(kStep, dim3(P.items), dim3(kTR), 0, st, P.a, (const PlainState*)P.s);
  hipLaunchKernelGGL(kGather<1>, dim3(P.bodies + kHeavyBlocks), dim3(kGatherT), 0, st, P.a, (const PlainState*)P.s, P.bodies);
  hipLaunchKernelGGL(kProduct<true>, dim3(P.items), dim3(kTR), 0, st, P.a, (const PlainState*)P.s);
  hipLaunchKernelGGL(kDots7, dim3(P.rows), dim3(kT), 0, st, P.a, (const PlainState*)P.s);
  hipLaunchKernelGGL(kPlainDecide, dim3(1), dim3(64 * (kDots + 1)), 0, st, P.a, P.s);
  if (P.antiRelax) {
    hipLaunchKernelGGL(kGather<4>, dim3(P.bodies + kHeavyBlocks), dim3(kGatherT), 0, st, P.a, (const PlainState*)P.s, P.bodies);
    hipLaunchKernelGGL(kRelaxRows, dim3(P.items), dim3(kTR), 0, st, P.a, (const PlainState*)P.s);
    hipLaunchKernelGGL(kRelaxR, dim3(P.rows), dim3(kT), 0, st, P.a, (const PlainState*)P.s);
  }
}

}  // namespace

void solvePlain(Scene& s) {
  const long R = s.R, cap = 3L * s.ncCap + s.nbil;
  const long S = std::max<long>(cap, 1);
  s.work.reserve((size_t)9 * S);
  const int nblkCap = blocksFor(S, kT), itemsCap = blocksFor((long)s.ncCap + s.nbil, kTR);
  s.partials.reserve((size_t)kDots * nblkCap + itemsCap);
  s.plainState.reserve(sizeof(PlainArgs) + sizeof(PlainState));
  PlainArgs a;
  std::memset(&a, 0, sizeof(a));
  a.ga = gatherArgs(s);
  a.nc = s.nc; a.nbil = s.nbil; a.R = R;
  a.nblk = blocksFor(R, kT);
  a.nMax = blocksFor((long)s.nc + s.nbil, kTR);
  a.maxIt = s.maxIt; a.antiRelax = s.antiRelax ? 1 : 0;
  a.mu = s.mu; a.tol = s.tol;
  const double cnt = (double)((long)s.nc + s.nbil);
  a.gdiff = 1.0 / (cnt * cnt);
  a.cA = s.cA.p; a.cB = s.cB.p; a.bilA = s.bilA.p; a.bilB = s.bilB.p;
  a.r = s.r.p;
  double* W = s.work.p;
  for (int k = 0; k < 4; ++k) a.ring[k] = W + k * S;
  a.Ny = W + 4 * S; a.g = W + 5 * S; a.Ng = W + 6 * S; a.y = W + 7 * S; a.ar = W + 8 * S;
  a.tmp = s.tmp.p; a.fc = s.fContact.p; a.v = s.v.p; a.k = s.k.p;
  a.part = s.partials.p;
  PlainGrid P;
  std::memset(&P, 0, sizeof(P));
  P.a = reinterpret_cast<const PlainArgs*>(s.plainState.p);
  P.s = reinterpret_cast<PlainState*>(s.plainState.p + sizeof(PlainArgs));
  P.bodies = gatherBlocks(a.ga);
  P.items = itemsCap;
  P.rows = nblkCap;
  P.antiRelax = a.antiRelax;
  const hipStream_t st = s.stream;
  if (!s.plainHost) DV_HIP(hipHostMalloc(&s.plainHost, 2 * sizeof(PlainState) + sizeof(PlainArgs), hipHostMallocDefault));
  PlainState* host = static_cast<PlainState*>(s.plainHost);
  std::memcpy(host + 2, &a, sizeof(a));
  DV_HIP(hipMemcpyAsync(s.plainState.p, host + 2, sizeof(a), hipMemcpyHostToDevice, st));
  const PlainState* sp = P.s;
  double* gamma = s.gamma.p;
  const int warm = s.warm ? 1 : 0;
  hipLaunchKernelGGL(kDotsEnds<0>, dim3(a.nblk), dim3(kT), 0, st, P.a, sp, gamma, warm);
  hipLaunchKernelGGL(kGather<2>, dim3(P.bodies + kHeavyBlocks), dim3(kGatherT), 0, st, P.a, sp, P.bodies);
  hipLaunchKernelGGL(kProduct<false>, dim3(a.nMax), dim3(kTR), 0, st, P.a, sp);
  hipLaunchKernelGGL(kDotsEnds<1>, dim3(a.nblk), dim3(kT), 0, st, P.a, sp, gamma, warm);
  hipLaunchKernelGGL(kPlainSetup, dim3(1), dim3(64 * (kDots + 1)), 0, st, P.a, P.s);
  if (!s.noGraph && !s.plainGraph.matches(&P, sizeof(P))) {
    s.plainGraph.reset();
    hipGraph_t graph;
    DV_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    for (int k = 0; k < kPassesPerChunk; ++k) enqueuePass(P, st);
    DV_HIP(hipStreamEndCapture(st, &graph));
    s.plainGraph.instantiate(graph, "hipGraphInstantiate(plain passes)");
    s.plainGraph.setKey(&P, sizeof(P));
  }
  hipEvent_t polled[2] = {s.ev[5], s.ev[6]};
  auto launch = [&](int b) {  // a chunk, then the copy of the state after it
    if (s.noGraph)
      for (int k = 0; k < kPassesPerChunk; ++k) enqueuePass(P, st);
    else
      s.plainGraph.launch(st);
    DV_HIP(hipMemcpyAsync(host + b, P.s, sizeof(PlainState), hipMemcpyDeviceToHost, st));
    DV_HIP(hipEventRecord(polled[b], st));
  };
  // the next chunk is queued before this one's state is read (after the solve
  // has ended its passes exit at once)
  launch(0);
  for (int b = 0;; b ^= 1) {
    launch(b ^ 1);
    DV_HIP(hipEventSynchronize(polled[b]));
    if (host[b].done) break;
  }
  hipLaunchKernelGGL(kGather<3>, dim3(P.bodies + kHeavyBlocks), dim3(kGatherT), 0, st, P.a, sp, P.bodies);
  hipLaunchKernelGGL(kProduct<false>, dim3(a.nMax), dim3(kTR), 0, st, P.a, sp);
  hipLaunchKernelGGL(kDotsEnds<2>, dim3(a.nblk), dim3(kT), 0, st, P.a, sp, gamma, warm);
  hipLaunchKernelGGL(kPlainEnd, dim3(1), dim3(64 * (kDots + 1)), 0, st, P.a, P.s);
  DV_HIP(hipMemcpyAsync(host, P.s, sizeof(PlainState), hipMemcpyDeviceToHost, st));
  DV_HIP(hipStreamSynchronize(st));
  DV_HIP(hipGetLastError());
  if (s.verbose) printf("  Iterations: %d Residual: %g\n", host->it, host->best);
  s.stats.objective = host->objective;
  s.stats.iterations = host->it;
  s.stats.residual = host->best;
  s.stats.backtracks = host->backtracks;
}

}  // namespace dv
