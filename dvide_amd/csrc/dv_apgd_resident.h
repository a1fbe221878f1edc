// The resident passes: thousands of passes of a slot in one launch, its
// contacts' state in registers and its workgroups exchanging what the other
// half of a pass needs through device-scope stores and flags.
//
// Included by dv_apgd_fused.hip after the pass kernels, whose arithmetic and
// summation orders it repeats bit for bit (a slot may run some chunks here
// and others as P1/P2 launches, and ends in the same state).
//
// Why: a pass as two launches costs two kernel boundaries and a reload of the
// whole state.  A grid barrier used to cost more, because an agent-scope
// release writes back the L2; but the data that crosses workgroups is small
// (J and tmp), and stored at device scope it needs no write-back.  Such a
// barrier takes 1.1 us among 8 workgroups, 1.3 among 32, 2.0 among 64 and 3.0
// among 256, and an exchange of 16 bytes per thread another 0.9 to 2.7.
// us per pass, launches -> resident (piles of the given contacts):
//   contacts    200   2,400   18,000  64,000  126,000  160,000  256,000
//   FP64       10.7    13.9     15.5    17.1     21.0     26.0     27.2
//          ->   5.4     9.2     10.2    11.8     14.2     18.3     23.3
//   mixed       8.8    11.7     12.9    13.6     16.1     18.9     20.7
//          ->   4.5     7.9      8.4    10.0     11.9     14.6     17.8
// What a pass waits for (18,000 contacts, mixed): P1 0.8 us, draining J 0.8,
// the partial sums under the flags' flight 1.1, P2 1.5, draining tmp and the
// flags 1.6, the totals and the decision 1.1.
#pragma once

// A workgroup's place: member `rank` of the `members` of slot `slot`'s team.
struct TeamItem {
  int slot, rank, members, pad;
};

// Per slot, in 64-bit words: the formation's outcome, then one flag per
// member.  Flags hold epochs that only grow, so nothing is cleared between
// launches.
constexpr int kTeamMax = 256;
constexpr int kTeamSync = 16 + kTeamMax;
// A team whose members are not all running after this long gives up (the
// 100 MHz wall clock): the slot's passes then run as launches.
constexpr unsigned long long kFormTicks = 200000ull;         // 2 ms
constexpr unsigned long long kFormTicksMany = 10000000ull;   // 100 ms: several scenes' teams wait for room
// No wait of a formed team lasts this long; a member that sees it ends.
constexpr unsigned long long kBarrierTicks = 1000000000ull;  // 10 s

using u64 = unsigned long long;

// Device-scope accesses: stores write through to where every XCD sees them
// and loads never return a line another workgroup has replaced, so exchanged
// data needs no cache write-back (which an agent-scope release does for the
// whole L2, and which made a grid barrier cost more than a kernel boundary).
constexpr int kDeviceScope = 16;  // the sc1 bit of the buffer instructions' cache policy
__device__ __forceinline__ u64 coLoad(const u64* p) {
  return __hip_atomic_load(gl(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void coStore(u64* p, u64 v) {
  __hip_atomic_store(gl(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double coLoad(const double* p) {
  return __builtin_bit_cast(double, coLoad(reinterpret_cast<const u64*>(p)));
}
__device__ __forceinline__ void coStore(double* p, double v) {
  coStore(reinterpret_cast<u64*>(p), __builtin_bit_cast(u64, v));
}
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
template <typename TM>
struct V3 {
  TM x, y, z;
};
// An exchanged array of n 3-vectors.  FP32: padded to 16 bytes.  FP64: the x
// and y of all entries, then the z, so that a wavefront's stores are two
// contiguous runs (padded to 32 bytes they were two half-filled ones, and took
// twice as long to drain).  Entry kNone reads as zero without touching
// memory: its offset lies past the bound that the hardware checks.
constexpr int kNone = -1;
template <typename TM>
struct CoArray {
  static constexpr int kSplit = sizeof(TM) == 8;
  __amdgpu_buffer_rsrc_t r, rz;
  __device__ CoArray(void* p, long n)
      : r(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)(16 * n), 0x00027000)),
        rz(__builtin_amdgcn_make_buffer_rsrc((char*)p + 16 * n, 0, kSplit ? (int)(8 * n) : 0, 0x00027000)) {}
  __device__ __forceinline__ V3<TM> ld(int i) const {
    const i32x4 a = __builtin_amdgcn_raw_buffer_load_b128(r, i == kNone ? 0x7FFFFF00 : 16 * i, 0, kDeviceScope);
    if constexpr (kSplit) {
      const i32x2 b = __builtin_amdgcn_raw_buffer_load_b64(rz, i == kNone ? 0x7FFFFF00 : 8 * i, 0, kDeviceScope);
      return V3<TM>{__builtin_bit_cast(double, i32x2{a.x, a.y}), __builtin_bit_cast(double, i32x2{a.z, a.w}),
                    __builtin_bit_cast(double, b)};
    } else {
      const int x = a.x, y = a.y, z = a.z;
      return V3<TM>{__builtin_bit_cast(float, x), __builtin_bit_cast(float, y), __builtin_bit_cast(float, z)};
    }
  }
  __device__ __forceinline__ void st(int i, TM x, TM y, TM z) const {
    if constexpr (kSplit) {
      const i32x2 a = __builtin_bit_cast(i32x2, x), b = __builtin_bit_cast(i32x2, y);
      __builtin_amdgcn_raw_buffer_store_b128(i32x4{a.x, a.y, b.x, b.y}, r, 16 * i, 0, kDeviceScope);
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(i32x2, z), rz, 8 * i, 0, kDeviceScope);
    } else {
      const V4<TM> v{x, y, z, (TM)0};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, v), r, 16 * i, 0, kDeviceScope);
    }
  }
};

// Waits until this wavefront's stores have reached device scope (vmcnt 0;
// not as inline asm, beside which the compiler keeps half of the registers
// for itself).
__device__ __forceinline__ void drainStores() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Every member's flag at `epoch`, or false after `ticks`.
__device__ __forceinline__ bool teamWait(const u64* flags, int W, u64 epoch, u64 ticks, int* bad) {
  for (int i = threadIdx.x; i < W; i += kTC) {
    if (coLoad(flags + i) >= epoch) continue;
    const u64 t0 = wall_clock64();
    for (int k = 1; coLoad(flags + i) < epoch; ++k)
      if ((k & 63) == 0 && wall_clock64() - t0 > ticks) {
        *bad = 1;
        break;
      }
  }
  __syncthreads();
  return *bad == 0;
}

// Barrier of a formed team, in two halves: what a member stored before it
// arrives, every member loads after the wait; work that the others do not
// need yet goes between the two.
__device__ __forceinline__ void teamArrive(u64* flags, int rank, int W, u64 epoch) {
  drainStores();
  __syncthreads();
  if (W > 1 && threadIdx.x == 0) coStore(flags + rank, epoch);
}
__device__ __forceinline__ bool teamWait(const u64* flags, int W, u64 epoch, int* bad) {
  if (W == 1) {
    __syncthreads();
    return true;
  }
  return teamWait(flags, W, epoch, kBarrierTicks, bad);
}

// All members are running, or none goes on: a member that has seen every
// flag proposes to go, one that has waited too long proposes to give up, and
// the first proposal of the launch holds for all.  Members wait for nothing
// else before this, so a team that cannot be placed whole (other work holds
// part of the chip) ends instead of waiting for ever.
__device__ __forceinline__ bool teamForm(u64* sync, int rank, int W, u64 epoch, u64 launch, u64 ticks, int* bad) {
  __shared__ u64 outcome;
  if (W == 1) return true;
  u64* flags = sync + 16;
  if (threadIdx.x == 0) coStore(flags + rank, epoch);
  const bool all = teamWait(flags, W, epoch, ticks, bad);
  if (threadIdx.x == 0) {
    u64 cur = coLoad(sync);
    while ((cur >> 1) != launch) {
      const u64 want = 2 * launch + (all ? 1 : 0);
      if (__hip_atomic_compare_exchange_strong(gl(sync), &cur, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT))
        cur = want;
    }
    outcome = cur;
    *bad = 0;
  }
  __syncthreads();
  return (outcome & 1) != 0;
}

// One body's place in P2: its contacts in ascending order, the nd it has as
// body B (listed from inc[k0]), then its own run from c0; and its bilateral
// rows.
template <typename TM>
struct BodyRuns {
  int g, k0, nd, n, c0, b0, b1;
  TM mi;
  bool sums;  // a movable body that is not on the heavy list
};
template <typename TM>
__device__ __forceinline__ BodyRuns<TM> bodyRuns(const Args<TM>& a, long g) {
  BodyRuns<TM> b;
  const bool own = g < a.dims.nb;
  b.g = own ? (int)g : 0;
  b.k0 = gl(a.iStart)[b.g];
  b.n = gl(a.iStart)[b.g + 1] - b.k0;
  b.c0 = gl(a.cStart)[b.g];
  b.nd = b.n - (gl(a.cStart)[b.g + 1] - b.c0);
  b.b0 = gl(a.bilIncStart)[b.g];
  b.b1 = gl(a.bilIncStart)[b.g + 1];
  b.mi = gl(a.minv)[b.g];
  b.sums = own && b.n <= kHeavyDegree && b.mi != (TM)0;
  if (!b.sums) {
    b.n = 0;
    b.b1 = b.b0;
  }
  return b;
}
template <typename TM>
__device__ __forceinline__ int contactOf(const Args<TM>& a, const BodyRuns<TM>& b, int k) {
  return k >= b.n ? kNone : k < b.nd ? gl(a.inc)[b.k0 + k] >> 1 : b.c0 + k - b.nd;
}
// A body's contacts in flight together.  A settled pile has 4.7 to a body and
// seldom more than 8, and each load more costs every body of the wavefront
// its issue (two runs of 8 loaded side by side took P2 0.5 us longer).
constexpr int kRun = 8;

// Wavefront totals in waveSum's and waveMax's order, valid in lane 63 only:
// past the rows of 16 lanes the partners come by row broadcasts instead of
// eight lane reads.
constexpr int kDppBcast15 = 0x142, kDppBcast31 = 0x143;
__device__ __forceinline__ double lastSum(double v) {
  v += dppMove<kDppXor1>(v);
  v += dppMove<kDppXor2>(v);
  v += dppMove<kDppHalfMirror>(v);
  v += dppMove<kDppMirror>(v);
  v += dppMove<kDppBcast15>(v);
  v += dppMove<kDppBcast31>(v);
  return v;
}
__device__ __forceinline__ double lastMax(double v) {
  v = fmax(v, dppMove<kDppXor1>(v));
  v = fmax(v, dppMove<kDppXor2>(v));
  v = fmax(v, dppMove<kDppHalfMirror>(v));
  v = fmax(v, dppMove<kDppMirror>(v));
  v = fmax(v, dppMove<kDppBcast15>(v));
  v = fmax(v, dppMove<kDppBcast31>(v));
  return v;
}
constexpr int kLast = 63;

// What decideStep computes for either outcome, from the state alone, ahead of
// the decision.
struct StepNext {
  double Lb, tb, La, ta, thetaNew, beta;
  __device__ explicit StepNext(const ApgdState& S) {
    const LazyNext n(S);
    Lb = n.backL(); tb = n.backT(Lb);
    La = n.nextL(); ta = n.nextT(La);
    thetaNew = n.nextTheta();
    beta = n.nextBeta(thetaNew);
  }
  __device__ explicit StepNext(const double* p) : Lb(p[0]), tb(p[1]), La(p[2]), ta(p[3]), thetaNew(p[4]), beta(p[5]) {}
  __device__ void store(double* p) const {
    p[0] = Lb; p[1] = tb; p[2] = La; p[3] = ta; p[4] = thetaNew; p[5] = beta;
  }
  __device__ double backL() const { return Lb; }
  __device__ double backT(double) const { return tb; }
  __device__ double nextL() const { return La; }
  __device__ double nextT(double) const { return ta; }
  __device__ double nextTheta() const { return thetaNew; }
  __device__ double nextBeta(double) const { return beta; }
};

// A view every thread reads alike, in scalar registers.
__device__ __forceinline__ double uniformDouble(double v) { return laneValue(v, 0); }
__device__ __forceinline__ PassView uniformView(const PassView& s) {
  PassView v;
  v.cur = __builtin_amdgcn_readfirstlane(s.cur);
  v.prev = __builtin_amdgcn_readfirstlane(s.prev);
  v.nxt = __builtin_amdgcn_readfirstlane(s.nxt);
  v.flags = __builtin_amdgcn_readfirstlane(s.flags);
  v.t = uniformDouble(s.t);
  v.beta = uniformDouble(s.beta);
  return v;
}

// `passes` passes (fewer once the solve has ended) of every slot in items, R
// row tiles per workgroup (R rows per thread).  Per pass a member
//   takes P1's step on its tiles, from registers (the iterates, N gamma and r
//     stay there, the frame in LDS), stores J and arrives; then, while the others
//     arrive, writes the iterate and N gamma back (memory is complete at
//     every pass end) and forms its partial sums;
//   takes P2 on its body units (64 bodies to a wavefront, the team's units
//     dealt out evenly), stores tmp and the units' Lipschitz sums, arrives,
//     and computes the next step sizes of either outcome while it waits;
//   decides the pass from the team's partial sums, as kDecide does.
// Two wavefronts per SIMD (up to 256 VGPRs, one workgroup to a CU): held to
// 128, so that a CU takes two, the mixed kernel spilled 20 and took 26.3 us
// per pass on 256,000 contacts, where two rows per thread take 17.8.
template <typename TM, bool kBil, int R>
__global__ __launch_bounds__(kTC, 2) void kTeam(const Args<TM>* __restrict__ A, Tables T, const TeamItem* items,
                                                u64* sync, u64 epoch, u64 launch, int passes, u64 formTicks) {
  constexpr bool kMixed = sizeof(TM) < sizeof(double);
  constexpr int NF = kMixed ? 6 : 3;
  constexpr unsigned kUsed = kP1Slots<TM>;
  constexpr int kW = kTC / 64;       // wavefronts
  constexpr int kWT = kTP / 64;      // of a heavy body's sum
  constexpr int kUnits = kTB / 64;   // body units of a body tile
  static_assert(kW == kSlots && kSlots == 8 && kUnits == 4, "a wavefront for each total; two loads to a body tile");
  const TeamItem me = items ? items[blockIdx.x] : TeamItem{0, (int)blockIdx.x, (int)gridDim.x, 0};
  const Args<TM>& a = A[me.slot];
  const SolveDims& D = a.dims;
  const int W = me.members, rank = me.rank, nTiles = a.nTiles;
  u64* sy = sync + (long)me.slot * kTeamSync;
  u64* flags = sy + 16;
  __shared__ int bad;
  __shared__ double shP[R][kW][kSlots], shTot[kW], shH[kWT][3];
  __shared__ ApgdState shS;  // the state and its view: registers are for the rows and bodies
  __shared__ PassView shV;
  __shared__ double shNext[6];
  // per thread, kept here instead of in registers: the rows' frames and the
  // first body's contacts
  __shared__ TM shF[R][9][kTC];
  __shared__ int shIds[kRun][kTC];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) {
    bad = 0;
    shS = STATE(T, me.slot, 1);
    shV = viewOf(shS);
  }
  __syncthreads();
  if (shS.done) return;  // the same for every member
  PassView V = uniformView(shV);
  const CoArray<TM> J(a.J, a.cap), tmp(kMixed ? (void*)a.tmp : (void*)a.tmpSplit, D.nb);
  const int nBT = a.nBodyTiles, nHeavy = gl(a.counters)[2], nl = nBT + nHeavy;
  const int nU = kUnits * nBT, u0 = rank + W * wave;  // body units (below)
  if (!kMixed) {  // M^-1 D^T gamma as the launches left it, into the exchanged form
    for (int u = u0; u < nU; u += W * kW) {
      const int g = u * 64 + lane;
      if (g >= D.nb) continue;
      const V4<TM> t = ld4(a.tmp, g);
      tmp.st(g, t.x, t.y, t.z);
    }
    drainStores();
    __syncthreads();
  }
  if (!teamForm(sy, rank, W, epoch, launch, formTicks, &bad)) return;

  // this thread's rows: row u of tile R rank + u
  struct Row {
    int c, ia, ib, f0, fs;  // the contact and its bodies; row 0, and the step to rows 1 and 2
    bool valid, bil;
    TM rv[3], nk[3], nm[3];
    double gk[3], gm[3], gn[3];
  };
  Row row[R];
  const long cap = a.cap;
#pragma unroll
  for (int u = 0; u < R; ++u) {
    Row& w = row[u];
    const long q = ((long)rank * R + u) * kTC + tid;
    w.valid = q < (long)D.nc + D.nbil;
    w.bil = kBil && q >= D.nc;
    w.c = w.valid && !w.bil ? (int)q : 0;
    w.f0 = w.valid ? (int)(w.bil ? BROW(a, q - D.nc) : q) : 0;
    w.fs = w.valid && !w.bil ? (int)cap : 0;
    w.ia = gl(a.cA)[w.c];
    w.ib = gl(a.cB)[w.c];
    if (kBil && w.valid && w.bil) {  // the two DOFs
      w.ia = gl(a.bilA)[q - D.nc];
      w.ib = gl(a.bilB)[q - D.nc];
    }
    TM fc[6], F[9];
#pragma unroll
    for (int k = 0; k < 6; ++k) fc[k] = k < NF ? gl(a.frame)[k * cap + w.c] : (TM)0;
    frameFrom(fc, D.geomMode, F);
#pragma unroll
    for (int k = 0; k < 9; ++k) shF[u][k][tid] = F[k];
#pragma unroll
    for (int rr = 0; rr < 3; ++rr) {
      const long f = w.f0 + (long)rr * w.fs;
      w.rv[rr] = gl(a.r)[f];
      w.gk[rr] = gl(a.ring[0] + V.cur * a.ringStride)[f];
      w.gm[rr] = gl(a.ring[0] + V.prev * a.ringStride)[f];
      w.nk[rr] = gl(a.rn[0] + V.cur * a.ringStride)[f];  // (not formed yet if fresh: replaced below)
      w.nm[rr] = gl(a.rn[0] + V.prev * a.ringStride)[f];
      w.gn[rr] = 0;
    }
  }
  auto tmpOf = [&](int dof) {
    const V3<TM> t = tmp.ld(dof / 3);
    const int k = dof % 3;
    return k == 0 ? t.x : (k == 1 ? t.y : t.z);
  };

  // body units: unit rank + W (wave + kW j) in iteration j.  A unit without a
  // movable light body is left out: its tmp is zero from the setup on, and so
  // are its sums.
  const BodyRuns<TM> first = bodyRuns(a, u0 < nU ? (long)u0 * 64 + lane : (long)D.nb);
#pragma unroll
  for (int k = 0; k < kRun; ++k) shIds[k][tid] = contactOf(a, first, k);
  // (the launches read the D^T gamma ring of fixed bodies too, times zero)
  if (kMixed)
    for (int u = u0; u < nU; u += W * kW) {
      const int g = u * 64 + lane;
      if (g < D.nb && gl(a.minv)[g] == (TM)0)
#pragma unroll
        for (int k = 0; k < 4; ++k) st4(a.sr, (long)k * D.nb + g, V4<TM>{0, 0, 0, 0});
    }
  unsigned live = 0;
  for (int j = 0, u = u0; u < nU; ++j, u += W * kW) {
    if (__any(bodyRuns(a, (long)u * 64 + lane).sums)) live |= 1u << j;
    else if (lane == 0) {
      coStore(a.lqw[0] + u, 0.0);
      coStore(a.lqw[1] + u, 0.0);
    }
  }
  bool liveHeavy = false;
  for (int h = rank; h < nHeavy; h += W) {
    if (gl(a.minv)[gl(a.heavy)[h]] != (TM)0) liveHeavy = true;
    else if (tid == 0) {
      coStore(a.lq[0] + nBT + h, 0.0);
      coStore(a.lq[1] + nBT + h, 0.0);
    }
  }

  u64 ep = epoch;
  for (int p = 0; p < passes; ++p) {
    const int par = p & 1;
    const bool mom = !(V.flags & kViewRestart), fresh = (V.flags & kViewFresh) != 0;
    const double bp = 1.0 + V.beta, bm = -V.beta;
    double* const Gn = a.ring[0] + V.nxt * a.ringStride;
    // y, N y and g of a row (formed once for the step and again for the sums,
    // rather than kept across the arrival)
    auto momentum = [&](const Row& w, int rr, double& y, double& ny, double& gg) {
      if (mom) {
        y = bp * w.gk[rr] + bm * w.gm[rr];
        ny = bp * (double)w.nk[rr] + bm * (double)w.nm[rr];
      } else {
        y = w.gk[rr];
        ny = (double)w.nk[rr];
      }
      gg = 1.0 * ny + 1.0 * (double)w.rv[rr];
    };
    // ---- P1
    if (fresh) {
      V3<TM> tA[R], tB[R];
#pragma unroll
      for (int u = 0; u < R; ++u)
        if (!row[u].bil) {
          tA[u] = tmp.ld(row[u].valid ? row[u].ia : kNone);
          tB[u] = tmp.ld(row[u].valid ? row[u].ib : kNone);
        }
#pragma unroll
      for (int u = 0; u < R; ++u) {
        Row& w = row[u];
        if (!w.valid) continue;
        if (w.bil) {
          w.nk[0] = tmpOf(w.ia);
          if (w.ib >= 0) w.nk[0] -= tmpOf(w.ib);
        } else {
          TM F[9];
#pragma unroll
          for (int k = 0; k < 9; ++k) F[k] = shF[u][k][tid];
          rowsOfTmp(F, V4<TM>{tA[u].x, tA[u].y, tA[u].z, (TM)0}, V4<TM>{tB[u].x, tB[u].y, tB[u].z, (TM)0}, w.nk[0],
                    w.nk[1], w.nk[2]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < R; ++u) {
      Row& w = row[u];
      if (!w.valid) continue;
#pragma unroll
      for (int rr = 0; rr < 3; ++rr) {
        if (w.bil && rr) continue;
        double y, ny, gg;
        momentum(w, rr, y, ny, gg);
        w.gn[rr] = 1.0 * y + (-V.t) * gg;
      }
      if (w.bil) {
        coStore(Gn + w.f0, w.gn[0]);  // P2 reads it
      } else {
        projectCone<double>(w.gn[0], w.gn[1], w.gn[2], D.mu);
        const TM x0 = (TM)w.gn[0], x1 = (TM)w.gn[1], x2 = (TM)w.gn[2];
        TM F[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) F[k] = shF[u][k][tid];
        J.st(w.c, F[0] * x0 + F[3] * x1 + F[6] * x2, F[1] * x0 + F[4] * x1 + F[7] * x2,
             F[2] * x0 + F[5] * x1 + F[8] * x2);
      }
    }
    teamArrive(flags, rank, W, ++ep);
    // what the others need only after P2: N gamma_k, gamma_new and the
    // partial sums, in P1's order
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const Row& w = row[u];
      double acc[kSlots];
      zero(acc);
      if (w.valid) {
        const int nr = w.bil ? 1 : 3;
        DV_GLOBAL TM* Nw = gl(a.rn[0] + V.cur * a.ringStride);
#pragma unroll
        for (int rr = 0; rr < 3; ++rr) {
          if (rr >= nr) continue;
          const long f = w.f0 + (long)rr * w.fs;
          if (fresh) Nw[f] = w.nk[rr];
          if (!w.bil) gl(Gn)[f] = w.gn[rr];
        }
        const double w0 = (double)w.nk[0] + (double)w.rv[0];
        if (w.bil) {
          double e;
          if (D.nc) {
            const double z = 1.0 * w.gk[0] + (-D.gdiff) * w0;
            const double ig = D.igdiff;
            e = fabs(ig * w.gk[0] + (-ig) * z);
          } else {
            e = fabs(w0);
          }
          acc[7] = fmax(acc[7], e == e ? e : INFINITY);
        } else {
          const double w1 = (double)w.nk[1] + (double)w.rv[1];
          const double w2 = (double)w.nk[2] + (double)w.rv[2];
          acc[7] = fmax(acc[7], residualContact(w.gk[0], w.gk[1], w.gk[2], w0, w1, w2, D.mu, D.gdiff, D.igdiff));
        }
#pragma unroll
        for (int rr = 0; rr < 3; ++rr) {
          if (rr >= nr) continue;
          double y, ny, gg;
          momentum(w, rr, y, ny, gg);
          const double dy = w.gn[rr] - y;
          if (!kMixed) {
            acc[0] += w.gn[rr] * (double)w.rv[rr];
            acc[1] += y * ny;
            acc[2] += y * (double)w.rv[rr];
            acc[3] += gg * dy;
          }
          acc[4] += dy * dy;
          acc[5] += gg * (w.gn[rr] - w.gk[rr]);
        }
      }
#pragma unroll
      for (int s = 0; s < kSlots; ++s) {
        if (!((kUsed >> s) & 1u)) continue;
        const double v = s == kSlots - 1 ? lastMax(acc[s]) : lastSum(acc[s]);
        if (lane == kLast) shP[u][wave][s] = v;
      }
    }
    if (!teamWait(flags, W, ep, &bad)) break;

    // ---- P2 (every load before a store: a wait for a load also waits for
    // the stores before it)
    const double* X = Gn + 3 * cap;  // bilateral rows of gamma_new
    for (int j = 0, u = u0; u < nU; ++j, u += W * kW) {
      if (!((live >> j) & 1u)) continue;
      const BodyRuns<TM> b = j == 0 ? first : bodyRuns(a, (long)u * 64 + lane);
      int id[kRun];
      if (j == 0) {
#pragma unroll
        for (int k = 0; k < kRun; ++k) id[k] = shIds[k][tid];
      } else {
#pragma unroll
        for (int k = 0; k < kRun; ++k) id[k] = contactOf(a, b, k);
      }
      V3<TM> v[kRun];
#pragma unroll
      for (int k = 0; k < kRun; ++k) v[k] = J.ld(id[k]);
      TM s0 = 0, s1 = 0, s2 = 0;
      for (int k = b.b0; kBil && k < b.b1; ++k) {
        const int e = gl(a.bilInc)[k];
        const double x = coLoad(X + (e >> 3));
        const TM t = (TM)((e & 1) ? -x : x);
        const int comp = (e >> 1) & 3;
        if (comp == 0) s0 += t; else if (comp == 1) s1 += t; else s2 += t;
      }
      for (int kb = 0;;) {
#pragma unroll
        for (int k = 0; k < kRun; ++k) {
          if (kb + k >= b.n) continue;
          if (kb + k < b.nd) {
            s0 -= v[k].x; s1 -= v[k].y; s2 -= v[k].z;
          } else {
            s0 += v[k].x; s1 += v[k].y; s2 += v[k].z;
          }
        }
        kb += kRun;
        if (kb >= b.n) break;
#pragma unroll
        for (int k = 0; k < kRun; ++k) v[k] = J.ld(contactOf(a, b, kb + k));
      }
      const double term = lastSum(b.sums ? lipschitzTerm(a, b.g, V, b.mi, s0, s1, s2) : 0.0);
      if (b.sums) tmp.st(b.g, b.mi * s0, b.mi * s1, b.mi * s2);
      if (lane == kLast) coStore(a.lqw[par] + u, term);
    }
    // movable bodies with many contacts, by the first kTP threads
    for (int h = rank; liveHeavy && h < nHeavy; h += W) {
      const int g = gl(a.heavy)[h];
      const TM mi = gl(a.minv)[g];
      if (mi == (TM)0) continue;
      const int k0 = gl(a.iStart)[g], n = gl(a.iStart)[g + 1] - k0;
      const int c0 = gl(a.cStart)[g], c1 = gl(a.cStart)[g + 1];
      const int nd = n - (c1 - c0);
      if (tid < kTP) {
        double hx = 0, hy = 0, hz = 0;
        for (int kb = tid; kb < n; kb += 4 * kTP) {
          V3<TM> v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int k = kb + i * kTP;
            v[i] = J.ld(k < nd ? gl(a.inc)[k0 + k] >> 1 : k < n ? c0 + k - nd : kNone);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int k = kb + i * kTP;
            if (k >= n) continue;
            const double sg = k < nd ? -1.0 : 1.0;
            hx += sg * (double)v[i].x;
            hy += sg * (double)v[i].y;
            hz += sg * (double)v[i].z;
          }
        }
        if (kBil && tid == 0) {
          for (int k = gl(a.bilIncStart)[g]; k < gl(a.bilIncStart)[g + 1]; ++k) {
            const int e = gl(a.bilInc)[k];
            const double x = coLoad(X + (e >> 3)), t = (e & 1) ? -x : x;
            const int comp = (e >> 1) & 3;
            if (comp == 0) hx += t; else if (comp == 1) hy += t; else hz += t;
          }
        }
        hx = lastSum(hx); hy = lastSum(hy); hz = lastSum(hz);
        if (lane == kLast) {
          shH[wave][0] = hx; shH[wave][1] = hy; shH[wave][2] = hz;
        }
      }
      __syncthreads();
      if (tid == 0) {
        TM t[3];
        for (int s = 0; s < 3; ++s) {
          double v = shH[0][s];
          for (int w = 1; w < kWT; ++w) v += shH[w][s];
          t[s] = (TM)v;
        }
        tmp.st(g, mi * t[0], mi * t[1], mi * t[2]);
        coStore(a.lq[par] + nBT + h, lipschitzTerm(a, g, V, mi, t[0], t[1], t[2]));
      }
      __syncthreads();
    }
    // the tiles' partial sums, by the last wavefront (which has the fewest
    // body units)
    if (wave == kW - 1 && lane < R * kSlots && ((kUsed >> (lane % kSlots)) & 1u)) {
      const int u = lane / kSlots, s = lane % kSlots;
      double v = shP[u][0][s];
      for (int w = 1; w < kW; ++w) v = s == kSlots - 1 ? fmax(v, shP[u][w][s]) : v + shP[u][w][s];
      if (R * rank + u < nTiles) coStore(a.part1[par] + ((long)R * rank + u) * kSlots + s, v);
    }
    teamArrive(flags, rank, W, ++ep);
    if (tid == 0) StepNext(shS).store(shNext);
    if (!teamWait(flags, W, ep, &bad)) break;

    // ---- the decision, by every member.  Wavefront s totals slot s of P1's
    // partials, and wavefront 6 (whose slot is not used) the Lipschitz terms,
    // in reduceSlots' order: lane l of its wavefront w adds entries 64 w + l,
    // 64 w + l + kTP, ..., and the wavefronts' sums are added in order (past
    // the entries they are zero, and left out).
    if (wave == 6) {
      const auto rq = __builtin_amdgcn_make_buffer_rsrc(a.lqw[par], 0, 8 * nU, 0x00027000);
      const auto rh = __builtin_amdgcn_make_buffer_rsrc(a.lq[par], 0, 8 * nl, 0x00027000);
      double v[kWT] = {0, 0, 0, 0};
      for (int b0 = 0; b0 < nl; b0 += kTP) {
        i32x4 x[kWT][2];  // a body tile's units, or a heavy body's term and zeros; all loads first
#pragma unroll
        for (int i = 0; i < kWT; ++i) {
          if (b0 + 64 * i >= nl) break;
          const int w = b0 + 64 * i + lane;
          if (w < nBT) {
            x[i][0] = __builtin_amdgcn_raw_buffer_load_b128(rq, 8 * kUnits * w, 0, kDeviceScope);
            x[i][1] = __builtin_amdgcn_raw_buffer_load_b128(rq, 8 * kUnits * w, 16, kDeviceScope);
          } else {  // (past nl: zero, by the bound)
            const i32x2 t = __builtin_amdgcn_raw_buffer_load_b64(rh, 8 * w, 0, kDeviceScope);
            x[i][0] = i32x4{t.x, t.y, 0, 0};
            x[i][1] = i32x4{0, 0, 0, 0};
          }
        }
#pragma unroll
        for (int i = 0; i < kWT; ++i) {
          if (b0 + 64 * i >= nl) break;
          double t = __builtin_bit_cast(double, i32x2{x[i][0].x, x[i][0].y});
          t += __builtin_bit_cast(double, i32x2{x[i][0].z, x[i][0].w});
          t += __builtin_bit_cast(double, i32x2{x[i][1].x, x[i][1].y});
          t += __builtin_bit_cast(double, i32x2{x[i][1].z, x[i][1].w});
          v[i] += t;
        }
      }
      double total = lastSum(v[0]);
      for (int i = 1; i < kWT && 64 * i < nl; ++i) total += lastSum(v[i]);
      if (lane == kLast) shTot[wave] = total;
    } else if ((kUsed >> wave) & 1u) {
      const auto rp = __builtin_amdgcn_make_buffer_rsrc(a.part1[par], 0, 8 * kSlots * nTiles, 0x00027000);
      double v[kWT] = {0, 0, 0, 0};
      for (int b0 = 0; b0 < nTiles; b0 += kTP) {
        double x[kWT];
#pragma unroll
        for (int i = 0; i < kWT; ++i) {
          if (b0 + 64 * i >= nTiles) break;
          const int w = b0 + 64 * i + lane;  // (past nTiles: zero, by the bound)
          x[i] = __builtin_bit_cast(double, (i32x2)__builtin_amdgcn_raw_buffer_load_b64(rp, 8 * kSlots * w + 8 * wave, 0,
                                                                                        kDeviceScope));
        }
#pragma unroll
        for (int i = 0; i < kWT; ++i) {
          if (b0 + 64 * i >= nTiles) break;
          v[i] = wave == kSlots - 1 ? fmax(v[i], x[i]) : v[i] + x[i];
        }
      }
      double total = wave == kSlots - 1 ? lastMax(v[0]) : lastSum(v[0]);
      for (int i = 1; i < kWT && 64 * i < nTiles; ++i)
        total = wave == kSlots - 1 ? fmax(total, lastMax(v[i])) : total + lastSum(v[i]);
      if (lane == kLast) shTot[wave] = total;
    }
    __syncthreads();
    if (tid == 0) {
      double tot[2 * kSlots];
#pragma unroll
      for (int s = 0; s < 2 * kSlots; ++s) tot[s] = 0.0;
#pragma unroll
      for (int s = 0; s < kSlots; ++s)
        if ((kUsed >> s) & 1u) tot[s] = shTot[s];
      tot[kSlots + 6] = shTot[6];
      ApgdState S = shS;
      decideStep<kMixed>(S, tot, D, StepNext(shNext));
      shS = S;
      shV = viewOf(S);
    }
    __syncthreads();
    V = uniformView(shV);
    if (V.flags & kViewDone) break;
    if (V.flags & kViewFresh) {  // accepted: gamma_new becomes gamma_k (a backtrack keeps both)
#pragma unroll
      for (int u = 0; u < R; ++u)
#pragma unroll
        for (int rr = 0; rr < 3; ++rr) {
          row[u].gm[rr] = row[u].gk[rr];
          row[u].nm[rr] = row[u].nk[rr];
          row[u].gk[rr] = row[u].gn[rr];
        }
    }
  }
  if (!kMixed) {  // M^-1 D^T gamma back for the launches
    for (int u = u0; u < nU; u += W * kW) {
      const int g = u * 64 + lane;
      if (g >= D.nb) continue;
      const V3<TM> t = tmp.ld(g);
      st4(a.tmp, g, V4<TM>{t.x, t.y, t.z, (TM)0});
    }
  }
  if (rank == 0 && tid == 0) {
    ApgdState S = shS;
    if (bad) {  // a member was lost (never seen): the solve ends as diverged
      S.done = 1;
      S.best = INFINITY;
    }
    STATE(T, me.slot, 0) = S;
    STATE(T, me.slot, 1) = S;
    VIEW(T, me.slot, 0) = viewOf(S);
    VIEW(T, me.slot, 1) = viewOf(S);
    T.out[me.slot] = S;
  }
}
