// The resident passes: thousands of passes of a slot in one launch, its
// contacts' state in registers and its workgroups exchanging what the other
// half of a pass needs through device-scope stores.
//
// Included by dv_apgd_fused.hip after the pass kernels, whose arithmetic and
// summation orders it repeats bit for bit (a slot may run some chunks here
// and others as P1/P2 launches, and ends in the same state).
//
// Why: a pass as two launches costs two kernel boundaries and a reload of the
// whole state.  What crosses workgroups is small (J, tmp and the sums), and
// stored at device scope it needs no write-back of the L2.  Exchanged under a
// grid barrier it still cost a chain of store, drain, flag, poll and load,
// 2.5 to 3 us twice a pass; so the entries carry the pass's tag themselves, a
// reader waits for just those that it needs, and the step of the next pass and
// its bodies' sums are taken before this one is decided.
// us per pass as launches, resident with two barriers a pass, with the step
// alone taken ahead, and so (piles of the given contacts):
//   contacts    134     440   1,630  11,900  41,800  82,400  168,000
//   FP64       10.7            13.9    15.5    17.1    21.0    27.2
//               5.4             9.2    10.2    11.8    14.2    23.3
//               4.6     5.7     6.6     7.2     8.1     9.8    17.5
//               4.6     5.2     5.7     6.8     7.8     9.4    14.6
//   mixed       8.8            11.7    12.9    13.6    16.1    20.7
//               4.5             7.9     8.4    10.0    11.9    17.8
//               3.7     4.1     5.1     5.4     6.0     6.8    10.8
//               3.8     3.8     4.3     4.9     5.4     5.8     9.6
// Where a pass of 11,900 contacts spends its 11,700 cycles (mixed, a wavefront
// with bodies): tmp's arrival 1,300, the next step 1,000, its sums 1,900, the
// contacts' J and the bodies' sums 2,500, the totals and the barrier 800, the
// decision and the change of registers 2,000, steps taken again (13% of the
// passes) 700.
#pragma once

// A workgroup's place: member `rank` of the `members` of slot `slot`'s team.
struct TeamItem {
  int slot, rank, members, pad;
};

// Per slot, in 64-bit words: the formation's outcome, then one flag per
// member.  Flags hold the launch's number, which only grows, so nothing is
// cleared between launches.
constexpr int kTeamMax = 256;
constexpr int kTeamSync = 16 + kTeamMax;
// A team whose members are not all running after this long gives up (0: at
// once): the slot's passes then run as launches.
constexpr double kFormMs = 2;
// Several scenes' teams wait for room: until a team before them has run its
// 512 passes, 13 ms at most.  (With 100 ms, two batches of two 112,000-sphere
// scenes on threads of their own, whose teams of 250 can each hold half of the
// chip, made 187 scene-steps/s in such a run, with 30 229, as launches 201.)
constexpr double kFormMsMany = 30;
constexpr double kFormMsMost = 1000;
constexpr double kTicksPerMs = 1e5;  // of the wall clock

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
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
template <typename TM>
struct V3 {
  TM x, y, z;
};
// What crosses workgroups carries its own arrival: every aligned 8-byte word
// of an exchanged entry holds 48 bits of it and a 16-bit tag that names the
// pass, and a reader loads until all words carry the tag it waits for.  A word
// of 8 bytes arrives whole, and no order between words or stores is needed,
// so nothing is drained and no flag follows the data.  A launch clears the
// tags before its members meet, so tags need not differ between launches.
__device__ __forceinline__ int lowTagged(int hi, unsigned tag) { return (hi & 0xFFFF) | (int)tag; }
__device__ __forceinline__ int highTagged(int hi, unsigned tag) { return (int)((unsigned)hi >> 16 | tag); }
// (a's low half above b's, and a's high half above b's low half)
__device__ __forceinline__ int lowLow(int a, int b) { return (int)__builtin_amdgcn_perm((unsigned)a, (unsigned)b, 0x05040100u); }
__device__ __forceinline__ int highLow(int a, int b) { return (int)__builtin_amdgcn_perm((unsigned)a, (unsigned)b, 0x07060100u); }
__device__ __forceinline__ i32x2 wordsOf(double v) { return __builtin_bit_cast(i32x2, v); }
__device__ __forceinline__ double doubleOf(int lo, int hi) { return __builtin_bit_cast(double, i32x2{lo, hi}); }
constexpr int kNone = -1;  // no entry: reads as zero and stores nothing, without touching memory
constexpr int kPastEnd = 0x7FFFFF00;  // an offset past every bound, which the hardware checks

// n 3-vectors.  FP32: 16 bytes, (x, y's high half) and (z, y's low half).
// FP64: 32 bytes, the low 48 bits of x, y and z, then the high 16 of the
// three, as two arrays of 16-byte halves, so that a wavefront's stores are
// contiguous runs.
template <typename TM>
struct CoArray {
  static constexpr int kSplit = sizeof(TM) == 8;
  static constexpr int kHalves = kSplit ? 2 : 1;
  struct Raw {
    i32x4 h[kHalves];
  };
  __amdgpu_buffer_rsrc_t r, r1;
  __device__ CoArray(void* p, long n)
      : r(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)(16 * n), 0x00027000)),
        r1(__builtin_amdgcn_make_buffer_rsrc((char*)p + (kSplit ? 16 * n : 0), 0, (int)(16 * n), 0x00027000)) {}
  __device__ __forceinline__ Raw ld(int i) const {
    const int o = i == kNone ? kPastEnd : 16 * i;
    Raw w;
    w.h[0] = __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, kDeviceScope);
    if constexpr (kSplit) w.h[1] = __builtin_amdgcn_raw_buffer_load_b128(r1, o, 0, kDeviceScope);
    return w;
  }
  __device__ __forceinline__ void st(int i, TM x, TM y, TM z, unsigned tag) const {
    const int o = i == kNone ? kPastEnd : 16 * i;
    if constexpr (kSplit) {
      const i32x2 a = wordsOf(x), b = wordsOf(y), c = wordsOf(z);
      const i32x4 h0{a.x, lowTagged(a.y, tag), b.x, lowTagged(b.y, tag)};
      const i32x4 h1{c.x, lowTagged(c.y, tag), (int)((unsigned)a.y >> 16 | ((unsigned)b.y & 0xFFFF0000u)), highTagged(c.y, tag)};
      __builtin_amdgcn_raw_buffer_store_b128(h0, r, o, 0, kDeviceScope);
      __builtin_amdgcn_raw_buffer_store_b128(h1, r1, o, 0, kDeviceScope);
    } else {
      const int b = __builtin_bit_cast(int, y);
      const i32x4 h{__builtin_bit_cast(int, x), highTagged(b, tag), __builtin_bit_cast(int, z), lowTagged(b, tag)};
      __builtin_amdgcn_raw_buffer_store_b128(h, r, o, 0, kDeviceScope);
    }
  }
  static __device__ __forceinline__ V3<TM> value(const Raw& w) {
    const i32x4 a = w.h[0];
    if constexpr (kSplit) {
      const i32x4 b = w.h[1];
      return V3<TM>{doubleOf(a.x, lowLow(b.z, a.y)), doubleOf(a.z, highLow(b.z, a.w)), doubleOf(b.x, lowLow(b.w, b.y))};
    } else {
      const int x = a.x, y = lowLow(a.y, a.w), z = a.z;
      return V3<TM>{__builtin_bit_cast(float, x), __builtin_bit_cast(float, y), __builtin_bit_cast(float, z)};
    }
  }
  // 0 in the upper half where the entry carries the tag
  static __device__ __forceinline__ unsigned missing(int i, const Raw& w, unsigned tag) {
    unsigned m = 0;
#pragma unroll
    for (int h = 0; h < kHalves; ++h) m |= ((unsigned)w.h[h].y ^ tag) | ((unsigned)w.h[h].w ^ tag);
    return i == kNone ? 0u : m;
  }
  // a bilateral row's gamma in the same form
  __device__ __forceinline__ void stDouble(int i, double v, unsigned tag) const {
    const i32x2 a = wordsOf(v);
    const int lo = a.x, hi = a.y;  // (a vector's element, bit-cast in place, reads element 0)
    if constexpr (kSplit) st(i, v, 0.0, 0.0, tag);
    else st(i, __builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi), 0.0f, tag);
  }
  static __device__ __forceinline__ double asDouble(const Raw& w) {
    const V3<TM> v = value(w);
    if constexpr (kSplit) return v.x;
    else return doubleOf(__builtin_bit_cast(int, v.x), __builtin_bit_cast(int, v.y));
  }
};
// One double as an exchanged entry of 16 bytes.
__device__ __forceinline__ i32x4 taggedDouble(double v, unsigned tag) {
  const i32x2 a = wordsOf(v);
  return i32x4{a.x, lowTagged(a.y, tag), (int)((unsigned)a.y >> 16), (int)tag};
}
__device__ __forceinline__ double valueOf(const i32x4& w) { return doubleOf(w.x, lowLow(w.z, w.y)); }
__device__ __forceinline__ unsigned missing(const i32x4& w, unsigned tag) {
  return ((unsigned)w.y ^ tag) | ((unsigned)w.w ^ tag);
}

__device__ __forceinline__ float exactFma(float x, float y, float z) { return __builtin_fmaf(x, y, z); }
__device__ __forceinline__ double exactFma(double x, double y, double z) { return __builtin_fma(x, y, z); }

// projectCone<double> without its branches, which every wavefront takes all
// of, and with 1 / mu and mu^2 + 1 formed once: the same results.
struct Cone {
  double mu, inverse, den;
  __device__ explicit Cone(double m) : mu(m), inverse(1.0 / m), den(m * m + 1.0) {}
  __device__ __forceinline__ void project(double& g0, double& g1, double& g2) const {
    const double gn = g0;
    if (mu == 0) {
      g1 = 0; g2 = 0;
      if (gn < 0) g0 = 0;
      return;
    }
    const double gt = __builtin_sqrt(g1 * g1 + g2 * g2);
    const bool inside = gt < mu * gn;
    const bool polar = (gt < -inverse * gn) | (fabs(gn) < 10e-15);
    const double gnp = (gt * mu + gn) / den;
    const double q = gnp * mu / gt;
    g0 = inside ? g0 : polar ? 0.0 : gnp;
    g1 = inside ? g1 : polar ? 0.0 : q * g1;
    g2 = inside ? g2 : polar ? 0.0 : q * g2;
  }
  __device__ __forceinline__ double residual(double g0, double g1, double g2, double w0, double w1, double w2,
                                             double gdiff, double ig) const {
    double z0 = 1.0 * g0 + (-gdiff) * w0, z1 = 1.0 * g1 + (-gdiff) * w1, z2 = 1.0 * g2 + (-gdiff) * w2;
    project(z0, z1, z2);
    const double e0 = ig * g0 + (-ig) * z0, e1 = ig * g1 + (-ig) * z1, e2 = ig * g2 + (-ig) * z2;
    const double sum = e0 + e1 + e2;
    return sum == sum ? fmax(fabs(e0), fmax(fabs(e1), fabs(e2))) : INFINITY;
  }
};

// A wait of the whole wavefront: load() until nothing is missing() in any lane,
// which loads of what has been asked for already may show at once; with kLanes
// only lanes with something missing load again (us per pass of 82,400 contacts
// in FP64 without and with: 11.1 and 10.5; with two rows a thread it costs
// registers, and 17.4 became 18.0).  It ends after
// kMostLoads loads (at 0.2 us or more each, some seconds) and then marks the
// member lost, whose other waits end after one.  (One way out, for all lanes
// together: loops with more kept what they load in three copies of its
// registers.)
constexpr int kMostLoads = 1 << 25;
__device__ __forceinline__ bool someMissing(unsigned m, unsigned least = 0x10000u) { return __any(m >= least); }
// An entry of a step taken on a guess is also there once the right step has
// replaced it (its tag is the guess's, plus one): what it holds is not used.
constexpr unsigned kOrReplaced = 0x20000u;
// (Otherwise the compiler carries the parts of what was loaded out of the wait
// in further registers.)
__device__ __forceinline__ void pinned(i32x4& w) { asm volatile("" : "+v"(w)); }
// Ends the wait for loads here.  Loads and stores complete in their order, so
// one that is left unused on some path is waited for, with every store since,
// wherever the compiler uses its registers next.
template <typename TM>
__device__ __forceinline__ void settled(const V4<TM>& v) { asm volatile("" : : "v"(v.x), "v"(v.y), "v"(v.z)); }
template <bool kLanes, class Missing, class Load>
__device__ __forceinline__ void waitFor(int* bad, unsigned least, const Missing& missing, const Load& load) {
  unsigned m = missing();
  if (!someMissing(m, least)) return;
  int left = __builtin_amdgcn_readfirstlane(__hip_atomic_load(bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) ? 1 : kMostLoads;
  do {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);  // (the loads stay in the loop)
    __builtin_amdgcn_s_sleep(10);  // (others' loads first: 0.1 to 0.6 us a pass)
    if (!kLanes || m >= least) load();
    m = missing();
    --left;
  } while ((int)someMissing(m, least) & (int)(left > 0));
  if (left <= 0) __hip_atomic_store(bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// N entries of an array, once each carries the tag (kNone: nothing to wait
// for).
template <typename TM, int N>
__device__ __forceinline__ void loadEntries(const CoArray<TM>& A, const int (&id)[N], typename CoArray<TM>::Raw (&w)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) w[k] = A.ld(id[k]);
}
template <bool kLanes, typename TM, int N>
__device__ __forceinline__ void await(const CoArray<TM>& A, const int (&id)[N], unsigned tag, int* bad,
                                      typename CoArray<TM>::Raw (&w)[N], unsigned least = 0x10000u) {
  loadEntries(A, id, w);
  waitFor<kLanes>(
      bad, least,
      [&] {
        unsigned m = 0;
#pragma unroll
        for (int k = 0; k < N; ++k) m |= A.missing(id[k], w[k], tag);
        return m;
      },
      [&] { loadEntries(A, id, w); });
#pragma unroll
  for (int k = 0; k < N; ++k)
#pragma unroll
    for (int h = 0; h < CoArray<TM>::kHalves; ++h) pinned(w[k].h[h]);
}

// Waits until this wavefront's stores have reached device scope (vmcnt 0;
// not as inline asm, beside which the compiler keeps half of the registers
// for itself).
__device__ __forceinline__ void drainStores() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// All members are running and have cleared their entries, or none goes on: a
// member that has seen every flag proposes to go, one that has waited too
// long proposes to give up, and the first proposal of the launch holds for
// all.  Members wait for nothing else before this, so a team that cannot be
// placed whole (other work holds part of the chip) ends instead of waiting
// for ever.
__device__ __forceinline__ bool teamForm(u64* sync, int rank, int W, u64 launch, u64 ticks) {
  __shared__ u64 outcome;
  __shared__ int late;
  if (threadIdx.x == 0) late = ticks == 0;
  drainStores();
  __syncthreads();
  if (W == 1) return true;
  u64* flags = sync + 16;
  if (threadIdx.x == 0) coStore(flags + rank, launch);
  for (int i = threadIdx.x; ticks && i < W; i += kTC) {
    const u64 t0 = wall_clock64();
    for (int k = 1; coLoad(flags + i) < launch; ++k)
      if ((k & 63) == 0 && wall_clock64() - t0 > ticks) {
        late = 1;
        break;
      }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    u64 cur = coLoad(sync);
    while ((cur >> 1) != launch) {
      const u64 want = 2 * launch + (late ? 0 : 1);
      if (__hip_atomic_compare_exchange_strong(gl(sync), &cur, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT))
        cur = want;
    }
    outcome = cur;
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
// A body's contacts in flight together.  A settled pile has 4.7 to a body, but
// of 64 bodies some have more than 8, and a second round of loads costs them
// all another flight: us per pass with 6, 8, 10 and 12 at 18,000 contacts 6.6,
// 6.3, 6.1 and 6.1 (mixed), 8.9, 8.5, 8.1 and 8.8 (FP64).
constexpr int kRunMost = 10;
// Two rows a thread in FP64 (and three, mixed) have no registers for ten: with 10, 8, 6, 5 and 4 at
// 168,000 contacts 16.6, 15.7, 14.9, 14.6 and 14.8 us, at 216,000 17.7, 17.7,
// 16.8, 16.2 and 16.3 (one row a thread, 11,900: 6.9 with 10, 7.0 with 9, 7.3
// with 8; mixed with two rows, 9.6 with 10, 10.0 with 8, 9.8 with 6).
constexpr int kRunTwo = 5;

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
  __device__ StepNext(double L, double theta) {
    const LazyNext n(L, theta);
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
//   has P1's step on its tiles, from registers (the iterates, N gamma and r
//     stay there, the frame in LDS), and J stored; forms its partial sums;
//   takes P2 on its body units (64 bodies to a wavefront, the team's units
//     dealt out evenly) as their contacts' J arrive; stores tmp and the units'
//     Lipschitz sums;
//   takes the next pass's step as its bodies' tmp arrive, on the guess that
//     this pass is accepted without a restart (then the next step size and
//     momentum do not depend on the pass's sums), and stores its J; and, on
//     the same guess, P2 on the wavefront's first unit, whose tmp is then on
//     its way while the pass is decided;
//   decides the pass from the team's partial sums, as kDecide does, and takes
//     the step and the unit again where the guess was wrong, under a second
//     tag.
// What keeps a member from storing over what another still reads: J of a
// contact is stored again only after tmp of its bodies, which is formed from
// it, has arrived, and tmp only after J of the body's contacts, formed from
// it; a step taken again stores over one that a slower member may still wait
// for, which takes either for its guess and drops what it made of it.  The
// partial sums alternate between two places, and are stored after a decision,
// which takes every member's.
// The iterates go back to memory when the launch ends, and gammaHat's when it
// leaves the registers.
// Two wavefronts per SIMD (up to 256 VGPRs, one workgroup to a CU): held to
// 128, so that a CU takes two, the mixed kernel spilled 20 and took 26.3 us
// per pass on 256,000 contacts, where two rows per thread take 10.7.  So, two
// rows mixed spill 4 VGPRs (15 with bilateral rows), three 26 (39), one in FP64
// 5 (8), the others none.
// Two rows in FP64 have room for the second step with gamma_{k-1} and its
// N gamma in LDS and five contacts of a body in flight: 17.4 us without the
// step, 14.6 with it.  (Mixed they stay in registers: 9.4 us, in LDS 9.6.)
// Three rows, mixed: 268,000 contacts 22.4 us as launches and 16.8 so, 327,000
// 24.0 and 18.0, 383,000 25.4 and 19.6.  (In FP64 the frames and the old
// iterates of three rows do not fit LDS.)
// In FP64 a large team's members wait for J, twice as long, with loads that
// take the others' room: us per pass with the unit taken ahead and not, 82
// members (41,800 contacts) 8.2 and 7.8, 162 (82,400) 10.5 and 9.4, but 24
// (11,900) 6.8 and 7.2; mixed 5.4 and 6.0, 5.8 and 6.8, 4.9 and 5.4.
// Where bodies outnumber contacts so far that both wavefronts of a SIMD have a
// unit, their waits cannot hide behind each other's steps: a shell's 19,200
// spheres with 20,100 contacts 6.4 ahead and 6.1 not.  With two rows a thread
// all units go ahead: 112,000 spheres, 256,000 contacts 10.7 ahead and 12.0
// not (mixed); 168,000 contacts 16.7 and 17.7 (FP64).
constexpr int kAheadMost = 64;
template <typename TM, bool kBil, int R>
__global__ __launch_bounds__(kTC, 2) void kTeam(const Args<TM>* __restrict__ A, Tables T, const TeamItem* items, int stride,
                                                u64* sync, u64 launch, int passes, u64 formTicks) {
  constexpr bool kMixed = sizeof(TM) < sizeof(double);
  constexpr int kRun = R == 1 || (kMixed && R == 2) ? kRunMost : kRunTwo;
  constexpr bool kOldInLds = R > (kMixed ? 2 : 1);
  constexpr bool kLanes = R == 1;
  constexpr int NF = kMixed ? 6 : 3;
  constexpr unsigned kUsed = kP1Slots<TM>;
  constexpr int kW = kTC / 64;       // wavefronts
  constexpr int kStateWave = kW - 2;
  constexpr int kWT = kTP / 64;      // of a heavy body's sum
  constexpr int kUnits = kTB / 64;   // body units of a body tile
  using Raw = typename CoArray<TM>::Raw;
  static_assert(kW == 2 * kUnits && kW == kSlots && kSlots == 8 && kUnits == 4, "a wavefront for each total; a body tile's units to a lane");
  // (a single team needs no list: every stride-th workgroup is a member)
  if (!items && (int)blockIdx.x % stride) return;
  const TeamItem me = items ? items[blockIdx.x] : TeamItem{0, (int)blockIdx.x / stride, (int)gridDim.x / stride, 0};
  const Args<TM>& a = A[me.slot];
  const SolveDims& D = a.dims;
  const int W = me.members, rank = me.rank, nTiles = a.nTiles;
  u64* sy = sync + (long)me.slot * kTeamSync;
  __shared__ int bad;
  __shared__ double shP[2][R][kW][kSlots], shTot[2][kW], shLq[2][kWT], shH[kWT][3];
  // the state before and after a pass; and, like the sums, for either parity:
  // a pass has one barrier, before its decision, which every wavefront takes
  __shared__ ApgdState shS[2];
  __shared__ double shTol;
  __shared__ int shMaxIt;
  __shared__ double shNext[3][6];  // (a pass's, the next one's, and the last one's, still read)
  __shared__ double shUnit[32][kW];  // the units' Lipschitz sums, and how many of a tile's are there
  __shared__ int unitCount[32][2];
  __shared__ u64 liveTiles;  // bit t: tile rank + W t has a unit with a movable light body
  // per thread, kept here instead of in registers: the rows' frames and the
  // first body's contacts
  __shared__ TM shF[R][9][kTC];
  __shared__ int shIds[kRun][kTC];
  // and gamma_{k-1} and its N gamma, which only a step taken again reads
  __shared__ double shGm[kOldInLds ? R : 1][3][kOldInLds ? kTC : 1];
  __shared__ TM shNm[kOldInLds ? R : 1][3][kOldInLds ? kTC : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < 64) unitCount[tid / 2][tid % 2] = 0;
  if (tid == 0) {
    bad = 0;
    liveTiles = 0;
    shTol = a.dims.tol;
    shMaxIt = a.dims.maxIt;
    shS[0] = STATE(T, me.slot, 1);
  }
  __syncthreads();
  if (shS[0].done) return;  // the same for every member
  PassView V = uniformView(viewOf(shS[0]));
  const long cap = a.cap;
  const CoArray<TM> J(a.J, cap + D.nbil), tmp(a.tmpX, D.nb);
  const int nBT = a.nBodyTiles, nHeavy = gl(a.counters)[2], nl = nBT + nHeavy;
  // body units of 64 bodies: a wavefront's in iteration j is of tile
  // rank + W (2 j + half)
  const int half = wave / kUnits, nU = kUnits * nBT;
  const int u0 = kUnits * (rank + W * half) + wave % kUnits, uStep = 2 * kUnits * W;
  // P1's partial sums (slot s of tile k at s nTiles + k) and the body tiles'
  // and the heavy bodies' Lipschitz sums, by pass parity
  const __amdgpu_buffer_rsrc_t rPart = __builtin_amdgcn_make_buffer_rsrc(a.partX, 0, 2 * 16 * kSlots * nTiles, 0x00027000);
  const __amdgpu_buffer_rsrc_t rLq = __builtin_amdgcn_make_buffer_rsrc(a.lqX, 0, 2 * 16 * nl, 0x00027000);
  auto postPart = [&](int par, int i, double v, unsigned tag) {
    __builtin_amdgcn_raw_buffer_store_b128(taggedDouble(v, tag), rPart, 16 * i, par * 16 * kSlots * nTiles, kDeviceScope);
  };
  auto postLq = [&](int par, int i, double v, unsigned tag) {
    __builtin_amdgcn_raw_buffer_store_b128(taggedDouble(v, tag), rLq, 16 * i, par * 16 * nl, kDeviceScope);
  };

  // this thread's rows: row u of tile R rank + u
  struct Row {
    int e, ia, ib;  // its entry of J, and the tmp of its bodies (kNone: fixed)
    int ca, cb;     // bilateral: the components
    bool valid, bil;
    TM rv[3], nk[3], nm[3], nn[3];
    double gk[3], gm[3], gn[3], gs[3];
  };
  Row row[R];
  auto keepOld = [&](int u, const double (&g)[3], const TM (&n)[3]) {
#pragma unroll
    for (int rr = 0; rr < 3; ++rr) {
      if constexpr (kOldInLds) {
        shGm[u][rr][tid] = g[rr];
        shNm[u][rr][tid] = n[rr];
      } else {
        row[u].gm[rr] = g[rr];
        row[u].nm[rr] = n[rr];
      }
    }
  };
  auto loadOld = [&](int u, double (&g)[3], TM (&n)[3]) {
#pragma unroll
    for (int rr = 0; rr < 3; ++rr) {
      if constexpr (kOldInLds) {
        g[rr] = shGm[u][rr][tid];
        n[rr] = shNm[u][rr][tid];
      } else {
        g[rr] = row[u].gm[rr];
        n[rr] = row[u].nm[rr];
      }
    }
  };
  auto flatOf = [&](int u, int rr) {  // row rr's place in a row vector
    const long q = ((long)rank * R + u) * kTC + tid;
    return kBil && q >= D.nc ? (long)BROW(a, q - D.nc) : ROW(a, rr, q);
  };
#pragma unroll
  for (int u = 0; u < R; ++u) {
    Row& w = row[u];
    const long q = ((long)rank * R + u) * kTC + tid;
    w.valid = q < (long)D.nc + D.nbil;
    w.bil = kBil && w.valid && q >= D.nc;
    const int c = w.valid && !w.bil ? (int)q : 0;
    w.e = w.bil ? (int)(cap + (q - D.nc)) : w.valid ? c : kNone;
    w.ia = gl(a.cA)[c];
    w.ib = gl(a.cB)[c];
    w.ca = w.cb = 0;
    if (kBil && w.bil) {  // the two DOFs
      const int da = gl(a.bilA)[q - D.nc], db = gl(a.bilB)[q - D.nc];
      w.ia = da / 3;
      w.ca = da % 3;
      w.ib = db < 0 ? w.ia : db / 3;
      w.cb = db < 0 ? -1 : db % 3;
    }
    if (!w.valid || gl(a.minv)[w.ia] == (TM)0) w.ia = kNone;
    if (!w.valid || w.cb < 0 || gl(a.minv)[w.ib] == (TM)0) w.ib = kNone;
    TM fc[6], F[9];
#pragma unroll
    for (int k = 0; k < 6; ++k) fc[k] = k < NF ? gl(a.frame)[k * cap + c] : (TM)0;
    frameFrom(fc, D.geomMode, F);
    // (no contact, no frame: without contacts in the scene the memory of
    // contact 0 may hold anything, and NaN times the row's zeros is NaN)
#pragma unroll
    for (int k = 0; k < 9; ++k) shF[u][k][tid] = w.valid && !w.bil ? F[k] : (TM)0;
    double gm[3];
    TM nm[3];
#pragma unroll
    for (int rr = 0; rr < 3; ++rr) {
      // (a thread without a row has one of zeros, which adds zero to every sum)
      const bool on = w.valid && !(w.bil && rr);
      const long f = on ? flatOf(u, rr) : 0;
      w.rv[rr] = on ? gl(a.r)[f] : (TM)0;
      w.gk[rr] = on ? gl(a.ring[0] + V.cur * a.ringStride)[f] : 0.0;
      gm[rr] = on ? gl(a.ring[0] + V.prev * a.ringStride)[f] : 0.0;
      w.nk[rr] = on ? gl(a.rn[0] + V.cur * a.ringStride)[f] : (TM)0;  // (not formed yet if fresh: replaced below)
      nm[rr] = on ? gl(a.rn[0] + V.prev * a.ringStride)[f] : (TM)0;
      w.gn[rr] = w.gs[rr] = 0;
      w.nn[rr] = 0;
    }
    keepOld(u, gm, nm);
    J.st(w.e, 0, 0, 0, 0);
  }
  // the iterate in registers back to its ring slot
  auto storeIterate = [&](int slot, int u, const double (&g)[3]) {
    const Row& w = row[u];
    if (!w.valid) return;
#pragma unroll
    for (int rr = 0; rr < 3; ++rr)
      if (!(w.bil && rr)) gl(a.ring[0] + slot * a.ringStride)[flatOf(u, rr)] = g[rr];
  };

  const BodyRuns<TM> first = bodyRuns(a, u0 < nU ? (long)u0 * 64 + lane : (long)D.nb);
#pragma unroll
  for (int k = 0; k < kRun; ++k) shIds[k][tid] = contactOf(a, first, k);
  unsigned live = 0;
  for (int j = 0, u = u0; u < nU; ++j, u += uStep) {
    const int g = u * 64 + lane;
    if (__any(bodyRuns(a, (long)g).sums)) {
      live |= 1u << j;
      if (lane == 0) __hip_atomic_fetch_or(&liveTiles, 1ull << (2 * j + half), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (g < D.nb) tmp.st(g, 0, 0, 0, 0);
    if (wave % kUnits == 0 && lane == kLast)
      for (int k = 0; k < 2; ++k) postLq(k, u / kUnits, 0.0, 0);
    // (the launches read the D^T gamma ring of fixed bodies too, times zero)
    if (kMixed && g < D.nb && gl(a.minv)[g] == (TM)0)
#pragma unroll
      for (int k = 0; k < 4; ++k) st4(a.sr, (long)k * D.nb + g, V4<TM>{0, 0, 0, 0});
  }
  for (int h = rank + W * tid; h < nHeavy; h += W * kTC)
    for (int k = 0; k < 2; ++k) postLq(k, nBT + h, 0.0, 0);
  bool liveHeavy = false;
  for (int h = rank; h < nHeavy; h += W) liveHeavy = liveHeavy || gl(a.minv)[gl(a.heavy)[h]] != (TM)0;
  // lane l of the last wavefront posts the zero sum of fixed body rank + W l
  auto isFixed = [&](int h) { return h < nHeavy && gl(a.minv)[gl(a.heavy)[h]] == (TM)0; };
  const bool fixedHeavy = wave == kW - 1 && isFixed(rank + W * lane);
  if (tid < R * kSlots) {
    const int u = tid / kSlots, s = tid % kSlots;
    if (R * rank + u < nTiles)
      for (int k = 0; k < 2; ++k) postPart(k, s * nTiles + R * rank + u, 0.0, 0);
  }
  if (!teamForm(sy, rank, W, launch, formTicks)) return;
  // The zero sums of tiles of fixed bodies only are posted by lane t of the
  // last wavefront; of the others, a unit without a movable light body has a
  // zero sum.
  const u64 tiles = liveTiles;
  unsigned units = 0;  // this wavefront's units of live tiles
  for (int j = 0, u = u0; u < nU; ++j, u += uStep)
    if ((tiles >> (2 * j + half)) & 1u) units |= 1u << j;
  units = __builtin_amdgcn_readfirstlane(units);
  const bool fixedTile = wave == kW - 1 && rank + W * lane < nBT && !((tiles >> lane) & 1u);

  // y, N y and g of a row (formed once for the step and again for the sums,
  // rather than kept)
  auto momentum = [&](bool mom, double beta, double gk, double gm, TM nk, TM nm, TM rv, double& y, double& ny,
                      double& gg) {
    if (mom) {
      const double bp = 1.0 + beta, bm = -beta;
      y = bp * gk + bm * gm;
      ny = bp * (double)nk + bm * (double)nm;
    } else {
      y = gk;
      ny = (double)nk;
    }
    gg = 1.0 * ny + 1.0 * (double)rv;
  };
  const Cone cone(D.mu);
  // P1's step of row u from (gk, gm, nk, nm) into out, and its J
  auto step = [&](int u, const double (&gk)[3], const double (&gm)[3], const TM (&nk)[3], const TM (&nm)[3], bool mom,
                  double beta, double t, double (&out)[3], unsigned tag) {
    const Row& w = row[u];
#pragma unroll
    for (int rr = 0; rr < 3; ++rr) {
      double y, ny, gg;
      momentum(mom, beta, gk[rr], gm[rr], nk[rr], nm[rr], w.rv[rr], y, ny, gg);
      out[rr] = 1.0 * y + (-t) * gg;
    }
    if (w.bil) {
      J.stDouble(w.e, out[0], tag);
    } else {
      cone.project(out[0], out[1], out[2]);
      const TM x0 = (TM)out[0], x1 = (TM)out[1], x2 = (TM)out[2];
      TM F[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) F[k] = shF[u][k][tid];
      J.st(w.e, F[0] * x0 + F[3] * x1 + F[6] * x2, F[1] * x0 + F[4] * x1 + F[7] * x2,
           F[2] * x0 + F[5] * x1 + F[8] * x2, tag);
    }
  };
  // N gamma of row u from its bodies' M^-1 D^T gamma
  auto rowsN = [&](int u, const V3<TM>& tA, const V3<TM>& tB, TM (&out)[3]) {
    const Row& w = row[u];
    if (w.bil) {
      auto comp = [](const V3<TM>& t, int k) { return k == 0 ? t.x : (k == 1 ? t.y : t.z); };
      out[0] = comp(tA, w.ca) - (w.cb < 0 ? (TM)0 : comp(tB, w.cb));
    } else {
      TM F[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) F[k] = shF[u][k][tid];
      rowsOfTmp(F, V4<TM>{tA.x, tA.y, tA.z, (TM)0}, V4<TM>{tB.x, tB.y, tB.z, (TM)0}, out[0], out[1], out[2]);
    }
  };
  auto rowsOfArrived = [&](unsigned tag) {
    int id[2 * R];
    Raw t[2 * R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
      id[2 * u] = row[u].ia;
      id[2 * u + 1] = row[u].ib;
    }
    await<kLanes>(tmp, id, tag, &bad, t);
#pragma unroll
    for (int u = 0; u < R; ++u) rowsN(u, tmp.value(t[2 * u]), tmp.value(t[2 * u + 1]), row[u].nn);
  };

  // the partial sums of the step from (gk, gm, nk, nm) to gn, in P1's order
  auto sumsOf = [&](int to, int u, const double (&gk)[3], const double (&gm)[3], const double (&gn)[3],
                    const TM (&nk)[3], const TM (&nm)[3], bool mom, double beta) {
    const Row& w = row[u];
    double acc[kSlots];
    zero(acc);
    const double w0 = (double)nk[0] + (double)w.rv[0];
    if (w.bil) {
      double e;
      if (D.nc) {
        const double z = 1.0 * gk[0] + (-D.gdiff) * w0;
        const double ig = D.igdiff;
        e = fabs(ig * gk[0] + (-ig) * z);
      } else {
        e = fabs(w0);
      }
      acc[7] = fmax(acc[7], e == e ? e : INFINITY);
    } else {
      const double w1 = (double)nk[1] + (double)w.rv[1];
      const double w2 = (double)nk[2] + (double)w.rv[2];
      acc[7] = fmax(acc[7], cone.residual(gk[0], gk[1], gk[2], w0, w1, w2, D.gdiff, D.igdiff));
    }
#pragma unroll
    for (int rr = 0; rr < 3; ++rr) {
      double y, ny, gg;
      momentum(mom, beta, gk[rr], gm[rr], nk[rr], nm[rr], w.rv[rr], y, ny, gg);
      const double dy = gn[rr] - y;
      if (!kMixed) {
        acc[0] += gn[rr] * (double)w.rv[rr];
        acc[1] += y * ny;
        acc[2] += y * (double)w.rv[rr];
        acc[3] += gg * dy;
      }
      acc[4] += dy * dy;
      acc[5] += gg * (gn[rr] - gk[rr]);
    }
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      if (!((kUsed >> s) & 1u)) continue;
      const double v = s == kSlots - 1 ? lastMax(acc[s]) : lastSum(acc[s]);
      if (lane == kLast) shP[to][u][wave][s] = v;
    }
  };

  auto bilateral = [&](const BodyRuns<TM>& b, unsigned tagJ, unsigned least, TM (&s)[3]) {
    for (int k = b.b0; kBil && k < b.b1; ++k) {
      const int e = gl(a.bilInc)[k];
      const int i[1] = {(int)cap + (e >> 3)};
      Raw x[1];
      await<kLanes>(J, i, tagJ, &bad, x, least);
      const double g = J.asDouble(x[0]);
      const TM t = (TM)((e & 1) ? -g : g);
      const int comp = (e >> 1) & 3;
      if (comp == 0) s[0] += t; else if (comp == 1) s[1] += t; else s[2] += t;
    }
  };
  auto contacts = [&](const BodyRuns<TM>& b, int kb, const Raw (&v)[kRun], TM (&s)[3]) {
#pragma unroll
    for (int k = 0; k < kRun; ++k) {
      // (past the body's contacts zero, which changes no sum that began with zero)
      const V3<TM> t = J.value(v[k]);
      const TM sign = kb + k < b.nd ? -1 : 1;  // (times it is exact)
      s[0] = exactFma(t.x, sign, s[0]); s[1] = exactFma(t.y, sign, s[1]); s[2] = exactFma(t.z, sign, s[2]);
    }
  };
  auto moreContacts = [&](const BodyRuns<TM>& b, int kb, unsigned tagJ, unsigned least, TM (&s)[3]) {  // from its kb-th on
    for (; __any(kb < b.n); kb += kRun) {
      int id[kRun];
      Raw v[kRun];
#pragma unroll
      for (int k = 0; k < kRun; ++k) id[k] = contactOf(a, b, kb + k);
      await<kLanes>(J, id, tagJ, &bad, v, least);
      contacts(b, kb, v, s);
    }
  };
  // P2 on this wavefront's first unit, whose D^T gamma_k and D^T gamma_{k-1}
  // stay in registers (mixed; dn the pass's, dg the guessed pass's)
  V4<TM> dc{0, 0, 0, 0}, dp{0, 0, 0, 0}, dn{0, 0, 0, 0}, dg{0, 0, 0, 0};
  double firstTerm = 0;
  if (kMixed && first.sums) {
    dc = ld4(a.sr, V.cur * (long)D.nb + first.g);
    dp = ld4(a.sr, V.prev * (long)D.nb + first.g);
  }
  const bool ahead = (R > 1 || __popcll(tiles) <= 1) && (kMixed || R > 1 || W <= kAheadMost);
  auto firstUnit = [&](unsigned tagJ, unsigned least, const V4<TM>& c, const V4<TM>& p, bool mom, double beta, V4<TM>& out) {
    if (!(live & 1u)) return;
    int id[kRun];
    Raw v[kRun];
#pragma unroll
    for (int k = 0; k < kRun; ++k) id[k] = shIds[k][tid];
    await<kLanes>(J, id, tagJ, &bad, v, least);
    TM s[3] = {0, 0, 0};
    bilateral(first, tagJ, least, s);
    contacts(first, 0, v, s);
    moreContacts(first, kRun, tagJ, least, s);
    if (first.sums) tmp.st(first.g, first.mi * s[0], first.mi * s[1], first.mi * s[2], tagJ);
    firstTerm = lastSum(first.sums ? lipschitzOf(first.mi, s[0], s[1], s[2], c, p, mom, beta) : 0.0);
    if (kMixed) out = V4<TM>{s[0], s[1], s[2], 0};
  };

  // the step sizes of a pass's either outcome, by a wavefront that has time
  // (as for the state)
  auto stepSizes = [&](int to, double fromL, double fromTheta) {
    if (wave != kStateWave) return;
    const StepNext n(fromL, fromTheta);
    if (lane == 0) n.store(shNext[to]);
  };

  int ends = 0;        // which state is the last
  bool taken = false;  // this pass's step was taken on the last one's guess
  for (int p = 0, sizes = 0; p < passes; ++p, sizes = sizes == 2 ? 0 : sizes + 1) {
    const int par = p & 1;
    const unsigned tag = (unsigned)(2 * p + 2) << 16;
    unsigned tagJ = tag;
    const bool mom = !(V.flags & kViewRestart);
    // ---- P1
    if (!taken) {
      if (p == 0) {
        if (V.flags & kViewFresh) {  // tmp as the launches or the last resident passes left it
#pragma unroll
          for (int u = 0; u < R; ++u) {
            const V4<TM> z{0, 0, 0, 0};
            const V4<TM> tA = row[u].ia == kNone ? z : ld4(a.tmp, row[u].ia);
            const V4<TM> tB = row[u].ib == kNone ? z : ld4(a.tmp, row[u].ib);
            rowsN(u, V3<TM>{tA.x, tA.y, tA.z}, V3<TM>{tB.x, tB.y, tB.z}, row[u].nk);
          }
        }
      } else {
        tagJ |= 1u << 16;
      }
#pragma unroll
      for (int u = 0; u < R; ++u) {
        Row& w = row[u];
        double gm[3];
        TM nm[3];
        loadOld(u, gm, nm);
        step(u, w.gk, gm, w.nk, nm, mom, V.beta, V.t, w.gn, tagJ);
        sumsOf(par, u, w.gk, gm, w.gn, w.nk, nm, mom, V.beta);
      }
      stepSizes(sizes, shS[par].L, shS[par].theta);  // (which its wavefront has stored)
      __syncthreads();
    }
    // the tiles' partial sums, by the last wavefront (which has the fewest
    // body units)
    if (wave == kW - 1 && lane < R * kSlots && ((kUsed >> (lane % kSlots)) & 1u)) {
      const int u = lane / kSlots, s = lane % kSlots;
      double t[kW];
#pragma unroll
      for (int w = 0; w < kW; ++w) t[w] = shP[par][u][w][s];
      double v = t[0];
#pragma unroll
      for (int w = 1; w < kW; ++w) v = s == kSlots - 1 ? fmax(v, t[w]) : v + t[w];
      if (R * rank + u < nTiles) postPart(par, s * nTiles + R * rank + u, v, tag);
    }
    if (fixedTile) postLq(par, rank + W * lane, 0.0, tag);
    if (fixedHeavy) postLq(par, nBT + rank + W * lane, 0.0, tag);
    for (int h = rank + W * (64 + lane); wave == kW - 1 && h < nHeavy; h += W * 64)
      if (isFixed(h)) postLq(par, nBT + h, 0.0, tag);

    // ---- P2
    // a unit's Lipschitz sum; the last of a tile's four posts the tile's
    auto postUnit = [&](int j, int u, double term) {
      if (lane != kLast) return;
      shUnit[j][wave] = term;
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      const int before = __hip_atomic_fetch_add(&unitCount[j][half], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      if (before != kUnits - 1) return;
      __hip_atomic_store(&unitCount[j][half], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      const double* t = &shUnit[j][kUnits * half];
      postLq(par, u / kUnits, ((t[0] + t[1]) + t[2]) + t[3], tag);
    };
    auto finish = [&](const BodyRuns<TM>& b, int j, int u, const TM (&s)[3], const V4<TM>& c, const V4<TM>& p) {
      if (b.sums) tmp.st(b.g, b.mi * s[0], b.mi * s[1], b.mi * s[2], tagJ);
      const double term = lastSum(b.sums ? lipschitzTerm(a, b.g, V, b.mi, s[0], s[1], s[2], c, p) : 0.0);
      postUnit(j, u, term);
    };
    auto loadRing = [&](int g, V4<TM>& c, V4<TM>& p) {  // D^T gamma_k and D^T gamma_{k-1}
      if (!kMixed) return;
      c = ld4(a.sr, V.cur * (long)D.nb + g);
      p = ld4(a.sr, V.prev * (long)D.nb + g);
    };
    if (!(taken && ahead)) firstUnit(tagJ, 0x10000u, dc, dp, mom, V.beta, dn);
    if (units & 1u) postUnit(0, u0, firstTerm);  // (zero where nothing is live)
    for (unsigned left = units & ~1u; left; left &= left - 1) {
      const int j = __builtin_ctz(left), u = u0 + j * uStep;
      if (!((live >> j) & 1u)) {
        postUnit(j, u, 0.0);
        continue;
      }
      const BodyRuns<TM> b = bodyRuns(a, (long)u * 64 + lane);
      V4<TM> c, p;
      loadRing(b.g, c, p);
      TM s[3] = {0, 0, 0};
      bilateral(b, tagJ, 0x10000u, s);
      moreContacts(b, 0, tagJ, 0x10000u, s);
      if (kMixed) {
        settled(c);
        settled(p);
      }
      finish(b, j, u, s, c, p);
    }
    // bodies with many contacts, by the first kTP threads
    for (int h = rank; liveHeavy && h < nHeavy; h += W) {
      const int g = gl(a.heavy)[h];
      const TM mi = gl(a.minv)[g];
      if (mi == (TM)0) continue;
      const int k0 = gl(a.iStart)[g], n = gl(a.iStart)[g + 1] - k0;
      const int c0 = gl(a.cStart)[g], c1 = gl(a.cStart)[g + 1];
      const int nd = n - (c1 - c0);
      V4<TM> c, p;
      loadRing(g, c, p);
      if (tid < kTP) {
        double hx = 0, hy = 0, hz = 0;
        for (int kb = tid; kb < n; kb += 4 * kTP) {
          int id[4];
          Raw v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int k = kb + i * kTP;
            id[i] = k < nd ? gl(a.inc)[k0 + k] >> 1 : k < n ? c0 + k - nd : kNone;
          }
          await<kLanes>(J, id, tagJ, &bad, v);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int k = kb + i * kTP;
            if (k >= n) continue;
            const double sg = k < nd ? -1.0 : 1.0;
            const V3<TM> t = J.value(v[i]);
            hx += sg * (double)t.x;
            hy += sg * (double)t.y;
            hz += sg * (double)t.z;
          }
        }
        if (kBil && tid == 0) {
          for (int k = gl(a.bilIncStart)[g]; k < gl(a.bilIncStart)[g + 1]; ++k) {
            const int e = gl(a.bilInc)[k];
            const int i[1] = {(int)cap + (e >> 3)};
            Raw x[1];
            await<kLanes>(J, i, tagJ, &bad, x);
            const double v = J.asDouble(x[0]), t = (e & 1) ? -v : v;
            const int comp = (e >> 1) & 3;
            if (comp == 0) hx += t; else if (comp == 1) hy += t; else hz += t;
          }
        }
        hx = lastSum(hx); hy = lastSum(hy); hz = lastSum(hz);
        if (lane == kLast) {
          shH[wave][0] = hx; shH[wave][1] = hy; shH[wave][2] = hz;
        }
      }
      if (kMixed) {
        settled(c);
        settled(p);
      }
      __syncthreads();
      if (tid == 0) {
        TM t[3];
        for (int s = 0; s < 3; ++s) {
          double v = shH[0][s];
          for (int w = 1; w < kWT; ++w) v += shH[w][s];
          t[s] = (TM)v;
        }
        tmp.st(g, mi * t[0], mi * t[1], mi * t[2], tagJ);
        postLq(par, nBT + h, lipschitzTerm(a, g, V, mi, t[0], t[1], t[2], c, p), tag);
      }
      __syncthreads();
    }

    // ---- the next pass's step, should this one be accepted without a restart
    const bool guess = p + 1 < passes;
    if (guess) rowsOfArrived(tagJ);
    const double tNext = uniformDouble(shNext[sizes][3]), betaNext = uniformDouble(shNext[sizes][5]);
    // The team's sums, in reduceSlots' order: lane l of its wavefront i adds
    // entries 64 i + l, 64 i + l + kTP, ..., and the wavefronts' sums are added
    // in order (past the entries they are zero, and left out).  Here wavefront
    // s totals slot s of P1's partials, and wavefront 6 - i is wavefront i for
    // the Lipschitz terms.
    const int il = 6 - wave;
    const bool sumsPart = (kUsed >> wave) & 1u, sumsLq = il >= 0 && il < kWT && 64 * il < nl;
    i32x4 xp[kWT], xl;  // a slot of four tiles; a body tile's or a heavy body's sum
    auto loadPart = [&](int b0) {
#pragma unroll
      for (int i = 0; i < kWT; ++i) {
        const int w = b0 + 64 * i + lane;
        xp[i] = __builtin_amdgcn_raw_buffer_load_b128(rPart, w >= nTiles ? kPastEnd : 16 * (wave * nTiles + w),
                                                      par * 16 * kSlots * nTiles, kDeviceScope);
      }
    };
    auto loadLq = [&](int b0) {
      const int w = b0 + 64 * il + lane;
      xl = __builtin_amdgcn_raw_buffer_load_b128(rLq, w >= nl ? kPastEnd : 16 * w, par * 16 * nl, kDeviceScope);
    };
    if (guess) {
#pragma unroll
      for (int u = 0; u < R; ++u) {
        Row& w = row[u];
        step(u, w.gn, w.gk, w.nn, w.nk, true, betaNext, tNext, w.gs, tag + (2u << 16));
      }
    }
    if (guess)
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const Row& w = row[u];
        sumsOf(par ^ 1, u, w.gn, w.gk, w.gs, w.nn, w.nk, true, betaNext);
      }
    if (guess) stepSizes(sizes == 2 ? 0 : sizes + 1, shNext[sizes][2], shNext[sizes][4]);  // (those of the guessed outcome)
    if (sumsPart) loadPart(0);
    if (sumsLq) loadLq(0);
    if (guess && ahead) firstUnit(tag + (2u << 16), kOrReplaced, dn, dc, true, betaNext, dg);
    if (sumsPart) {
      double v[kWT] = {0, 0, 0, 0};
      for (int b0 = 0; b0 < nTiles; b0 += kTP) {
        if (b0) loadPart(b0);
        waitFor<false>(
            &bad, 0x10000u,
            [&] {
              unsigned m = 0;
#pragma unroll
              for (int i = 0; i < kWT; ++i) m |= b0 + 64 * i + lane < nTiles ? missing(xp[i], tag) : 0u;
              return m;
            },
            [&] { loadPart(b0); });
#pragma unroll
        for (int i = 0; i < kWT; ++i) pinned(xp[i]);
#pragma unroll
        for (int i = 0; i < kWT; ++i) v[i] = wave == kSlots - 1 ? fmax(v[i], valueOf(xp[i])) : v[i] + valueOf(xp[i]);
      }
      double total = wave == kSlots - 1 ? lastMax(v[0]) : lastSum(v[0]);
      for (int i = 1; i < kWT && 64 * i < nTiles; ++i)
        total = wave == kSlots - 1 ? fmax(total, lastMax(v[i])) : total + lastSum(v[i]);
      if (lane == kLast) shTot[par][wave] = total;
    }
    if (sumsLq) {
      double v = 0;
      for (int b0 = 0; b0 + 64 * il < nl; b0 += kTP) {
        if (b0) loadLq(b0);
        const int w = b0 + 64 * il + lane;
        waitFor<false>(
            &bad, 0x10000u, [&] { return w < nl ? missing(xl, tag) : 0u; }, [&] { loadLq(b0); });
        pinned(xl);
        v += valueOf(xl);
      }
      const double total = lastSum(v);
      if (lane == kLast) shLq[par][il] = total;
    }


    // ---- the decision, by every member's every wavefront
    __syncthreads();
    const bool lost = __builtin_amdgcn_readfirstlane(bad) != 0;  // (set by waits only, which all lie before this point)
    const ApgdState& before = shS[par];
    double lq = shLq[par][0];
#pragma unroll
    for (int i = 1; i < kWT; ++i) {
      const double more = lq + shLq[par][i];
      lq = 64 * i < nl ? more : lq;
    }
    const int dropped = V.prev;
    bool keep = false;  // gammaHat leaves the registers
    // most passes are accepted without a restart, as decideStep has it
    // (all loads at once, and no branch between them)
    const double res = shTot[par][kSlots - 1], best = before.best, tol = shTol, stepL = before.L;
    const int pending = before.pendingRes, it = before.it, maxIt = shMaxIt, hatBefore = before.hatSrc;
    double t[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) t[k] = (kUsed >> k) & 1u ? shTot[par][k] : 0.0;
    const bool better = res < best;
    bool goesOn = (pending != 0) & (res < INFINITY) & !((better ? res : best) < tol) & (it < maxIt) & !(t[5] > 0);
    if (kMixed) {
      goesOn = goesOn & !(lq >= stepL * t[4]);
    } else {
      const double obj1 = 0.5 * lq + t[0], nrm = sqrt(t[4]);
      double obj2 = 0.5 * t[1] + t[2];
      obj2 += t[3] + 0.5 * stepL * (nrm * nrm);
      goesOn = goesOn & !(obj1 >= obj2);
    }
    if (__any(goesOn)) {  // (alike in all lanes)
      const int hat = __any(better) ? V.cur : __builtin_amdgcn_readfirstlane(hatBefore);
      V.prev = V.cur;
      V.cur = V.nxt;
      V.nxt = __builtin_ctz(~(1u << V.cur | 1u << V.prev | 1u << hat));
      V.flags = kViewFresh;
      V.t = tNext;
      V.beta = betaNext;
      keep = hat == dropped;
      if (wave == kStateWave) {
        ApgdState S = before;
        const StepNext n(shNext[sizes]);
        S.passes++;
        S.best = better ? res : best;
        S.hatSrc = hat;
        S.beta = n.beta;
        S.restart = 0;
        S.L = n.La;
        S.t = n.ta;
        S.theta = n.thetaNew;
        S.prev = V.prev;
        S.cur = V.cur;
        S.nxt = V.nxt;
        S.it++;
        S.bt = 0;
        S.pendingRes = 1;
        S.fresh = 1;
        if (lane == 0) shS[par ^ 1] = S;
      }
    } else {
      double tot[2 * kSlots];
#pragma unroll
      for (int k = 0; k < 2 * kSlots; ++k) tot[k] = 0.0;
#pragma unroll
      for (int k = 0; k < kSlots; ++k)
        if ((kUsed >> k) & 1u) tot[k] = shTot[par][k];
      tot[kSlots + 6] = lq;
      ApgdState S = before;
      SolveDims limits = D;  // (of these two only, and not from memory)
      limits.tol = shTol;
      limits.maxIt = shMaxIt;
      decideStep<kMixed>(S, tot, limits, StepNext(shNext[sizes]));
      if (wave == kStateWave && lane == 0) shS[par ^ 1] = S;
      V = uniformView(viewOf(S));
      keep = __builtin_amdgcn_readfirstlane(S.hatSrc) == dropped;
    }
    ends = par ^ 1;
    if (lost || (V.flags & kViewDone)) break;
    taken = false;
    if (V.flags & kViewFresh) {  // accepted: gamma_new becomes gamma_k (a backtrack keeps both)
      taken = !(V.flags & kViewRestart) && V.t == tNext && V.beta == betaNext;
      if (kMixed) {
        dp = dc;
        dc = dn;
        dn = dg;
      }
#pragma unroll
      for (int u = 0; u < R; ++u) {
        Row& w = row[u];
        if (keep) {
          double gm[3];
          TM nm[3];
          loadOld(u, gm, nm);
          storeIterate(dropped, u, gm);
        }
        keepOld(u, w.gk, w.nk);
#pragma unroll
        for (int rr = 0; rr < 3; ++rr) {
          w.gk[rr] = w.gn[rr];
          w.nk[rr] = w.nn[rr];
          w.gn[rr] = w.gs[rr];
        }
      }
    }
  }
  // what the launches, or the next resident passes, read
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const Row& w = row[u];
    double gm[3];
    TM nm[3];
    loadOld(u, gm, nm);
    if (V.prev != V.cur) storeIterate(V.prev, u, gm);
    storeIterate(V.cur, u, w.gk);
    if (!w.valid) continue;
#pragma unroll
    for (int rr = 0; rr < 3; ++rr) {
      if (w.bil && rr) continue;
      const long f = flatOf(u, rr);
      if (V.prev != V.cur) gl(a.rn[0] + V.prev * a.ringStride)[f] = nm[rr];
      if (!(V.flags & kViewFresh)) gl(a.rn[0] + V.cur * a.ringStride)[f] = w.nk[rr];
    }
  }
  if (kMixed && first.sums) {
    if (V.prev != V.cur) st4(a.sr, V.prev * (long)D.nb + first.g, dp);
    st4(a.sr, V.cur * (long)D.nb + first.g, dc);
  }
  // (from the thread's own stores; after the last decision of a solve nothing
  // reads tmp, and it may hold a guess)
  if ((V.flags & (kViewFresh | kViewDone)) == kViewFresh) {
    for (int u = u0; u < nU; u += uStep) {
      const BodyRuns<TM> b = bodyRuns(a, (long)u * 64 + lane);
      if (!b.sums) continue;
      const V3<TM> t = tmp.value(tmp.ld(b.g));
      st4(a.tmp, b.g, V4<TM>{t.x, t.y, t.z, (TM)0});
    }
    for (int h = rank; tid == 0 && h < nHeavy; h += W) {
      const int g = gl(a.heavy)[h];
      if (gl(a.minv)[g] == (TM)0) continue;
      const V3<TM> t = tmp.value(tmp.ld(g));
      st4(a.tmp, g, V4<TM>{t.x, t.y, t.z, (TM)0});
    }
  }
  if (rank == 0 && tid == 64 * kStateWave) {
    ApgdState S = shS[ends];
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
