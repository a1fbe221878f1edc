// Collision detection for gfx950: a spatial-hash broadphase fused with the
// narrowphase, emitting contacts directly in canonical (idA, idB) order, plus
// the body-major incidence lists used for D^T products.
//
// Reference behaviour (CollisionDetector.cu):
//   * AABBs are geometry +- (radius or half extents + envelope)      (:24-79)
//   * candidate pairs exclude the same body and equal families != -1 (:131-132)
//   * the kept set is {pen >= -envelope} of the sphere-sphere and
//     sphere-box narrowphase; box-box never collides                 (:287-328)
//   * contacts are ordered by the 64-bit key (idA << 32) | idB after a
//     stable sort + unique of the candidates                           (:166-173, 621-622)
// The kept set does not depend on the bins (every kept pair's AABBs overlap
// with a margin of one envelope), so any complete broadphase yields the same
// contacts.  Here:
//   1. small spheres are sorted into the slots of a hash of cells of edge
//      2*(r_max + envelope), so a kept partner lies in one of the 27
//      neighbouring cells; boxes and large spheres form a short "big" list
//      tested against every geometry;
//   2. one walk of the neighbouring cells, sixteen lanes to a sphere, finds
//      each sphere's partners, sorts them by id and keeps them (up to kList);
//   3. one prefix sum over the bodies gives each geometry's contact row and
//      incidence offsets and the list of heavy bodies;
//   4. each sphere's row is written at its final canonical position from the
//      kept partners (no global key sort and no second walk), with the
//      incidences of both of its bodies: a body's incidences are listed in
//      ascending contact order, first the contacts where it is B (its place
//      among B's partners below is its place in B's list), then its own row.
// The keep test and the contact record are evaluated with the shared
// dv_geom.h code (no fused multiply-add), bit-identical to the oracle.
#include "dv_geom.h"
#include "dv_internal.h"

#include <algorithm>
#include <cmath>

namespace dv {
namespace {

constexpr int kT = 256;

// What a walk reads of a small geometry, in the order of the cells: its
// position and radius (posR), and its id, row of cells and family (meta).
struct alignas(32) PosR {
  double x, y, z, r;
};

struct CdArgs {
  const double* p;
  const double* geom;
  const int* family;
  const int* smallIds;
  const int* bigIds;
  int nb, nsmall, nbig;
  double cs, envelope;
  unsigned mask;
  int mode;
  const unsigned* slotStart;
  PosR* posR;
  int4* meta;
};

// A cell's slot: a hash of its row (the cells along x) plus its place in the
// row, so that the three cells beside each other are three slots in a row and
// a walk takes nine ranges instead of 27.
__device__ __forceinline__ unsigned rowHash(int cy, int cz) {
  return ((unsigned)cy * 19349663u) ^ ((unsigned)cz * 83492791u);
}
// A row of cells, modulo 2^16 rows each way: among a sphere's nine rows no
// two are equal, so a candidate belongs to one of them at most, and one
// whose row lies 2^16 rows away is refused by the keep test.
__device__ __forceinline__ int rowKey(int cy, int cz) {
  return (int)(((unsigned)cy << 16) | ((unsigned)cz & 0xFFFFu));
}

__device__ __forceinline__ int cellCoord(double x, double cs) {
  double c = floor(x / cs);
  c = fmin(fmax(c, -1073741824.0), 1073741824.0);
  return (int)c;
}

__device__ __forceinline__ d3 ldPos(const double* p, int g) {
  return mk3(p[3 * g], p[3 * g + 1], p[3 * g + 2]);
}

// keep test of the pair {a, b}, evaluated in canonical order (min, max)
__device__ __forceinline__ bool keepPair(const CdArgs& a, int x, int y) {
  int lo = x < y ? x : y, hi = x < y ? y : x;
  int fl = a.family[lo], fh = a.family[hi];
  if (fl == fh && fl != -1) return false;
  d3 pA = ldPos(a.p, lo), pB = ldPos(a.p, hi);
  d3 gA = ldPos(a.geom, lo), gB = ldPos(a.geom, hi);
  return narrowphase(pA, gA, pB, gB, a.envelope, a.mode, (d3*)0, (double*)0, (d3*)0) != 0;
}

__device__ void insertionSort(int* x, int n) {
  for (int i = 1; i < n; ++i) {
    int v = x[i], j = i - 1;
    while (j >= 0 && x[j] > v) {
      x[j + 1] = x[j];
      --j;
    }
    x[j + 1] = v;
  }
}

__global__ __launch_bounds__(kT) void clearCells(unsigned* x, long n, int* counters) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0u;
  if (i < 8) counters[i] = 0;
}

// each small geometry's slot and its place there
__global__ __launch_bounds__(kT) void hashSmall(CdArgs a, unsigned* slotOf, unsigned* slotCount) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.nsmall) return;
  const d3 pg = ldPos(a.p, a.smallIds[t]);
  const unsigned s =
      (rowHash(cellCoord(pg.y, a.cs), cellCoord(pg.z, a.cs)) + (unsigned)cellCoord(pg.x, a.cs)) & a.mask;
  slotOf[2 * (size_t)t] = s;
  slotOf[2 * (size_t)t + 1] = atomicAdd(&slotCount[s], 1u);
}

__global__ __launch_bounds__(kT) void scatterSmall(CdArgs a, const unsigned* slotOf) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.nsmall) return;
  const int g = a.smallIds[t];
  const d3 pg = ldPos(a.p, g);
  const unsigned pos = a.slotStart[slotOf[2 * (size_t)t]] + slotOf[2 * (size_t)t + 1];
  a.posR[pos] = PosR{pg.x, pg.y, pg.z, a.geom[3 * (size_t)g]};
  a.meta[pos] = make_int4(g, rowKey(cellCoord(pg.y, a.cs), cellCoord(pg.z, a.cs)), a.family[g], 0);
}

// The same in one workgroup, the counts in LDS, for a table of up to kSortMost
// slots: clearing, hashing, two scan kernels and scattering are five launches
// of 3 to 5 us each, whatever the scene's size.  Collision detection of a step
// with the launches and so (and with the merged ones below): one sphere 66 and
// 40 us, 1,000 spheres 85 and 52, 4,000 78 and 67; with a larger table one
// workgroup takes longer than the launches: 8,001 spheres 96, against 77.
constexpr int kSortT = 1024;
constexpr int kSortMost = 8192;  // slots: 4,096 small geometries at most
__global__ __launch_bounds__(kSortT) void sortSmall(CdArgs a, unsigned* slotStart, int* counters) {
  constexpr int kPer = kSortMost / kSortT;       // slots of a thread
  constexpr int kOwn = kSortMost / 2 / kSortT;   // its geometries
  __shared__ unsigned count[kSortMost];
  __shared__ unsigned waveSums[kSortT / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int T = (int)a.mask + 1;
  for (int k = tid; k < T; k += kSortT) count[k] = 0;
  if (tid < 8) counters[tid] = 0;
  __syncthreads();
  int id[kOwn], key[kOwn];
  unsigned slot[kOwn], place[kOwn];
  d3 pos[kOwn];
#pragma unroll
  for (int q = 0; q < kOwn; ++q) {
    const int t = q * kSortT + tid;
    id[q] = t < a.nsmall ? a.smallIds[t] : -1;
    if (id[q] < 0) continue;
    pos[q] = ldPos(a.p, id[q]);
    const int cy = cellCoord(pos[q].y, a.cs), cz = cellCoord(pos[q].z, a.cs);
    slot[q] = (rowHash(cy, cz) + (unsigned)cellCoord(pos[q].x, a.cs)) & a.mask;
    key[q] = rowKey(cy, cz);
    place[q] = atomicAdd(&count[slot[q]], 1u);
  }
  __syncthreads();
  // exclusive scan: T / kSortT slots to a thread
  const int per = T / kSortT;
  unsigned sum = 0, v[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    v[q] = q < per ? count[tid * per + q] : 0u;
    sum += v[q];
  }
  unsigned x = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) waveSums[wave] = x;
  __syncthreads();
  unsigned at = x - sum;
#pragma unroll
  for (int w = 0; w < kSortT / 64; ++w) at += w < wave ? waveSums[w] : 0u;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    if (q >= per) continue;
    count[tid * per + q] = at;
    slotStart[tid * per + q] = at;
    at += v[q];
  }
  if (tid == kSortT - 1) slotStart[T] = at;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kOwn; ++q) {
    if (id[q] < 0) continue;
    const unsigned k = count[slot[q]] + place[q];
    a.posR[k] = PosR{pos[q].x, pos[q].y, pos[q].z, a.geom[3 * (size_t)id[q]]};
    a.meta[k] = make_int4(id[q], key[q], a.family[id[q]], 0);
  }
}

// The partners of small geometries, sixteen lanes to each: nine lanes walk a
// row of three cells, the others test the big list.  A candidate is refused
// by the squared distance first (with a margin far above the rounding of the
// exact test), so that few take the exact test's square root.  The partners
// are sorted by id and kept in lists[g * kList]; with kCsr (a sphere has more
// than kList) every geometry's partners go to csr[iStart[g]...] instead.
// Bound by latency at every size (dependent loads: the slots, then the
// candidates), so by the lanes in flight; one lane to a sphere walking 27
// cells one by one, twice, took 285 + 338 us at 112,000 spheres and 130 + 142
// at 8,000.
constexpr int kList = 24;
constexpr int kLanes = 16;
constexpr int kGroups = kT / kLanes;
template <bool kCsr>
__device__ void walkSmall(const CdArgs& a, int block, int* cntUp, int* cntDown, int* lists, int* over, const int* iStart,
                          int* csr) {
  __shared__ int found[kGroups], above[kGroups], ids[kGroups][kList];
  const int lane = threadIdx.x % kLanes, grp = threadIdx.x / kLanes;
  const int t = block * kGroups + grp;
  const bool on = t < a.nsmall;
  if (lane == 0) found[grp] = above[grp] = 0;
  __syncthreads();
  const int4 me = a.meta[on ? t : 0];
  const PosR pr = a.posR[on ? t : 0];
  const int g = me.x;
  int* const out = kCsr ? csr + (on ? iStart[g] : 0) : nullptr;
  auto keep = [&](int j) {
    const int k = atomicAdd(&found[grp], 1);
    if (j > g) atomicAdd(&above[grp], 1);
    if (kCsr) out[k] = j;
    else if (k < kList) ids[grp][k] = j;
  };
  if (on && lane < 9) {
    const int cx = cellCoord(pr.x, a.cs), cy = cellCoord(pr.y, a.cs) + lane % 3 - 1;
    const int cz = cellCoord(pr.z, a.cs) + lane / 3 - 1;
    const int key = rowKey(cy, cz);
    const unsigned first = (rowHash(cy, cz) + (unsigned)cx - 1u) & a.mask;
    // slots first .. first + 2, which may wrap round the table's end
    const unsigned T = a.mask + 1u, wrap = first + 3u > T ? first + 3u - T : 0u;
    unsigned k = a.slotStart[first], end = a.slotStart[first + 3u - wrap];
    for (int part = 0; part < (wrap ? 2 : 1); ++part) {
      if (part) {
        k = 0;
        end = a.slotStart[wrap];
      }
      for (; k < end; ++k) {
        const int4 m = a.meta[k];
        const PosR q = a.posR[k];
        if (m.y != key || m.x == g || (m.z == me.z && m.z != -1)) continue;
        const d3 d = mk3(q.x - pr.x, q.y - pr.y, q.z - pr.z);
        const double rr = pr.r + q.r, far = rr + a.envelope;
        if (!(dot3(d, d) <= far * far * 1.00001 + 1e-30)) continue;
        if (rr - lengthOf(d, a.mode) >= -a.envelope) keep(m.x);
      }
    }
  } else if (on) {
    for (int q = lane - 9; q < a.nbig; q += kLanes - 9) {
      const int b = a.bigIds[q];
      if (keepPair(a, g, b)) keep(b);
    }
  }
  __syncthreads();
  const int n = found[grp];
  if (!on) return;
  if (kCsr) {
    __threadfence_block();
    if (lane == 0) insertionSort(out, n);
    return;
  }
  if (lane == 0) {
    cntUp[g] = above[grp];
    cntDown[g] = n - above[grp];
    if (n > kList) {
      *over = 1;
      lists[(size_t)g * kList] = 0;  // not a big geometry's mark
    }
  }
  if (n > kList) return;
  for (int e = lane; e < n; e += kLanes) {
    const int id = ids[grp][e];
    int rank = 0;
    for (int f = 0; f < n; ++f) rank += ids[grp][f] < id ? 1 : 0;
    lists[(size_t)g * kList + rank] = id;
  }
}

__device__ int blockSum(int v) {
  __shared__ int red[kT / 64];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  int s = 0;
#pragma unroll
  for (int w = 0; w < kT / 64; ++w) s += red[w];
  __syncthreads();
  return s;
}

// Big geometries (boxes, large spheres) are paired with every geometry in
// chunks of kChunk partners: block (chunk, b) counts the kept partners of big
// geometry b in its chunk; a per-big scan over the chunks then gives each
// block its output offsets, so the emit pass writes the row in order.  Two
// rounds of a workgroup to a chunk: with eight, few workgroups each waited
// for eight rounds in turn (26 + 11 us at 112,000 spheres).  Past kChunksMany
// chunks there are workgroups enough, and eight rounds to a chunk keep the
// counts' memory, which grows with the square of the big geometries, small;
// past kChunksMost larger chunks keep their number an int.
constexpr int kChunk = 512, kChunkMany = 2048;
constexpr long kChunksMany = 1L << 20, kChunksMost = 1L << 30;
struct Chunks {
  int size, n;  // partners of a chunk, chunks of a big geometry
  int all;      // chunks of all of them
};
Chunks chunksOf(const CdArgs& a) {
  auto all = [&](int size) { return (long)a.nbig * blocksFor(a.nb, size); };
  Chunks c;
  c.size = all(kChunk) > kChunksMany ? kChunkMany : kChunk;
  while (all(c.size) > kChunksMost) c.size *= 2;
  c.n = blocksFor(a.nb, c.size);
  c.all = (int)all(c.size);
  return c;
}

// A workgroup to each of `items`, in launches of at most 2^31 threads (a
// dimension of a grid holds less than 2^32).
template <class Launch>
void launchItems(int items, const Launch& launch) {
  constexpr int kMost = 1 << 23;
  for (int first = 0; first < items; first += kMost) launch(first, dim3(std::min(kMost, items - first)));
}

__device__ void countBigChunk(const CdArgs& a, int q, int chunk, const Chunks& ch, int* chUp, int* chDown, int* cntUp,
                              int* cntDown) {
  const int b = a.bigIds[q];
  const int j0 = chunk * ch.size, j1 = min(a.nb, j0 + ch.size);
  int up = 0, down = 0;
  for (int j = j0 + threadIdx.x; j < j1; j += kT) {
    if (j == b) continue;
    if (keepPair(a, b, j)) {
      if (j > b) ++up; else ++down;
    }
  }
  up = blockSum(up);
  down = blockSum(down);
  if (threadIdx.x == 0) {
    const bool only = ch.n == 1;  // then there is nothing to scan
    chUp[q * ch.n + chunk] = only ? 0 : up;
    chDown[q * ch.n + chunk] = only ? 0 : down;
    if (only) {
      cntUp[b] = up;
      cntDown[b] = down;
    }
  }
}

// The walk of the small geometries in the first walkBlocks workgroups and the
// big ones' chunks in the others, which need nothing of each other.
__global__ __launch_bounds__(kT) void countPartners(CdArgs a, int first, int walkBlocks, Chunks ch, int* cntUp,
                                                    int* cntDown, int* lists, int* over, int* chUp, int* chDown) {
  const int w = first + (int)blockIdx.x;
  if (w < walkBlocks) {
    walkSmall<false>(a, w, cntUp, cntDown, lists, over, nullptr, nullptr);
  } else {
    const int k = w - walkBlocks;
    countBigChunk(a, k / ch.n, k % ch.n, ch, chUp, chDown, cntUp, cntDown);
  }
}
__global__ __launch_bounds__(kT) void listPartners(CdArgs a, int first, int* over, const int* iStart, int* csr) {
  walkSmall<true>(a, first + (int)blockIdx.x, nullptr, nullptr, nullptr, over, iStart, csr);
}

// per big geometry: exclusive scan of its chunk counts (in place) and totals,
// a wavefront to each
__global__ __launch_bounds__(64) void scanBigChunks(CdArgs a, int nchunks, int* chUp, int* chDown, int* cntUp,
                                                    int* cntDown) {
  const int q = blockIdx.x, lane = threadIdx.x;
  int baseUp = 0, baseDown = 0;
  for (int k0 = 0; k0 < nchunks; k0 += 64) {
    const int k = k0 + lane;
    const int at = q * nchunks + k;
    const int u = k < nchunks ? chUp[at] : 0, d = k < nchunks ? chDown[at] : 0;
    int su = u, sd = d;  // inclusive over the wavefront
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) {
      const int yu = __shfl_up(su, w, 64), yd = __shfl_up(sd, w, 64);
      if (lane >= w) { su += yu; sd += yd; }
    }
    if (k < nchunks) {
      chUp[at] = baseUp + su - u;
      chDown[at] = baseDown + sd - d;
    }
    baseUp += __shfl(su, 63, 64);
    baseDown += __shfl(sd, 63, 64);
  }
  if (lane == 0) {
    cntUp[a.bigIds[q]] = baseUp;
    cntDown[a.bigIds[q]] = baseDown;
  }
}

// Offsets of every body's contact row (cStart) and incidences (iStart), and
// the heavy bodies (more than kHeavyDegree incidences) in ascending order, so
// that everything summed over them is summed in a fixed order: one scan of
// three counts, tile sums and then the tiles, each workgroup of which adds up
// the tiles before its own (past kDirectTiles, scanBodyTiles does that for
// all; up to kCountTiles, the counts before it themselves, a launch less).  The totals go to the host's pinned memory as well.
constexpr int kBodyTile = 1024;
constexpr int kDirectTiles = 1024;
constexpr int kCountTiles = 8;
struct Counts3 {
  int up, all, heavy;
};
__device__ __forceinline__ Counts3 countsOf(const int* cntUp, const int* cntDown, int g, int nb) {
  if (g >= nb) return Counts3{0, 0, 0};
  const int u = cntUp[g], n = u + cntDown[g];
  return Counts3{u, n, n > kHeavyDegree ? 1 : 0};
}
__device__ __forceinline__ Counts3 add3c(const Counts3& a, const Counts3& b) {
  return Counts3{a.up + b.up, a.all + b.all, a.heavy + b.heavy};
}
__global__ __launch_bounds__(kT) void bodyTileSums(int nb, const int* cntUp, const int* cntDown, int* sums) {
  Counts3 s{0, 0, 0};
#pragma unroll
  for (int q = 0; q < kBodyTile / kT; ++q)
    s = add3c(s, countsOf(cntUp, cntDown, blockIdx.x * kBodyTile + q * kT + threadIdx.x, nb));
  const int u = blockSum(s.up), n = blockSum(s.all), h = blockSum(s.heavy);
  if (threadIdx.x == 0) {
    sums[3 * blockIdx.x] = u;
    sums[3 * blockIdx.x + 1] = n;
    sums[3 * blockIdx.x + 2] = h;
  }
}
// in-place exclusive scan of many tile sums by one workgroup
__global__ __launch_bounds__(64) void scanBodyTiles(int* sums, int tiles) {
  int base[3] = {0, 0, 0};
  for (int k0 = 0; k0 < tiles; k0 += 64) {
    const int k = k0 + (int)threadIdx.x;
    for (int c = 0; c < 3; ++c) {
      const int x = k < tiles ? sums[3 * (size_t)k + c] : 0;
      int y = x;
#pragma unroll
      for (int w = 1; w < 64; w <<= 1) {
        const int z = __shfl_up(y, w, 64);
        if ((int)threadIdx.x >= w) y += z;
      }
      if (k < tiles) sums[3 * (size_t)k + c] = base[c] + y - x;
      base[c] += __shfl(y, 63, 64);
    }
  }
}
__global__ __launch_bounds__(kT) void scanBodies(int nb, const int* cntUp, const int* cntDown, const int* sums,
                                                 int tiles, int* cStart, int* iStart, int* heavy, int* counters,
                                                 int* host) {
  __shared__ int waveUp[kT / 64], waveAll[kT / 64], waveHeavy[kT / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tile = blockIdx.x;
  Counts3 base{0, 0, 0};
  if (tiles <= kCountTiles) {
    Counts3 s{0, 0, 0};
    for (int g = threadIdx.x; g < tile * kBodyTile; g += kT) s = add3c(s, countsOf(cntUp, cntDown, g, nb));
    base = Counts3{blockSum(s.up), blockSum(s.all), blockSum(s.heavy)};
  } else if (tiles > kDirectTiles) {
    base = Counts3{sums[3 * (size_t)tile], sums[3 * (size_t)tile + 1], sums[3 * (size_t)tile + 2]};
  } else {
    Counts3 s{0, 0, 0};
    for (int k = threadIdx.x; k < tile; k += kT) s = add3c(s, Counts3{sums[3 * k], sums[3 * k + 1], sums[3 * k + 2]});
    base = Counts3{blockSum(s.up), blockSum(s.all), blockSum(s.heavy)};
  }
  constexpr int kPer = kBodyTile / kT;
  const int g0 = tile * kBodyTile + (int)threadIdx.x * kPer;
  Counts3 v[kPer], s{0, 0, 0};
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    v[q] = countsOf(cntUp, cntDown, g0 + q, nb);
    s = add3c(s, v[q]);
  }
  Counts3 x = s;  // inclusive over the wavefront
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) {
    const Counts3 y{__shfl_up(x.up, w, 64), __shfl_up(x.all, w, 64), __shfl_up(x.heavy, w, 64)};
    if (lane >= w) x = add3c(x, y);
  }
  if (lane == 63) {
    waveUp[wave] = x.up; waveAll[wave] = x.all; waveHeavy[wave] = x.heavy;
  }
  __syncthreads();
  Counts3 e = add3c(base, Counts3{x.up - s.up, x.all - s.all, x.heavy - s.heavy});
#pragma unroll
  for (int w = 0; w < kT / 64; ++w)
    if (w < wave) e = add3c(e, Counts3{waveUp[w], waveAll[w], waveHeavy[w]});
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int g = g0 + q;
    if (g < nb) {
      cStart[g] = e.up;
      iStart[g] = e.all;
      if (v[q].heavy) heavy[e.heavy] = g;
    }
    e = add3c(e, v[q]);
    if (g == nb - 1) {
      cStart[nb] = e.up;
      iStart[nb] = e.all;
      counters[2] = e.heavy;
      host[0] = e.up;
      host[1] = e.all;
      host[2] = counters[3];  // a sphere's partners exceed kList
    }
  }
}

struct EmitOut {
  int* cA;
  int* cB;
  double* frame;  // 9 SoA, stride cap
  double* gap;
  double* loc;    // 3 SoA, stride cap
  int cap;
  int* inc;
  int* posB;
  const int* lists;  // kList sorted partners per small geometry; a big geometry's first is -1
  const int* csr;    // or every geometry's, at iStart
  const int* cStart;
  const int* iStart;
  const int* cntUp;
  const int* cntDown;
};

__device__ __forceinline__ const int* listOf(const EmitOut& o, int g) {
  return o.csr ? o.csr + o.iStart[g] : o.lists + (size_t)g * kList;
}
__device__ __forceinline__ bool isBig(const EmitOut& o, int g) { return o.lists[(size_t)g * kList] < 0; }

// Contact c = (A, B) among the incidences of B, a small geometry: in the
// order of B's partners below it.
__device__ __forceinline__ void placeB(const EmitOut& o, int c, int A, int B) {
  const int* L = listOf(o, B);
  int lo = 0, hi = o.cntDown[B];
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (L[mid] < A) lo = mid + 1; else hi = mid;
  }
  const int i0 = o.iStart[B];
  o.inc[i0 + lo] = (c << 1) | 1;
  o.posB[c] = i0 - o.cStart[B] + lo;
}

__device__ __forceinline__ void writeRecord(const CdArgs& a, const EmitOut& o, int c, int A, int B) {
  d3 n, l;
  double w;
  narrowphase(ldPos(a.p, A), ldPos(a.geom, A), ldPos(a.p, B), ldPos(a.geom, B), a.envelope, a.mode,
              &n, &w, &l);
  d3 u, v;
  contactFrame(n, a.mode, &u, &v);
  const long S = o.cap;
  o.frame[0 * S + c] = n.x; o.frame[1 * S + c] = n.y; o.frame[2 * S + c] = n.z;
  o.frame[3 * S + c] = u.x; o.frame[4 * S + c] = u.y; o.frame[5 * S + c] = u.z;
  o.frame[6 * S + c] = v.x; o.frame[7 * S + c] = v.y; o.frame[8 * S + c] = v.z;
  o.gap[c] = w;
  o.loc[0 * S + c] = l.x; o.loc[1 * S + c] = l.y; o.loc[2 * S + c] = l.z;
  o.cA[c] = A;
  o.cB[c] = B;
}

// Rows of the small geometries, in id order and four lanes to each, so that a
// wavefront writes one run of contacts.
__device__ void emitSmall(const CdArgs& a, const EmitOut& o, int block) {
  const int t = (block * kT + (int)threadIdx.x) >> 2, lane = threadIdx.x & 3;
  if (t >= a.nsmall) return;
  const int g = a.smallIds[t];
  const int nu = o.cntUp[g], nd = o.cntDown[g], c0 = o.cStart[g], i0 = o.iStart[g];
  const int* L = listOf(o, g);
  for (int k = lane; k < nu; k += 4) {
    const int j = L[nd + k], c = c0 + k;
    writeRecord(a, o, c, g, j);
    o.inc[i0 + nd + k] = c << 1;
    if (!isBig(o, j)) placeB(o, c, g, j);
  }
}

// Contact c = (A, B) of a small geometry A with a big one B above it: A's
// contacts are its partners above it, in order.
__device__ __forceinline__ int contactWith(const EmitOut& o, int A, int B) {
  const int* L = listOf(o, A);
  const int nd = o.cntDown[A];
  int lo = nd, hi = nd + o.cntUp[A];
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (L[mid] < B) lo = mid + 1; else hi = mid;
  }
  return o.cStart[A] + lo - nd;
}

// big geometry rows: ordered stream compaction of each chunk's partners, and
// its incidences as body B (of big partners below it, ~id for now: placeBig)
__device__ void emitBigChunk(const CdArgs& a, const EmitOut& o, int q, int chunk, const Chunks& ch, const int* chUp,
                             const int* chDown) {
  const int b = a.bigIds[q];
  const int j0 = chunk * ch.size, j1 = min(a.nb, j0 + ch.size);
  __shared__ int baseUp, baseDown;
  if (threadIdx.x == 0) {
    baseUp = o.cStart[b] + chUp[q * ch.n + chunk];
    baseDown = o.iStart[b] + chDown[q * ch.n + chunk];
  }
  __syncthreads();
  __shared__ int wUp[kT / 64], wDown[kT / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int jb = j0; jb < j1; jb += kT) {
    const int j = jb + threadIdx.x;
    const bool kept = (j < j1 && j != b) ? keepPair(a, b, j) : false;
    const bool isUp = kept && j > b, isDown = kept && j < b;
    const unsigned long long mUp = __ballot(isUp), mDown = __ballot(isDown);
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int rUp = __popcll(mUp & below), rDown = __popcll(mDown & below);
    if (lane == 0) { wUp[wave] = __popcll(mUp); wDown[wave] = __popcll(mDown); }
    __syncthreads();
    int offUp = baseUp, offDown = baseDown, totUp = 0, totDown = 0;
#pragma unroll
    for (int w = 0; w < kT / 64; ++w) {
      if (w < wave) { offUp += wUp[w]; offDown += wDown[w]; }
      totUp += wUp[w];
      totDown += wDown[w];
    }
    if (isUp) {
      const int c = offUp + rUp;
      writeRecord(a, o, c, b, j);
      o.inc[o.iStart[b] + o.cntDown[b] + (c - o.cStart[b])] = c << 1;
      if (!isBig(o, j)) placeB(o, c, b, j);
    }
    if (isDown) {
      const int i = offDown + rDown;
      if (isBig(o, j)) {
        o.inc[i] = ~j;
      } else {
        const int c = contactWith(o, j, b);
        o.inc[i] = (c << 1) | 1;
        o.posB[c] = i - o.cStart[b];
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) { baseUp += totUp; baseDown += totDown; }
    __syncthreads();
  }
}

// All rows: the small geometries' in the first smallBlocks workgroups.
__global__ __launch_bounds__(kT) void emitContacts(CdArgs a, EmitOut o, int first, int smallBlocks, Chunks ch,
                                                   const int* chUp, const int* chDown) {
  const int w = first + (int)blockIdx.x;
  if (w < smallBlocks) {
    emitSmall(a, o, w);
  } else {
    const int k = w - smallBlocks;
    emitBigChunk(a, o, k / ch.n, k % ch.n, ch, chUp, chDown);
  }
}

// The incidences a big geometry has as body B with other big ones, from the
// ids left there, once the rows are written: the contact is found in the
// partner's row.  (Boxes never collide with each other.)
__global__ __launch_bounds__(kT) void placeBig(CdArgs a, EmitOut o) {
  const int b = a.bigIds[blockIdx.y];
  const int i0 = o.iStart[b], nd = o.cntDown[b];
  for (int q = blockIdx.x * kT + threadIdx.x; q < nd; q += gridDim.x * kT) {
    if (o.inc[i0 + q] >= 0) continue;
    const int j = ~o.inc[i0 + q];
    int lo = o.cStart[j], hi = lo + o.cntUp[j];
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (o.cB[mid] < b) lo = mid + 1; else hi = mid;
    }
    o.inc[i0 + q] = (lo << 1) | 1;
    o.posB[lo] = i0 - o.cStart[b] + q;
  }
}

__global__ void markBig(CdArgs a, int* lists) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < a.nbig) lists[(size_t)a.bigIds[q] * kList] = -1;
}

}  // namespace

namespace {

CdArgs cdArgs(Scene& s) {
  CdArgs a;
  a.p = s.p.p;
  a.geom = s.geom.p;
  a.family = s.family.p;
  a.smallIds = s.smallIds.p;
  a.bigIds = s.bigIds.p;
  a.nb = s.nb;
  a.nsmall = s.nsmall;
  a.nbig = s.nbig;
  a.cs = 2.0 * (s.cellSize + s.envelope);
  if (!(a.cs > 0)) a.cs = 1.0;
  a.envelope = s.envelope;
  a.mask = s.hashSize - 1;
  a.mode = s.geomMode;
  a.slotStart = s.slotStart.p;
  a.posR = reinterpret_cast<PosR*>(s.cellPosR.p);
  a.meta = reinterpret_cast<int4*>(s.cellMeta.p);
  return a;
}

}  // namespace

void collideInit(Scene& s) {
  // classify: spheres up to 4x the median radius of the caller's spheres are
  // hashed, the rest (boxes, large spheres) are tested against every
  // geometry; the shells' contact points (bodies from nUser on, spheres of
  // half the shell's thickness) are always hashed
  std::vector<double> radii;
  for (int i = 0; i < s.nUser; ++i)
    if (s.hGeom[3 * i + 1] == 0) radii.push_back(s.hGeom[3 * i]);
  double rmed = 0;
  if (!radii.empty()) {
    std::vector<double> tmp = radii;
    std::nth_element(tmp.begin(), tmp.begin() + tmp.size() / 2, tmp.end());
    rmed = tmp[tmp.size() / 2];
  }
  std::vector<int> small, big;
  double rmax = 0;
  for (int i = 0; i < s.nb; ++i) {
    bool sphere = s.hGeom[3 * i + 1] == 0;
    if (sphere && (i >= s.nUser || s.hGeom[3 * i] <= 4.0 * rmed)) {
      small.push_back(i);
      rmax = std::max(rmax, s.hGeom[3 * i]);
    } else {
      big.push_back(i);
    }
  }
  s.nsmall = (int)small.size();
  s.nbig = (int)big.size();
  s.bigPairs = false;
  for (int i : big) s.bigPairs = s.bigPairs || (s.nbig > 1 && s.hGeom[3 * i + 1] == 0);
  s.cellSize = rmax;  // scaled with the envelope at each step
  unsigned T = 1024;
  while (T < 2u * (unsigned)std::max(1, s.nsmall)) T <<= 1;
  s.hashSize = T;
  s.smallIds.reserve(std::max(1, s.nsmall));
  s.bigIds.reserve(std::max(1, s.nbig));
  if (s.nsmall)
    DV_HIP(hipMemcpyAsync(s.smallIds.p, small.data(), sizeof(int) * s.nsmall, hipMemcpyHostToDevice, s.stream));
  if (s.nbig)
    DV_HIP(hipMemcpyAsync(s.bigIds.p, big.data(), sizeof(int) * s.nbig, hipMemcpyHostToDevice, s.stream));
  s.slotOf.reserve(2 * (size_t)std::max(1, s.nsmall));
  s.slotCount.reserve(T);
  s.slotStart.reserve(T + 1);
  s.cellPosR.reserve(4 * (size_t)std::max(1, s.nsmall));
  s.cellMeta.reserve(4 * (size_t)std::max(1, s.nsmall));
  s.lists.reserve((size_t)kList * std::max(1, s.nb));
  s.cntUp.reserve(s.nb + 1);
  s.cntDown.reserve(s.nb + 1);
  s.cStart.reserve(s.nb + 1);
  s.iStart.reserve(s.nb + 1);
  s.counters.reserve(8);
  s.heavy.reserve(s.nb + 1);
  const CdArgs a = cdArgs(s);
  hipLaunchKernelGGL(markBig, dim3(blocksFor(s.nbig, 64)), dim3(64), 0, s.stream, a, s.lists.p);
  DV_HIP(hipStreamSynchronize(s.stream));
}

void collideCount(Scene& s) {
  const hipStream_t st = s.stream;
  const CdArgs a = cdArgs(s);
  const unsigned T = s.hashSize;

  if (T <= (unsigned)kSortMost) {
    hipLaunchKernelGGL(sortSmall, dim3(1), dim3(kSortT), 0, st, a, s.slotStart.p, s.counters.p);
  } else {
    hipLaunchKernelGGL(clearCells, dim3(blocksFor(T, kT)), dim3(kT), 0, st, s.slotCount.p, (long)T, s.counters.p);
    hipLaunchKernelGGL(hashSmall, dim3(blocksFor(s.nsmall, kT)), dim3(kT), 0, st, a, s.slotOf.p, s.slotCount.p);
    exclusiveScanU(s, s.slotCount.p, s.slotStart.p, (int)T);
    hipLaunchKernelGGL(scatterSmall, dim3(blocksFor(s.nsmall, kT)), dim3(kT), 0, st, a, (const unsigned*)s.slotOf.p);
  }
  const Chunks ch = chunksOf(a);
  s.bigChunks.reserve(2 * (size_t)std::max(1, ch.all));
  int* chUp = s.bigChunks.p;
  int* chDown = s.bigChunks.p + std::max(1, ch.all);
  const int walkBlocks = s.nsmall ? blocksFor(s.nsmall, kGroups) : 0;
  launchItems(walkBlocks + ch.all, [&](int first, dim3 grid) {
    hipLaunchKernelGGL(countPartners, grid, dim3(kT), 0, st, a, first, walkBlocks, ch, s.cntUp.p, s.cntDown.p,
                       s.lists.p, s.counters.p + 3, chUp, chDown);
  });
  if (s.nbig && ch.n > 1)
    hipLaunchKernelGGL(scanBigChunks, dim3(s.nbig), dim3(64), 0, st, a, ch.n, chUp, chDown, s.cntUp.p, s.cntDown.p);
  // contact rows and incidence offsets, heavy bodies, and the totals for the host
  const int tiles = blocksFor(s.nb, kBodyTile);
  s.scanTmp.reserve(3 * (size_t)tiles);
  s.pinned[0] = s.pinned[1] = s.pinned[2] = 0;  // (a scene without bodies)
  if (tiles > kCountTiles)
    hipLaunchKernelGGL(bodyTileSums, dim3(tiles), dim3(kT), 0, st, s.nb, (const int*)s.cntUp.p, (const int*)s.cntDown.p,
                       s.scanTmp.p);
  if (tiles > kDirectTiles) hipLaunchKernelGGL(scanBodyTiles, dim3(1), dim3(64), 0, st, s.scanTmp.p, tiles);
  hipLaunchKernelGGL(scanBodies, dim3(tiles), dim3(kT), 0, st, s.nb, (const int*)s.cntUp.p, (const int*)s.cntDown.p,
                     (const int*)s.scanTmp.p, tiles, s.cStart.p, s.iStart.p, s.heavy.p,
                     s.counters.p, s.pinned);
  DV_HIP(hipGetLastError());
}

void collideEmit(Scene& s) {
  const hipStream_t st = s.stream;
  const CdArgs a = cdArgs(s);
  const Chunks ch = chunksOf(a);
  int* chUp = s.bigChunks.p;
  int* chDown = s.bigChunks.p + std::max(1, ch.all);
  DV_HIP(hipStreamSynchronize(st));  // the counts of collideCount
  const int nc = s.pinned[0];
  const int ninc = s.pinned[1];
  if (nc < 0 || ninc < 0 || nc > kMaxContacts)
    throw DvError{DV_ERR_UNSUPPORTED, "more than 2^28 contacts in one scene"};
  if (ninc != 2 * nc) throw DvError{DV_ERR_STATE, "collision detection: asymmetric pair counts"};
  s.nc = nc;
  if (nc > s.ncCap || s.ncCap == 0) {
    int cap = std::max(1024, nc + nc / 4);
    s.cA.release(); s.cB.release(); s.frame.release(); s.gap.release(); s.loc.release();
    s.frame32.release(); s.inc.release(); s.posB.release();
    s.cA.reserve(cap); s.cB.reserve(cap);
    s.frame.reserve((size_t)9 * cap);
    s.gap.reserve(cap);
    s.loc.reserve((size_t)3 * cap);
    s.inc.reserve((size_t)2 * cap);
    s.posB.reserve(cap);
    s.ncCap = cap;
  }
  const bool csr = s.pinned[2] != 0;
  if (csr) {
    s.csr.reserve(std::max(1, ninc));
    launchItems(blocksFor(s.nsmall, kGroups), [&](int first, dim3 grid) {
      hipLaunchKernelGGL(listPartners, grid, dim3(kT), 0, st, a, first, s.counters.p + 3, (const int*)s.iStart.p,
                         s.csr.p);
    });
  }
  EmitOut o;
  o.cA = s.cA.p; o.cB = s.cB.p; o.frame = s.frame.p; o.gap = s.gap.p; o.loc = s.loc.p;
  o.cap = s.ncCap;
  o.inc = s.inc.p; o.posB = s.posB.p;
  o.lists = s.lists.p; o.csr = csr ? s.csr.p : nullptr;
  o.cStart = s.cStart.p; o.iStart = s.iStart.p; o.cntUp = s.cntUp.p; o.cntDown = s.cntDown.p;
  const int smallBlocks = s.nsmall ? blocksFor(4L * s.nsmall, kT) : 0;
  launchItems(smallBlocks + ch.all, [&](int first, dim3 grid) {
    hipLaunchKernelGGL(emitContacts, grid, dim3(kT), 0, st, a, o, first, smallBlocks, ch, (const int*)chUp,
                       (const int*)chDown);
  });
  if (s.bigPairs) hipLaunchKernelGGL(placeBig, dim3(16, s.nbig), dim3(kT), 0, st, a, o);
  DV_HIP(hipGetLastError());
}

void collide(Scene& s) {
  collideCount(s);
  collideEmit(s);
}

}  // namespace dv
