// fof_engine.hip -- Friends-of-Friends linking pipeline for gfx950.
//
// Replaces the reference's cell lists + serial sweep + ring merge
// (src_v2/FOF.c:44-161, Befriend :341-376) and computes what the host's
// retrieval / Checkhalo / Output_Halos loops (src_v2/FOF.c:188-203,
// :378-430, :797-847) derive from the ring.
//
// Pipeline (one launch per phase for all volumes of a batch):
//   1 k_pa_count     reference cell of every particle (src_v2/FOF.c:79-83),
//                    per-tile histograms of cell buckets
//   2 scan           (bucket, tile) offsets
//   3 k_pa_scatter, k_pb_scatter, k_pc_sort   one LDS-staged partition into
//                    fine buckets of 2^11 to 2^14 cells, or two (coarse
//                    buckets, then 256 fine ones in each), then a counting sort
//                    per fine bucket -> cell starts, dense-cell lists and
//                    float4 {x,y,z,index} in cell order
//                    (sparse addressing: composite keys, radix sort, cell list)
//   4 k_subsort      cells with >= max(T, 256) particles: counting sort by
//                    sub-cell; sub-cells have side <= l/sqrt(3), so each is a
//                    clique and its particles start in one union-find set
//                    ("runs")
//   5 k_link_sparse  one thread per particle of a sparse cell: own cell and
//                    the 13 forward cells (src_v2/FOF.c:112-153); with sparse
//                    addressing k_link_rows, a wave per 512 particles
//   6 k_link_dense   dense cells of 256 particles or more, each linked by
//                    one workgroup that took it from a queue: run pairs with
//                    early exit
//     k_link_small   dense cells below 256 particles, one wave each: every
//                    pair tested from LDS broadcasts, components by BFS over
//                    a bit matrix in registers
//   7 union-find finish: flatten, group minimum index, sizes
//   8 groups of two or more ranked by label through a label bitmap, each
//     given a segment of the member list; labels (written by index,
//     straight or through scatter_u32) while every member goes to its
//     group's segment; each segment sorted by index (a wave in registers,
//     or a workgroup)
//   9 ring in ascending index order (written the same way), halo list,
//     FP64 halo sums
//
// Pair rule (src_v2/FOF.c:351-357): dx = fl32(xi - xj) widened to double,
// distsq = (dx^2 + dy^2) + dz^2 in FP64, linked iff !(distsq > linksq).
// dx^2 is exact in FP64, so only the two additions round.  The FP32 test
// d2 = fma(dz,dz,fma(dy,dy,dx*dx)) has relative error < 2e-7; outside the
// band |d2/l2 - 1| >= band (>= 1e-6) it decides exactly as the FP64
// expression would, inside it the FP64 expression is evaluated as written.
#include <math.h>
#include <string.h>

#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "fof_internal.h"
#include "fof_pairwalk.h"

namespace fof {

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ int vol_of(const uint32_t *__restrict__ vbeg, int nvol,
                                      uint32_t p) {
  int lo = 0, hi = nvol - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (vbeg[mid] <= p) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Volume lookups for waves whose active lanes hold ascending elements (a
// grid-stride loop over 64-aligned runs, a tile, a label-sorted list): the
// volumes of the wave's first and last element are found with scalar loads,
// starting from the previous iteration's volume (hint, wave-uniform), and the
// lanes only search between them -- in a batch nearly every wave lies in one
// volume, and a cold binary search is six dependent loads.
__device__ __forceinline__ int vol_from(const uint32_t *__restrict__ vbeg, int nvol, uint32_t a,
                                        int hint) {
  if (vbeg[hint] <= a && a < vbeg[hint + 1]) return hint;
  return vol_of(vbeg, nvol, a);
}

__device__ __forceinline__ int vol_between(const uint32_t *__restrict__ vbeg, int nvol,
                                           uint32_t p, uint32_t a, uint32_t b, int &hint) {
  const int lo0 = vol_from(vbeg, nvol, a, hint);
  const int hi0 = (b < vbeg[lo0 + 1]) ? lo0 : vol_of(vbeg, nvol, b);
  hint = hi0;
  int lo = lo0, hi = hi0;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (vbeg[mid] <= p) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// lanes hold consecutive elements p (n elements in all)
__device__ __forceinline__ int vol_of_run(const uint32_t *__restrict__ vbeg, int nvol,
                                          uint32_t p, uint32_t n, int &hint) {
  if (nvol == 1) return 0;
  const uint32_t a = __builtin_amdgcn_readfirstlane(p);
  return vol_between(vbeg, nvol, p, a, min(a + 63u, n - 1u), hint);
}

// lanes hold ascending elements p
__device__ __forceinline__ int vol_of_sorted(const uint32_t *__restrict__ vbeg, int nvol,
                                             uint32_t p, int &hint) {
  if (nvol == 1) return 0;
  const uint32_t a = __builtin_amdgcn_readfirstlane(p);
  const int last = 63 - __clzll(__ballot(1));
  return vol_between(vbeg, nvol, p, a, __builtin_amdgcn_readlane(p, last), hint);
}

// Reference cell coordinate along one axis (src_v2/FOF.c:79-81), clamped.
__device__ __forceinline__ int cell1(double x, double rmin_buff, double lcell, int n,
                                     double *u) {
  double t = (x - rmin_buff) / lcell;
  *u = t;
  int i = (int)floor(t);
  return i < 0 ? 0 : (i >= n ? n - 1 : i);
}

struct CellPos {
  int ix, iy, iz;   // reference cell
  int fx, fy, fz;   // fine (sub-cell) coordinate = i*m + s
};

__device__ __forceinline__ int sub1(double u, int i, int m) {
  int s = (int)floor((u - (double)i) * (double)m);
  return s < 0 ? 0 : (s >= m ? m - 1 : s);
}

__device__ __forceinline__ CellPos cell_pos(const VolDev &V, float x, float y, float z) {
  CellPos c;
  double ux, uy, uz;
  c.ix = cell1((double)x, V.rmin_buff[0], V.lcell[0], V.nx, &ux);
  c.iy = cell1((double)y, V.rmin_buff[1], V.lcell[1], V.ny, &uy);
  c.iz = cell1((double)z, V.rmin_buff[2], V.lcell[2], V.nz, &uz);
  if (V.m[0] > 0) {
    c.fx = c.ix * V.m[0] + sub1(ux, c.ix, V.m[0]);
    c.fy = c.iy * V.m[1] + sub1(uy, c.iy, V.m[1]);
    c.fz = c.iz * V.m[2] + sub1(uz, c.iz, V.m[2]);
  } else {
    c.fx = c.ix, c.fy = c.iy, c.fz = c.iz;
  }
  return c;
}

// A float4 load rebuilt from its components: copies of the vector type
// itself into a private array keep the array in scratch memory.
__device__ __forceinline__ float4 ld4(const float4 *p) {
  const float4 v = *p;
  return make_float4(v.x, v.y, v.z, v.w);
}

// Fine (sub-cell) coordinates of a particle of a dense cell, 21 bits per axis,
// recorded once by k_subsort and read by the link kernels.
__device__ __forceinline__ unsigned long long pack_fine(int fx, int fy, int fz) {
  return (unsigned long long)fx | ((unsigned long long)fy << 21) | ((unsigned long long)fz << 42);
}
__device__ __forceinline__ int fine_x(unsigned long long f) { return (int)(f & 0x1FFFFFull); }
__device__ __forceinline__ int fine_y(unsigned long long f) { return (int)((f >> 21) & 0x1FFFFFull); }
__device__ __forceinline__ int fine_z(unsigned long long f) { return (int)((f >> 42) & 0x1FFFFFull); }

__device__ __forceinline__ uint32_t cell_id(const VolDev &V, int ix, int iy, int iz) {
  return V.cbeg + ((uint32_t)iz * (uint32_t)V.ny + (uint32_t)iy) * (uint32_t)V.nx +
         (uint32_t)ix;
}

// Cell addressing.  Dense: a table of cell starts over every cell of every
// volume (cell id = cbeg + linear index).  Sparse: only occupied cells, in
// (volume, linear index) order, listed with their composite keys
// (volume << volshift) | linear index and found by binary search.
struct Grid {
  const uint32_t *start;       // cell start offsets (+1 entry)
  const uint32_t *cell_of;     // sparse: cell of each sorted particle
  const uint32_t *klo, *khi;   // sparse: key of each cell
  const uint32_t *ncell;       // sparse: cells in the list
  const uint32_t *err;         // not 0: a particle lies outside its volume (see cell_of_xyz)
  int sparse;
  int volshift;
};

__device__ __forceinline__ unsigned long long comp_key(const Grid &G, const VolDev &V, int ix,
                                                       int iy, int iz) {
  return ((unsigned long long)V.vid << G.volshift) |
         (((unsigned long long)iz * (unsigned)V.ny + (unsigned)iy) * (unsigned)V.nx +
          (unsigned)ix);
}

__device__ __forceinline__ unsigned long long cell_key(const Grid &G, uint32_t c) {
  return (unsigned long long)G.klo[c] | ((unsigned long long)G.khi[c] << 32);
}

// First occupied cell with a key >= k.
__device__ __forceinline__ uint32_t cell_lower(const Grid &G, uint32_t U, unsigned long long k) {
  uint32_t lo = 0, hi = U;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (cell_key(G, mid) < k) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Cell index of (ix,iy,iz) (in range), kNone when a sparse cell is empty.
__device__ __forceinline__ uint32_t cell_index(const Grid &G, const VolDev &V, int ix, int iy,
                                               int iz) {
  if (!G.sparse) return cell_id(V, ix, iy, iz);
  const uint32_t U = *G.ncell;
  const unsigned long long k = comp_key(G, V, ix, iy, iz);
  const uint32_t c = cell_lower(G, U, k);
  return c < U && cell_key(G, c) == k ? c : kNone;
}

// Particle range covering cells (x0..x1, iy, iz) of a dense grid.
__device__ __forceinline__ void row_range(const Grid &G, const VolDev &V, int x0, int x1, int iy,
                                          int iz, uint32_t &r0, uint32_t &r1) {
  const uint32_t c0 = cell_id(V, x0, iy, iz);
  r0 = G.start[c0];
  r1 = G.start[c0 + (uint32_t)(x1 - x0) + 1];
}

// Squared linking length of a home cell: constant, or the variable rule
// (same operation order as the oracle; built with -ffp-contract=off).
__device__ __forceinline__ double cell_linksq(const VolDev &V, int ix, int iy, int iz) {
  if (V.vntab == 0) return V.linksq;
  double c0 = V.rmin_buff[0] + ((double)ix + 0.5) * V.lcell[0];
  double c1 = V.rmin_buff[1] + ((double)iy + 0.5) * V.lcell[1];
  double c2 = V.rmin_buff[2] + ((double)iz + 0.5) * V.lcell[2];
  double e0 = c0 - V.vorigin[0], e1 = c1 - V.vorigin[1], e2 = c2 - V.vorigin[2];
  double r2 = e0 * e0 + e1 * e1 + e2 * e2;
  double top = (double)(V.vntab - 1);
  double t = r2 / V.vr2max * top;
  if (!(t < top)) return V.vtab[V.vntab - 1];
  int k = (int)floor(t);
  double f = t - (double)k;
  return V.vtab[k] + f * (V.vtab[k + 1] - V.vtab[k]);
}

struct Rule {
  double linksq;  // FP64 threshold (src_v2/FOF.c:357)
  double prune2;  // squared sub-cell gap beyond which no pair can link
  float lo, hi;   // FP32 decision thresholds
};

__device__ __forceinline__ Rule make_rule(const VolDev &V, int ix, int iy, int iz) {
  Rule r;
  if (V.vntab == 0) {
    r.linksq = V.linksq;
    r.lo = V.lo;
    r.hi = V.hi;
  } else {
    r.linksq = cell_linksq(V, ix, iy, iz);
    r.lo = (float)(r.linksq * (1.0 - (double)V.band));
    r.hi = (float)(r.linksq * (1.0 + (double)V.band));
  }
  r.prune2 = r.linksq * (1.0 + 1e-4);
  return r;
}

// The reference's test in FP64 (src_v2/FOF.c:345-357): dx = fl32(xi - xj),
// distsq summed in double, linked unless distsq > linksq.
__device__ __forceinline__ bool pair_exact(float ax, float ay, float az, float bx, float by,
                                           float bz, double linksq) {
  const float dx = ax - bx, dy = ay - by, dz = az - bz;
  const double ex = dx, ey = dy, ez = dz;
  double ds = ex * ex + ey * ey;
  ds = ds + ez * ez;
  return !(ds > linksq);
}

// The reference predicate with the FP32 fast path.
__device__ __forceinline__ bool pair_linked(const float4 a, const float4 b, const Rule &r,
                                            uint32_t &nre) {
  const float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
  const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
  if (d2 < r.lo) return true;
  if (d2 > r.hi) return false;
  nre++;
  return pair_exact(a.x, a.y, a.z, b.x, b.y, b.z, r.linksq);
}

// Union-find on cell-sorted indices; roots are hooked larger-under-smaller,
// so every root is the smallest sorted index of its set and parent[x] <= x.
// Loads are agent-coherent (skip the non-coherent per-CU cache); a stale
// value can only be an older (larger) ancestor, so walks still terminate.
__device__ __forceinline__ uint32_t ld_par(uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_par(uint32_t *p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint32_t uf_find(uint32_t *par, uint32_t x) {
  uint32_t cur = ld_par(par + x);
  if (cur == x) return x;
  uint32_t prev = x, nxt;
  while (cur > (nxt = ld_par(par + cur))) {
    st_par(par + prev, nxt);  // path halving
    prev = cur;
    cur = nxt;
  }
  return cur;
}

// The roots of a and b, the two walks advancing together so that their
// loads overlap (path halving on both).
__device__ __forceinline__ void uf_find2(uint32_t *par, uint32_t &a, uint32_t &b) {
  uint32_t ca = ld_par(par + a), cb = ld_par(par + b);
  uint32_t qa = a, qb = b;
  bool fa = (ca == a), fb = (cb == b);
  while (!fa || !fb) {
    const uint32_t na = fa ? ca : ld_par(par + ca);
    const uint32_t nb = fb ? cb : ld_par(par + cb);
    if (!fa) {
      if (ca > na) st_par(par + qa, na), qa = ca, ca = na;
      else fa = true;
    }
    if (!fb) {
      if (cb > nb) st_par(par + qb, nb), qb = cb, cb = nb;
      else fb = true;
    }
  }
  a = ca, b = cb;
}

__device__ __forceinline__ void uf_union(uint32_t *par, uint32_t a, uint32_t b) {
  for (;;) {
    uf_find2(par, a, b);
    if (a == b) return;
    if (a > b) {
      uint32_t t = a;
      a = b;
      b = t;
    }
    uint32_t old = atomicCAS(par + b, b, a);
    if (old == b) return;
    b = old;
  }
}

// Join j to the set whose root (or an ancestor of it) is rx; returns the
// current root.  Skips the hook when j is already in the set.
__device__ __forceinline__ uint32_t uf_join(uint32_t *par, uint32_t rx, uint32_t j) {
  uint32_t b = uf_find(par, j);
  for (;;) {
    uint32_t a = uf_find(par, rx);
    if (a == b) return a;
    if (a > b) {
      const uint32_t t = a;
      a = b;
      b = t;
    }
    const uint32_t old = atomicCAS(par + b, b, a);
    if (old == b) return a;
    rx = a;
    b = uf_find(par, old);
  }
}

// LDS written by some lanes of a wave and read by others afterwards: the
// wave's LDS operations execute in order; this keeps the compiler from
// moving them across.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Statistics counters are spread over kCtrSlots copies, one 128-byte line
// each, picked by workgroup: a million waves adding to one address serialise
// at one L2 channel.  The host sums the copies.  Counter k of a slot:
constexpr int kCtrTestsSparse = 0;  // pair tests in k_link_sparse
constexpr int kCtrRechecks = 1;     // tests re-decided in FP64 (all kernels)
constexpr int kCtrGroups = 2;       // groups of any size
constexpr int kCtrOwned = 3;        // owned halos
constexpr int kCtrTestsBig = 4;     // pair tests in k_link_dense
constexpr int kCtrTestsSmall = 5;   // pair tests in k_link_small
constexpr int kCtrJoined = 6;       // candidate run pairs found already joined
constexpr int kCtrSlots = 64;
constexpr int kCtrStride = 16;  // u64 per slot
constexpr int kCtrWide = 8;     // of these the second half: listed pairs of long runs
__device__ __forceinline__ void ctr_add(unsigned long long *ctr, int k, unsigned long long v) {
  atomicAdd(ctr + (blockIdx.x & (kCtrSlots - 1)) * kCtrStride + k, v);
}

__device__ __forceinline__ void add_counters(unsigned long long *ctr, int ktests, uint32_t tests,
                                             uint32_t rechecks, uint32_t joined = 0) {
  uint64_t t = tests, r = rechecks, j = joined;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    t += __shfl_down(t, o, 64);
    r += __shfl_down(r, o, 64);
    j += __shfl_down(j, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    if (t) ctr_add(ctr, ktests, t);
    if (r) ctr_add(ctr, kCtrRechecks, r);
    if (j) ctr_add(ctr, kCtrJoined, j);
  }
}

// Device-side counts and flags of a call (u32 words of the `small` block);
// the counters follow at word kSmCtr.
constexpr int kSmErr = 0;       // bit 0: particle outside [rmin_buff, rmax_buff]
constexpr int kSmNDense = 1;    // dense cells below kBigCell particles
constexpr int kSmM = 2;         // members of groups of two or more (member list)
constexpr int kSmH = 3;         // halos
constexpr int kSmWide = 4;      // listed pairs of long runs (may pass kWideCap)
constexpr int kSmU = 5;         // occupied cells (sparse addressing)
constexpr int kSmNBig = 7;      // dense cells from kBigCell particles
constexpr int kSmR = 8;         // groups of two or more (their roots)
constexpr int kSmNtB = 10;      // tiles of the fine partition pass
constexpr int kSmDq = 11;       // next cell of k_link_dense's queue
constexpr int kSmCtr = 64;

// Dense cells with at least this many particles are linked by a workgroup each
// (of 256 to 1024 threads), smaller ones by a wave or a few of them.
constexpr uint32_t kBigCell = 256;

// ---------------------------------------------------------------------------
// 1-3 (dense grid): counting sort by cell without global atomics.
// Cells are grouped into fine buckets of 2^fb consecutive cells and, where
// there are more than kMaxBuckets of those, into coarse buckets of 256.
//   A: per tile of particles, cell keys and an LDS histogram of the (coarse)
//      buckets; scan; scatter {key}, {x,y,z,index} by bucket
//   B: (coarse buckets only) the same inside each coarse bucket, 256 ways
//   C: one workgroup per fine bucket: LDS counters for its 2^fb cells,
//      scan -> cell starts and dense-cell lists, LDS cursors -> cell order
// 256-way partitions keep a tile's open output lines few enough to be
// combined in L2; all counting is in LDS.
//
// Sizes: tiles of kPartTile particles and buckets of 2^14 cells at most;
// smaller calls shrink both (part_tile, fine_bits) until about 1024
// tiles and 256 buckets are in flight, since one workgroup's serial pass over
// 32768 particles is what a small call waits for (64^3 box, 11 tiles and 22
// buckets, passes A, B and C: 57 + 94, 35 + 44 and 35 us; now 7 + 8 and 15).
// Up to kMaxBuckets fine buckets pass A places them directly and pass B is
// not run: with the 1100 buckets of a 256^3 box 333 us for A's scatter, less
// than the two scatters' reads and writes take (and seven launches fewer),
// although a sub-tile then holds six particles a bucket.
//
// The scatters write a run per bucket and sub-tile, and C's writes are random
// inside its bucket; what bounds all three is lines that leave L2 partly
// written.  So a sub-tile is as much as LDS holds (kSub: 512^3 box, 2048
// particles 1.88 ms for A's scatter and 2.07 for B's, 4096 1.68 and 1.80, 7168
// 1.67 and 1.66; 256^3 box 444, 369 and 333 us), one workgroup of 1024 threads
// a compute unit.  With two levels a bucket is 2^12 cells where that leaves
// at most kMaxCoarse coarse buckets: passes A, B and C of the 512^3 box take
// 1.67 + 1.66 + 2.73 ms with 2^14 cells, 1.72 + 1.53 + 2.34 with 2^13, 1.85 +
// 1.52 + 2.12 with 2^12, 2.06 + 1.58 + 2.19 with 2^11.
// ---------------------------------------------------------------------------
constexpr uint32_t kSub = 7168;  // particles a partition kernel lays out in LDS at a time
constexpr uint32_t kPartTile = 5 * kSub;
constexpr int kFineBits = 14;  // of the largest fine buckets
constexpr uint32_t kFineCells = 1u << kFineBits;
constexpr int kMaxBuckets = 1280;  // of pass A
constexpr int kMaxCoarse = 1024;   // coarse buckets (C < 2^31 cells: at most 512 of 2^22)

static uint32_t part_tile(uint64_t N) {
  const uint64_t n = N / 1024;
  if (n >= kSub) return (uint32_t)std::min<uint64_t>(kPartTile, n / kSub * kSub);
  return (uint32_t)std::min<uint64_t>(kSub, std::max<uint64_t>(1, (n + 2047) / 2048) * 2048);
}
static int fine_bits(uint64_t C) {
  int fb = kFineBits;
  while (fb > 11 && (C >> fb) < 256) fb--;
  if ((C + (1u << fb) - 1) >> fb > (uint64_t)kMaxBuckets)  // two levels
    while (fb > 12 && (C + (1ull << (fb + 7)) - 1) >> (fb + 7) <= (uint64_t)kMaxCoarse) fb--;
  return fb;
}

__device__ __forceinline__ uint32_t cell_of_xyz(float x, float y, float z, const VolDev &V,
                                                uint32_t *__restrict__ err) {
  // src_v2/read_data.c:810-812 bounds; non-finite values are rejected too.
  // Such a particle is sorted as one of cell 0 while its coordinates say another
  // cell, or none: ranges, sub-cells and key order made from them would not
  // hold.  So a call with one lists no dense cell and links nothing (its
  // answer is FOF_E_DOMAIN).
  const bool ok = ((double)x >= V.rmin_buff[0]) && ((double)x <= V.rmax_buff[0]) &&
                  ((double)y >= V.rmin_buff[1]) && ((double)y <= V.rmax_buff[1]) &&
                  ((double)z >= V.rmin_buff[2]) && ((double)z <= V.rmax_buff[2]);
  if (!ok) atomicOr(err, 1u);
  double u;
  const int ix = ok ? cell1((double)x, V.rmin_buff[0], V.lcell[0], V.nx, &u) : 0;
  const int iy = ok ? cell1((double)y, V.rmin_buff[1], V.lcell[1], V.ny, &u) : 0;
  const int iz = ok ? cell1((double)z, V.rmin_buff[2], V.lcell[2], V.nz, &u) : 0;
  return cell_id(V, ix, iy, iz);
}

// A, count: keys, validation, hist[b * ntiles + tile] (bucket-major, so one
// exclusive scan gives each (bucket, tile) its first output slot), and the
// outputs' defaults (own label, own 1-based ring entry) where given.
__global__ __launch_bounds__(256) void k_pa_count(const uint8_t *__restrict__ base,
                                                  uint32_t stride, uint32_t offpos, uint32_t N,
                                                  const VolDev *__restrict__ vols,
                                                  const uint32_t *__restrict__ vbeg, int nvol,
                                                  uint32_t Bc, uint32_t ntiles,
                                                  uint32_t ptile, int shift,
                                                  uint32_t *__restrict__ key,
                                                  uint32_t *__restrict__ hist,
                                                  uint32_t *__restrict__ label_out,
                                                  uint32_t *__restrict__ next_out,
                                                  uint32_t *__restrict__ err) {
  __shared__ uint32_t h[kMaxBuckets];
  const uint32_t tile = blockIdx.x;
  for (uint32_t b = threadIdx.x; b < Bc; b += blockDim.x) h[b] = 0;
  __syncthreads();
  const uint32_t p0 = tile * ptile, p1 = min(N, p0 + ptile);
  int hint = 0;
  // kCnt records per thread loaded before any is used; the volume's
  // constants are read once per batch when the batch lies in one volume
  // (read per element, their loads were the pass's critical path: 11 ms
  // against 7.5 at 1024^3)
  constexpr int kCnt = 8;
  for (uint32_t q0 = p0; q0 < p1; q0 += kCnt * 256) {
    float x[kCnt], y[kCnt], z[kCnt];
#pragma unroll
    for (int k = 0; k < kCnt; k++) {
      const uint32_t p = min(q0 + threadIdx.x + k * 256, p1 - 1);
      const float *pp = reinterpret_cast<const float *>(base + (uint64_t)p * stride + offpos);
      x[k] = pp[0], y[k] = pp[1], z[k] = pp[2];
    }
    const uint32_t qe = min(q0 + kCnt * 256, p1) - 1;
    int va = 0;
    bool one = true;
    if (nvol > 1) {
      va = vol_from(vbeg, nvol, q0, hint);
      hint = va;
      one = qe < vbeg[va + 1];
    }
    uint32_t c[kCnt], b[kCnt];
    if (one) {
      const VolDev V = vols[va];
#pragma unroll
      for (int k = 0; k < kCnt; k++) b[k] = V.pbeg;
#pragma unroll
      for (int k = 0; k < kCnt; k++)
        c[k] = q0 + threadIdx.x + k * 256 < p1 ? cell_of_xyz(x[k], y[k], z[k], V, err) : 0u;
    } else {
#pragma unroll
      for (int k = 0; k < kCnt; k++) {
        const uint32_t p = q0 + threadIdx.x + k * 256;
        c[k] = b[k] = 0;
        if (p < p1) {
          const VolDev &V = vols[vol_of_run(vbeg, nvol, p, N, hint)];
          c[k] = cell_of_xyz(x[k], y[k], z[k], V, err);
          b[k] = V.pbeg;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kCnt; k++) {
      const uint32_t p = q0 + threadIdx.x + k * 256;
      if (p < p1) {
        key[p] = c[k];
        if (label_out) label_out[p] = p - b[k];
        if (next_out) next_out[p] = p - b[k] + 1u;
        atomicAdd(&h[c[k] >> shift], 1u);
      }
    }
  }
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < Bc; b += blockDim.x) hist[(uint64_t)b * ntiles + tile] = h[b];
}

// Partition scatter through LDS: a sub-tile of kSub elements is laid out in
// bucket order in LDS, then each bucket's elements leave as one contiguous
// run at the bucket's cursor.  cur[] holds the block's global cursors.
// 7168 elements (7 per thread) give each of 256 buckets 28 per flush,
// so that most output lines are complete before L2 evicts them.
constexpr int kPartNT = 1024;            // threads of the partition scatter kernels
constexpr int kPer = kSub / kPartNT;     // elements a thread holds per sub-tile

template <int NB>
__device__ __forceinline__ void staged_part(uint32_t nsub, const uint32_t (&kk)[kPer],
                                            const float4 (&pp)[kPer],
                                            int shift, uint32_t mask, uint32_t nbk,
                                            uint32_t *cur, uint32_t *lcnt, uint32_t *loff,
                                            uint32_t *skey, float4 *spos, uint32_t *ws,
                                            uint32_t *__restrict__ okey,
                                            float4 *__restrict__ opos) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t rank[kPer];
#pragma unroll
  for (int k = 0; k < kPer; k++)
    if (threadIdx.x + k * kPartNT < nsub)
      rank[k] = atomicAdd(&lcnt[(kk[k] >> shift) & mask], 1u);
  __syncthreads();
  // exclusive scan of lcnt over the buckets (kB consecutive per thread)
  constexpr int kB = (NB + kPartNT - 1) / kPartNT;
  uint32_t c[kB], loc = 0;
#pragma unroll
  for (int q = 0; q < kB; q++) {
    const uint32_t b = threadIdx.x * kB + q;
    c[q] = b < nbk ? lcnt[b] : 0u;
    loc += c[q];
  }
  uint32_t inc = loc;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) ws[w] = inc;
  __syncthreads();
  uint32_t pre = inc - loc;
  for (int q = 0; q < w; q++) pre += ws[q];
#pragma unroll
  for (int q = 0; q < kB; q++) {
    const uint32_t b = threadIdx.x * kB + q;
    if (b < nbk) loff[b] = pre;
    pre += c[q];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPer; k++)
    if (threadIdx.x + k * kPartNT < nsub) {
      const uint32_t j = loff[(kk[k] >> shift) & mask] + rank[k];
      skey[j] = kk[k];
      spos[j] = pp[k];
    }
  __syncthreads();
  for (uint32_t j = threadIdx.x; j < nsub; j += kPartNT) {
    const uint32_t key = skey[j], b = (key >> shift) & mask;
    const uint32_t g = cur[b] + (j - loff[b]);
    okey[g] = key;
    opos[g] = spos[j];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kB; q++) {
    const uint32_t b = threadIdx.x * kB + q;
    if (b < nbk) cur[b] += lcnt[b], lcnt[b] = 0;
  }
  __syncthreads();
}

// A, scatter: keys and {x,y,z,index} to the tile's slots of each of at most
// NB buckets.
__global__ __launch_bounds__(kPartNT) void k_pa_scatter(const uint8_t *__restrict__ base,
                                                    uint32_t stride, uint32_t offpos, uint32_t N,
                                                    uint32_t Bc, uint32_t ntiles,
                                                    uint32_t ptile, int shift,
                                                    const uint32_t *__restrict__ key,
                                                    const uint32_t *__restrict__ off,
                                                    uint32_t *__restrict__ okey,
                                                    float4 *__restrict__ opos) {
  constexpr int NB = kMaxBuckets;
  __shared__ uint32_t cur[NB], lcnt[NB], loff[NB];
  __shared__ uint32_t skey[kSub];
  __shared__ float4 spos[kSub];
  __shared__ uint32_t ws[kPartNT / 64];
  const uint32_t tile = blockIdx.x;
  for (uint32_t b = threadIdx.x; b < NB; b += blockDim.x) {
    cur[b] = b < Bc ? off[(uint64_t)b * ntiles + tile] : 0u;
    lcnt[b] = 0;
  }
  __syncthreads();
  const uint32_t p0 = tile * ptile, p1 = min(N, p0 + ptile);
  for (uint32_t q0 = p0; q0 < p1; q0 += kSub) {
    const uint32_t nsub = min(kSub, p1 - q0);
    uint32_t kk[kPer];
    float4 pp[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      const uint32_t i = threadIdx.x + k * kPartNT;
      if (i < nsub) {
        const uint32_t p = q0 + i;
        const uint32_t c = key[p];
        const float *fp = reinterpret_cast<const float *>(base + (uint64_t)p * stride + offpos);
        kk[k] = c;
        pp[k] = make_float4(fp[0], fp[1], fp[2], __uint_as_float(p));
      }
    }
    staged_part<NB>(nsub, kk, pp, shift, ~0u, Bc, cur, lcnt, loff, skey, spos, ws, okey, opos);
  }
}

// Coarse bucket starts (Bc + 1 entries) out of the scanned A histogram.
__global__ void k_pa_starts(uint32_t Bc, uint32_t ntiles, const uint32_t *__restrict__ off,
                            uint32_t *__restrict__ cstart) {
  for (uint32_t b = blockIdx.x * blockDim.x + threadIdx.x; b <= Bc; b += gridDim.x * blockDim.x)
    cstart[b] = off[(uint64_t)b * ntiles];
}

// B: tiles inside coarse buckets.  tinfo[t] = coarse bucket of tile t;
// t0[c] = first tile of bucket c (t0[Bc] = number of tiles, also left in
// *ntb).  Built on the device from the coarse bucket starts; the pass-B
// kernels are launched for the most tiles the buckets can need
// (ntiles_A + Bc) and the blocks past t0[Bc] do no work.
__global__ __launch_bounds__(kMaxCoarse) void k_pb_tiles(uint32_t Bc, uint32_t ntmax,
                                                         uint32_t ptile,
                                                         const uint32_t *__restrict__ cstart,
                                                         uint32_t *__restrict__ t0,
                                                         uint32_t *__restrict__ tinfo,
                                                         uint32_t *__restrict__ ntb) {
  __shared__ uint32_t ws[kMaxCoarse / 64];
  const uint32_t c = threadIdx.x, lane = c & 63, w = c >> 6;
  const uint32_t nt = c < Bc ? (cstart[c + 1] - cstart[c] + ptile - 1) / ptile : 0u;
  uint32_t inc = nt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) ws[w] = inc;
  __syncthreads();
  uint32_t pre = inc - nt, tot = 0;
  for (uint32_t q = 0; q < kMaxCoarse / 64; q++) {
    pre += q < w ? ws[q] : 0u;
    tot += ws[q];
  }
  if (c < Bc) {
    t0[c] = pre;
    for (uint32_t k = 0; k < nt; k++) tinfo[pre + k] = c;
  }
  if (c == 0) {
    t0[Bc] = tot;
    *ntb = tot;
  }
  for (uint32_t t = tot + c; t < ntmax; t += blockDim.x) tinfo[t] = kNone;
}
__device__ __forceinline__ void pb_tile(uint32_t t, uint32_t ptile,
                                        const uint32_t *__restrict__ tinfo,
                                        const uint32_t *__restrict__ t0,
                                        const uint32_t *__restrict__ cstart, uint32_t &c,
                                        uint32_t &i0, uint32_t &i1, uint32_t &nt, uint32_t &k) {
  c = tinfo[t];
  k = t - t0[c];
  nt = t0[c + 1] - t0[c];
  i0 = cstart[c] + k * ptile;
  i1 = min(cstart[c + 1], i0 + ptile);
}

__global__ __launch_bounds__(256) void k_pb_count(uint32_t ptile, int fb,
                                                  const uint32_t *__restrict__ tinfo,
                                                  const uint32_t *__restrict__ t0,
                                                  const uint32_t *__restrict__ cstart,
                                                  const uint32_t *__restrict__ ikey,
                                                  uint32_t *__restrict__ hist) {
  __shared__ uint32_t h[256];
  if (tinfo[blockIdx.x] == kNone) {  // past the last tile: zero its histogram slots
    hist[256ull * blockIdx.x + threadIdx.x] = 0;
    return;
  }
  uint32_t c, i0, i1, nt, k;
  pb_tile(blockIdx.x, ptile, tinfo, t0, cstart, c, i0, i1, nt, k);
  h[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t i = i0 + threadIdx.x; i < i1; i += blockDim.x)
    atomicAdd(&h[(ikey[i] >> fb) & 255u], 1u);
  __syncthreads();
  hist[256ull * t0[c] + (uint64_t)threadIdx.x * nt + k] = h[threadIdx.x];
}

__global__ __launch_bounds__(kPartNT) void k_pb_scatter(uint32_t ptile, int fb,
                                                    const uint32_t *__restrict__ tinfo,
                                                    const uint32_t *__restrict__ t0,
                                                    const uint32_t *__restrict__ cstart,
                                                    const uint32_t *__restrict__ off,
                                                    const uint32_t *__restrict__ ikey,
                                                    const float4 *__restrict__ ipos,
                                                    uint32_t *__restrict__ okey,
                                                    float4 *__restrict__ opos) {
  __shared__ uint32_t cur[256], lcnt[256], loff[256];
  __shared__ uint32_t skey[kSub];
  __shared__ float4 spos[kSub];
  __shared__ uint32_t ws[kPartNT / 64];
  if (tinfo[blockIdx.x] == kNone) return;  // past the last tile
  uint32_t c, i0, i1, nt, k;
  pb_tile(blockIdx.x, ptile, tinfo, t0, cstart, c, i0, i1, nt, k);
  for (uint32_t b = threadIdx.x; b < 256; b += kPartNT) {
    cur[b] = off[256ull * t0[c] + (uint64_t)b * nt + k];
    lcnt[b] = 0;
  }
  __syncthreads();
  for (uint32_t q0 = i0; q0 < i1; q0 += kSub) {
    const uint32_t nsub = min(kSub, i1 - q0);
    uint32_t kk[kPer];
    float4 pp[kPer];
#pragma unroll
    for (int q = 0; q < kPer; q++) {
      // loads clamped to the sub-tile (the extra elements are masked in
      // staged_part), so the arrays live in registers, not scratch
      const uint32_t i = min(threadIdx.x + q * kPartNT, nsub - 1);
      kk[q] = ikey[q0 + i];
      const float4 v = ipos[q0 + i];
      pp[q] = make_float4(v.x, v.y, v.z, v.w);
    }
    staged_part<256>(nsub, kk, pp, fb, 255u, 256, cur, lcnt, loff, skey, spos, ws, okey, opos);
  }
}

// Fine bucket starts (F + 1 entries).
__global__ void k_pb_starts(uint32_t F, const uint32_t *__restrict__ t0,
                            const uint32_t *__restrict__ cstart, const uint32_t *__restrict__ off,
                            uint32_t N, uint32_t *__restrict__ fstart) {
  for (uint32_t f = blockIdx.x * blockDim.x + threadIdx.x; f <= F; f += gridDim.x * blockDim.x) {
    if (f == F) {
      fstart[f] = N;
      continue;
    }
    const uint32_t c = f >> 8, sub = f & 255u, nt = t0[c + 1] - t0[c];
    fstart[f] = nt ? off[256ull * t0[c] + (uint64_t)sub * nt] : cstart[c];
  }
}

__device__ __forceinline__ int vol_of_cell(const VolDev *__restrict__ vols, int nvol, uint32_t c) {
  int lo = 0, hi = nvol - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (vols[mid].cbeg <= c) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// C: one workgroup per fine bucket, all counting in LDS.  The dense-cell
// lists are gathered per workgroup in LDS and appended with one atomic per
// list (per-wave appends to the two global counters were a third of the
// kernel's time); a workgroup whose lists outgrow LDS appends the rest per
// wave.
constexpr int kPcThreads = 1024;
constexpr uint32_t kPcListS = 1536, kPcListB = 512;

// The bucket's particles start at fstart[f * fstride].  Also each particle's
// union-find start (par, run_end, gsize).
__global__ __launch_bounds__(kPcThreads) void k_pc_sort(uint64_t C, int fb,
                                                 const uint32_t *__restrict__ fstart,
                                                 uint32_t fstride,
                                                 const uint32_t *__restrict__ ikey,
                                                 const float4 *__restrict__ ipos,
                                                 uint32_t *__restrict__ start,
                                                 float4 *__restrict__ pos4,
                                                 const VolDev *__restrict__ vols, int nvol,
                                                 const uint32_t *__restrict__ err,
                                                 uint32_t T, uint32_t *__restrict__ dense,
                                                 uint32_t *__restrict__ ndense,
                                                 uint32_t *__restrict__ dbig,
                                                 uint32_t *__restrict__ nbig,
                                                 uint32_t *__restrict__ par,
                                                 uint32_t *__restrict__ run_end,
                                                 uint32_t *__restrict__ gsize) {
  // counters padded by one word per 64 so that the per-thread segments of
  // the scan fall in different LDS banks
  __shared__ uint32_t lc[kFineCells + kFineCells / 64 + 1];
  auto P = [](uint32_t e) { return e + (e >> 6); };
  __shared__ uint32_t ws[kPcThreads / 64];
  __shared__ uint32_t lsml[kPcListS], lbig[kPcListB];
  // entries reserved, first reservation that did not fit, global bases
  __shared__ uint32_t nres[2], nfit[2], gbase[2];
  if (*err) T = kNone;  // no cell is dense
  const uint32_t f = blockIdx.x;
  const uint32_t q0 = fstart[(uint64_t)f * fstride], q1 = fstart[(uint64_t)(f + 1) * fstride];
  const uint64_t c0 = (uint64_t)f << fb;
  const uint32_t cells = 1u << fb;
  const uint32_t nc = (uint32_t)min((uint64_t)cells, C - c0);
  for (uint32_t e = threadIdx.x; e < cells + cells / 64 + 1; e += blockDim.x) lc[e] = 0;
  if (threadIdx.x < 2) nres[threadIdx.x] = 0, nfit[threadIdx.x] = threadIdx.x ? kPcListB : kPcListS;
  __syncthreads();
  for (uint32_t i = q0 + threadIdx.x; i < q1; i += blockDim.x)
    atomicAdd(&lc[P(ikey[i] & (cells - 1))], 1u);
  __syncthreads();
  // exclusive scan of the 2^fb counters: kPer consecutive per thread
  const uint32_t kPer = cells / kPcThreads;
  const uint32_t e0 = threadIdx.x * kPer;
  uint32_t loc = 0;
  for (uint32_t q = 0; q < kPer; q++) loc += lc[P(e0 + q)];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t inc = loc;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) ws[w] = inc;
  __syncthreads();
  uint32_t pre = inc - loc;
  for (int q = 0; q < w; q++) pre += ws[q];
  for (uint32_t q = 0; q < kPer; q++) {
    const uint32_t v = lc[P(e0 + q)];
    lc[P(e0 + q)] = pre;
    pre += v;
  }
  if (threadIdx.x == kPcThreads - 1) lc[P(cells)] = pre;  // bucket total
  __syncthreads();
  // one wave's dense cells of one kind: into the LDS list while it fits
  // (the fitting reservations are a prefix of the list), else appended
  auto append = [&](int kind, bool mine, uint32_t cell) {
    const unsigned long long bal = __ballot(mine);
    if (!bal) return;
    const uint32_t cnt = (uint32_t)__popcll(bal), below = (uint32_t)__popcll(bal & ((1ull << lane) - 1));
    const uint32_t cap = kind ? kPcListB : kPcListS;
    uint32_t base = 0;
    if (lane == 0) {
      base = atomicAdd(&nres[kind], cnt);
      if (base + cnt > cap) {
        atomicMin(&nfit[kind], base);
        base = 0x80000000u | atomicAdd(kind ? nbig : ndense, cnt);
      }
    }
    base = __shfl(base, 0, 64);
    if (!mine) return;
    if (base & 0x80000000u) (kind ? dbig : dense)[(base & 0x7FFFFFFFu) + below] = cell;
    else (kind ? lbig : lsml)[base + below] = cell;
  };
  // cell starts (coalesced) and the dense-cell lists
  for (uint32_t e0 = threadIdx.x & ~63u; e0 < nc; e0 += blockDim.x) {
    const uint32_t e = e0 + lane;
    bool sml = false, big = false;
    if (e < nc) {
      const uint32_t s = lc[P(e)], n = lc[P(e + 1)] - s;
      start[c0 + e] = q0 + s;
      if (n >= T) {  // dense: below kBigCell always, from it only with sub-cells
        sml = n < kBigCell;
        big = !sml && vols[vol_of_cell(vols, nvol, (uint32_t)(c0 + e))].m[0] > 0;
      }
    }
    append(0, sml, (uint32_t)(c0 + e));
    append(1, big, (uint32_t)(c0 + e));
  }
  if (c0 + nc == C && threadIdx.x == 0) start[C] = q1;
  __syncthreads();
  if (threadIdx.x < 2) {
    const uint32_t k = threadIdx.x, m = min(nres[k], nfit[k]);
    nfit[k] = m;
    gbase[k] = m ? atomicAdd(k ? nbig : ndense, m) : 0u;
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < nfit[0]; k += blockDim.x) dense[gbase[0] + k] = lsml[k];
  for (uint32_t k = threadIdx.x; k < nfit[1]; k += blockDim.x) dbig[gbase[1] + k] = lbig[k];
  // scatter with LDS cursors
  for (uint32_t i = q0 + threadIdx.x; i < q1; i += blockDim.x) {
    const uint32_t slot = q0 + atomicAdd(&lc[P(ikey[i] & (cells - 1))], 1u);
    pos4[slot] = ipos[i];
    par[i] = i;
    run_end[i] = i + 1;
    gsize[i] = 0;
  }
}

// 1-3 (sparse addressing): composite keys, sorted, occupied cells.
__global__ __launch_bounds__(256) void k_keys_sparse(const uint8_t *__restrict__ base,
                                                     uint32_t stride, uint32_t offpos, uint32_t N,
                                                     const VolDev *__restrict__ vols,
                                                     const uint32_t *__restrict__ vbeg, int nvol,
                                                     Grid G, uint32_t *__restrict__ klo,
                                                     uint32_t *__restrict__ khi,
                                                     uint32_t *__restrict__ val,
                                                     uint32_t *__restrict__ label_out,
                                                     uint32_t *__restrict__ next_out,
                                                     uint32_t *__restrict__ err) {
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < N;
       p += gridDim.x * blockDim.x) {
    const VolDev &V = vols[vol_of(vbeg, nvol, p)];
    const float *pp = reinterpret_cast<const float *>(base + (uint64_t)p * stride + offpos);
    const float x = pp[0], y = pp[1], z = pp[2];
    const bool ok = ((double)x >= V.rmin_buff[0]) && ((double)x <= V.rmax_buff[0]) &&
                    ((double)y >= V.rmin_buff[1]) && ((double)y <= V.rmax_buff[1]) &&
                    ((double)z >= V.rmin_buff[2]) && ((double)z <= V.rmax_buff[2]);
    if (!ok) atomicOr(err, 1u);
    double u;
    const int ix = ok ? cell1((double)x, V.rmin_buff[0], V.lcell[0], V.nx, &u) : 0;
    const int iy = ok ? cell1((double)y, V.rmin_buff[1], V.lcell[1], V.ny, &u) : 0;
    const int iz = ok ? cell1((double)z, V.rmin_buff[2], V.lcell[2], V.nz, &u) : 0;
    const unsigned long long k = comp_key(G, V, ix, iy, iz);
    klo[p] = (uint32_t)k;
    khi[p] = (uint32_t)(k >> 32);
    val[p] = p;
    if (label_out) label_out[p] = p - V.pbeg;
    if (next_out) next_out[p] = p - V.pbeg + 1u;
  }
}

__global__ __launch_bounds__(256) void k_gather_u32(uint32_t N, const uint32_t *__restrict__ src,
                                                    const uint32_t *__restrict__ idx,
                                                    uint32_t *__restrict__ dst) {
  for (uint32_t x = blockIdx.x * blockDim.x + threadIdx.x; x < N; x += gridDim.x * blockDim.x)
    dst[x] = src[idx[x]];
}

__global__ __launch_bounds__(256) void k_scatter_sparse(const uint8_t *__restrict__ base,
                                                        uint32_t stride, uint32_t offpos,
                                                        uint32_t N, const uint32_t *__restrict__ perm,
                                                        const VolDev *__restrict__ vols,
                                                        const uint32_t *__restrict__ vbeg,
                                                        int nvol, Grid G,
                                                        float4 *__restrict__ pos4,
                                                        uint32_t *__restrict__ sklo,
                                                        uint32_t *__restrict__ skhi) {
  for (uint32_t x = blockIdx.x * blockDim.x + threadIdx.x; x < N;
       x += gridDim.x * blockDim.x) {
    const uint32_t p = perm[x];
    const float *pp = reinterpret_cast<const float *>(base + (uint64_t)p * stride + offpos);
    const float4 q = make_float4(pp[0], pp[1], pp[2], __uint_as_float(p));
    pos4[x] = q;
    const VolDev &V = vols[vol_of(vbeg, nvol, p)];
    const CellPos c = cell_pos(V, q.x, q.y, q.z);
    const unsigned long long k = comp_key(G, V, c.ix, c.iy, c.iz);
    sklo[x] = (uint32_t)k;
    skhi[x] = (uint32_t)(k >> 32);
  }
}

__global__ __launch_bounds__(256) void k_cell_flags(uint32_t N, const uint32_t *__restrict__ sklo,
                                                    const uint32_t *__restrict__ skhi,
                                                    uint32_t *__restrict__ flags) {
  for (uint32_t x = blockIdx.x * blockDim.x + threadIdx.x; x < N;
       x += gridDim.x * blockDim.x)
    flags[x] = (x == 0 || sklo[x] != sklo[x - 1] || skhi[x] != skhi[x - 1]) ? kFlag : 0u;
}

// Per occupied cell: close the start list, record the cell's key, list dense
// cells.  (Each particle's cell comes with the list; the dense cells' 26
// neighbours are found by binary search over the keys.  Writing the former
// here, one thread to a cell's particles, inserting the keys into a hash table
// for the latter and appending to the lists wave by wave took 1.0 ms for the
// 9.8e6 cells of a lightcone.)
constexpr uint32_t kCellTile = 4096;  // cells of a block: two appends a block at most

__global__ __launch_bounds__(256) void k_cells_finish(
    const uint32_t *__restrict__ dU, uint32_t N, uint32_t *__restrict__ cstart,
    const uint32_t *__restrict__ sklo, const uint32_t *__restrict__ skhi,
    uint32_t *__restrict__ klo, uint32_t *__restrict__ khi,
    const VolDev *__restrict__ vols,
    const uint32_t *__restrict__ vbeg, int nvol, const uint32_t *__restrict__ err, uint32_t T,
    uint32_t *__restrict__ dense, uint32_t *__restrict__ ndense, uint32_t *__restrict__ dbig,
    uint32_t *__restrict__ nbig) {
  // the tile's dense cells: the small ones from the front, the others from the back
  __shared__ uint16_t lst[kCellTile];
  __shared__ uint32_t cnt[2], base[2];
  const uint32_t U = *dU;
  const uint64_t t0 = (uint64_t)blockIdx.x * kCellTile;
  if (t0 >= U) return;
  if (*err) T = kNone;  // no cell is dense
  if (threadIdx.x < 2) cnt[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < kCellTile && t0 + q < U; q += 256) {
    const uint32_t c = (uint32_t)t0 + q;
    const uint32_t s = cstart[c], e = (c + 1 < U) ? cstart[c + 1] : N;
    if (c + 1 == U) cstart[U] = N;
    klo[c] = sklo[s], khi[c] = skhi[s];
    if (e - s < T) continue;
    // dense: below kBigCell always, from it only with sub-cells
    if (e - s < kBigCell) lst[atomicAdd(&cnt[0], 1u)] = (uint16_t)q;
    else if (vols[vol_of(vbeg, nvol, s)].m[0] > 0)
      lst[kCellTile - 1 - atomicAdd(&cnt[1], 1u)] = (uint16_t)q;
  }
  __syncthreads();
  if (threadIdx.x < 2 && cnt[threadIdx.x])
    base[threadIdx.x] = atomicAdd(threadIdx.x ? nbig : ndense, cnt[threadIdx.x]);
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < cnt[0]; k += 256) dense[base[0] + k] = (uint32_t)t0 + lst[k];
  for (uint32_t k = threadIdx.x; k < cnt[1]; k += 256)
    dbig[base[1] + k] = (uint32_t)t0 + lst[kCellTile - 1 - k];
}

__global__ __launch_bounds__(256) void k_init_uf(uint32_t N, uint32_t *__restrict__ par,
                                                 uint32_t *__restrict__ run_end) {
  for (uint32_t x = blockIdx.x * blockDim.x + threadIdx.x; x < N;
       x += gridDim.x * blockDim.x) {
    par[x] = x;
    run_end[x] = x + 1;
  }
}

// ---------------------------------------------------------------------------
// 4: sub-cell counting sort of dense cells; runs become cliques.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int sub_bin(const VolDev &V, const float4 p) {
  double ux, uy, uz;
  const int ix = cell1((double)p.x, V.rmin_buff[0], V.lcell[0], V.nx, &ux);
  const int iy = cell1((double)p.y, V.rmin_buff[1], V.lcell[1], V.ny, &uy);
  const int iz = cell1((double)p.z, V.rmin_buff[2], V.lcell[2], V.nz, &uz);
  return (sub1(uz, iz, V.m[2]) * V.m[1] + sub1(uy, iy, V.m[1])) * V.m[0] + sub1(ux, ix, V.m[0]);
}

// Sub-cell counting sort, one workgroup of NT threads per dense cell of the
// list (cells of 256 particles or more; smaller dense cells stay unsorted:
// k_link_small tests all their pairs).
constexpr int kMaxCellBins = 12 * 12 * 12;  // m <= 12 per axis

template <int NT>
__global__ __launch_bounds__(NT) void k_subsort(const uint32_t *__restrict__ dense,
                                                const uint32_t *__restrict__ ndense,
                                                const uint32_t *__restrict__ start,
                                                const VolDev *__restrict__ vols,
                                                const uint32_t *__restrict__ vbeg, int nvol,
                                                float4 *__restrict__ pos4,
                                                float4 *__restrict__ tmp4,
                                                uint32_t *__restrict__ par,
                                                uint32_t *__restrict__ run_end,
                                                unsigned long long *__restrict__ fine,
                                                uint32_t *__restrict__ rtoff,
                                                uint32_t *__restrict__ rtab) {
  constexpr int kWaves = NT / 64;
  constexpr int kPer = (kMaxCellBins + NT - 1) / NT;  // bins per thread in the scans
  __shared__ uint32_t bcur[kMaxCellBins];    // cursors
  __shared__ uint32_t bstart[kMaxCellBins];  // run starts
  __shared__ uint32_t ws[kWaves];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // block-wide exclusive scan of one value per thread; returns (prefix, total)
  auto block_scan = [&](uint32_t loc, uint32_t &tot) -> uint32_t {
    uint32_t inc = loc;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    uint32_t off = 0;
    tot = 0;
#pragma unroll
    for (int q = 0; q < kWaves; q++) {
      off += (q < w) ? ws[q] : 0u;
      tot += ws[q];
    }
    return off + inc - loc;
  };
  const uint32_t nd = *ndense;
  for (uint32_t d = blockIdx.x; d < nd; d += gridDim.x) {
    const uint32_t c = dense[d];
    const uint32_t s = start[c], e = start[c + 1], n = e - s;
    const VolDev &V = vols[vol_of(vbeg, nvol, s)];
    if (V.m[0] == 0) continue;  // no sub-cells in this volume (uniform per block)
    const int nbins = V.m[0] * V.m[1] * V.m[2];
    for (int b = threadIdx.x; b < kMaxCellBins; b += NT) bcur[b] = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += NT) atomicAdd(&bcur[sub_bin(V, pos4[s + i])], 1u);
    __syncthreads();
    // exclusive scan of the counts -> starts and cursors (kPer bins a thread)
    {
      const int b0 = threadIdx.x * kPer;
      uint32_t loc = 0, tot;
      for (int q = 0; q < kPer; q++)
        if (b0 + q < nbins) loc += bcur[b0 + q];
      uint32_t pre = block_scan(loc, tot);
      for (int q = 0; q < kPer; q++)
        if (b0 + q < nbins) {
          const uint32_t cc = bcur[b0 + q];
          bstart[b0 + q] = pre;
          bcur[b0 + q] = pre;
          pre += cc;
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += NT) {
      const float4 p = pos4[s + i];
      tmp4[s + atomicAdd(&bcur[sub_bin(V, p)], 1u)] = p;
    }
    __syncthreads();
    // run table of the cell: heads in sub-cell order at rtab[s ..), their
    // number at rtoff[s] (a cell has at most as many runs as particles)
    {
      const int b0 = threadIdx.x * kPer;
      uint32_t loc = 0, tot;
      for (int q = 0; q < kPer; q++)
        if (b0 + q < nbins && bcur[b0 + q] != bstart[b0 + q]) loc++;
      const uint32_t pre = block_scan(loc, tot);
      if (threadIdx.x == 0) rtoff[s] = tot;
      uint32_t r = s + pre;
      for (int q = 0; q < kPer; q++)
        if (b0 + q < nbins && bcur[b0 + q] != bstart[b0 + q]) rtab[r++] = s + bstart[b0 + q];
    }
    for (uint32_t i = threadIdx.x; i < n; i += NT) {
      const float4 p = tmp4[s + i];
      const CellPos cp = cell_pos(V, p.x, p.y, p.z);
      const int b = ((cp.fz - cp.iz * V.m[2]) * V.m[1] + (cp.fy - cp.iy * V.m[1])) * V.m[0] +
                    (cp.fx - cp.ix * V.m[0]);
      pos4[s + i] = p;
      par[s + i] = s + bstart[b];
      run_end[s + i] = s + bcur[b];
      fine[s + i] = pack_fine(cp.fx, cp.fy, cp.fz);
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// 5: sparse cells -- one thread per particle.
// ---------------------------------------------------------------------------
// A particle against the particles j .. je - 1, each joined where it links.  rx:
// the particle's root, refreshed by every join.
__device__ __forceinline__ void scan_range(const float4 px, const Rule &R, uint32_t j, uint32_t je,
                                           const float4 *__restrict__ pos4,
                                           uint32_t *__restrict__ par, uint32_t &rx,
                                           uint32_t &tests, uint32_t &rechecks) {
  for (; j + 4 <= je; j += 4) {
    float4 q[4];
#pragma unroll
    for (int k = 0; k < 4; k++) q[k] = ld4(pos4 + j + k);
    uint32_t hit = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) hit |= pair_linked(px, q[k], R, rechecks) ? (1u << k) : 0u;
    tests += 4;
    while (hit) {
      const int k = __builtin_ctz(hit);
      hit &= hit - 1;
      rx = uf_join(par, rx, j + k);
    }
  }
  for (; j < je; j++) {
    tests++;
    if (pair_linked(px, pos4[j], R, rechecks)) rx = uf_join(par, rx, j);
  }
}

// A particle against the particle ranges r0[k] .. r1[k) of its forward
// neighbours where dense cells are scanned run by run (sub-sorted cells) or
// particle by particle.
__device__ __forceinline__ void scan_rows(const float4 px, const CellPos &cp, const VolDev &V,
                                          const Rule &R, const uint32_t (&r0)[5],
                                          const uint32_t (&r1)[5], int nr, uint32_t T,
                                          const float4 *__restrict__ pos4,
                                          const uint32_t *__restrict__ run_end,
                                          const unsigned long long *__restrict__ fine,
                                          uint32_t *__restrict__ par, uint32_t &rx,
                                          uint32_t &tests, uint32_t &rechecks) {
  const bool subcells = V.m[0] > 0;
  for (int r = 0; r < nr; r++) {
    uint32_t j = r0[r];
    const uint32_t je = r1[r];
    if (!subcells || je - j < T) {
      // fewer than T particles: no dense cell here, every particle is a run
      scan_range(px, R, j, je, pos4, par, rx, tests, rechecks);
      continue;
    }
    while (j < je) {
      const uint32_t re = run_end[j];
      if (re == j + 1) {
        tests++;
        if (pair_linked(px, pos4[j], R, rechecks)) rx = uf_join(par, rx, j);
        j++;
        continue;
      }
      // a clique run of a dense cell: skip it when out of reach or joined
      const unsigned long long fj = fine[j];
      const int gx = max(abs(fine_x(fj) - cp.fx) - 1, 0);
      const int gy = max(abs(fine_y(fj) - cp.fy) - 1, 0);
      const int gz = max(abs(fine_z(fj) - cp.fz) - 1, 0);
      const double g2 = (double)(gx * gx) * V.s2[0] + (double)(gy * gy) * V.s2[1] +
                        (double)(gz * gz) * V.s2[2];
      if (!(g2 > R.prune2) && uf_find(par, rx) != uf_find(par, j)) {
        for (uint32_t k = j; k < re; k++) {
          tests++;
          if (pair_linked(px, pos4[k], R, rechecks)) {
            rx = uf_join(par, rx, k);
            break;
          }
        }
      }
      j = re;
    }
  }
}

// FAST: every volume of the call has a constant l, a dense grid and
// sub-cells, so only the first branch below is compiled (it then fits 8
// waves per SIMD without spilling); otherwise both branches.  Both run at 8
// waves per SIMD (the full kernel spills a little: at 6 waves without spills
// it was 15% slower on a lightcone).
template <bool FAST>
__global__ __launch_bounds__(256, 8) void k_link_sparse(uint32_t N, const float4 *__restrict__ pos4,
                                                     const Grid G,
                                                     const uint32_t *__restrict__ run_end,
                                                     const unsigned long long *__restrict__ fine,
                                                     uint32_t *__restrict__ par,
                                                     const VolDev *__restrict__ vols,
                                                     const uint32_t *__restrict__ vbeg,
                                                     int nvol, uint32_t T,
                                                     unsigned long long *__restrict__ ctr) {
  if (*G.err) return;  // a particle's cell may not be the one it is sorted in
  uint32_t tests = 0, rechecks = 0;
  int hint = 0;
  for (uint32_t x = blockIdx.x * blockDim.x + threadIdx.x; x < N;
       x += gridDim.x * blockDim.x) {
    const float4 px = pos4[x];
    const VolDev &V = vols[vol_of_run(vbeg, nvol, x, N, hint)];
    const CellPos cp = cell_pos(V, px.x, px.y, px.z);
    const uint32_t c = cell_id(V, cp.ix, cp.iy, cp.iz);
    const uint32_t s = G.start[c], e = G.start[c + 1];
    // dense cells are linked by k_link_small (below kBigCell particles) and
    // k_link_dense (from it, with sub-cells)
    if (e - s >= T && (e - s < kBigCell || V.m[0] > 0)) continue;
    const Rule R = make_rule(V, cp.ix, cp.iy, cp.iz);
    uint32_t rx = x;  // x's root, refreshed by every join
    const int nx = V.nx, ny = V.ny, nz = V.nz;
    const int xl = (cp.ix > 0) ? 1 : 0, xr = (cp.ix + 1 < nx) ? 1 : 0;
    if (FAST || (V.vntab == 0 && V.m[0] > 0)) {
      // Constant l on a dense grid: k_link_dense links every pair that has a
      // particle in a dense cell (its forward cells, and its backward cells
      // that are sparse).  Here: the sparse cells among the own cell (after
      // x) and the 13 forward cells, partners loaded four at a time.
      // Row segments: own row (ix, ix+1); (iy+1, iz) and (iy-1..iy+1, iz+1)
      // over ix-1..ix+1.  b[r][0..3] are the segment's cell boundaries.
      uint32_t b[5][4];
      bool ok[5];
      b[0][0] = x + 1, b[0][1] = e, b[0][2] = xr ? G.start[c + 2] : e, b[0][3] = b[0][2];
      ok[0] = true;
#pragma unroll
      for (int r = 1; r < 5; r++) {
        const int ry = (r == 1) ? cp.iy + 1 : cp.iy + (r - 3);
        const int rz = (r == 1) ? cp.iz : cp.iz + 1;
        ok[r] = ry >= 0 && ry < ny && rz < nz;
        const uint32_t c0 = ok[r] ? cell_id(V, cp.ix - xl, ry, rz) : 0u;
        const int ncell = xl + 1 + xr;
        // the four cell starts from c0 in one load (the table has slack
        // behind its last entry)
        uint32_t q[4];
        __builtin_memcpy(q, G.start + c0, sizeof(q));
        b[r][0] = ok[r] ? q[0] : 0u;
        b[r][1] = ok[r] ? q[1] : 0u;
        b[r][2] = ok[r] ? (ncell >= 2 ? q[2] : q[1]) : 0u;
        b[r][3] = ok[r] ? (ncell >= 3 ? q[3] : b[r][2]) : 0u;
      }
#pragma unroll
      for (int r = 0; r < 5; r++) {
        if (!ok[r]) continue;
        // a dense cell (own row: only ix+1 can be) is skipped
        const bool d0 = r > 0 && b[r][1] - b[r][0] >= T;
        const bool d1 = b[r][2] - b[r][1] >= T;
        const bool d2 = r > 0 && b[r][3] - b[r][2] >= T;
        uint32_t j = b[r][0];
        for (;;) {
          if (d0 && j < b[r][1]) j = b[r][1];
          if (d1 && j >= b[r][1] && j < b[r][2]) j = b[r][2];
          if (d2 && j >= b[r][2]) j = b[r][3];
          if (j >= b[r][3]) break;
          uint32_t je = min(j + 4u, b[r][3]);
          if (d1 && j < b[r][1]) je = min(je, b[r][1]);
          if (d2 && j < b[r][2]) je = min(je, b[r][2]);
          const uint32_t n = je - j;
          float4 q[4];
#pragma unroll
          for (int k = 0; k < 4; k++) q[k] = ((uint32_t)k < n) ? ld4(pos4 + j + k) : px;
          uint32_t hit = 0;
#pragma unroll
          for (int k = 0; k < 4; k++)
            hit |= ((uint32_t)k < n && pair_linked(px, q[k], R, rechecks)) ? (1u << k) : 0u;
          tests += n;
          while (hit) {
            const int k = __builtin_ctz(hit);
            hit &= hit - 1;
            rx = uf_join(par, rx, j + k);
          }
          j = je;
        }
      }
      continue;
    }
    if (FAST) continue;  // not reached: the branch above always continues
    // Up to five contiguous ranges cover the own cell (after x) and the 13
    // forward cells: (ix+1,iy,iz); row (iy+1,iz); rows (iy-1..iy+1, iz+1).
    uint32_t r0[5], r1[5];
    int nr = 0;
    r0[nr] = x + 1;
    r1[nr] = G.start[c + 1 + xr];
    nr++;
    if (cp.iy + 1 < ny) {
      row_range(G, V, cp.ix - xl, cp.ix + xr, cp.iy + 1, cp.iz, r0[nr], r1[nr]);
      nr++;
    }
    if (cp.iz + 1 < nz) {
      for (int dy = -1; dy <= 1; dy++) {
        if (cp.iy + dy < 0 || cp.iy + dy >= ny) continue;
        row_range(G, V, cp.ix - xl, cp.ix + xr, cp.iy + dy, cp.iz + 1, r0[nr], r1[nr]);
        nr++;
      }
    }
    scan_rows(px, cp, V, R, r0, r1, nr, T, pos4, run_end, fine, par, rx, tests, rechecks);
  }
  add_counters(ctr, kCtrTestsSparse, tests, rechecks);
}

// The same over occupied cells (sparse addressing).  Particles, cells and keys
// are in one order, and a neighbour row's keys are the cell's own plus a
// constant: the rows of consecutive particles are consecutive stretches of
// the key list.  A wave takes kRowRun consecutive particles, keeps a place in
// the list for each of the four rows above its own, reads the keys there 128
// at a time into LDS, and each lane finds its first key by binary search.
// Thirteen probes of a hash table a particle, each a random line of gigabytes,
// took 4.09 ms for a lightcone of 1.6e7 particles in 16 shells.  A dense cell of
// a row is linked by the whole wave for one particle after the other, a run a
// lane and runs above 8 particles 64 at a time: a lane that went through the
// hundreds of runs of a big cell alone kept 63 waiting (2.98 ms, now 2.16).
// What bounds it now: the chain of dependent loads of such cells and of the
// scans (search 13, scans 25 thousand cycles a wave's 64 particles).
constexpr uint32_t kRowRun = 512;  // particles of a wave
constexpr uint32_t kRowWin = 128;   // keys of a window

// A cell at or before the first one with key >= t in [lo, U) (t uniform), at
// most 64 before it: 64 samples a step.
__device__ __forceinline__ uint32_t wave_lower(const Grid &G, uint32_t lo, uint32_t U,
                                               unsigned long long t) {
  const uint32_t lane = threadIdx.x & 63;
  uint32_t hi = U;
  while (hi - lo > 64) {
    const uint32_t step = (hi - lo + 63) / 64;
    const uint32_t at = lo + (lane + 1) * step - 1;
    const bool below = at < hi && cell_key(G, at) < t;
    lo = min(hi, lo + (uint32_t)__popcll(__ballot(below)) * step);
    hi = min(hi, lo + step);
  }
  return lo;
}

__global__ __launch_bounds__(256, 6) void k_link_rows(uint32_t N, const float4 *__restrict__ pos4,
                                                   const Grid G,
                                                   const uint32_t *__restrict__ run_end,
                                                   const unsigned long long *__restrict__ fine,
                                                   const uint32_t *__restrict__ rtoff,
                                                   const uint32_t *__restrict__ rtab,
                                                   uint32_t *__restrict__ par,
                                                   const VolDev *__restrict__ vols,
                                                   const uint32_t *__restrict__ vbeg, int nvol,
                                                   uint32_t T,
                                                   unsigned long long *__restrict__ ctr) {
  __shared__ unsigned long long wins[4][kRowWin];
  __shared__ uint32_t rowc[4][5][64];  // a lane's first cell in each row
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  unsigned long long *const win = wins[wv];
  uint32_t(*const row)[64] = rowc[wv];
  if (*G.err) return;  // the key list may be out of order
  const uint32_t U = *G.ncell;
  const uint64_t x0 = ((uint64_t)blockIdx.x * 4 + wv) * kRowRun;
  uint32_t tests = 0, rechecks = 0;
  uint32_t place[4] = {kNone, kNone, kNone, kNone};
  int hint = 0, last_v = -1;
  for (uint32_t q = 0; q < kRowRun && x0 + q < N; q += 64) {
    const uint32_t x = (uint32_t)(x0 + q) + lane;
    const bool valid = x < N;
    const uint32_t xc = min(x, N - 1);
    const float4 px = ld4(pos4 + xc);
    const int v = vol_of_run(vbeg, nvol, xc, N, hint);
    const VolDev &V = vols[v];
    const CellPos cp = cell_pos(V, px.x, px.y, px.z);
    const uint32_t c = G.cell_of[xc];
    const uint32_t s = G.start[c], e = G.start[c + 1];
    // dense cells are linked by k_link_small and k_link_dense
    const bool active = valid && !(e - s >= T && (e - s < kBigCell || V.m[0] > 0));
    if (!__ballot(active)) continue;
    // a wave in two volumes looks each row up on its own
    const int v0 = __builtin_amdgcn_readfirstlane(v);
    const bool one = __ballot(v != v0) == 0;
    if (!one || v0 != last_v) place[0] = place[1] = place[2] = place[3] = kNone;
    last_v = one ? v0 : -1;
    const int nx = V.nx, ny = V.ny, nz = V.nz;
    const unsigned long long key = cell_key(G, c);
    uint32_t ncell[5];  // occupied cells of each row (own row: behind the own cell)
    row[0][lane] = c + 1;
    ncell[0] = active && cp.ix + 1 < nx && c + 1 < U && cell_key(G, c + 1) == key + 1 ? 1u : 0u;
#pragma unroll
    for (int r = 1; r < 5; r++) {
      ncell[r] = 0;
      const int dy = r == 1 ? 1 : r - 3, dz = r == 1 ? 0 : 1;
      const bool want = active && cp.iy + dy >= 0 && cp.iy + dy < ny && cp.iz + dz < nz;
      const long long d = ((long long)dz * ny + dy) * nx;
      // the row's keys a .. b (ascending over the lanes of one volume)
      const unsigned long long a = key + (unsigned long long)(d - (cp.ix > 0 ? 1 : 0));
      const unsigned long long b = key + (unsigned long long)(d + (cp.ix + 1 < nx ? 1 : 0));
      unsigned long long need = __ballot(want);
      if (!need) continue;
      if (one) {
        auto first = [&]() -> unsigned long long {
          const int l = __builtin_ctzll(need);
          return (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)a, l) |
                 ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(a >> 32), l) << 32);
        };
        uint32_t w = place[r - 1] == kNone ? wave_lower(G, 0, U, first()) : place[r - 1];
        for (;;) {
          wave_sync();
          win[lane] = w + lane < U ? cell_key(G, w + lane) : ~0ull;
          win[lane + 64] = w + 64 + lane < U ? cell_key(G, w + 64 + lane) : ~0ull;
          wave_sync();
          // resolved when the first key >= a and the two behind it are here
          const bool here = ((need >> lane) & 1ull) && a <= win[kRowWin - 4];
          if (here) {
            uint32_t lo = 0;
#pragma unroll
            for (uint32_t st = kRowWin / 2; st > 0; st >>= 1)
              if (win[lo + st - 1] < a) lo += st;
            uint32_t n = 0;
#pragma unroll
            for (uint32_t k = 0; k < 3; k++) n += win[lo + k] <= b ? 1u : 0u;
            ncell[r] = n;
            row[r][lane] = w + lo;
          }
          const unsigned long long done = __ballot(here);
          need &= ~done;
          if (!need) break;
          // the next window behind this one, or where the first lane left lies
          w = done ? w + kRowWin - 3 : wave_lower(G, w + kRowWin - 3, U, first());
        }
        place[r - 1] = w;
      } else if (want) {
        const uint32_t lo = cell_lower(G, U, a);
        uint32_t n = 0;
        while (n < 3 && lo + n < U && cell_key(G, lo + n) <= b) n++;
        ncell[r] = n;
        row[r][lane] = lo;
      }
    }
    Rule R;
    uint32_t rx = x, dcells = 0;  // bit 3 r + k: cell k of row r is dense
    if (active) {
      R = make_rule(V, cp.ix, cp.iy, cp.iz);
      const bool subcells = V.m[0] > 0;
      scan_range(px, R, x + 1, e, pos4, par, rx, tests, rechecks);
#pragma unroll
      for (int r = 0; r < 5; r++) {
        if (!ncell[r]) continue;
        const uint32_t cf = row[r][lane];
        uint32_t j = G.start[cf], je = G.start[cf + ncell[r]];
        if (subcells && je - j >= T) {
          // sub-sorted cells among them are left to the wave where the
          // particle's sub-cell is within reach of the cell
          const int dy = r == 0 ? 0 : r == 1 ? 1 : r - 3, dz = r < 2 ? 0 : 1;
          const unsigned long long mid = key + (unsigned long long)(((long long)dz * ny + dy) * nx);
          const int gy = dy > 0 ? (cp.iy + 1) * V.m[1] - cp.fy - 1 : dy < 0 ? cp.fy - cp.iy * V.m[1] : 0;
          const int gz = dz > 0 ? (cp.iz + 1) * V.m[2] - cp.fz - 1 : 0;
          for (uint32_t k = 0; k < ncell[r]; k++) {
            const uint32_t ke = G.start[cf + k + 1];
            if (ke - j >= T) {
              const int dx = (int)(long long)(cell_key(G, cf + k) - mid);
              const int gx = dx > 0 ? (cp.ix + 1) * V.m[0] - cp.fx - 1 : dx < 0 ? cp.fx - cp.ix * V.m[0] : 0;
              const double g2 = (double)(gx * gx) * V.s2[0] + (double)(gy * gy) * V.s2[1] +
                                (double)(gz * gz) * V.s2[2];
              if (!(g2 > R.prune2)) dcells |= 1u << (3 * r + k);
            } else {
              scan_range(px, R, j, ke, pos4, par, rx, tests, rechecks);
            }
            j = ke;
          }
          continue;
        }
        scan_range(px, R, j, je, pos4, par, rx, tests, rechecks);
      }
    }
    wave_sync();
    while (const unsigned long long pend = __ballot(dcells != 0)) {
      // the lowest lane's next dense cell
      const int l = __builtin_ctzll(pend);
      const uint32_t dl = (uint32_t)__builtin_amdgcn_readlane((int)dcells, l);
      const uint32_t t = (uint32_t)__builtin_ctz(dl);
      if ((int)lane == l) dcells &= dcells - 1;
      auto lf = [&](float f) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), l)); };
      auto li = [&](int i) { return __builtin_amdgcn_readlane(i, l); };
      auto ld = [&](double q) { return __hiloint2double(li(__double2hiint(q)), li(__double2loint(q))); };
      const VolDev &W = vols[li(v)];
      const float4 q = make_float4(lf(px.x), lf(px.y), lf(px.z), 0.f);
      const Rule Q = {ld(R.linksq), ld(R.prune2), lf(R.lo), lf(R.hi)};
      const int qx = li(cp.fx), qy = li(cp.fy), qz = li(cp.fz);
      const uint32_t xl = (uint32_t)li((int)x), sB = G.start[row[t / 3][l] + t % 3];
      const uint32_t runs = rtoff[sB];
      for (uint32_t i0 = 0; i0 < runs; i0 += 64) {
        uint32_t j = 0, je = 0;
        if (i0 + lane < runs) {
          j = rtab[sB + i0 + lane];
          const unsigned long long fj = fine[j];
          const int gx = max(abs(fine_x(fj) - qx) - 1, 0);
          const int gy = max(abs(fine_y(fj) - qy) - 1, 0);
          const int gz = max(abs(fine_z(fj) - qz) - 1, 0);
          const double g2 = (double)(gx * gx) * W.s2[0] + (double)(gy * gy) * W.s2[1] +
                            (double)(gz * gz) * W.s2[2];
          je = g2 > Q.prune2 ? j : run_end[j];
        }
        // short runs a lane each, longer ones 64 particles at a time
        unsigned long long big = __ballot(je - j > 8);
        if (je - j <= 8)
          for (; j < je; j++) {
            tests++;
            if (pair_linked(q, pos4[j], Q, rechecks)) {
              uf_union(par, xl, j);
              break;
            }
          }
        while (big) {
          const int b = __builtin_ctzll(big);
          big &= big - 1;
          const uint32_t bj = (uint32_t)__builtin_amdgcn_readlane((int)j, b);
          const uint32_t be = (uint32_t)__builtin_amdgcn_readlane((int)je, b);
          for (uint32_t k0 = bj; k0 < be; k0 += 64) {
            bool hit = false;
            if (k0 + lane < be) {
              tests++;
              hit = pair_linked(q, pos4[k0 + lane], Q, rechecks);
            }
            const unsigned long long h = __ballot(hit);
            if (!h) continue;
            if (lane == 0) uf_union(par, xl, k0 + (uint32_t)__builtin_ctzll(h));
            break;
          }
        }
      }
    }
  }
  add_counters(ctr, kCtrTestsSparse, tests, rechecks);
}

// ---------------------------------------------------------------------------
// 6: dense cells -- one workgroup per cell, run pairs with early exit.
// ---------------------------------------------------------------------------
// Run-table capacities.  The home cell has one run per occupied sub-cell,
// at most 12^3 (and at most one per particle); neighbour runs (dense
// neighbours) or particles (sparse neighbours) are taken a chunk at a time.
constexpr int kMaxRuns = 1728;
constexpr uint32_t kMaxT = 512;
// Default dense threshold: on clumpy 1024^3 boxes (b = 0.2, about one
// particle per cell) the link and sub-sort phases take 148-149 ms for T = 16,
// 20 and 24, 153 ms at 32 and 155 ms at 40.
constexpr uint32_t kDefaultT = 24;

__device__ __forceinline__ uint32_t pack_rel(int a, int b, int c) {
  return ((uint32_t)(a & 255)) | ((uint32_t)(b & 255) << 8) | ((uint32_t)(c & 255) << 16);
}
__device__ __forceinline__ int rel_x(uint32_t r) { return (int)(int8_t)(r & 255); }
__device__ __forceinline__ int rel_y(uint32_t r) { return (int)(int8_t)((r >> 8) & 255); }
__device__ __forceinline__ int rel_z(uint32_t r) { return (int)(int8_t)((r >> 16) & 255); }

// Union-find over run slots in LDS (A's runs 0..na-1, the neighbour's runs
// after them).  Hooking larger-under-smaller keeps A's roots inside A, so the
// neighbour's slots can be reset for the next neighbour.
__device__ __forceinline__ uint32_t lfind(volatile uint32_t *lp, uint32_t x) {
  for (;;) {
    const uint32_t p = lp[x];
    if (p == x) return x;
    const uint32_t gp = lp[p];
    if (gp == p) return p;
    lp[x] = gp;
    x = gp;
  }
}

__device__ __forceinline__ void lunion(volatile uint32_t *lp, uint32_t a, uint32_t b) {
  for (;;) {
    a = lfind(lp, a);
    b = lfind(lp, b);
    if (a == b) return;
    if (a > b) {
      const uint32_t t = a;
      a = b;
      b = t;
    }
    if (atomicCAS((uint32_t *)&lp[b], b, a) == b) return;
  }
}

// Home-cell sub-cell coordinates (0..11) packed 4 bits per axis.
__device__ __forceinline__ uint16_t pack_home(int x, int y, int z) {
  return (uint16_t)(x | (y << 4) | (z << 8));
}

// Cells with more runs than this enumerate candidates through a bitmap of
// A's occupied sub-cells, one x-row of the window at a time; cells with fewer
// test every run pair.  The window is walked twice: first the sub-cells that
// touch the run's own (|offset| <= 1 on every axis), whose pairs link most
// often, so that their merges prune the second walk over the rest.
constexpr int kMapRuns = 24;

// 0, 1, -1, 2, -2, ...: window rows visited from the centre out.
__device__ __forceinline__ int zig(int k) { return (k & 1) ? (k + 1) >> 1 : -(k >> 1); }

// Cell offset of neighbour k of the dense kernels' table: k < 13 the 13
// forward cells of src_v2/FOF.c:122-153 ((1,0,0); (-1..1,1,0); (-1..1,-1..1,1)),
// k >= 13 the same offsets negated.
__device__ __forceinline__ void nb_offset(int k, int dd[3]) {
  const int kf = k % 13, sg = k < 13 ? 1 : -1;
  dd[0] = dd[1] = dd[2] = 0;
  if (kf == 0) dd[0] = 1;
  else if (kf < 4) dd[1] = 1, dd[0] = kf - 2;
  else dd[2] = 1, dd[1] = (kf - 4) / 3 - 1, dd[0] = (kf - 4) % 3 - 1;
  dd[0] *= sg, dd[1] *= sg, dd[2] *= sg;
}

// Bytes of dynamic LDS for ra home-run slots and MAXRUNSB neighbour slots:
// ahead (and the cell's end), agr, lp (ra + MAXRUNSB), arel (u16).
constexpr size_t dense_lds(uint32_t ra, uint32_t maxrunsb) {
  return 4 * ((size_t)3 * ra + 1 + maxrunsb) + 2 * (size_t)ra + 8;
}

// a / d for a < 2^23 (inv = 1 / d in float): the quotient in float is off by
// at most one.
__device__ __forceinline__ uint32_t div_small(uint32_t a, uint32_t d, float inv) {
  uint32_t q = (uint32_t)((float)a * inv);
  const uint32_t r = a - q * d;
  if ((int)r < 0) q--;
  else if (r >= d) q++;
  return q;
}

// Run pairs of many particles, {first, number} of the home cell's run and of the
// other's: listed by k_link_dense, tested by k_init_groups.  The list lies in
// the unused half of the counters' lines, four pairs each, so that it costs
// k_link_dense no register for an address of its own.
constexpr uint32_t kWideCap = 4 * kCtrSlots;  // further pairs are tested where they are found
__device__ __forceinline__ uint32_t *wide_count(unsigned long long *ctr) {
  return reinterpret_cast<uint32_t *>(ctr) - kSmCtr + kSmWide;
}
__device__ __forceinline__ uint4 *wide_pair(unsigned long long *ctr, uint32_t k) {
  return reinterpret_cast<uint4 *>(ctr + (k >> 2) * kCtrStride + kCtrWide) + (k & 3);
}

// WPE: waves per SIMD to fit (the register budget; LDS per workgroup is
// sized at launch to the runs a cell of the batch can have).
//
// The cell's data (run heads, window bitmaps, union-find) is shared by the
// workgroup; the waves take 64 slots at a time -- (row of the window, run) or
// (row, neighbour item) -- from a counter in LDS and work on their own: a lane
// walks its row's occupied sub-cells, candidate pairs not yet joined go to the
// wave's queue, and 64 queued pairs are tested together, a lane each (the
// first kTile x kTile particles, which settles nearly all), what is left by
// 16-lane groups.  Enumerating reads no global memory and no barrier stands
// between enumerating and testing.
//
// What bounds it: one cell's chain of dependent steps while there are few
// cells, VALU issue and latency (LDS finds, positions) when many.  Before, the
// workgroup went through rounds of 768 slots, tested single pairs where they
// were found and drained a common queue four pairs a wave at a time, each
// behind two walks of the global union-find: the kernel took 630 us for the
// 64^3 box (132 cells), 2.88 ms for 256^3 and 7.25 ms for 512^3; now 0.74 and
// 3.36 ms, and 160 us for the 64^3 box with 1024 threads a cell.  Walking whole rows first instead of the touching sub-cells made
// half as many pairs again (30 against 15 G cycles at 512^3).  Six waves per
// SIMD: at eight (64 registers) the spills doubled the cycles per cell, five
// was 10% slower.
template <int NT, int WPE, int MAXRUNS, int MAXRUNSB>
__global__ __launch_bounds__(NT, WPE) void k_link_dense(const uint32_t *__restrict__ dense,
                                                    const uint32_t *__restrict__ ndense,
                                                    const float4 *__restrict__ pos4,
                                                    const Grid G,
                                                    const uint32_t *__restrict__ run_end,
                                                    const unsigned long long *__restrict__ fine,
                                                    const uint32_t *__restrict__ rtoff,
                                                    const uint32_t *__restrict__ rtab,
                                                    uint32_t T,
                                                    uint32_t *__restrict__ par,
                                                    const VolDev *__restrict__ vols,
                                                    const uint32_t *__restrict__ vbeg,
                                                    int nvol,
                                                    unsigned long long *__restrict__ ctr,
                                                    uint32_t ra, uint32_t *__restrict__ dq) {
  // per-run slots of the home cell (ra <= MAXRUNS of them: the most
  // sub-cells of a cell in the batch), in dynamic LDS
  extern __shared__ uint32_t dyn[];
  uint32_t *const ahead = dyn, *const agr = dyn + ra + 1, *const lp = dyn + 2 * ra + 1;
  uint16_t *const arel = reinterpret_cast<uint16_t *>(dyn + 3 * ra + 1 + MAXRUNSB);
  __shared__ uint32_t bhead[MAXRUNSB], brel[MAXRUNSB], bgr[MAXRUNSB];
  __shared__ uint32_t wq[NT / 64][128];  // the waves' queues of pairs to test
  // occupied sub-cells of A (<= 12^3) and the occupied count before each
  // word: A's runs are listed in sub-cell order, so the run slot of an
  // occupied sub-cell is its rank in the bitmap
  constexpr int kOccW = kMaxRuns / 64 + 1;
  __shared__ unsigned long long occ[kOccW];
  __shared__ uint16_t wpre[kOccW];
  // after the touching pairs: the dominant LDS set (mainr, kNone if none)
  // and a bitmap of the occupied sub-cells whose runs were outside it
  // ("stragglers"); a pair of two runs of the dominant set is joined, so a
  // run or neighbour item in it needs only the stragglers of a window row
  __shared__ unsigned long long smap[kOccW];
  __shared__ uint32_t mainr;
  __shared__ uint32_t nbS[26], nbOff[27];
  __shared__ uint8_t nbDense[26];
  __shared__ uint32_t cntx, cnty, slots[3], dnext;
  uint32_t tests = 0, rechecks = 0, joined = 0;
  const uint32_t lane = threadIdx.x & 63;
  const unsigned long long lt = (1ull << lane) - 1;
  uint32_t *const wqw = wq[__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))];
  const uint32_t nd = *ndense;
  // cells are taken from a queue (*dq, zero at launch) one at a time: their
  // costs differ by orders of magnitude, and a fixed share per workgroup
  // left a tail (51.2 against 49.4 ms on the clumpy 1024^3 box)
  if (threadIdx.x == 0) dnext = atomicAdd(dq, 1u);
  __syncthreads();
  for (uint32_t d = dnext; d < nd; d = dnext) {
    const uint32_t c = dense[d];
    const uint32_t sA = G.start[c];
    const VolDev &V = vols[vol_of(vbeg, nvol, sA)];
    const unsigned long long f0 = fine[sA];
    const int mm[3] = {V.m[0], V.m[1], V.m[2]};
    const int ix = fine_x(f0) / mm[0], iy = fine_y(f0) / mm[1], iz = fine_z(f0) / mm[2];
    const Rule R = make_rule(V, ix, iy, iz);
    const int ox = ix * mm[0], oy = iy * mm[1], oz = iz * mm[2];
    int reach[3];
    for (int a = 0; a < 3; a++)  // largest sub-cell offset whose gap can be within reach
      reach[a] = min((int)floor(sqrt(R.prune2 / V.s2[a])) + 1, mm[a]);
    // Sub-cell gap pruning in FP32: the prune radius carries a 1e-4 margin,
    // far above the FP32 rounding of the gap.
    const float gs0 = (float)V.s2[0], gs1 = (float)V.s2[1], gs2 = (float)V.s2[2];
    const float gp2 = (float)R.prune2;
    auto gap_ok = [&](int dx, int dy, int dz) {
      const int gx = max(abs(dx) - 1, 0), gy = max(abs(dy) - 1, 0), gz = max(abs(dz) - 1, 0);
      return (float)(gx * gx) * gs0 + (float)(gy * gy) * gs1 + (float)(gz * gz) * gs2 <= gp2;
    };
    // neighbour table: the 13 forward cells of src_v2/FOF.c:122-153 and,
    // for a constant l on a dense grid, the 13 backward cells when sparse
    // (k_link_sparse leaves their pairs with dense cells to this kernel);
    // their items (runs of dense neighbours, particles of sparse ones) and
    // the window of sub-cells that can reach A
    if (threadIdx.x < 64) {  // wave 0: one neighbour a lane, then a scan of the counts
      const int k = threadIdx.x;
      uint32_t items = 0;
      if (k < 26) {
        int dd[3];
        nb_offset(k, dd);
        const int bx = ix + dd[0], by = iy + dd[1], bz = iz + dd[2];
        uint32_t sB = 0, eB = 0;
        const bool want = k < 13 || (!G.sparse && V.vntab == 0);
        if (want && !(bx < 0 || bx >= V.nx || by < 0 || by >= V.ny || bz < 0 || bz >= V.nz)) {
          const uint32_t cb = cell_index(G, V, bx, by, bz);
          if (cb != kNone) sB = G.start[cb], eB = G.start[cb + 1];
        }
        if (k >= 13 && eB - sB >= T) eB = sB;  // a dense backward cell links this pair itself
        // runs of a cell sub-sorted into runs, particles of any other: dense
        // cells of kBigCell particles or more always are; the smaller ones
        // only where k_link_sparse scans runs (sparse addressing or a
        // variable l)
        const bool dn = (eB - sB >= T) && (eB - sB >= kBigCell || G.sparse || V.vntab != 0);
        nbS[k] = sB;
        nbDense[k] = dn ? 1 : 0;
        items = dn ? rtoff[sB] : eB - sB;  // runs of a dense cell, else particles
      }
#pragma unroll
      for (int o = 1; o < 32; o <<= 1) {
        const uint32_t t = __shfl_up(items, o, 64);
        if (k >= o) items += t;
      }
      if (k < 26) nbOff[k + 1] = items;
      if (k == 0) nbOff[0] = 0;
    }
    // the home cell's runs (one per occupied sub-cell, in sub-cell order)
    // from its run table; runs <= min(particles, sub-cells) <= ra
    const int na = (int)rtoff[sA];
    if (threadIdx.x == 0) {
      mainr = kNone, slots[0] = slots[1] = 0;
      ahead[na] = G.start[c + 1];  // runs follow one another: each ends where the next begins
    }
    if (threadIdx.x < kOccW) occ[threadIdx.x] = 0, smap[threadIdx.x] = 0;
    __syncthreads();
    const int wy = 2 * reach[1] + 1, wz = 2 * reach[2] + 1;
    for (uint32_t k = threadIdx.x; k < (uint32_t)na; k += blockDim.x) {
      const uint32_t j = rtab[sA + k];
      const unsigned long long f = fine[j];
      const int rx = fine_x(f) - ox, ry = fine_y(f) - oy, rz = fine_z(f) - oz;
      ahead[k] = j;
      arel[k] = pack_home(rx, ry, rz);
      agr[k] = uf_find(par, j);  // snapshot of the global root
      lp[k] = k;
      const int bin = (rz * mm[1] + ry) * mm[0] + rx;
      atomicOr(&occ[bin >> 6], 1ull << (bin & 63));
    }
    __syncthreads();
    if (threadIdx.x < kOccW) {
      uint32_t n = 0;
      for (uint32_t w = 0; w < threadIdx.x; w++) n += __popcll(occ[w]);
      wpre[threadIdx.x] = (uint16_t)n;
    }
    __syncthreads();
    // run slot of the first occupied sub-cell at or after bin
    auto rank = [&](int bin) -> uint32_t {
      const int w = bin >> 6;
      return wpre[w] + (uint32_t)__popcll(occ[w] & ((1ull << (bin & 63)) - 1));
    };
    // bits of the occupied sub-cells [bin0, bin0 + len) of A (len <= 25)
    auto rowbits = [&](int bin0, int len) -> uint32_t {
      const int w = bin0 >> 6, sh = bin0 & 63;
      unsigned long long v = occ[w] >> sh;
      if (sh + len > 64) v |= occ[w + 1] << (64 - sh);
      return (uint32_t)(v & ((1ull << len) - 1));
    };
    // the same for the stragglers
    auto srowbits = [&](int bin0, int len) -> uint32_t {
      const int w = bin0 >> 6, sh = bin0 & 63;
      unsigned long long v = smap[w] >> sh;
      if (sh + len > 64) v |= smap[w + 1] << (64 - sh);
      return (uint32_t)(v & ((1ull << len) - 1));
    };
    const bool bmap = na > kMapRuns;
    // bits of x in [c - 1, c + 1] for a row starting at x0, given s = c - 1 - x0
    auto touchbits = [](int s) -> uint32_t { return s >= 0 ? 7u << s : 7u >> -s; };
    // the run of an LDS slot: particles [h, h + n)
    auto run_of = [&](uint32_t sl, uint32_t &h, uint32_t &n) {
      if (sl < (uint32_t)na) {
        h = ahead[sl], n = ahead[sl + 1] - h;
      } else {
        h = bhead[sl - na], n = brel[sl - na] >> 24;
        if (n == 255) n = run_end[h] - h;  // the packed size saturates
      }
    };
    uint32_t qn = 0;  // pairs in the wave's queue (uniform)
    // test the last m (<= 64) queued pairs of LDS slots, a lane each
    constexpr uint32_t kTile = 4;
    // particle pairs from which two walks of the global union-find cost less
    // than the tests they may spare (1024: 32 steps of a group; 1e6 particles
    // in 10 clumps of sigma 5 l: 0.79 ms with the walks, 0.81 without), and
    // from which a pair is left to a wave of its own (0.9 ms of a group's time)
    constexpr unsigned long long kLongPair = 1024, kWidePair = 65536;
    auto flush = [&](uint32_t m) {
      wave_sync();
      qn -= m;
      uint32_t sa = 0, sb = 0, ha = 0, hb = 0, n1 = 0, n2 = 0;
      bool live = lane < m, link = false;
      if (live) {
        const uint32_t e = wqw[qn + lane];
        sa = e >> 16, sb = e & 0xFFFFu;
        if (lfind(lp, sa) == lfind(lp, sb)) live = false, joined++;
      }
      if (live) {
        run_of(sa, ha, n1), run_of(sb, hb, n2);
        const uint32_t t1 = min(n1, kTile), t2 = min(n2, kTile);
        uint32_t spare = 0;
        float4 a[kTile];
#pragma unroll
        for (uint32_t k = 0; k < kTile; k++) a[k] = ld4(pos4 + ha + min(k, t1 - 1));
        for (uint32_t j = 0; j < t2 && !link; j++) {
          const float4 q = ld4(pos4 + hb + j);
#pragma unroll
          for (uint32_t k = 0; k < kTile; k++)  // past the run's end its last once more, not counted
            link |= pair_linked(a[k], q, R, k < t1 ? rechecks : spare);
          tests += t1;
        }
        if (link) lunion(lp, sa, sb);
      }
      // pairs with more particles, not linked so far: four at a time
      unsigned long long rest = __ballot(live && !link && (n1 > kTile || n2 > kTile));
      const uint32_t gl = lane & 15;
      while (rest) {
        uint32_t src = 0;  // the group's pair: the grp-th set bit
        unsigned long long left = rest;
        bool mine = false;
#pragma unroll
        for (uint32_t g = 0; g < 4; g++) {
          if (left) {
            const uint32_t l = (uint32_t)__builtin_ctzll(left);
            left &= left - 1;
            if (g == (lane >> 4)) src = l, mine = true;
          }
        }
        rest = left;
        const uint32_t xa = __shfl(sa, src, 64), xb = __shfl(sb, src, 64);
        const uint32_t ga = __shfl(ha, src, 64), gb = __shfl(hb, src, 64);
        const uint32_t m1 = __shfl(n1, src, 64), m2 = __shfl(n2, src, 64);
        // joined by now?  (the group's first lane asks: one answer a group; of
        // a long pair also whether other cells have joined the runs since, and
        // the longest are listed for k_init_groups while the list has room)
        bool done = !mine;
        if (mine && gl == 0) {
          const unsigned long long all = (unsigned long long)m1 * m2;
          done = lfind(lp, xa) == lfind(lp, xb);
          if (!done && all >= kLongPair && uf_find(par, ga) == uf_find(par, gb))
            lunion(lp, xa, xb), done = true;
          joined += done ? 1u : 0u;
          if (!done && all >= kWidePair) {
            const uint32_t k = atomicAdd(wide_count(ctr), 1u);
            if (k < kWideCap) *wide_pair(ctr, k) = make_uint4(ga, m1, gb, m2), done = true;
          }
        }
        done = __shfl((int)done, lane & ~15u, 64) != 0;
        uint32_t rows = done ? 0u : m1;
        const float4 *const qa = pos4 + ga, *const qb = pos4 + gb;
        PairWalk p(gl, max(m2, 1u));
        while (__ballot(p.i < rows)) {
          bool l = false;
#pragma unroll
          for (int k = 0; k < 2; k++) {
            if (p.i < rows) {
              l |= pair_linked(qa[p.i], qb[p.j], R, rechecks);
              tests++;
            }
            p.step();
          }
          const uint32_t gbits = (uint32_t)(__ballot(l) >> (lane & ~15u)) & 0xFFFFu;
          if (gbits) rows = 0;
        }
        if (mine && !done && rows == 0 && gl == 0) lunion(lp, xa, xb);
      }
      wave_sync();
    };
    // one candidate a lane (all lanes call): a pair of slots not joined yet
    // is joined on equal snapshots of the global roots, else queued
    auto offer = [&](bool any, uint32_t sa, uint32_t sb, uint32_t ga, uint32_t gb) {
      bool want = false;
      if (any) {
        if (lfind(lp, sa) == lfind(lp, sb)) {
          joined++;
        } else if (ga == gb) {
          joined++;
          lunion(lp, sa, sb);
        } else {
          want = true;
        }
      }
      const unsigned long long bal = __ballot(want);
      if (want) wqw[qn + (uint32_t)__popcll(bal & lt)] = (sa << 16) | sb;
      qn += (uint32_t)__popcll(bal);
      if (qn >= 64) flush(64);
    };
    // the wave's next 64 slots of a phase (its first)
    auto take = [&](int ph) -> uint32_t {
      uint32_t p = 0;
      if (lane == 0) p = atomicAdd(&slots[ph], 64u);
      return (uint32_t)__builtin_amdgcn_readfirstlane((int)p);
    };
    // the occupied sub-cells `bits` (of `all`, from x0, first slot r0) of a
    // lane's row against its run or item: offset dxo from it in x
    auto walk = [&](uint32_t bits, uint32_t all, uint32_t r0, int x0, int bx, int dy, int dz,
                    uint32_t other, uint32_t gother) {
      while (__ballot(bits != 0)) {
        bool any = false;
        uint32_t sa = 0, sb = 0, ga = 0, gb = 0;
        if (bits) {
          const int b = __builtin_ctz(bits);
          bits &= bits - 1;
          if (gap_ok(x0 + b - bx, dy, dz)) {
            const uint32_t ia = r0 + __popc(all & ((1u << b) - 1));
            any = true;
            sa = min(ia, other), sb = max(ia, other);
            ga = agr[ia], gb = gother;
          }
        }
        offer(any, sa, sb, ga, gb);
      }
    };
    // (A, A)
    const float ina = 1.0f / (float)na;
    if (bmap) {
      // slots (row of the forward window, run), row-major, rows centre-out;
      // the first walk (touching sub-cells: the 5 forward rows at |dy|, dz
      // <= 1) before the second (every forward row)
      const int ry = reach[1], rz = reach[2];
      const uint32_t nrow1 = 5, nrow2 = (uint32_t)(ry + 1 + rz * wy);
      auto aa_slots = [&](bool first) {
        const uint32_t to = (first ? nrow1 : nrow2) * (uint32_t)na;
        for (uint32_t p0 = take(first ? 0 : 1); p0 < to; p0 = take(first ? 0 : 1)) {
          const uint32_t p = p0 + lane;
          uint32_t bits = 0, all = 0, r0 = 0, ia = 0;
          int x0 = 0, ax = 0, dy = 0, dz = 0;
          if (p < to) {
            const uint32_t r2 = div_small(p, (uint32_t)na, ina);
            ia = p - r2 * (uint32_t)na;
            if (first) {
              dz = r2 < 2 ? 0 : 1;
              dy = zig((int)(r2 < 2 ? r2 : r2 - 2));
            } else if (r2 <= (uint32_t)ry) {
              dy = (int)r2;
            } else {
              const uint32_t t = r2 - (uint32_t)(ry + 1);
              dz = 1 + (int)(t / (uint32_t)wy);
              dy = zig((int)(t % (uint32_t)wy));
            }
            const bool trow = dz <= 1 && dy >= -1 && dy <= 1;
            const uint32_t rr = arel[ia];
            const int ay = (rr >> 4) & 15, az = rr >> 8;
            ax = rr & 15;
            const int by = ay + dy, bz = az + dz;
            x0 = (dz == 0 && dy == 0) ? ax + 1 : max(ax - reach[0], 0);
            const int x1 = min(ax + reach[0], mm[0] - 1);
            if (bz < mm[2] && by >= 0 && by < mm[1] && x0 <= x1 && gap_ok(0, dy, dz)) {
              const int bin0 = (bz * mm[1] + by) * mm[0] + x0;
              bits = all = rowbits(bin0, x1 - x0 + 1);
              r0 = rank(bin0);
              if (trow) bits &= first ? touchbits(ax - 1 - x0) : ~touchbits(ax - 1 - x0);
              if (!first && mainr != kNone) {  // a run of the dominant set: only the stragglers
                const int abin = (az * mm[1] + ay) * mm[0] + ax;
                if (!((smap[abin >> 6] >> (abin & 63)) & 1ull)) bits &= srowbits(bin0, x1 - x0 + 1);
              }
            }
          }
          walk(bits, all, r0, x0, ax, dy, dz, ia, p < to ? agr[ia] : 0u);
        }
        if (qn) flush(qn);
        __syncthreads();
      };
      aa_slots(true);
      // the dominant set: a vote of 64 runs spread over the cell (wave 0);
      // kept when it holds at least a quarter of them
      if (threadIdx.x < 64) {
        const uint32_t r = lfind(lp, (uint32_t)(((uint64_t)threadIdx.x * (uint32_t)na) >> 6));
        uint32_t best = kNone, bestc = 0;
        unsigned long long pend = __ballot(true);
        while (pend) {
          const uint32_t rl = __shfl(r, __ffsll((long long)pend) - 1, 64);
          const unsigned long long m = __ballot(r == rl);
          const uint32_t cnt1 = (uint32_t)__popcll(m);
          if (cnt1 > bestc) bestc = cnt1, best = rl;
          pend &= ~m;
        }
        if (threadIdx.x == 0) mainr = bestc >= 16 ? best : kNone;
      }
      __syncthreads();
      if (mainr != kNone) {
        for (uint32_t k = threadIdx.x; k < (uint32_t)na; k += blockDim.x)
          if (lfind(lp, k) != mainr) {
            const uint32_t rk = arel[k];
            const int bin = ((rk >> 8) * mm[1] + ((rk >> 4) & 15)) * mm[0] + (rk & 15);
            atomicOr(&smap[bin >> 6], 1ull << (bin & 63));
          }
      }
      __syncthreads();
      aa_slots(false);
    } else {
      const uint32_t total = (uint32_t)na * (uint32_t)na;  // na <= kMapRuns
      for (uint32_t p0 = take(0); p0 < total; p0 = take(0)) {
        const uint32_t p = p0 + lane;
        const uint32_t ia = div_small(p, (uint32_t)na, ina), ib = p - ia * (uint32_t)na;
        bool any = p < total && ib > ia;
        if (any) {
          const uint32_t rra = arel[ia], rrb = arel[ib];
          any = gap_ok((int)(rrb & 15) - (int)(rra & 15),
                       (int)((rrb >> 4) & 15) - (int)((rra >> 4) & 15),
                       (int)(rrb >> 8) - (int)(rra >> 8));
        }
        offer(any, ia, ib, any ? agr[ia] : 0u, any ? agr[ib] : 0u);
      }
      if (qn) flush(qn);
      __syncthreads();
    }
    // (A, B): the neighbours' items in chunks of MAXRUNSB
    const uint32_t ntot = nbOff[26];
    for (uint32_t c0 = 0; c0 < ntot; c0 += MAXRUNSB) {
      const uint32_t c1 = min(ntot, c0 + (uint32_t)MAXRUNSB);
      if (threadIdx.x == 0) cntx = cnty = slots[2] = 0;
      __syncthreads();
      for (uint32_t g = c0 + threadIdx.x; g < c1; g += blockDim.x) {
        int q = 0, qh = 25;  // the last neighbour whose items start at or before g
        while (q < qh) {
          const int mid = (q + qh + 1) >> 1;
          if (nbOff[mid] <= g) q = mid;
          else qh = mid - 1;
        }
        const uint32_t item = g - nbOff[q];
        const uint32_t j = nbDense[q] ? rtab[nbS[q] + item] : nbS[q] + item;
        int fx, fy, fz;
        uint32_t len = 1;
        if (nbDense[q]) {
          const unsigned long long f = fine[j];
          len = min(run_end[j] - j, 255u);
          fx = fine_x(f), fy = fine_y(f), fz = fine_z(f);
        } else {
          const float4 pj = pos4[j];
          const CellPos cj = cell_pos(V, pj.x, pj.y, pj.z);
          fx = cj.fx, fy = cj.fy, fz = cj.fz;
        }
        // within reach of A: at most reach sub-cells beyond A's face
        const int rr[3] = {fx - ox, fy - oy, fz - oz};
        int dd[3];
        nb_offset(q, dd);
        bool far = false;
        for (int a = 0; a < 3; a++)
          far |= (dd[a] == 1 && rr[a] > mm[a] - 1 + reach[a]) || (dd[a] == -1 && rr[a] < -reach[a]);
        if (far) continue;
        // the x neighbours' items from the front, the others' from the back
        // (MAXRUNSB items at most)
        const uint32_t k = dd[1] == 0 && dd[2] == 0 ? atomicAdd(&cntx, 1u)
                                                    : MAXRUNSB - 1 - atomicAdd(&cnty, 1u);
        bhead[k] = j;
        brel[k] = pack_rel(rr[0], rr[1], rr[2]) | len << 24;
        bgr[k] = uf_find(par, j);
        lp[na + k] = na + k;
      }
      __syncthreads();
      const uint32_t nbx = cntx, nb = nbx + cnty;
      // slot of the chunk's item j
      auto item = [&](uint32_t j) -> uint32_t { return j < nbx ? j : MAXRUNSB - 1 - (j - nbx); };
      const float inb = 1.0f / (float)max(nb, 1u), inbx = 1.0f / (float)max(nbx, 1u);
      // every (home run, neighbour item) pair within reach
      if (bmap) {
        // slots (row of A, item), row-major: the touching sub-cells first,
        // then every row.  Of A's rows an item can reach, a neighbour in y
        // (z) has at most reach planes of ay (az), nearest first, on any
        // other axis the 2 reach + 1 around its own; so an x neighbour's
        // items have wy wz rows, the others' at most nr
        const uint32_t nr1 = 3, nr2 = (uint32_t)max(reach[2] * wy, reach[1] * wz);
        const uint32_t t1 = nr1 * nb + (9 - nr1) * nbx;
        const uint32_t total = t1 + nr2 * nb + ((uint32_t)(wy * wz) - nr2) * nbx;
        for (uint32_t p0 = take(2); p0 < total; p0 = take(2)) {
          const uint32_t p = p0 + lane;
          const uint32_t mr = mainr == kNone ? kNone : lfind(lp, mainr);
          uint32_t bits = 0, all = 0, r0 = 0, jb = 0;
          int x0 = 0, bx = 0, dy = 0, dz = 0;
          if (p < total) {
            const bool first = p < t1;
            const uint32_t q = first ? p : p - t1, nr = first ? nr1 : nr2, both = nr * nb;
            const int py = first ? 1 : reach[1], pz = first ? 1 : reach[2];
            uint32_t r, j;
            if (q < both) r = div_small(q, nb, inb), j = q - r * nb;
            else r = div_small(q - both, nbx, inbx), j = q - both - r * nbx, r += nr;
            jb = item(j);
            const uint32_t rb = brel[jb];
            bx = rel_x(rb);
            const int by = rel_y(rb), bz = rel_z(rb);
            const bool iny = by >= 0 && by < mm[1], inz = bz >= 0 && bz < mm[2];
            const int ny = iny ? 2 * py + 1 : py;
            const int kz = (int)r / ny, ky = (int)r - kz * ny;
            const int az = inz ? bz + zig(kz) : (bz < 0 ? kz : mm[2] - 1 - kz);
            const int ay = iny ? by + zig(ky) : (by < 0 ? ky : mm[1] - 1 - ky);
            dz = az - bz, dy = ay - by;
            const bool trow = dz >= -1 && dz <= 1 && dy >= -1 && dy <= 1;
            x0 = max(bx - reach[0], 0);
            const int x1 = min(bx + reach[0], mm[0] - 1);
            if (kz < (inz ? 2 * pz + 1 : pz) && az >= 0 && az < mm[2] && ay >= 0 && ay < mm[1] &&
                x0 <= x1 && (!first || trow) && gap_ok(0, dy, dz)) {
              const int bin0 = (az * mm[1] + ay) * mm[0] + x0;
              bits = all = rowbits(bin0, x1 - x0 + 1);
              r0 = rank(bin0);
              if (trow) bits &= first ? touchbits(bx - 1 - x0) : ~touchbits(bx - 1 - x0);
              // an item already in the dominant set: only the stragglers
              if (bits && mr != kNone && lfind(lp, na + jb) == mr) bits &= srowbits(bin0, x1 - x0 + 1);
            }
          }
          walk(bits, all, r0, x0, bx, dy, dz, na + jb, p < total ? bgr[jb] : 0u);
        }
      } else {
        const uint32_t total = (uint32_t)na * nb;
        for (uint32_t p0 = take(2); p0 < total; p0 = take(2)) {
          const uint32_t p = p0 + lane;
          const uint32_t ib = div_small(p, (uint32_t)na, ina), ia = p - ib * (uint32_t)na;
          bool any = p < total;
          uint32_t jb = 0;
          if (any) {
            jb = item(ib);
            const uint32_t rra = arel[ia], rb = brel[jb];
            any = gap_ok(rel_x(rb) - (int)(rra & 15), rel_y(rb) - (int)((rra >> 4) & 15),
                         rel_z(rb) - (int)(rra >> 8));
          }
          offer(any, ia, na + jb, any ? agr[ia] : 0u, any ? bgr[jb] : 0u);
        }
      }
      if (qn) flush(qn);
      __syncthreads();
      // commit: a neighbour run joined in LDS joins its (home-cell) root's run
      for (uint32_t j = threadIdx.x; j < nb; j += blockDim.x) {
        const uint32_t ib = item(j);
        const uint32_t r = lfind(lp, na + ib);
        if (r != na + ib) uf_union(par, bhead[ib], ahead[r]);
      }
      if (c1 < ntot) __syncthreads();  // the slots are reused by the next chunk
    }
    // commit the home cell's runs (all their merges)
    for (int ia = threadIdx.x; ia < na; ia += blockDim.x) {
      const uint32_t r = lfind(lp, ia);
      if (r != (uint32_t)ia) uf_union(par, ahead[ia], ahead[r]);
    }
    if (threadIdx.x == 0) dnext = atomicAdd(dq, 1u);
    __syncthreads();
  }
  add_counters(ctr, kCtrTestsBig, tests, rechecks, joined);
}

// ---------------------------------------------------------------------------
// 6b: small dense cells (T <= n < kBigCell particles) -- one wave per cell,
// every pair tested in registers, components by bit-matrix closure.
// ---------------------------------------------------------------------------
// At about one particle per sub-cell (the usual case for cells below 256
// particles) the sub-cell cliques of k_link_dense save few tests, while their
// run-pair enumeration costs each lane a divergent walk per candidate.  Here
// a wave tests 64 pairs per step with no branch and no memory access: each
// lane holds one particle, the partners are held one per lane and broadcast
// with readlane.  Pairs the FP32 test leaves undecided (within the band
// around l^2) are re-decided in FP64 afterwards.  Links inside the cell form a
// symmetric bit matrix in registers (lane i: rows i, i+64, ...; a ballot gives
// the transposed columns), closed transitively (Warshall: for every k, the
// rows holding k absorb row k), so each particle knows its component without
// one union per link.  Neighbour particles within reach of the cell's box are
// then tested 64 at a time against the cell; each joins the first particle it
// links to, and one that links two components merges them in an LDS
// union-find seeded with the components (the four largest components' masks
// are kept in scalar registers, so a candidate skips whole components).
// Which pairs belong to this kernel is the rule of k_link_dense: the cell's
// own pairs, its 13 forward neighbours (src_v2/FOF.c:122-153) and, for a
// constant l on a dense grid, its backward neighbours that are sparse.
//
// Each wave of a workgroup works on its own cells (no workgroup barriers);
// the neighbours' particles are read as one index space over the 26 ranges,
// two 64-particle chunks in flight, and the next cell's bounds are fetched
// while the current one is linked.
constexpr int kSmallQ = 128;    // neighbour candidates queued in LDS (< 64 + 64)
constexpr int kSmallWaves = 4;  // waves per workgroup
constexpr float kFar = 1e18f;   // position of an absent particle: links nothing

constexpr int kBlk = 4;  // partners per block of a wave's pair tests
struct SmallLds {
  // the cell's particles, x, y and z apart (the w field is not needed; the
  // float4 table cost 6 KB more per workgroup and 6% of the kernel's time),
  // then kBlk absent ones
  float ax[kBigCell + kBlk], ay[kBigCell + kBlk], az[kBigCell + kBlk];
  unsigned long long cm[4][4];       // the four largest components (bit masks)
  uint32_t lp[kBigCell];             // union-find over the cell's components
  float qx[kSmallQ], qy[kSmallQ], qz[kSmallQ];  // queued neighbour candidates
  uint32_t qidx[kSmallQ];
};

// The lane's particle (xi, yi, zi) against the kBlk partners p[0..kBlk-1]
// in LDS, the same for every lane (broadcast reads, all issued before the
// tests).  Past the cell's last particle the table holds kBlk absent ones at
// -kFar (absent lanes sit at +kFar), so a short last block needs no masking:
// nothing links them.  Returns bit k = linked under the reference's test: the FP32
// decision outside the band; when any lane has a pair inside the band, the
// block is re-decided pair by pair with pair_linked.  With COLS, cols[k] is
// the lane mask of partner k's links (the transposed block).  A re-decision
// counts in the lanes below from + k: in a tile against itself each pair comes
// up twice, and counts where the lane is the lower one.
template <bool COLS>
__device__ __forceinline__ uint32_t testblk(float xi, float yi, float zi,
                                           const float *__restrict__ px,
                                           const float *__restrict__ py,
                                           const float *__restrict__ pz, const Rule &R,
                                           uint32_t &rechecks,
                                           unsigned long long (&cols)[kBlk], int from) {
  uint32_t lk = 0;
  unsigned long long band = 0;  // lanes with an undecided pair (uniform)
  float qx[kBlk], qy[kBlk], qz[kBlk];
#pragma unroll
  for (int k = 0; k < kBlk; k++) qx[k] = px[k], qy[k] = py[k], qz[k] = pz[k];
#pragma unroll
  for (int k = 0; k < kBlk; k++) {
    const float dx = xi - qx[k], dy = yi - qy[k], dz = zi - qz[k];
    const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
    const bool l = d2 < R.lo;
    const unsigned long long c = __ballot(l);
    if (COLS) cols[k] = c;
    lk |= l ? (1u << k) : 0u;
    band |= __ballot(d2 <= R.hi) & ~c;
  }
  if (band) {  // rare: re-decide the block exactly
    lk = 0;
#pragma unroll
    for (int k = 0; k < kBlk; k++) {
      const float4 q = make_float4(qx[k], qy[k], qz[k], 0.f);
      uint32_t again = 0;
      const bool l = pair_linked(make_float4(xi, yi, zi, 0.f), q, R, again);
      if ((int)(threadIdx.x & 63) < from + k) rechecks += again;
      if (COLS) cols[k] = __ballot(l);
      lk |= l ? (1u << k) : 0u;
    }
  }
  return lk;
}

// The cell's own pairs (NW 64-particle tiles, 64 (NW - 1) < nA <= 64 NW;
// the particles in S.ax, S.ay, S.az): the link matrix, its components (breadth-first,
// by pulling: a particle joins when its row meets the frontier), each
// particle's component root (the lowest member) into lp, and the four
// largest components' masks into S.cm.
template <int NW>
__device__ __forceinline__ void small_cell_own(SmallLds &S, uint32_t nA, const Rule &R,
                                               uint32_t &rechecks) {
  const uint32_t lane = threadIdx.x & 63;
  float xr[NW], yr[NW], zr[NW];
#pragma unroll
  for (int r = 0; r < NW; r++) {
    const uint32_t i = 64 * r + lane;
    const uint32_t ic = i < nA ? i : 0;
    xr[r] = i < nA ? S.ax[ic] : kFar, yr[r] = i < nA ? S.ay[ic] : kFar;
    zr[r] = i < nA ? S.az[ic] : kFar;
  }
  unsigned long long rows[NW][NW];  // rows[r][w]: links of 64 r + lane to 64 w ..
#pragma unroll
  for (int r = 0; r < NW; r++)
#pragma unroll
    for (int w = 0; w < NW; w++) rows[r][w] = 0;
#pragma unroll
  for (int ta = 0; ta < NW; ta++) {
#pragma unroll
    for (int tb = ta; tb < NW; tb++) {
      const uint32_t jn = min(64u, nA - 64 * tb);
      for (uint32_t j0 = 0; j0 < jn; j0 += kBlk) {
        unsigned long long cols[kBlk];
        const uint32_t o = 64 * tb + j0;
        const uint32_t h =
            testblk<true>(xr[ta], yr[ta], zr[ta], S.ax + o, S.ay + o, S.az + o, R, rechecks, cols,
                          ta == tb ? (int)j0 : 64);
        rows[ta][tb] |= (unsigned long long)h << j0;
        if (tb != ta) {  // the transposed block: rows of 64 tb + j0 + k, word ta
#pragma unroll
          for (int k = 0; k < kBlk; k++)
            if (lane == j0 + k) rows[tb][ta] = cols[k];
        }
      }
    }
  }
  // particles present, and those linked to none (their own component)
  unsigned long long unv[NW];
#pragma unroll
  for (int r = 0; r < NW; r++) {
    const uint32_t n = min(64u, nA - 64 * r);
    const unsigned long long present = n >= 64 ? ~0ull : ((1ull << n) - 1);
    unsigned long long other = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) other |= (w == r) ? (rows[r][w] & ~(1ull << lane)) : rows[r][w];
    const unsigned long long iso = __ballot(other == 0) & present;
    if ((iso >> lane) & 1ull) S.lp[64 * r + lane] = 64 * r + lane;
    unv[r] = present & ~iso;
  }
  uint32_t csz[4] = {0, 0, 0, 0};
  unsigned long long cmask[4][NW];
#pragma unroll
  for (int c = 0; c < 4; c++)
#pragma unroll
    for (int w = 0; w < NW; w++) cmask[c][w] = 0;
  for (;;) {
    int sw = -1;
#pragma unroll
    for (int w = NW - 1; w >= 0; w--)
      if (unv[w]) sw = w;
    if (sw < 0) break;
    unsigned long long comp[NW], F[NW];
#pragma unroll
    for (int w = 0; w < NW; w++) {
      comp[w] = (w == sw) ? (unv[w] & (~unv[w] + 1)) : 0ull;  // the seed: lowest unvisited
      F[w] = comp[w];
      unv[w] &= ~comp[w];
    }
    uint32_t seed = 0;
#pragma unroll
    for (int w = 0; w < NW; w++)
      if (comp[w]) seed = 64 * w + (uint32_t)__builtin_ctzll(comp[w]);
    for (;;) {
      unsigned long long nx[NW], any = 0;
#pragma unroll
      for (int r = 0; r < NW; r++) {
        unsigned long long meet = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) meet |= rows[r][w] & F[w];
        nx[r] = __ballot(meet != 0) & unv[r];
        any |= nx[r];
      }
      if (!any) break;
#pragma unroll
      for (int r = 0; r < NW; r++) comp[r] |= nx[r], unv[r] &= ~nx[r], F[r] = nx[r];
    }
    uint32_t size = 0;
#pragma unroll
    for (int r = 0; r < NW; r++) {
      if ((comp[r] >> lane) & 1ull) S.lp[64 * r + lane] = seed;
      size += (uint32_t)__popcll(comp[r]);
    }
    // keep the four largest (descending)
#pragma unroll
    for (int c = 0; c < 4; c++) {
      if (size > csz[c]) {
        const uint32_t ts = csz[c];
        csz[c] = size;
        size = ts;
#pragma unroll
        for (int w = 0; w < NW; w++) {
          const unsigned long long tm = cmask[c][w];
          cmask[c][w] = comp[w];
          comp[w] = tm;
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 4; c++)
#pragma unroll
    for (int w = 0; w < NW; w++)
      if (lane == 0) S.cm[c][w] = cmask[c][w];
}

// One cell of NW 64-particle tiles (64 (NW - 1) < nA <= 64 NW): its own
// pairs, its neighbours' particles, the commit.  nxt: the wave's next cell
// (kNone: none), whose bounds are fetched into nS, nE on the way.
template <int NW>
__device__ __forceinline__ void small_cell(SmallLds &S, uint32_t sA, uint32_t nA,
                                           const VolDev &V, const CellPos &cp, const Rule &R,
                                           uint32_t nbS, uint32_t nbN,
                                           const float4 *__restrict__ pos4, const Grid &G,
                                           uint32_t *__restrict__ par, uint32_t nxt,
                                           uint32_t part, uint32_t parts, uint32_t &nS, uint32_t &nE, uint32_t &tests,
                                           uint32_t &rechecks) {
  const uint32_t lane = threadIdx.x & 63;
  volatile uint32_t *const lp = S.lp;
  // (A, A), in every part and counted in the first
  uint32_t again = 0;
  small_cell_own<NW>(S, nA, R, again);
  rechecks += part == 0 ? again : 0u;
  tests += (lane == 0 && part == 0) ? nA * (nA - 1) / 2 : 0u;
  wave_sync();
  // the next cell's bounds (its index has arrived by now)
  if (nxt != kNone) nS = G.start[nxt], nE = G.start[nxt + 1];
  // (A, B): the 26 ranges as one index space: off = exclusive prefix
  uint32_t off = nbN;
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) {
    const uint32_t t = __shfl_up(off, o, 64);
    if (lane >= (uint32_t)o) off += t;
  }
  const uint32_t total = __shfl(off, 25, 64);
  off -= nbN;
  // the bounding box of the cell's particles: a neighbour particle farther
  // than l from it links to none of them (prune2 carries a 1e-4 margin on
  // l^2; the gap is evaluated in FP64 from the float coordinates)
  double lo[3], hi[3];
  {
    float mn[3] = {kFar, kFar, kFar}, mx[3] = {-kFar, -kFar, -kFar};
#pragma unroll
    for (int r = 0; r < NW; r++) {
      const uint32_t i = 64 * r + lane;
      if (i < nA) {
        const float qx = S.ax[i], qy = S.ay[i], qz = S.az[i];
        mn[0] = fminf(mn[0], qx), mn[1] = fminf(mn[1], qy), mn[2] = fminf(mn[2], qz);
        mx[0] = fmaxf(mx[0], qx), mx[1] = fmaxf(mx[1], qy), mx[2] = fmaxf(mx[2], qz);
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
      for (int a = 0; a < 3; a++) {
        mn[a] = fminf(mn[a], __shfl_xor(mn[a], o, 64));
        mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], o, 64));
      }
#pragma unroll
    for (int a = 0; a < 3; a++) lo[a] = mn[a], hi[a] = mx[a];
  }
  // index g of the space -> particle, for the 64 consecutive indices g0 +
  // lane: only the ranges from the one holding g0 to the one holding the
  // chunk's last index are scanned
  auto locate = [&](uint32_t g0) -> uint32_t {
    const uint32_t g = g0 + lane, gl = min(g0 + 63u, total - 1u);
    const unsigned long long la = __ballot(lane < 26 && off <= g0);
    const unsigned long long lb = __ballot(lane < 26 && off <= gl);
    const int ka = 63 - __clzll(la), kb = 63 - __clzll(lb);
    uint32_t base = (uint32_t)__builtin_amdgcn_readlane((int)nbS, ka) -
                    (uint32_t)__builtin_amdgcn_readlane((int)off, ka);
    for (int k = ka + 1; k <= kb; k++) {
      const uint32_t ok = (uint32_t)__builtin_amdgcn_readlane((int)off, k);
      const uint32_t sk = (uint32_t)__builtin_amdgcn_readlane((int)nbS, k);
      if (g >= ok) base = sk - ok;
    }
    return base + g;
  };
  uint32_t qn = 0;  // uniform
  auto flush = [&](uint32_t cnt) {
    wave_sync();
    const bool vb = lane < cnt;
    const uint32_t lq = vb ? lane : 0;
    const uint32_t jb = S.qidx[lq];
    const float bx = vb ? S.qx[lq] : kFar, by = vb ? S.qy[lq] : kFar, bz = vb ? S.qz[lq] : kFar;
    tests += vb ? nA : 0u;
    unsigned long long m[NW];
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const uint32_t jn = min(64u, nA - 64 * w);
      unsigned long long mw = 0;
      for (uint32_t j0 = 0; j0 < jn; j0 += kBlk) {
        unsigned long long cols[kBlk];
        const uint32_t o = 64 * w + j0;
        mw |= (unsigned long long)testblk<false>(bx, by, bz, S.ax + o, S.ay + o, S.az + o, R,
                                                 rechecks, cols, 64)
              << j0;
      }
      m[w] = vb ? mw : 0ull;
    }
    // join the first linked particle; every further component linked
    // merges with its component
    bool any = false;
#pragma unroll
    for (int q = 0; q < NW; q++) any |= m[q] != 0;
    if (any) {
      int i0 = -1;
#pragma unroll
      for (int q = NW - 1; q >= 0; q--)
        if (m[q]) i0 = 64 * q + __builtin_ctzll(m[q]);
      uf_union(par, jb, sA + (uint32_t)i0);
#pragma unroll
      for (int c = 0; c < 4; c++) {
        bool hit = false;
#pragma unroll
        for (int q = 0; q < NW; q++) hit |= (m[q] & S.cm[c][q]) != 0;
        if (!hit) continue;
        int ic0 = -1;
#pragma unroll
        for (int q = NW - 1; q >= 0; q--)
          if (m[q] & S.cm[c][q]) ic0 = 64 * q + __builtin_ctzll(m[q] & S.cm[c][q]);
        lunion(lp, (uint32_t)i0, (uint32_t)ic0);
#pragma unroll
        for (int q = 0; q < NW; q++) m[q] &= ~S.cm[c][q];
      }
      // members of smaller components, one at a time
      for (;;) {
        int i = -1;
#pragma unroll
        for (int q = NW - 1; q >= 0; q--)
          if (m[q]) i = 64 * q + __builtin_ctzll(m[q]);
        if (i < 0) break;
        lunion(lp, (uint32_t)i0, (uint32_t)i);
#pragma unroll
        for (int q = 0; q < NW; q++)
          if (q == (i >> 6)) m[q] &= m[q] - 1;
      }
    }
    wave_sync();
  };
  auto push = [&](float4 pb, uint32_t j, bool valid) {
    bool keep = false;
    if (valid) {
      const double x = pb.x, y = pb.y, z = pb.z;
      const double gx = fmax(fmax(lo[0] - x, x - hi[0]), 0.0);
      const double gy = fmax(fmax(lo[1] - y, y - hi[1]), 0.0);
      const double gz = fmax(fmax(lo[2] - z, z - hi[2]), 0.0);
      keep = !(gx * gx + gy * gy + gz * gz > R.prune2);
    }
    const unsigned long long bal = __ballot(keep);
    if (keep) {
      const uint32_t at = qn + (uint32_t)__popcll(bal & ((1ull << lane) - 1));
      S.qx[at] = pb.x, S.qy[at] = pb.y, S.qz[at] = pb.z;
      S.qidx[at] = j;
    }
    qn += (uint32_t)__popcll(bal);
    if (qn >= 64) {
      flush(64);
      // move the overflow down (qn - 64 < 64 entries)
      const bool mv = lane < qn - 64;
      const uint32_t lm = 64 + (mv ? lane : 0);
      const float tx = S.qx[lm], ty = S.qy[lm], tz = S.qz[lm];
      const uint32_t ti = S.qidx[lm];
      wave_sync();
      if (mv) S.qx[lane] = tx, S.qy[lane] = ty, S.qz[lane] = tz, S.qidx[lane] = ti;
      qn -= 64;
    }
  };
  for (uint32_t g0 = 128 * part; g0 < total; g0 += 128 * parts) {
    const uint32_t ga = g0 + lane, gb = g0 + 64 + lane;
    const bool va = ga < total, vb = gb < total;
    const uint32_t ja = locate(g0);
    const uint32_t jb = g0 + 64 < total ? locate(g0 + 64) : 0u;
    const float4 pa = va ? ld4(pos4 + ja) : make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 pb = vb ? ld4(pos4 + jb) : make_float4(0.f, 0.f, 0.f, 0.f);
    push(pa, ja, va);
    if (g0 + 64 < total) push(pb, jb, vb);
  }
  if (qn) flush(qn);
  wave_sync();
  // commit the cell's components (and the merges made through
  // neighbours): a particle still its own global root is hooked under its
  // component's root with one CAS (the root is lower: larger-under-
  // smaller), any other joins by union
  for (uint32_t i = lane; i < nA; i += 64) {
    const uint32_t r = lfind(lp, i);
    if (r != i && atomicCAS(par + sA + i, sA + i, sA + r) != sA + i) uf_union(par, sA + i, sA + r);
  }
  wave_sync();
}

// Five waves per SIMD (at most 96 VGPRs, a few spilled).  On the clumpy
// 1024^3 box: 33.4 ms with blocks of 8 partners and no cap (134 VGPRs, three
// waves), 28.3 ms at four waves, 25.0 ms with blocks of 4 at five, 23.5 ms
// with the x, y, z tables; six waves (80 VGPRs) spill enough to take 31.4 ms.
// Waves a cell's neighbour particles are split over while there are few cells
// (each part links the cell's own particles anew).  The kernel then waits for
// its largest cell, whose candidates one wave tests 64 at a time: in the 64^3
// box 230 particles against 1096 candidates took all of its 290 us, eight times
// the mean cell.  Eight parts while all still run at once, beyond that only for
// the larger cells: 64^3 box (815 cells) 291 -> 125 us, 144^3 (8e3) 427 -> 269,
// 192^3 (2.2e4) 565 -> 434, 256^3 (4.2e4) 881 -> 754; 512^3 (3.2e5) is not split
// (3.6 ms either way).
__device__ __forceinline__ uint32_t small_parts(uint32_t cells) {
  return cells <= 512u ? 8u : cells <= 16384u ? 4u : cells <= 49152u ? 2u : 1u;
}

__global__ __launch_bounds__(64 * kSmallWaves) __attribute__((amdgpu_waves_per_eu(5))) void k_link_small(
    const uint32_t *__restrict__ dense, const uint32_t *__restrict__ ndense,
    const float4 *__restrict__ pos4, const Grid G, uint32_t T, uint32_t *__restrict__ par,
    const VolDev *__restrict__ vols, const uint32_t *__restrict__ vbeg, int nvol,
    unsigned long long *__restrict__ ctr) {
  // the wave's index, made visibly uniform so that the cell's bounds, its
  // particles as partners and the scan state live in scalar registers
  const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  __shared__ SmallLds Sall[kSmallWaves];
  SmallLds &S = Sall[wv];
  uint32_t tests = 0, rechecks = 0;
  const uint32_t lane = threadIdx.x & 63;
  // work items: (cell, part), `parts` (a power of two) to a cell
  const uint32_t parts = small_parts(*ndense);
  const uint32_t psh = (uint32_t)__builtin_ctz(parts);
  const uint32_t nd = *ndense << psh;
  const uint32_t w0 = blockIdx.x * kSmallWaves + wv;
  const uint32_t ws = gridDim.x * kSmallWaves;
  // bounds of the wave's next cell, fetched ahead
  uint32_t nS = 0, nE = 0;
  if (w0 < nd) {
    const uint32_t c = dense[w0 >> psh];
    nS = G.start[c], nE = G.start[c + 1];
  }
  for (uint32_t d = w0; d < nd; d += ws) {
    const uint32_t part = d & (parts - 1);
    const uint32_t sA = nS, nA = nE - nS;  // T <= nA < kBigCell
    const uint32_t cN = (d + ws < nd) ? dense[(d + ws) >> psh] : 0u;
    // only cells worth it: the others are their first part's alone
    const uint32_t mine = parts == 8 ? 8u : min(parts, nA >= 160 ? 4u : nA >= 96 ? 2u : 1u);
    if (part >= mine) {
      if (d + ws < nd) nS = G.start[cN], nE = G.start[cN + 1];
      continue;
    }
    const VolDev &V = vols[vol_of(vbeg, nvol, sA)];
    const float4 p0 = pos4[sA];
    for (uint32_t i = lane; i < nA; i += 64) {
      const float4 q = ld4(pos4 + sA + i);
      S.ax[i] = q.x, S.ay[i] = q.y, S.az[i] = q.z;
    }
    if (lane < (uint32_t)kBlk) S.ax[nA + lane] = -kFar, S.ay[nA + lane] = -kFar, S.az[nA + lane] = -kFar;
    const CellPos cp = cell_pos(V, p0.x, p0.y, p0.z);
    const Rule R = make_rule(V, cp.ix, cp.iy, cp.iz);
    // neighbour k of the table (lane k): its particle range
    uint32_t nbS = 0, nbN = 0;
    if (lane < 26) {
      int dd[3];
      nb_offset((int)lane, dd);
      const int bx = cp.ix + dd[0], by = cp.iy + dd[1], bz = cp.iz + dd[2];
      const bool want = lane < 13 || (!G.sparse && V.vntab == 0 && V.m[0] > 0);
      if (want && !(bx < 0 || bx >= V.nx || by < 0 || by >= V.ny || bz < 0 || bz >= V.nz)) {
        const uint32_t cb = cell_index(G, V, bx, by, bz);
        if (cb != kNone) nbS = G.start[cb], nbN = G.start[cb + 1] - nbS;
      }
      if (lane >= 13 && nbN >= T) nbN = 0;  // a dense backward cell links this pair itself
    }
    wave_sync();
    const uint32_t nw = (nA + 63) >> 6;
    const uint32_t nxt = (d + ws < nd) ? cN : kNone;
    if (nw <= 1) small_cell<1>(S, sA, nA, V, cp, R, nbS, nbN, pos4, G, par, nxt, part, mine, nS, nE, tests, rechecks);
    else if (nw == 2) small_cell<2>(S, sA, nA, V, cp, R, nbS, nbN, pos4, G, par, nxt, part, mine, nS, nE, tests, rechecks);
    else if (nw == 3) small_cell<3>(S, sA, nA, V, cp, R, nbS, nbN, pos4, G, par, nxt, part, mine, nS, nE, tests, rechecks);
    else small_cell<4>(S, sA, nA, V, cp, R, nbS, nbN, pos4, G, par, nxt, part, mine, nS, nE, tests, rechecks);
  }
  add_counters(ctr, kCtrTestsSmall, tests, rechecks);
}

// ---------------------------------------------------------------------------
// 7: union-find finish
// ---------------------------------------------------------------------------
// Particle ID of input record p (the reference's P[p].ID, src_v2/vars.h:36-47).
__device__ __forceinline__ unsigned long long rec_id(const uint8_t *__restrict__ base,
                                                     uint32_t stride, uint32_t offid, uint32_t p) {
  const uint32_t *q = reinterpret_cast<const uint32_t *>(base + (uint64_t)p * stride + offid);
  return (unsigned long long)q[0] | ((unsigned long long)q[1] << 32);
}

// Flatten every particle to its root; the other members of a group
// accumulate their minimum input index and their count at the root (minorig
// and gsize start at ~0 and 0; the root itself is added in k_label).  With
// idroot, the members' minimum particle ID is accumulated the same way.
__global__ __launch_bounds__(256) void k_flatten(uint32_t N, uint32_t *__restrict__ par,
                                                 const float4 *__restrict__ pos4,
                                                 uint32_t *__restrict__ minorig,
                                                 uint32_t *__restrict__ gsize,
                                                 unsigned long long *__restrict__ ctr,
                                                 const uint8_t *__restrict__ base, uint32_t stride,
                                                 uint32_t offid,
                                                 unsigned long long *__restrict__ idroot) {
  uint32_t roots = 0;
  const uint32_t lane = threadIdx.x & 63;
  // wave-uniform loop: lanes of a wave reduce together
  for (uint32_t xb = blockIdx.x * blockDim.x + (threadIdx.x & ~63u); xb < N;
       xb += gridDim.x * blockDim.x) {
    const uint32_t x = xb + lane;
    uint32_t r = x;
    bool member = false;
    if (x < N) {
      uint32_t p = par[x];
      while (p != r) {
        r = p;
        p = par[r];
      }
      member = (r != x);
      if (member) par[x] = r;
      else roots++;
    }
    const uint32_t o = member ? __float_as_uint(pos4[x].w) : 0xFFFFFFFFu;
    // members of one group are mostly neighbours in the cell order: one
    // atomicMin / atomicAdd per distinct root in the wave
    unsigned long long pend = __ballot(member);
    while (pend) {
      const int leader = __ffsll((long long)pend) - 1;
      const uint32_t rl = __shfl(r, leader, 64);
      const bool mine = member && r == rl;
      const unsigned long long m = __ballot(mine);
      uint32_t v = mine ? o : 0xFFFFFFFFu;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) v = min(v, (uint32_t)__shfl_xor(v, off, 64));
      if ((int)lane == leader) {
        atomicMin(minorig + rl, v);
        atomicAdd(gsize + rl, (uint32_t)__popcll(m));
      }
      if (idroot) {
        unsigned long long id = mine ? rec_id(base, stride, offid, o) : ~0ull;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
          const unsigned long long t = __shfl_xor(id, off, 64);
          id = t < id ? t : id;
        }
        if ((int)lane == leader) atomicMin(idroot + rl, id);
      }
      pend &= ~m;
    }
  }
  uint64_t t = roots;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o, 64);
  if ((threadIdx.x & 63) == 0 && t) ctr_add(ctr, kCtrGroups, t);
}

// Does a particle of run a (na of them) link to one of run b?  By a whole
// wave: particles of a farther than l from the box of b are passed over 64 at
// a time, each of the others is tested against b.  prune2 (l^2 with a margin of
// 1e-4) is compared with differences of floats that are no larger than those
// of the pairs, so nothing that links is passed over.  Two sub-cells of 20001
// and 20000 particles 1.2 l apart took 5.2 s pair by pair, now 0.1 ms.
__device__ __forceinline__ bool wave_runs_link(const float4 *__restrict__ a, uint32_t na,
                                               const float4 *__restrict__ b, uint32_t nb,
                                               const Rule &R, uint32_t &tests,
                                               uint32_t &rechecks) {
  const uint32_t lane = threadIdx.x & 63;
  const float gp2 = (float)R.prune2;
  float lo[3], hi[3];
  {
    const float4 q = ld4(b);
    lo[0] = hi[0] = q.x, lo[1] = hi[1] = q.y, lo[2] = hi[2] = q.z;
  }
  for (uint32_t j = lane; j < nb; j += 64) {
    const float4 q = ld4(b + j);
    lo[0] = fminf(lo[0], q.x), lo[1] = fminf(lo[1], q.y), lo[2] = fminf(lo[2], q.z);
    hi[0] = fmaxf(hi[0], q.x), hi[1] = fmaxf(hi[1], q.y), hi[2] = fmaxf(hi[2], q.z);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int d = 0; d < 3; d++) {
      lo[d] = fminf(lo[d], __shfl_xor(lo[d], o, 64));
      hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], o, 64));
    }
  for (uint32_t i0 = 0; i0 < na; i0 += 64) {
    const float4 p = ld4(a + min(i0 + lane, na - 1));
    const float gx = fmaxf(fmaxf(lo[0] - p.x, p.x - hi[0]), 0.f);
    const float gy = fmaxf(fmaxf(lo[1] - p.y, p.y - hi[1]), 0.f);
    const float gz = fmaxf(fmaxf(lo[2] - p.z, p.z - hi[2]), 0.f);
    unsigned long long near = __ballot(i0 + lane < na && !(gx * gx + gy * gy + gz * gz > gp2));
    while (near) {
      const int l = __builtin_ctzll(near);
      near &= near - 1;
      auto at = [&](float f) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), l)); };
      const float4 q = make_float4(at(p.x), at(p.y), at(p.z), 0.f);
      for (uint32_t j = lane; j - lane < nb; j += 64) {
        bool hit = false;
        if (j < nb) {
          tests++;
          hit = pair_linked(q, ld4(b + j), R, rechecks);
        }
        if (__ballot(hit)) return true;
      }
    }
  }
  return false;
}

// The accumulators of k_flatten (minimum index, with idroot minimum ID; sizes
// where the bucket sort has not cleared them) and the label bitmap.  Also
// the listed pairs of long runs, a wave each unless they are joined by now:
// k_link_dense has no register to spare for them (10% slower) and a
// launch of their own costs every call 3 us.
__global__ __launch_bounds__(256) void k_init_groups(uint32_t N, uint32_t *__restrict__ minorig,
                                                     unsigned long long *__restrict__ idroot,
                                                     uint32_t *__restrict__ gsize,
                                                     uint32_t nw, uint32_t *__restrict__ bits,
                                                     const float4 *__restrict__ pos4,
                                                     uint32_t *__restrict__ par,
                                                     const VolDev *__restrict__ vols,
                                                     const uint32_t *__restrict__ vbeg, int nvol,
                                                     unsigned long long *__restrict__ ctr) {
  const uint32_t n = min(*wide_count(ctr), kWideCap);
  for (uint32_t x = blockIdx.x * blockDim.x + threadIdx.x; x < N; x += gridDim.x * blockDim.x) {
    minorig[x] = ~0u;
    if (idroot) idroot[x] = ~0ull;
    if (gsize) gsize[x] = 0;
    if (x < nw) bits[x] = 0;
  }
  const uint32_t w0 = blockIdx.x * 4 + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (w0 >= n) return;
  const uint32_t lane = threadIdx.x & 63;
  uint32_t tests = 0, rechecks = 0, joined = 0;
  for (uint32_t k = w0; k < n; k += gridDim.x * 4) {
    const uint4 e = *wide_pair(ctr, k);
    uint32_t v = 0;
    if (lane == 0) v = uf_find(par, e.x) == uf_find(par, e.z) ? 1u : 0u;
    if (__builtin_amdgcn_readfirstlane((int)v)) {
      joined += v;
      continue;
    }
    const VolDev &V = vols[vol_of(vbeg, nvol, e.x)];
    const float4 p = pos4[e.x];
    const CellPos cp = cell_pos(V, p.x, p.y, p.z);
    const Rule R = make_rule(V, cp.ix, cp.iy, cp.iz);
    if (wave_runs_link(pos4 + e.x, e.y, pos4 + e.z, e.w, R, tests, rechecks) && lane == 0)
      uf_union(par, e.x, e.z);
  }
  add_counters(ctr, kCtrTestsBig, tests, rechecks, joined);
}

// Members of groups of two or more: label[orig] = group minimum index |
// kFlag, and each member's (label, orig) at the next free slot of its group
// in the member list (the group's cursor, indexed by its label, starts
// at the group's first slot; lanes of one group take consecutive slots with
// one atomic).  The head's entry of hsize receives the group size.  Two ways
// to write the index-ordered label array from the cell-ordered particles:
//  DIRECT  random 4-byte writes straight into label -- when every volume's
//          label range is small enough to stay in the last-level cache
//          while its cells are processed (the 4^3-batched 1024^3 box: 11 ms
//          less than the partitioned writes); with label_out given (no
//          minimum-ID output wanted) straight into the caller's output, as
//          volume-local labels over the defaults the key pass wrote;
//  else    scatter_u32 from the member list afterwards, partitioned by index
//          (one 1.09e9-particle volume: 4 ms less than direct writes spread
//          over 4.4 GB).
constexpr uint32_t kLabTile = 4096;
// Largest volume (particles) written directly: 400 MB of labels, past the 256
// MB last-level cache.  Whole calls on one periodic box, direct against
// partitioned: 2.9e7 particles 5.74 against 5.87 ms, 3.8e7 7.46 / 7.70, 6.7e7
// 12.7 / 13.2, 1.39e8 27.4 / 27.4, 2.7e8 54.9 / 53.3; with minimum IDs 6.7e7
// 14.55 / 14.78, 9.5e7 21.1 / 21.1, 1.3e8 29.1 / 28.4.
constexpr uint64_t kDirectMax = 3ull << 25;

template <bool DIRECT>
__global__ __launch_bounds__(256) void k_label(uint32_t N, const uint32_t *__restrict__ par,
                                               const float4 *__restrict__ pos4,
                                               const uint32_t *__restrict__ minorig,
                                               const uint32_t *__restrict__ gsize,
                                               uint32_t *__restrict__ out,
                                               uint32_t *__restrict__ hsize,
                                               uint32_t *__restrict__ cursor,
                                               uint32_t *__restrict__ mkey,
                                               uint32_t *__restrict__ mval,
                                               const uint8_t *__restrict__ base, uint32_t stride,
                                               uint32_t offid,
                                               const unsigned long long *__restrict__ idroot,
                                               unsigned long long *__restrict__ idhead, int single,
                                               const VolDev *__restrict__ vols,
                                               const uint32_t *__restrict__ vbeg, int nvol,
                                               uint32_t *__restrict__ label_out) {
  const uint32_t lane = threadIdx.x & 63;
  const unsigned long long lt = (1ull << lane) - 1;
  const uint64_t x0 = (uint64_t)blockIdx.x * kLabTile;
  // the tile's volume base when the tile lies in one volume (volumes are
  // contiguous in the cell order too), else looked up per particle
  uint32_t btile = kNone;
  if (DIRECT && label_out && x0 < N) {
    const int va = vol_of(vbeg, nvol, (uint32_t)x0);
    if (min((uint64_t)N, x0 + kLabTile) <= vbeg[va + 1]) btile = vbeg[va];
  }
  for (uint32_t q = 0; q < kLabTile; q += 256) {
    const uint64_t xx = x0 + q + threadIdx.x;
    bool mem = false;
    uint32_t o = 0, lab = 0, r = 0;
    if (xx < N) {
      const uint32_t x = (uint32_t)xx;
      r = par[x];
      const uint32_t g = gsize[r];
      // singletons: their defaults are written, unless their volume keeps
      // groups of one (those join the member list)
      if (!(r == x && g == 0) || (single && !(1.0 < vols[vol_of(vbeg, nvol, x)].nphalomin))) {
        mem = true;
        o = __float_as_uint(pos4[x].w);
        const uint32_t orr = (r == x) ? o : __float_as_uint(pos4[r].w);
        lab = min(minorig[r], orr);
        if (DIRECT && label_out)  // straight to the output, volume-local
          label_out[o] = lab - (btile != kNone ? btile : vbeg[vol_of(vbeg, nvol, x)]);
        else if (DIRECT)
          out[o] = lab | kFlag;
        if (o == lab) {
          hsize[lab] = g + 1u;
          if (idhead) {  // the root's own ID joins the members' minimum
            const unsigned long long a = idroot[r], b = rec_id(base, stride, offid, orr);
            idhead[lab] = a < b ? a : b;
          }
        }
      }
    }
    // member-list slots: the wave's first few groups one atomic each (a
    // wave's particles are mostly in one or two groups), any other lane its own
    unsigned long long todo = __ballot(mem);
    for (int it = 0; it < 4 && todo; it++) {
      const int first = __builtin_ctzll(todo);
      const uint32_t l0 = (uint32_t)__builtin_amdgcn_readlane((int)lab, first);
      const bool mine = mem && lab == l0;
      const unsigned long long same = __ballot(mine);
      uint32_t b = 0;
      if ((int)lane == first) b = atomicAdd(cursor + l0, (uint32_t)__popcll(same));
      b = (uint32_t)__builtin_amdgcn_readlane((int)b, first);
      if (mine) {
        const uint32_t slot = b + (uint32_t)__popcll(same & lt);
        mkey[slot] = lab;
        mval[slot] = o;
      }
      todo &= ~same;
    }
    if ((todo >> lane) & 1ull) {
      const uint32_t slot = atomicAdd(cursor + lab, 1u);
      mkey[slot] = lab;
      mval[slot] = o;
    }
  }
}

// Streaming kernels whose elements' volumes are looked up per wave take one
// contiguous tile of kTileN elements per block, so that a wave's next
// elements usually lie in the volume of its last ones (the hint of
// vol_of_run); a grid-stride loop would jump across volumes every step.
constexpr uint32_t kTileN = 4096;
static inline uint32_t tiles_for(uint64_t n) { return (uint32_t)std::max<uint64_t>(1, (n + kTileN - 1) / kTileN); }

// Every particle as a singleton (label = own index, group size 1, kept only
// when Nphalomin <= 1); k_label overwrites the members of larger groups.
__global__ __launch_bounds__(256) void k_label_init(uint32_t N, const VolDev *__restrict__ vols,
                                                    const uint32_t *__restrict__ vbeg, int nvol,
                                                    uint32_t *__restrict__ label,
                                                    uint32_t *__restrict__ hsize) {
  const uint64_t i0 = (uint64_t)blockIdx.x * kTileN, i1 = min((uint64_t)N, i0 + kTileN);
  if (i0 >= i1) return;
  auto body = [&](uint32_t i, double nphalomin) {
    label[i] = i | (!(1.0 < nphalomin) ? kFlag : 0u);
    hsize[i] = 1u;
  };
  const int va = vol_of(vbeg, nvol, (uint32_t)i0);
  if (i1 <= vbeg[va + 1]) {  // the tile lies in one volume
    const double nph = vols[va].nphalomin;
    for (uint32_t i = (uint32_t)i0 + threadIdx.x; i < i1; i += blockDim.x) body(i, nph);
    return;
  }
  int hint = va;
  for (uint32_t i = (uint32_t)i0 + threadIdx.x; i < i1; i += blockDim.x)
    body(i, vols[vol_of_run(vbeg, nvol, i, N, hint)].nphalomin);
}

// Outputs for every particle: label_out (volume-local), for particles not in
// the sorted list the trivial ring entry next = self (1-based), and the
// group's minimum particle ID (own ID for a singleton).
__global__ __launch_bounds__(256) void k_out_init(uint32_t N, const uint32_t *__restrict__ label,
                                                  const uint32_t *__restrict__ vbeg, int nvol,
                                                  uint32_t *__restrict__ label_out,
                                                  uint32_t *__restrict__ next_out,
                                                  const uint32_t *__restrict__ hsize,
                                                  const uint8_t *__restrict__ base, uint32_t stride,
                                                  uint32_t offid,
                                                  const unsigned long long *__restrict__ idhead,
                                                  unsigned long long *__restrict__ minid_out) {
  const uint64_t i0 = (uint64_t)blockIdx.x * kTileN, i1 = min((uint64_t)N, i0 + kTileN);
  if (i0 >= i1) return;
  auto body = [&](uint32_t i, uint32_t b) {
    const uint32_t l = label[i];
    const uint32_t head = l & ~kFlag;
    if (label_out) label_out[i] = head - b;
    if (next_out && !(l & kFlag)) next_out[i] = i - b + 1u;
    if (minid_out)
      minid_out[i] = (head == i && hsize[i] == 1u) ? rec_id(base, stride, offid, i) : idhead[head];
  };
  const int va = vol_of(vbeg, nvol, (uint32_t)i0);
  if (i1 <= vbeg[va + 1]) {  // the tile lies in one volume
    const uint32_t b = vbeg[va];
    for (uint32_t i = (uint32_t)i0 + threadIdx.x; i < i1; i += blockDim.x) body(i, b);
    return;
  }
  int hint = va;
  for (uint32_t i = (uint32_t)i0 + threadIdx.x; i < i1; i += blockDim.x)
    body(i, vbeg[vol_of_run(vbeg, nvol, i, N, hint)]);
}

// Ring in ascending index order over the label-sorted list (1-based,
// volume-local successors), and halo starts.  The entries go straight into
// next_out, or, with pidx, leave as (index, successor) pairs in list order
// for scatter_u32 (the choice of k_label).
// ---------------------------------------------------------------------------
// The member list: every group of two or more as one segment, segments in
// ascending label (head index) order, members inside a segment in ascending
// input index -- the order of the reference's rings (src_v2/FOF.c:359-373
// joins rings so that each runs up the input order from its head) and of its
// halo loops (src_v2/FOF.c:797-847).  Built without sorting the members by
// label: the groups' roots are sorted by label (one entry per group), a scan
// of their sizes gives each segment's first slot, k_label puts every member
// in its segment, and each segment is then sorted by index on its own.
// ---------------------------------------------------------------------------
// The group list in label order without a sort: each group of two or more
// (and, where a volume keeps groups of one -- Nphalomin <= 1 -- each such
// particle) sets the bit of its label (the group's lowest input index) in a
// bitmap over the input indices and puts its size at lsize[label].  Blocks of
// consecutive words then total their groups, members and halos (groups passing
// the size cut) in k_group_sums, and k_group_emit, each block behind the totals
// of those before it, lists in label order each group's first member slot and
// the halos' first slots, and sets its cursor (by label).  Two launches
// in place of thirteen (bit counts, two scans, the list, the cursors, the halo
// flags and their compaction), which is what a small call waits for; the sizes
// are gathered twice for it.
__global__ __launch_bounds__(256) void k_group_bits(uint32_t N, const uint32_t *__restrict__ par,
                                                    const uint32_t *__restrict__ gsize,
                                                    const uint32_t *__restrict__ minorig,
                                                    const float4 *__restrict__ pos4,
                                                    uint32_t *__restrict__ bits,
                                                    uint32_t *__restrict__ lsize, int single,
                                                    const VolDev *__restrict__ vols,
                                                    const uint32_t *__restrict__ vbeg, int nvol) {
  for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < N; j += gridDim.x * blockDim.x) {
    if (par[j] != j) continue;
    const uint32_t g = gsize[j];
    if (g == 0 && (!single || 1.0 < vols[vol_of(vbeg, nvol, j)].nphalomin)) continue;
    const uint32_t lab = min(minorig[j], __float_as_uint(pos4[j].w));  // minorig: ~0 alone
    atomicOr(bits + (lab >> 5), 1u << (lab & 31));
    lsize[lab] = g + 1u;
  }
}

constexpr uint32_t kGroupBlocks = 4096;  // at most: each block reads the totals before it

// Words of a block: kGroupWords(nw) consecutive runs of 256.
static inline uint32_t group_runs(uint64_t nw) {
  return (uint32_t)((nw + 256ull * kGroupBlocks - 1) / (256ull * kGroupBlocks));
}

struct GroupTot {
  uint32_t groups, members, halos, pad;
};

// One bitmap word's groups, members and halos (labels ascend with the bits).
template <class F>
__device__ __forceinline__ void word_groups(uint32_t m, uint64_t w,
                                            const uint32_t *__restrict__ lsize,
                                            const VolDev *__restrict__ vols,
                                            const uint32_t *__restrict__ vbeg, int nvol, F f) {
  int v = -1;
  while (m) {
    const uint32_t lab = (uint32_t)(w * 32) + (uint32_t)__builtin_ctz(m);
    m &= m - 1;
    if (v < 0 || lab >= vbeg[v + 1]) v = vol_of(vbeg, nvol, lab);
    const uint32_t n = lsize[lab];
    f(lab, n, !((double)n < vols[v].nphalomin));  // src_v2/FOF.c:202, :290-298
  }
}

// Block-wide exclusive scan of (a, b) over 256 threads and their totals.
__device__ __forceinline__ void block_scan2(uint32_t &a, uint32_t &b, uint32_t &ta, uint32_t &tb,
                                            uint32_t (&ws)[2][4]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t ia = a, ib = b;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t x = __shfl_up(ia, o, 64), y = __shfl_up(ib, o, 64);
    if (lane >= o) ia += x, ib += y;
  }
  __syncthreads();
  if (lane == 63) ws[0][w] = ia, ws[1][w] = ib;
  __syncthreads();
  a = ia - a, b = ib - b;
  ta = tb = 0;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    if (q < w) a += ws[0][q], b += ws[1][q];
    ta += ws[0][q], tb += ws[1][q];
  }
}

__global__ __launch_bounds__(256) void k_group_sums(uint64_t nw, uint32_t runs,
                                                    const uint32_t *__restrict__ bits,
                                                    const uint32_t *__restrict__ lsize,
                                                    const VolDev *__restrict__ vols,
                                                    const uint32_t *__restrict__ vbeg, int nvol,
                                                    GroupTot *__restrict__ tot) {
  __shared__ uint32_t ws[2][4];
  GroupTot t = {0, 0, 0, 0};
  for (uint32_t j = 0; j < runs; j++) {
    const uint64_t w = ((uint64_t)blockIdx.x * runs + j) * 256 + threadIdx.x;
    if (w >= nw) break;
    word_groups(bits[w], w, lsize, vols, vbeg, nvol, [&](uint32_t, uint32_t n, bool halo) {
      t.groups++, t.members += n, t.halos += halo ? 1u : 0u;
    });
  }
  uint32_t g = t.groups, m = t.members, h = t.halos, z = 0;
  block_scan2(g, m, t.groups, t.members, ws);
  block_scan2(h, z, t.halos, t.pad, ws);
  if (threadIdx.x == 0) tot[blockIdx.x] = t;
}

__global__ __launch_bounds__(256) void k_group_emit(uint64_t nw, uint32_t runs,
                                                    const uint32_t *__restrict__ bits,
                                                    const uint32_t *__restrict__ lsize,
                                                    const VolDev *__restrict__ vols,
                                                    const uint32_t *__restrict__ vbeg, int nvol,
                                                    const GroupTot *__restrict__ tot,
                                                    uint32_t *__restrict__ offs,
                                                    uint32_t *__restrict__ cursor,
                                                    uint32_t *__restrict__ hk,
                                                    uint32_t *__restrict__ small) {
  __shared__ uint32_t ws[2][4];
  GroupTot pre = {0, 0, 0, 0};
  for (uint32_t b = threadIdx.x; b < blockIdx.x; b += 256) {
    const GroupTot t = tot[b];
    pre.groups += t.groups, pre.members += t.members, pre.halos += t.halos;
  }
  {
    uint32_t a = pre.groups, b = pre.members, c = pre.halos, d = 0, z;
    block_scan2(a, b, pre.groups, pre.members, ws);
    block_scan2(c, d, pre.halos, z, ws);
  }
  for (uint32_t j = 0; j < runs; j++) {
    const uint64_t w = ((uint64_t)blockIdx.x * runs + j) * 256 + threadIdx.x;
    if (w - threadIdx.x >= nw) break;
    const uint32_t m = w < nw ? bits[w] : 0u;
    uint32_t gh = 0, mem = 0, tgh, tmem;  // groups | halos << 16: at most 8192 each in a run
    word_groups(m, w, lsize, vols, vbeg, nvol, [&](uint32_t, uint32_t n, bool halo) {
      gh += halo ? 0x10001u : 1u, mem += n;
    });
    block_scan2(gh, mem, tgh, tmem, ws);
    uint32_t g = pre.groups + (gh & 0xFFFFu), h = pre.halos + (gh >> 16), at = pre.members + mem;
    word_groups(m, w, lsize, vols, vbeg, nvol, [&](uint32_t lab, uint32_t n, bool halo) {
      offs[g++] = at;
      cursor[lab] = at;
      if (halo && hk) hk[h++] = at;
      at += n;
    });
    pre.groups += tgh & 0xFFFFu, pre.halos += tgh >> 16, pre.members += tmem;
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
    offs[pre.groups] = pre.members;
    small[kSmR] = pre.groups;
    small[kSmM] = pre.members;
    if (hk) small[kSmH] = pre.halos;
  }
}

// Sorting each segment of the member list by index.  Groups of at most four
// members are sorted by a lane each; larger ones are listed, up to kSegWave
// members for a wave each (a bitonic network in registers; 64 E elements for E
// per lane, lane-major, so that the stages below distance E stay inside a lane
// and the others are lane shuffles), the rest for a workgroup each: an LSD
// radix sort in LDS with as many digits as the indices have bits, up to
// kSegLds members by 256 threads and up to kSegLdsBig by 1024; beyond that the
// same passes through scratch, kSegLdsBig members at a time.
//
// Why lists: groups come in label order and a label is the group's lowest
// index, so the first few hundred groups of a volume are its largest; a wave
// that took 64 consecutive groups sorted all of those alone.  64^3 box: 216 us
// there and 112 us in four radix passes through global memory over the largest
// group, now 5 + 33 + 23 us; 512^3 box 307 + 676 us, now 160 + 580 + 240 (of
// these, merging chunks in LDS by binary search in place of the radix passes
// took 45 us for the largest group of the 64^3 box, and a bitonic sort of
// kSegLds members by 256 threads 676).  Above kSegLdsBig one workgroup's pass
// over 2^20 members takes 1.4 ms (three passes 4.4; four with 256 threads and
// 256 members at a time took 16.4, and merging sorted runs of kSegLdsBig by
// binary search in scratch 22.4; for 32768 members 0.12, 0.41 and 0.14 ms).
// What bounds it now: the ranking of
// the largest group on one compute unit while there are few groups (eight
// ballots for 64 keys), shuffles and latency when many.  Four waves per SIMD:
// six spill (508 us at 512^3, 37 at 64^3).
constexpr uint32_t kSegWave = 1024;
constexpr uint32_t kSegLds = 4096, kSegLdsBig = 16384;
constexpr int kSmLarge = 9;  // groups listed for a workgroup each, up to kSegLds members
constexpr int kSmMid = 12;   // groups listed for a wave each
constexpr int kSmHuge = 13;  // larger groups, a workgroup of 1024 threads each

// n <= 64: one element a lane, the network only as wide as n needs
__device__ __forceinline__ void seg_sort_lane(uint32_t *__restrict__ p, uint32_t n, uint32_t lane) {
  uint32_t v = lane < n ? p[lane] : 0xFFFFFFFFu;
  uint32_t P = 2;
  while (P < n) P <<= 1;
  for (uint32_t k = 2; k <= P; k <<= 1)
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      const uint32_t u = (uint32_t)__shfl_xor((int)v, (int)j, 64);
      const bool up = (lane & k) == 0, lower = (lane & j) == 0;
      v = (lower == up) ? min(v, u) : max(v, u);
    }
  if (lane < n) p[lane] = v;
}

// n <= 64 E elements of p, in place: element a = E lane + e in register e of
// the lane
template <int E>
__device__ __forceinline__ void seg_sort_regs(uint32_t *p, uint32_t n, uint32_t lane) {
  constexpr uint32_t P = 64u * E;
  uint32_t v[E];
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t a = lane * E + e;
    v[e] = a < n ? p[a] : 0xFFFFFFFFu;
  }
#pragma unroll
  for (uint32_t k = 2; k <= P; k <<= 1)
#pragma unroll
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      if (j < (uint32_t)E) {
#pragma unroll
        for (int e = 0; e < E; e++) {
          if (e & j) continue;
          const bool up = ((lane * E + e) & k) == 0;
          const uint32_t x = v[e], y = v[e | j];
          v[e] = up ? min(x, y) : max(x, y);
          v[e | j] = up ? max(x, y) : min(x, y);
        }
      } else {
        const uint32_t lj = j / E;
        const bool lower = (lane & lj) == 0;
#pragma unroll
        for (int e = 0; e < E; e++) {
          const uint32_t u = (uint32_t)__shfl_xor((int)v[e], (int)lj, 64);
          const bool up = ((lane * E + e) & k) == 0;
          v[e] = (lower == up) ? min(v[e], u) : max(v[e], u);
        }
      }
    }
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t a = lane * E + e;
    if (a < n) p[a] = v[e];
  }
}

// The lanes sort the groups of at most four members and list the others
// (gathered per workgroup in LDS: one append a full list, so the two device
// counters see few atomics).
constexpr uint32_t kSegList = 1024;

__global__ __launch_bounds__(256) void k_seg_sort(const uint32_t *__restrict__ dR,
                                                  const uint32_t *__restrict__ offs,
                                                  uint32_t *__restrict__ mval,
                                                  uint32_t *__restrict__ mid,
                                                  uint32_t *__restrict__ dMid,
                                                  uint32_t *__restrict__ large,
                                                  uint32_t *__restrict__ dL,
                                                  uint32_t *__restrict__ huge,
                                                  uint32_t *__restrict__ dHuge) {
  __shared__ uint32_t lst[kSegList], nl, base;
  const uint32_t R = *dR;
  const uint32_t lane = threadIdx.x & 63;
  if (threadIdx.x == 0) nl = 0;
  __syncthreads();
  auto flush = [&]() {
    __syncthreads();
    if (threadIdx.x == 0) base = nl ? atomicAdd(dMid, nl) : 0u;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < nl; i += 256) mid[base + i] = lst[i];
    __syncthreads();
    if (threadIdx.x == 0) nl = 0;
    __syncthreads();
  };
  for (uint32_t c0 = blockIdx.x * 256; c0 < R; c0 += gridDim.x * 256) {
    const uint32_t g = c0 + threadIdx.x;
    uint32_t s = 0, n = 0;
    if (g < R) s = offs[g], n = offs[g + 1] - s;
    if (n <= 4) {  // a comparator network on the lane's own group
      uint32_t v[4];
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = (uint32_t)e < n ? mval[s + e] : 0xFFFFFFFFu;
      auto cas = [&](int a, int b) {
        const uint32_t x = v[a], y = v[b];
        v[a] = min(x, y), v[b] = max(x, y);
      };
      cas(0, 1), cas(2, 3), cas(0, 2), cas(1, 3), cas(1, 2);
#pragma unroll
      for (int e = 0; e < 4; e++)
        if ((uint32_t)e < n) mval[s + e] = v[e];
    }
    const bool m = n > 4 && n <= kSegWave;
    const unsigned long long bm = __ballot(m);
    if (bm) {
      uint32_t b = 0;
      if (lane == 0) b = atomicAdd(&nl, (uint32_t)__popcll(bm));
      b = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
      if (m) lst[b + (uint32_t)__popcll(bm & ((1ull << lane) - 1))] = g;
    }
    if (n > kSegLds) huge[atomicAdd(dHuge, 1u)] = g;
    else if (n > kSegWave) large[atomicAdd(dL, 1u)] = g;
    __syncthreads();
    if (nl > kSegList - 256) flush();  // uniform: nl is read after the barrier by all
    __syncthreads();
  }
  flush();
}

// Groups of list `large` by workgroups of NT threads, up to LDS members in LDS
// and (the form without MID) larger ones through scratch; then, with MID, the
// groups of list `mid` by waves.
template <int NT, uint32_t LDS, bool MID>
__global__ __launch_bounds__(NT, 4) void k_seg_sort_list(const uint32_t *__restrict__ dL,
                                                      const uint32_t *__restrict__ large,
                                                      const uint32_t *__restrict__ dMid,
                                                      const uint32_t *__restrict__ mid,
                                                      const uint32_t *__restrict__ offs,
                                                      uint32_t *__restrict__ mval,
                                                      uint32_t *__restrict__ scratch, int bits) {
  constexpr int kWaves = NT / 64, kR = LDS / NT;  // waves, elements a thread holds
  static_assert(NT >= 256, "a thread for each digit");
  __shared__ uint32_t sk[LDS], wcnt[kWaves][256], wsum[4], cur[MID ? 1 : 256];
  const uint32_t t = threadIdx.x, lane = t & 63;
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(t >> 6));
  const unsigned long long lt = (1ull << lane) - 1;
  const int passes = (bits + 7) / 8, width = (bits + passes - 1) / passes;
  const uint32_t mask = (1u << width) - 1;
  auto clear = [&]() {
    __syncthreads();
    for (uint32_t q = t; q < kWaves * 256u; q += NT) (&wcnt[0][0])[q] = 0;
    __syncthreads();
  };
  // A digit's number of counted keys, in its thread.
  auto digit_total = [&]() -> uint32_t {
    uint32_t c = 0;
    if (t < 256)
#pragma unroll
      for (int q = 0; q < kWaves; q++) c += wcnt[q][t];
    return c;
  };
  // Exclusive scan of one value of each of the first 256 threads.
  auto scan256 = [&](uint32_t c) -> uint32_t {
    uint32_t inc = c;
    if (t < 256) {
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(inc, o, 64);
        if (lane >= (uint32_t)o) inc += u;
      }
      if (lane == 63) wsum[w] = inc;
    }
    __syncthreads();
    uint32_t pre = inc - c;
    if (t < 256)
      for (uint32_t q = 0; q < w; q++) pre += wsum[q];
    return pre;
  };
  // The n elements at src in order: a stable pass a digit, LDS elements at a time.
  // A chunk's keys are in registers between ranking and placing: wave w has the
  // keys [w per, (w + 1) per) of it, 64 at a time, lanes of one digit found by
  // ballots, wcnt[w][d] counting the wave's keys of digit d so far and then
  // their first place.  Up to LDS elements stay in LDS between the passes
  // and return to src; more go from src to dst and back (far), the digits'
  // places counted ahead of each pass; the result's place is returned.
  auto sort = [&](uint32_t *src, uint32_t *dst, uint32_t n) -> uint32_t * {
    const bool far = !MID && n > LDS;
    for (int k = 0; k < passes; k++) {
      const int shift = k * width;
      if (far) {
        clear();  // (and the pass before is visible to the workgroup)
        for (uint32_t i = t; i < n; i += NT) atomicAdd(&wcnt[w][(src[i] >> shift) & mask], 1u);
        __syncthreads();
        const uint32_t pre = scan256(digit_total());
        if (!MID && t < 256) cur[t] = pre;
      }
      for (uint32_t c0 = 0; c0 < n; c0 += LDS) {
        const uint32_t m = min(LDS, n - c0);
        const uint32_t per = (m + NT - 1) / NT * 64, i0 = w * per, i1 = min(m, i0 + per);
        clear();
        uint32_t key[kR], rk[kR];
#pragma unroll
        for (int r = 0; r < kR; r++) {
          if (64u * r >= per) break;
          const uint32_t i = i0 + 64 * r + lane;
          key[r] = i < i1 ? (k && !far ? sk[i] : src[c0 + i]) : 0u;
        }
#pragma unroll
        for (int r = 0; r < kR; r++) {
          if (64u * r >= per) break;
          const bool valid = i0 + 64 * r + lane < i1;
          const uint32_t d = (key[r] >> shift) & mask;
          unsigned long long peers = __ballot(valid);
          for (int b = 0; b < width; b++) {
            const bool on = (d >> b) & 1u;
            const unsigned long long bb = __ballot(on);
            peers &= on ? bb : ~bb;
          }
          const uint32_t below = (uint32_t)__popcll(peers & lt);
          uint32_t old = 0;
          if (valid) old = wcnt[w][d];
          wave_sync();
          if (valid && below == 0) wcnt[w][d] = old + (uint32_t)__popcll(peers);
          wave_sync();
          rk[r] = old + below;
        }
        __syncthreads();
        uint32_t at = far ? (t < 256 ? cur[MID ? 0 : t] : 0u) : scan256(digit_total());
        if (t < 256) {
#pragma unroll
          for (int q = 0; q < kWaves; q++) {
            const uint32_t x = wcnt[q][t];
            wcnt[q][t] = at;
            at += x;
          }
          if (far) cur[MID ? 0 : t] = at;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kR; r++) {
          if (64u * r >= per) break;
          if (i0 + 64 * r + lane < i1) {
            const uint32_t o = wcnt[w][(key[r] >> shift) & mask] + rk[r];
            if (far) dst[o] = key[r];
            else sk[o] = key[r];
          }
        }
      }
      if (far) {
        uint32_t *x = src;
        src = dst, dst = x;
      }
    }
    __syncthreads();
    if (!far)
      for (uint32_t i = t; i < n; i += NT) src[i] = sk[i];
    return src;
  };
  const uint32_t nl = *dL;
  for (uint32_t q = blockIdx.x; q < nl; q += gridDim.x) {
    const uint32_t g = large[q];
    const uint32_t s = offs[g], n = offs[g + 1] - s;
    const uint32_t *const r = sort(mval + s, scratch + s, n);
    if (r != mval + s)
      for (uint32_t i = t; i < n; i += NT) mval[s + i] = r[i];
  }
  if (!MID) return;
  const uint32_t nm = *dMid;
  for (uint32_t q = blockIdx.x * (NT / 64) + w; q < nm; q += gridDim.x * (NT / 64)) {
    const uint32_t g = mid[q];
    const uint32_t s = (uint32_t)__builtin_amdgcn_readfirstlane((int)offs[g]);
    const uint32_t n = (uint32_t)__builtin_amdgcn_readfirstlane((int)offs[g + 1]) - s;
    uint32_t *p = mval + s;
    if (n <= 64) seg_sort_lane(p, n, lane);
    else if (n <= 128) seg_sort_regs<2>(p, n, lane);
    else if (n <= 256) seg_sort_regs<4>(p, n, lane);
    else if (n <= 512) seg_sort_regs<8>(p, n, lane);
    else seg_sort_regs<16>(p, n, lane);
  }
}

__global__ __launch_bounds__(256) void k_ring(const uint32_t *__restrict__ dM,
                                              const uint32_t *__restrict__ skey,
                                              const uint32_t *__restrict__ sval,
                                              const uint32_t *__restrict__ vbeg, int nvol,
                                              uint32_t *__restrict__ next_out,
                                              uint32_t *__restrict__ pidx,
                                              uint32_t *__restrict__ pval) {
  const uint32_t M = *dM;
  const uint64_t k0 = (uint64_t)blockIdx.x * kTileN, k1 = min((uint64_t)M, k0 + kTileN);
  if (k0 >= k1) return;
  auto body = [&](uint32_t k, uint32_t lab, uint32_t b) {
    const uint32_t i = sval[k];
    const uint32_t nx = (k + 1 < M && skey[k + 1] == lab) ? sval[k + 1] : lab;
    if (pidx) pidx[k] = i, pval[k] = nx - b + 1u;
    else if (next_out) next_out[i] = nx - b + 1u;
  };
  // the list is sorted by label, so by volume; a member shares its head's
  // volume, and a tile whose first and last labels share one has no other
  const int va = vol_of(vbeg, nvol, skey[k0]);
  if (skey[k1 - 1] < vbeg[va + 1]) {
    const uint32_t b = vbeg[va];
    for (uint32_t k = (uint32_t)k0 + threadIdx.x; k < k1; k += blockDim.x) body(k, skey[k], b);
    return;
  }
  int hint = va;
  for (uint32_t k = (uint32_t)k0 + threadIdx.x; k < k1; k += blockDim.x) {
    const uint32_t lab = skey[k];
    const int v = vol_of_sorted(vbeg, nvol, lab, hint);
    body(k, lab, vbeg[v]);
  }
}

// Halo sums: FP64 accumulation of the float Pos / Vel of the members in
// ascending index order from the head (the order the host walks the ring
// returned in next_out), so the host's Checkhalo / Output_Halos loops give
// the same bits.  One wavefront per halo: the 64 lanes stage 64 members at a
// time in LDS as doubles and then each of the first NQ lanes adds one
// quantity over them, in order.  Quantities (q = lane):
//   0-5    Pos x,y,z, Vel x,y,z                          (src_v2/FOF.c:805-810)
//   with MOM, the second moments (src_v2/FOF.c:811-824):
//   6-11   Pos xx,yy,zz,xy,xz,yz   12-17  Vel xx,...     raw products, ring order
//   18-20  Pos x,y,z - head        21-23  Vel - head     deviations from the head
//   24-29  Pos products of those   30-35  Vel products   (for centred moments)
// A float difference widened to double is exact here (same-halo members), and
// products of two such numbers (< 53 significant bits) are exact, so only the
// additions round.  Every quantity is the product of two staged rows: 0-5 the
// components, 6-11 the deviations (MOM), and a row of ones for those that are
// no product (times 1.0 is exact).  Members past the last are staged as zeros:
// a sum that began at +0.0 is never -0.0, so adding +0.0 changes no bit, and
// the adding loop runs eight members at a time with its LDS reads issued ahead
// of the additions.
//
// What bounds it: the largest halo's chain of dependent additions while
// there are few halos, the gather (one 128-byte line per member record) when
// there are many.  For halos above kHaloAhead blocks the records of the next
// 256 members are in registers and their list entries 256 further, every
// load unconditional, so that neither of the gather's two dependent loads is
// waited for in a block.  Before (float rows, one LDS read and one conversion
// ahead of every addition, the next 64 records loaded during the block):
// 437 us for the 64^3 box, whose largest halo has about 1e4 members, 2669 with
// MOM for a 144^3 box and 2.22 ms for a 512^3 box; now 72, 125 and 1.72 ms.
constexpr int kHaloAhead = 4;   // 64-member blocks in flight
constexpr int kHaloRow = 66;    // doubles a row: 16-byte aligned, rows in different banks

template <bool MOM>
__global__ __launch_bounds__(256) void k_halo_sums(const uint32_t *__restrict__ dH,
                                                   const uint32_t *__restrict__ hk,
                                                   const uint32_t *__restrict__ skey,
                                                   const uint32_t *__restrict__ sval,
                                                   const uint32_t *__restrict__ hsize,
                                                   const uint8_t *__restrict__ base,
                                                   uint32_t stride, uint32_t offpos,
                                                   uint32_t offvel,
                                                   const VolDev *__restrict__ vols,
                                                   const uint32_t *__restrict__ vbeg, int nvol,
                                                   fof_halo_v1 *__restrict__ out,
                                                   fof_moments_v1 *__restrict__ mout,
                                                   uint64_t cap, uint64_t *__restrict__ hoff,
                                                   unsigned long long *__restrict__ ctr) {
  constexpr int NQ = MOM ? 36 : 6;
  constexpr int kOnes = 12;
  constexpr int kRows = MOM ? 13 : 6;
  __shared__ __align__(16) double stage[4][kRows][kHaloRow];
  const uint32_t H = *dH;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t nw = gridDim.x * (blockDim.x >> 6);
  uint32_t owned_cnt = 0;
  int hint = 0;
  // the two rows whose product is the lane's quantity
  int ra = lane < 6 ? lane : 0, rb = kOnes;
  if (MOM && lane >= 6 && lane < NQ) {
    if (lane >= 18 && lane < 24) {
      ra = lane - 18 + 6;
    } else {  // component pairs of the products: xx yy zz xy xz yz
      const int r = lane < 18 ? lane - 6 : lane - 24, o = (r / 6) * 3 + (lane < 18 ? 0 : 6), k = r % 6;
      ra = o + (k < 3 ? k : (k < 5 ? 0 : 1));
      rb = o + (k < 3 ? k : (k == 3 ? 1 : 2));
    }
  }
  if constexpr (MOM) {
    stage[w][kOnes][lane] = 1.0;
    wave_sync();
  }
  const double *const pa = stage[w][ra], *const pb = stage[w][MOM ? rb : 0];
  // hoff[v] = first halo whose head lies in volume v or later
  for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v <= (uint64_t)nvol;
       v += (uint64_t)gridDim.x * blockDim.x) {
    uint32_t lo = v == (uint64_t)nvol ? H : 0, hi = v == 0 ? 0 : H;
    const uint32_t head = vbeg[v];
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (skey[hk[mid]] < head) lo = mid + 1;
      else hi = mid;
    }
    hoff[v] = lo;
  }
  for (uint32_t h = blockIdx.x * (blockDim.x >> 6) + w; h < H; h += nw) {
    // wave-uniform, visibly so: branches on them leave the loads in flight countable
    const uint32_t k0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)hk[h]);
    const uint32_t lab = (uint32_t)__builtin_amdgcn_readfirstlane((int)skey[k0]);
    const uint32_t n = (uint32_t)__builtin_amdgcn_readfirstlane((int)hsize[lab]);
    hint = vol_from(vbeg, nvol, lab, hint);  // halos ascend by head, per wave too
    const int v = hint;
    const VolDev &V = vols[v];
    const double elo[3] = {V.rmin_buff[0], V.rmin_buff[1], V.rmin_buff[2]};
    const double ehi[3] = {V.rmax_buff[0], V.rmax_buff[1], V.rmax_buff[2]}, el = V.linklength;
    double acc = 0;
    uint32_t warn = 0;
    double ref[6];
    // list entry and record of member k + lane; past the last, the last's again
    auto entry = [&](uint32_t k) -> uint32_t { return sval[k0 + min(k + (uint32_t)lane, n - 1)]; };
    auto fetch = [&](uint32_t i, float (&q)[6]) {
      const uint8_t *rec = base + (uint64_t)i * stride;
      const float *pp = reinterpret_cast<const float *>(rec + offpos);
      const float *vv = reinterpret_cast<const float *>(rec + offvel);
      q[0] = pp[0], q[1] = pp[1], q[2] = pp[2], q[3] = vv[0], q[4] = vv[1], q[5] = vv[2];
    };
    auto store = [&](uint32_t m, const float (&r)[6]) {
      const bool in = (uint32_t)lane < m;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        const double q = r[d];
        if (in && ((q - elo[d] < el) || (ehi[d] - q < el))) warn |= 1u << d;
      }
#pragma unroll
      for (int c = 0; c < 6; c++) {
        stage[w][c][lane] = in ? (double)r[c] : 0.0;
        if (MOM) stage[w][6 + c][lane] = in ? (double)r[c] - ref[c] : 0.0;
      }
    };
    auto add = [&](uint32_t m) {
      wave_sync();
      if (lane < NQ) {
        for (uint32_t q = 0; q < m; q += 8) {
          double a[8];
#pragma unroll
          for (int t = 0; t < 8; t++) a[t] = pa[q + t];
          if (MOM) {
            double b[8];
#pragma unroll
            for (int t = 0; t < 8; t++) b[t] = pb[q + t];
#pragma unroll
            for (int t = 0; t < 8; t++) a[t] = a[t] * b[t];
          }
#pragma unroll
          for (int t = 0; t < 8; t++) acc += a[t];
        }
      }
      wave_sync();  // the rows are written again
    };
    // the head (first member) is the reference point of the deviations
    auto set_ref = [&](const float (&r)[6]) {
#pragma unroll
      for (int c = 0; c < 6; c++) ref[c] = MOM ? (double)__shfl(r[c], 0, 64) : 0.0;
    };
    if (n <= 64u * kHaloAhead) {
      float r[6];
      fetch(entry(0), r);
      set_ref(r);
      for (uint32_t k = 0; k < n; k += 64) {
        store(n - k, r);
        if (k + 64 < n) fetch(entry(k + 64), r);
        add(min(64u, n - k));
      }
    } else {
      // every load unconditional (their indices stay in the halo), so that a
      // block waits for its own records only, not for those behind them
      float r[kHaloAhead][6];
      uint32_t at[kHaloAhead];
#pragma unroll
      for (int j = 0; j < kHaloAhead; j++) at[j] = entry(64 * j);
#pragma unroll
      for (int j = 0; j < kHaloAhead; j++) fetch(at[j], r[j]);
#pragma unroll
      for (int j = 0; j < kHaloAhead; j++) at[j] = entry(64 * (kHaloAhead + j));
      set_ref(r[0]);
      uint32_t k = 0;
      for (; k + 64 * kHaloAhead <= n; k += 64 * kHaloAhead) {
#pragma unroll
        for (int j = 0; j < kHaloAhead; j++) {
          store(64, r[j]);
          fetch(at[j], r[j]);
          at[j] = entry(k + 64 * (2 * kHaloAhead + j));
          add(64);
        }
      }
#pragma unroll
      for (int j = 0; j < kHaloAhead; j++)
        if (k + 64 * j < n) {
          store(n - k - 64 * j, r[j]);
          add(min(64u, n - k - 64 * j));
        }
    }
    const double s0 = __shfl(acc, 0, 64), s1 = __shfl(acc, 1, 64), s2 = __shfl(acc, 2, 64);
    const double s3 = __shfl(acc, 3, 64), s4 = __shfl(acc, 4, 64), s5 = __shfl(acc, 5, 64);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) warn |= __shfl_xor(warn, o, 64);
    // src_v2/FOF.c:394-401
    const double cx = s0 / (double)n, cy = s1 / (double)n, cz = s2 / (double)n;
    const bool own = !((cx < V.rmin[0]) || (cx >= V.rmax[0]) || (cy < V.rmin[1]) ||
                       (cy >= V.rmax[1]) || (cz < V.rmin[2]) || (cz >= V.rmax[2]));
    if (!own) warn = 0;
    if (MOM && mout && h < cap) {
      // raw products (lanes 6-17), centred products from the deviations:
      // sum (a - ma)(b - mb) = S_ab - S_a S_b / n with a, b taken about the head
      double dev[6];
#pragma unroll
      for (int c = 0; c < 6; c++) dev[c] = __shfl(acc, 18 + c, 64);
      double prod[12];
#pragma unroll
      for (int c = 0; c < 12; c++) prod[c] = __shfl(acc, 24 + c, 64);
      const double rawq = __shfl(acc, 6 + lane % 12, 64);  // every lane takes part
      if (lane < 12) {
        const int blk = lane / 6, k = lane % 6, o = blk * 3;
        const int ca = o + (k < 3 ? k : (k < 5 ? 0 : 1));
        const int cb = o + (k < 3 ? k : (k == 3 ? 1 : 2));
        double pc = 0, da = 0, db = 0;
#pragma unroll
        for (int c = 0; c < 12; c++) pc = (c == lane) ? prod[c] : pc;
#pragma unroll
        for (int c = 0; c < 6; c++) {
          da = (c == ca) ? dev[c] : da;
          db = (c == cb) ? dev[c] : db;
        }
        double *mo = reinterpret_cast<double *>(mout + h);
        mo[lane] = rawq;                            // pos2[6], vel2[6]
        mo[12 + lane] = pc - da * db / (double)n;   // cpos2[6], cvel2[6]
      }
    }
    if (lane == 0) {
      if (h < cap) {
        fof_halo_v1 H1;
        H1.head = lab - vbeg[v];
        H1.n = n;
        H1.owned = own ? 1u : 0u;
        H1.edge_warn = warn;
        H1.sum_pos[0] = s0, H1.sum_pos[1] = s1, H1.sum_pos[2] = s2;
        H1.sum_vel[0] = s3, H1.sum_vel[1] = s4, H1.sum_vel[2] = s5;
        out[h] = H1;
      }
      owned_cnt += own ? 1u : 0u;
    }
  }
  uint64_t t = owned_cnt;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o, 64);
  if ((threadIdx.x & 63) == 0 && t) ctr_add(ctr, kCtrOwned, t);
}

// ---------------------------------------------------------------------------
// host orchestration
// ---------------------------------------------------------------------------
static inline uint32_t grid_for(uint64_t n, uint32_t cap = 65535u * 4u) {
  uint64_t g = (n + 255) / 256;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (uint32_t)g;
}

static int bits_for(uint64_t n) {
  int b = 1;
  while (b < 32 && (1ull << b) < n) b++;
  return b;
}

// Host-side volume preparation: grid and thresholds, validated.
struct HostVol {
  VolDev d;
  uint64_t ncell;
  double ncell_d;
};

// Smallest l^2 of the cells holding particles, per volume with a variable
// l (as the bits of a non-negative double: their order is the doubles').
// Each wave takes kVlRun consecutive particles and keeps a running minimum
// per lane, flushed when the lane's volume changes and once at the end (an
// atomic per wave and step on one address per volume serialises).
constexpr uint32_t kVlRun = 2048;

__global__ __launch_bounds__(256) void k_varlink_min(const uint8_t *__restrict__ base,
                                                     uint32_t stride, uint32_t offpos, uint32_t N,
                                                     const VolDev *__restrict__ vols,
                                                     const uint32_t *__restrict__ vbeg, int nvol,
                                                     unsigned long long *__restrict__ vmin) {
  const int lane = threadIdx.x & 63;
  const uint64_t w0 = ((uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * kVlRun;
  int cv = -1, hint = 0;
  unsigned long long cm = ~0ull;
  for (uint32_t r = 0; r < kVlRun; r += 64) {
    const uint64_t pp64 = w0 + r + lane;
    if (pp64 >= N) break;
    const uint32_t p = (uint32_t)pp64;
    const int v = vol_of_run(vbeg, nvol, p, N, hint);
    const VolDev &V = vols[v];
    const float *pp = reinterpret_cast<const float *>(base + (uint64_t)p * stride + offpos);
    const double x = pp[0], y = pp[1], z = pp[2];
    const bool ok = V.vntab > 0 && x >= V.rmin_buff[0] && x <= V.rmax_buff[0] &&
                    y >= V.rmin_buff[1] && y <= V.rmax_buff[1] && z >= V.rmin_buff[2] &&
                    z <= V.rmax_buff[2];
    unsigned long long bits = ~0ull;
    if (ok) {
      double u;
      const int ix = cell1(x, V.rmin_buff[0], V.lcell[0], V.nx, &u);
      const int iy = cell1(y, V.rmin_buff[1], V.lcell[1], V.ny, &u);
      const int iz = cell1(z, V.rmin_buff[2], V.lcell[2], V.nz, &u);
      const double l2 = cell_linksq(V, ix, iy, iz);
      memcpy(&bits, &l2, 8);
    }
    if (v != cv) {
      if (cv >= 0 && cm != ~0ull) atomicMin(vmin + cv, cm);
      cv = v, cm = bits;
    } else if (bits < cm) {
      cm = bits;
    }
  }
  const int v0 = __shfl(cv, 0, 64);
  if (__ballot(cv != v0) == 0ull) {  // one volume: reduce over the wave first
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const unsigned long long t = __shfl_xor(cm, o, 64);
      cm = t < cm ? t : cm;
    }
    if (lane == 0 && v0 >= 0 && cm != ~0ull) atomicMin(vmin + v0, cm);
  } else if (cv >= 0 && cm != ~0ull) {
    atomicMin(vmin + cv, cm);
  }
}

// Sub-cells: side <= l_min (1 - 1e-6) / sqrt(3) so that any two particles
// of one sub-cell link (see file header).  Disabled (m = 0) when more than
// 12 per axis would be needed, or l_min = 0.
static void set_subcells(VolDev &V, double lmin2) {
  V.m[0] = V.m[1] = V.m[2] = 0;
  if (!(lmin2 > 0)) return;
  const double s = sqrt(lmin2) * (1.0 - 1e-6) / sqrt(3.0);
  int m[3];
  bool ok = true;
  for (int k = 0; k < 3; k++) {
    double q = ceil(V.lcell[k] / s);
    if (q < 1) q = 1;
    if (q > 12) ok = false;
    m[k] = (int)q;
  }
  const int nn[3] = {V.nx, V.ny, V.nz};
  for (int k = 0; k < 3; k++)
    if ((double)nn[k] * m[k] >= 2097152.0) ok = false;  // 21-bit fine coordinates
  if (ok)
    for (int k = 0; k < 3; k++) {
      V.m[k] = m[k];
      const double side = V.lcell[k] / m[k];
      V.s2[k] = side * side;
    }
}

int prepare_volume(const fof_volume_v1 &in, double band, HostVol &hv, std::vector<const fof_varlink_v1 *> &vl) {
  const fof_domain_v1 &D = in.domain;
  VolDev &V = hv.d;
  memset(&V, 0, sizeof(V));
  for (int k = 0; k < 3; k++) {
    V.rmin_buff[k] = D.rmin_buff[k];
    V.rmax_buff[k] = D.rmax_buff[k];
    V.rmin[k] = D.rmin[k];
    V.rmax[k] = D.rmax[k];
    V.lcell[k] = D.lcell[k];
    if (!(D.lcell[k] > 0) || !std::isfinite(D.lcell[k]) || !(D.rmax_buff[k] >= D.rmin_buff[k]))
      return FOF_E_ARG;
  }
  if (!(D.linklength >= 0) || !std::isfinite(D.linklength)) return FOF_E_ARG;
  V.linklength = D.linklength;
  V.linksq = D.linklength * D.linklength;  // src_v2/FOF.c:60
  V.nphalomin = D.nphalomin;
  V.band = (float)band;
  V.lo = (float)(V.linksq * (1.0 - band));
  V.hi = (float)(V.linksq * (1.0 + band));
  // An internal grid finer than the reference's, for a constant l well
  // inside the reference cells.  The reference predicate links a pair only
  // if its true distance is below l(1 + 1e-7) (dx = fl32(xi - xj) errs by
  // < 6e-8).  On an axis where lcell > l(1 + 1e-6), every such pair is at
  // most one cell apart on the reference grid and on any grid whose cells
  // are longer still, so both sweeps find the same linked pairs and the
  // groups do not depend on the choice.  Such an axis is cut into
  // r = ceil(lcell / 6.9 l) cells (so sub-cells, m <= 12, stay on: the
  // all-pairs scan of coarse cells is what a coarse grid otherwise costs).
  // A variable l keeps the reference grid: its cell's l^2 is part of the
  // rule (src_v2/FOF.c:102-109).
  if (!D.varlink && D.linklength > 0) {
    for (int k = 0; k < 3; k++) {
      const double L = D.lcell[k], l = D.linklength;
      if (!(L > l * (1.0 + 1e-6))) continue;
      double r = ceil(L / (6.9 * l));
      const double ext = D.rmax_buff[k] - D.rmin_buff[k];
      while (r > 1 && ceil(ext / (L / r)) + 1.0 > 1048576.0) r -= 1;  // at most 2^20 cells
      if (r > 1) V.lcell[k] = L / r;
    }
  }
  // src_v2/FOF.c:63-65 (on the grid in use)
  double e[3];
  for (int k = 0; k < 3; k++) e[k] = ceil((D.rmax_buff[k] - D.rmin_buff[k]) / V.lcell[k]) + 1.0;
  if (!(e[0] < 2e9 && e[1] < 2e9 && e[2] < 2e9)) return FOF_E_RANGE;
  V.nx = (int)e[0], V.ny = (int)e[1], V.nz = (int)e[2];
  hv.ncell_d = e[0] * e[1] * e[2];
  hv.ncell = (hv.ncell_d < 1.8e19) ? (uint64_t)V.nx * (uint64_t)V.ny * (uint64_t)V.nz : ~0ull;
  // Smallest linking length that any home cell can use.
  double lmin2 = V.linksq;
  if (D.varlink) {
    const fof_varlink_v1 *L = D.varlink;
    if (L->ntab < 2 || !L->l2tab || !(L->r2max > 0)) return FOF_E_ARG;
    vl.push_back(L);
    V.vntab = L->ntab;
    V.vr2max = L->r2max;
    for (int k = 0; k < 3; k++) V.vorigin[k] = L->origin[k];
    lmin2 = -1;  // set by the caller from the occupied cells
  }
  set_subcells(V, lmin2);
  return 0;
}

// Bump allocator over a workspace: run once with base == nullptr to size it,
// then over the allocated arena to carve it.  Every buffer is 256-byte
// aligned.
struct Carve {
  uint8_t *base = nullptr;
  size_t off = 0;
  template <class T>
  T *take(size_t bytes) {
    const size_t o = (off + 255) & ~(size_t)255;
    off = o + bytes;
    return base ? reinterpret_cast<T *>(base + o) : nullptr;
  }
};

// Host-side description of a call: volumes, grids, sizes of every buffer.
struct Plan {
  uint64_t N = 0, C = 0, Csz = 0;
  double Cd = 0;
  uint32_t nvol = 0;
  bool sparse = false;
  int key_bits = 0, volshift = 0;
  uint32_t T = kDefaultT;
  uint32_t big_grid = 8192;  // workgroups of k_link_dense and of its sub-cell sort
  double band = 1e-5;
  std::vector<HostVol> hv;
  std::vector<uint32_t> vbeg;
  std::vector<double> vt_host;
  std::vector<uint32_t> vt_off;  // per volume: first table entry (or ~0)
  size_t vt_entries = 0;
  bool varlink = false;
  // dense grid partitions
  uint32_t F = 0, Bc = 0, ntA = 0, ntBmax = 0, ptile = kPartTile;
  int fb = kFineBits;      // log2 of the cells of a fine bucket
  bool two_level = false;  // coarse buckets first (passes A and B)
  bool hist_in_fine = false;  // pass A's histogram shares a buffer
  uint64_t nA = 0, nB = 0;
  uint64_t ndense_cap = 0, Hbound = 0, Hstage = 0;
  bool single_halos = false;  // some volume keeps groups of one (Nphalomin <= 1)
  size_t tmpb = 0;
  // what the call produces
  uint32_t flags = 0;
  bool host_input = false, host_out = false;
  bool want_ring = false, want_label = false, want_minid = false, want_halos = false,
       want_mom = false;
  bool stage_halos = false;  // halos (and moments) into the workspace first
  bool direct_writes = true;  // labels and ring straight by index (k_label)
  uint32_t stride = 32, offpos = 8, offvel = 20;
  int32_t offid = 0;
};

// Device buffers of a call, carved from the arena.
struct Bufs {
  float4 *pos4;
  uint32_t *key, *start, *par, *runend, *rtab, *gsize, *label, *sortbuf, *dense, *hhead, *cnt,
      *part, *vbeg, *small;
  unsigned long long *fine, *idhead;
  void *tmp;
  VolDev *vols;
  double *vtab;
  uint64_t *hoff;
  uint8_t *input;
  uint32_t *st_next, *st_label;
  unsigned long long *st_minid;
  fof_halo_v1 *st_halo;
  fof_moments_v1 *st_mom;
};

constexpr size_t kSmallBytes = 256 + (size_t)kCtrSlots * kCtrStride * 8;

// The head block of a workspace: counts, flags and counters (zero at first),
// halo offsets, volume table, variable-l tables, volume starts -- one upload
// ahead of a call's kernels; the first two are read back in one copy after
// them.  Byte offsets in it:
struct HeadLayout {
  size_t hoff, vols, vtab, vbeg, bytes;
  HeadLayout(uint32_t nvol, size_t vt_entries) {
    hoff = kSmallBytes;
    vols = (hoff + (nvol + 1) * 8ull + 15) & ~(size_t)15;
    vtab = vols + nvol * sizeof(VolDev);
    vbeg = vtab + vt_entries * sizeof(double);
    bytes = vbeg + (nvol + 1) * 4ull;
  }
};

static size_t layout(const Plan &pl, uint8_t *base, Bufs &b) {
  Carve c;
  c.base = base;
  const uint64_t N = pl.N, q4 = (N + 63) / 64 * 64;
  b.pos4 = c.take<float4>(N * 16);
  b.key = c.take<uint32_t>(N * 4 + 64);
  b.start = c.take<uint32_t>((pl.Csz + 2) * 4 + 64);
  b.par = c.take<uint32_t>(N * 4 + 64);
  b.runend = c.take<uint32_t>(N * 4 + 64);
  b.fine = c.take<unsigned long long>(N * 8 + 64);
  b.rtab = c.take<uint32_t>(N * 4 + 64);
  b.gsize = c.take<uint32_t>(N * 4 + 64);
  b.label = c.take<uint32_t>(N * 4 + 64);
  b.sortbuf = c.take<uint32_t>(16 * q4 + 256);
  b.dense = c.take<uint32_t>(2 * pl.ndense_cap * 4 + 64);
  b.tmp = c.take<void>(pl.tmpb);
  const HeadLayout hl(pl.nvol, pl.vt_entries);
  uint8_t *head = c.take<uint8_t>(hl.bytes + 64);
  if (head) {
    b.small = reinterpret_cast<uint32_t *>(head);
    b.hoff = reinterpret_cast<uint64_t *>(head + hl.hoff);
    b.vols = reinterpret_cast<VolDev *>(head + hl.vols);
    b.vtab = reinterpret_cast<double *>(head + hl.vtab);
    b.vbeg = reinterpret_cast<uint32_t *>(head + hl.vbeg);
  }
  b.hhead = c.take<uint32_t>(pl.Hbound * 4 + 64);
  b.cnt = pl.sparse ? c.take<uint32_t>(N * 4 + 64) : nullptr;
  b.part = pl.sparse ? nullptr
                     : c.take<uint32_t>(((pl.hist_in_fine ? 0 : 2 * pl.nA) + 2 * pl.nB +
                                         2 * (uint64_t)pl.Bc + pl.ntBmax + pl.F + 512) * 4);
  b.input = pl.host_input ? c.take<uint8_t>(N * pl.stride) : nullptr;
  b.idhead = pl.want_minid ? c.take<unsigned long long>(N * 8 + 64) : nullptr;
  const bool ho = pl.host_out;
  b.st_next = ho && pl.want_ring ? c.take<uint32_t>(N * 4) : nullptr;
  b.st_label = ho && pl.want_label ? c.take<uint32_t>(N * 4) : nullptr;
  b.st_minid = ho && pl.want_minid ? c.take<unsigned long long>(N * 8) : nullptr;
  const bool hs = ho || pl.stage_halos;
  b.st_halo = hs && pl.want_halos ? c.take<fof_halo_v1>(pl.Hstage * sizeof(fof_halo_v1)) : nullptr;
  b.st_mom = hs && pl.want_mom ? c.take<fof_moments_v1>(pl.Hstage * sizeof(fof_moments_v1)) : nullptr;
  return c.off + 256;
}

static int make_plan(const fof_particles_v1 *P, const fof_volume_v1 *vols, uint32_t nvol,
                     const fof_opts_v1 *opts, const fof_outputs_v1 *out, Plan &pl) {
  pl.flags = opts ? opts->flags : 0u;
  pl.band = (opts && opts->band > 0) ? opts->band : 1e-5;
  if (!(pl.band >= 1e-6 && pl.band <= 0.1)) return FOF_E_ARG;
  pl.T = std::min(kMaxT, (opts && opts->dense_threshold) ? opts->dense_threshold : kDefaultT);
  pl.big_grid = (opts && opts->big_grid) ? std::min(opts->big_grid, 65536u) : 8192u;
  pl.nvol = nvol;
  pl.stride = P->stride, pl.offpos = P->off_pos, pl.offvel = P->off_vel, pl.offid = P->off_id;
  pl.host_input = P->location != FOF_MEM_DEVICE;
  pl.hv.resize(nvol);
  pl.vbeg.resize(nvol + 1);
  pl.vt_off.assign(nvol, ~0u);
  std::vector<const fof_varlink_v1 *> vls;
  double nphmin = 1e300;
  for (uint32_t v = 0; v < nvol; v++) {
    if (vols[v].offset != pl.N) return FOF_E_ARG;  // volumes must be back to back
    int rc = prepare_volume(vols[v], pl.band, pl.hv[v], vls);
    if (rc) return rc;
    pl.vbeg[v] = (uint32_t)pl.N;
    pl.hv[v].d.pbeg = (uint32_t)pl.N;
    pl.hv[v].d.vid = v;
    pl.N += vols[v].n;
    if (pl.N >= 0x7FFFFFFFull) return FOF_E_RANGE;
    pl.hv[v].d.pend = (uint32_t)pl.N;
    pl.Cd += pl.hv[v].ncell_d;
    // a size cut that is no number keeps every group (no n is below it)
    nphmin = std::min(nphmin, std::isnan(vols[v].domain.nphalomin) ? 0.0 : vols[v].domain.nphalomin);
  }
  pl.vbeg[nvol] = (uint32_t)pl.N;
  // labels and ring: straight random writes by index while every volume's
  // range is not much more than the last-level cache, else through an index
  // partition
  uint64_t maxvol = 0;
  for (uint32_t v = 0; v < nvol; v++) maxvol = std::max<uint64_t>(maxvol, pl.vbeg[v + 1] - pl.vbeg[v]);
  pl.direct_writes = (pl.flags & FOF_OPT_WRITE_PAIRS) ? false
                     : (pl.flags & FOF_OPT_WRITE_DIRECT) ? true
                                                          : maxvol <= kDirectMax;
  if (pl.N != P->n) return FOF_E_ARG;
  // Dense cell tables unless they would dwarf the particle arrays or reach
  // the 2^31 cells a u32 cell index (with room for the table's end) allows.
  pl.sparse = (pl.flags & FOF_OPT_SPARSE) || pl.Cd > 3.0 * (double)pl.N + 4194304.0 ||
              pl.Cd >= (double)0x7FFFFFF0u;
  if (pl.sparse) {
    int lb = 1, vb = 0;
    for (uint32_t v = 0; v < nvol; v++) {
      int b = 1;
      while (b < 64 && (double)(1ull << b) < pl.hv[v].ncell_d) b++;
      lb = std::max(lb, b);
    }
    while ((1u << vb) < nvol) vb++;
    for (uint32_t v = 0; v < nvol; v++)
      if (pl.hv[v].ncell_d > 1.8e19) return FOF_E_RANGE;
    if (lb + vb > 64) return FOF_E_RANGE;
    pl.volshift = lb;
    pl.key_bits = lb + vb;
  } else {
    for (uint32_t v = 0; v < nvol; v++) {
      pl.hv[v].d.cbeg = (uint32_t)pl.C;
      pl.hv[v].d.ncell = (uint32_t)pl.hv[v].ncell;
      pl.C += pl.hv[v].ncell;
    }
  }
  pl.Csz = pl.sparse ? pl.N : pl.C;
  for (uint32_t v = 0; v < nvol; v++)
    if (vols[v].domain.varlink) {
      pl.vt_off[v] = (uint32_t)pl.vt_entries;
      pl.vt_entries += vols[v].domain.varlink->ntab;
    }
  pl.varlink = pl.vt_entries > 0;
  // outputs
  const bool od = out->location == FOF_MEM_DEVICE;
  pl.host_out = !od;
  pl.want_ring = out->next && !(pl.flags & FOF_OPT_NO_RING);
  pl.want_label = out->label != nullptr;
  pl.want_minid = out->minid != nullptr;
  if (pl.want_minid && P->off_id < 0) return FOF_E_ARG;
  pl.want_halos = !(pl.flags & FOF_OPT_NO_HALOS);
  pl.want_mom = pl.want_halos && out->moments != nullptr;
  // sizes
  const uint64_t N = pl.N;
  pl.ndense_cap = N / (pl.T ? pl.T : 1) + 2;
  // kept groups have at least max(1, ceil(nphalomin)) members and are disjoint
  const double kmin = std::max(1.0, std::ceil(std::min(nphmin, 4e9)));
  pl.Hbound = std::min<uint64_t>(N, (uint64_t)((double)N / kmin) + 1);
  pl.single_halos = !(1.0 < nphmin);
  pl.Hstage = std::min<uint64_t>(pl.Hbound, out->halo_cap);
  pl.tmpb = std::max(sort_tmp_bytes(N), compact_tmp_bytes(N));
  if (!pl.sparse) {
    pl.ptile = part_tile(N);
    pl.fb = fine_bits(pl.C);
    pl.F = (uint32_t)((pl.C + (1u << pl.fb) - 1) >> pl.fb);
    pl.two_level = pl.F > (uint32_t)kMaxBuckets;
    pl.Bc = pl.two_level ? (pl.F + 255) >> 8 : pl.F;
    if (pl.two_level && pl.Bc > (uint32_t)kMaxCoarse) return FOF_E_RANGE;
    pl.ntA = (uint32_t)((N + pl.ptile - 1) / pl.ptile);
    pl.ntBmax = pl.two_level ? pl.ntA + pl.Bc : 0;
    pl.nA = (uint64_t)pl.Bc * pl.ntA;
    pl.nB = 256ull * pl.ntBmax;
    pl.hist_in_fine = pl.nA + 64 <= N;
    pl.tmpb = std::max(pl.tmpb, scan_tmp_bytes(std::max(pl.nA, pl.nB) + 1));
  }
  // varlink tables (checked on the host)
  pl.vt_host.resize(pl.vt_entries);
  for (uint32_t v = 0; v < nvol; v++) {
    const fof_varlink_v1 *L = vols[v].domain.varlink;
    if (!L) continue;
    double *dst = pl.vt_host.data() + pl.vt_off[v];
    if (L->location == FOF_MEM_DEVICE)
      FOF_HIP(hipMemcpy(dst, L->l2tab, L->ntab * sizeof(double), hipMemcpyDeviceToHost));
    else
      memcpy(dst, L->l2tab, L->ntab * sizeof(double));
    for (uint32_t k = 0; k < L->ntab; k++)
      if (!(dst[k] >= 0) || !std::isfinite(dst[k])) return FOF_E_ARG;
  }
  return 0;
}

// The volume table of the head block as uploaded.
static void build_vols(const Plan &pl, const Bufs &b, uint8_t *vols) {
  for (uint32_t v = 0; v < pl.nvol; v++) {
    VolDev V = pl.hv[v].d;
    if (pl.vt_off[v] != ~0u) V.vtab = b.vtab + pl.vt_off[v];
    memcpy(vols + v * sizeof(VolDev), &V, sizeof(VolDev));
  }
}

// The head block in the pipeline's page-locked buffer (its last upload is
// done: every call ends synchronised).
static int build_head(const Plan &pl, const Bufs &b, Pipe &pp) {
  const HeadLayout hl(pl.nvol, pl.vt_entries);
  int rc;
  if ((rc = ensure_host(pp.up, hl.bytes)) || (rc = ensure_host(pp.down, hl.vols))) return rc;
  uint8_t *h = static_cast<uint8_t *>(pp.up.ptr);
  memset(h, 0, hl.vols);
  build_vols(pl, b, h + hl.vols);
  if (pl.vt_entries) memcpy(h + hl.vtab, pl.vt_host.data(), pl.vt_entries * sizeof(double));
  memcpy(h + hl.vbeg, pl.vbeg.data(), (pl.nvol + 1) * 4);
  return 0;
}

// ---------------------------------------------------------------------------
// One pipeline's share of a call: plan, carved workspace, output pointers.
// ---------------------------------------------------------------------------
struct Run {
  Plan pl;
  Bufs B;
  Pipe *pp = nullptr;
  const uint8_t *dbase = nullptr;  // particle records on the device
  const void *host_src = nullptr;  // host records to upload first (host input)
  uint32_t *d_next = nullptr, *d_label = nullptr;
  unsigned long long *d_minid = nullptr;
  fof_halo_v1 *d_halo = nullptr;
  fof_moments_v1 *d_mom = nullptr;
  uint64_t hcap = 0;
  uint64_t poff = 0;    // first particle of this pipeline in the call
  uint32_t v0 = 0;      // first volume of this pipeline in the call
  bool timing = false;  // per-phase events on this pipeline's stream
  bool side = false;    // k_link_small on the pipeline's side stream
  uint32_t spans = 0;
  int first_span = -1, last_span = -1;
};

// Plan a pipeline over volumes [v0, v0 + nv) of the call (rebased so that
// the pipeline sees particles from 0) and carve its workspace.
static int prepare_run(Run &r, Pipe &pp, const fof_particles_v1 *P, const fof_volume_v1 *vols,
                       uint32_t v0, uint32_t nv, const fof_opts_v1 *opts,
                       const fof_outputs_v1 *out, bool stage_halos, uint8_t *fixed,
                       size_t fixed_bytes) {
  r.pp = &pp;
  r.v0 = v0;
  r.poff = vols[v0].offset;
  fof_particles_v1 Pg = *P;
  std::vector<fof_volume_v1> vg(vols + v0, vols + v0 + nv);
  uint64_t n = 0;
  for (auto &v : vg) {
    v.offset -= r.poff;
    n += v.n;
  }
  Pg.n = n;
  Pg.base = static_cast<const uint8_t *>(P->base) + r.poff * P->stride;
  int rc = make_plan(&Pg, vg.data(), nv, opts, out, r.pl);
  if (rc) return rc;
  Plan &pl = r.pl;
  pl.stage_halos = stage_halos && pl.want_halos;
  if (pl.N == 0) return 0;
  const size_t need = layout(pl, nullptr, r.B);
  if (fixed) {
    // the caller's fixed workspace: nothing is allocated
    if (need > fixed_bytes || pl.sparse) return FOF_E_RANGE;
    layout(pl, fixed, r.B);
  } else {
    // a workspace far larger than this call needs (a previous call with
    // fewer pipelines) is given back rather than kept beside the others
    if (pp.arena.bytes > 2 * need && pp.arena.bytes - need > (1ull << 30)) release(pp.arena);
    if ((rc = ensure(pp.arena, need))) return rc;
    layout(pl, static_cast<uint8_t *>(pp.arena.ptr), r.B);
  }
  if (pl.host_input) {
    r.host_src = Pg.base;
    r.dbase = r.B.input;
  } else {
    r.dbase = static_cast<const uint8_t *>(Pg.base);
  }
  const bool od = !pl.host_out;
  r.d_next = pl.want_ring ? (od ? out->next + r.poff : r.B.st_next) : nullptr;
  r.d_label = pl.want_label ? (od ? out->label + r.poff : r.B.st_label) : nullptr;
  r.d_minid = pl.want_minid ? (od ? reinterpret_cast<unsigned long long *>(out->minid) + r.poff
                                  : r.B.st_minid)
                            : nullptr;
  const bool direct = od && !pl.stage_halos;
  r.d_halo = pl.want_halos ? (direct ? out->halos : r.B.st_halo) : nullptr;
  r.d_mom = pl.want_mom ? (direct ? out->moments : r.B.st_mom) : nullptr;
  r.hcap = r.d_halo ? (direct ? out->halo_cap : pl.Hstage) : 0;
  return build_head(pl, r.B, pp);
}

// Is this host memory the device copies from as it is (page-locked)?
static bool page_locked(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type == hipMemoryTypeHost || a.type == hipMemoryTypeManaged;
}

// Copies between pageable host memory and the device through page-locked
// pieces, several threads each filling (or emptying) two of their own in turn.
// The runtime's own staging of such a copy reached 27 to 39 GB/s up and 18 down
// where a page-locked copy reaches 57: a call on 2.4e6 host records of 32 bytes
// took 5.0 ms with the domain check ahead of it, 4.8 with the check beside it, and
// takes 3.6 with pieces checked as they are filled.  Small copies stay the
// runtime's: a thread costs some 20 us to start.  Pieces hold whole records, unit
// bytes each.  seen(a, b): units [a, b) are about to go up.
constexpr size_t kStaged = 4 * kPiece;

// Is a copy of this host memory staged?  Not where the pieces cannot be had.
static bool staged(fof_ctx *ctx, const void *host, size_t bytes, size_t unit) {
  EngineState &S = ctx->st;
  if (bytes < kStaged || unit > kPiece || page_locked(host)) return false;
  if (ensure_host(S.pieces, 2 * kCopyThreads * kPiece)) {
    (void)hipGetLastError();
    return false;
  }
  for (auto &e : S.piece_ev)
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      e = nullptr;
      (void)hipGetLastError();
      return false;
    }
  return true;
}

static int staged_copy(fof_ctx *ctx, bool up, uint8_t *dev, uint8_t *host, size_t bytes,
                       size_t unit, hipStream_t st,
                       const std::function<void(uint64_t, uint64_t)> &seen) {
  EngineState &S = ctx->st;
  const uint64_t n = bytes / unit, per = std::max<uint64_t>(1, kPiece / unit);
  const uint64_t np = (n + per - 1) / per;
  const unsigned nth = (unsigned)std::min<uint64_t>(
      {kCopyThreads, std::max(1u, std::thread::hardware_concurrency()), np});
  std::atomic<int> err{(int)hipSuccess};
  run_threads(nth, [&](unsigned t) {
    hipError_t e = hipSetDevice(ctx->device);
    uint8_t *const buf = static_cast<uint8_t *>(S.pieces.ptr) + 2 * t * kPiece;
    hipEvent_t *const ev = S.piece_ev + 2 * t;
    auto empty = [&](uint64_t q, int b) {  // the piece that came down
      memcpy(host + q * per * unit, buf + b * kPiece, (std::min(n, (q + 1) * per) - q * per) * unit);
    };
    int k = 0;
    for (uint64_t q = t; q < np && e == hipSuccess; q += nth, k++) {
      const uint64_t a = q * per, z = std::min(n, a + per);
      uint8_t *const p = buf + (k & 1) * kPiece;
      if (k >= 2) e = hipEventSynchronize(ev[k & 1]);
      if (e != hipSuccess) break;
      if (up) {
        if (seen) seen(a, z);
        memcpy(p, host + a * unit, (z - a) * unit);
        e = hipMemcpyAsync(dev + a * unit, p, (z - a) * unit, hipMemcpyHostToDevice, st);
      } else {
        if (k >= 2) empty(q - 2 * (uint64_t)nth, k & 1);
        e = hipMemcpyAsync(p, dev + a * unit, (z - a) * unit, hipMemcpyDeviceToHost, st);
      }
      if (e == hipSuccess) e = hipEventRecord(ev[k & 1], st);
    }
    // the pieces in flight: up, the buffers are filled again by the next copy
    for (int m = std::max(0, k - 2); m < k; m++) {
      const hipError_t w = hipEventSynchronize(ev[m & 1]);
      if (e == hipSuccess) e = w;
      if (!up && e == hipSuccess) empty(t + (uint64_t)m * nth, m & 1);
    }
    if (e != hipSuccess) err = (int)e;
  });
  if (err.load() != (int)hipSuccess)
    return fof_set_hip_error((hipError_t)err.load(), "staged copy", __FILE__, __LINE__);
  return 0;
}

// An output to the host.
static int to_host(fof_ctx *ctx, void *host, const void *dev, size_t bytes, hipStream_t st) {
  if (staged(ctx, host, bytes, 4))
    return staged_copy(ctx, false, static_cast<uint8_t *>(const_cast<void *>(dev)),
                       static_cast<uint8_t *>(host), bytes, 4, st, nullptr);
  FOF_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st));
  return 0;
}

// Uploads that precede a pipeline's kernels: the head block and, for
// host-resident input, the particle records (checked on their way when staged).
static int upload_run(fof_ctx *ctx, Run &r, hipStream_t st, HostCheck *check, bool &all_seen) {
  if (r.pl.N == 0) return 0;
  if (r.host_src) {
    const size_t bytes = r.pl.N * r.pl.stride;
    if (staged(ctx, r.host_src, bytes, r.pl.stride)) {
      std::atomic<bool> bad{false};
      int rc = staged_copy(ctx, true, r.B.input,
                           static_cast<uint8_t *>(const_cast<void *>(r.host_src)), bytes,
                           r.pl.stride, st, [&](uint64_t a, uint64_t z) {
                             if (check && !check->range(r.poff + a, r.poff + z)) bad = true;
                           });
      if (bad && check) check->state = 2;
      if (rc) return rc;
    } else {
      all_seen = false;
      FOF_HIP(hipMemcpyAsync(r.B.input, r.host_src, bytes, hipMemcpyHostToDevice, st));
    }
  }
  const HeadLayout hl(r.pl.nvol, r.pl.vt_entries);
  FOF_HIP(hipMemcpyAsync(r.B.small, r.pp->up.ptr, hl.bytes, hipMemcpyHostToDevice, st));
  return 0;
}

// Every kernel of a pipeline, in stream order.  Without a variable linking
// length or occupied-cell addressing nothing here waits for the host, so the
// sequence can be captured in a graph.
static int enqueue_run(Run &r, hipStream_t st) {
  Plan &pl = r.pl;
  Bufs &B = r.B;
  Pipe &pp = *r.pp;
  const uint64_t N = pl.N;
  if (N == 0) return 0;
  const uint32_t nvol = pl.nvol;
  int rc = 0;
  const uint8_t *dbase = r.dbase;
  uint32_t *small = B.small;
  unsigned long long *ctr = reinterpret_cast<unsigned long long *>(small + kSmCtr);
  const bool timing = r.timing;
  if (timing && !pp.events) {
    for (auto &e : pp.ev) FOF_HIP(hipEventCreate(&e));
    pp.events = true;
  }
  r.spans = 0;
  r.first_span = r.last_span = -1;
  auto tb = [&](int k) -> int {
    if (timing) {
      FOF_HIP(hipEventRecord(pp.ev[2 * k], st));
      if (r.first_span < 0) r.first_span = k;
    }
    return 0;
  };
  auto te = [&](int k) -> int {
    if (timing) {
      FOF_HIP(hipEventRecord(pp.ev[2 * k + 1], st));
      r.spans |= 1u << k;
      r.last_span = k;
    }
    return 0;
  };
  if (pl.varlink) {
    // A variable l: the sub-cell size follows the smallest l of any occupied
    // cell (only occupied cells are home cells of a pair), not of the table.
    unsigned long long *dmin = reinterpret_cast<unsigned long long *>(B.hoff);
    if ((rc = fill_u32(reinterpret_cast<uint32_t *>(dmin), 2ull * nvol, ~0u, st))) return rc;
    k_varlink_min<<<(uint32_t)((N + 4 * kVlRun - 1) / (4 * kVlRun)), 256, 0, st>>>(
        dbase, pl.stride, pl.offpos, (uint32_t)N, B.vols, B.vbeg, (int)nvol, dmin);
    FOF_HIP(hipGetLastError());
    std::vector<unsigned long long> hmin(nvol);
    FOF_HIP(hipMemcpyAsync(hmin.data(), dmin, nvol * 8, hipMemcpyDeviceToHost, st));
    FOF_HIP(hipStreamSynchronize(st));
    for (uint32_t v = 0; v < nvol; v++) {
      if (pl.vt_off[v] == ~0u || hmin[v] == ~0ull) continue;
      double l2;
      memcpy(&l2, &hmin[v], 8);
      set_subcells(pl.hv[v].d, l2);
    }
    const HeadLayout hl(nvol, pl.vt_entries);
    build_vols(pl, B, static_cast<uint8_t *>(pp.up.ptr) + hl.vols);
    FOF_HIP(hipMemcpyAsync(B.vols, static_cast<uint8_t *>(pp.up.ptr) + hl.vols,
                           nvol * sizeof(VolDev), hipMemcpyHostToDevice, st));
  }

  const VolDev *dV = B.vols;
  const uint32_t *dVB = B.vbeg;
  float4 *pos4 = B.pos4;
  uint32_t *key = B.key, *start = B.start, *par = B.par, *runend = B.runend, *rtab = B.rtab;
  unsigned long long *fine = B.fine;
  uint32_t *rtoff = key;  // free between the cell sort and k_label (head sizes)
  uint32_t *gsize = B.gsize, *label = B.label;
  const uint64_t q4 = (N + 63) / 64 * 64;
  // four u32 arrays; viewed as float4[N] they are the sub-cell sort buffer
  uint32_t *sk0 = B.sortbuf, *sv0 = sk0 + q4, *sk1 = sk0 + 2 * q4, *sv1 = sk0 + 3 * q4;
  uint32_t *dense = B.dense, *dbig = dense + pl.ndense_cap;
  const uint32_t NN = (uint32_t)N;
  const uint32_t stride = pl.stride, offpos = pl.offpos, offvel = pl.offvel;
  const uint32_t offid = pl.offid >= 0 ? (uint32_t)pl.offid : 0u;
  const uint32_t gN = grid_for(N);
  const uint32_t T = pl.T;
  const bool direct = pl.direct_writes;
  // direct writes and no minimum IDs: the key pass writes the outputs'
  // defaults and k_label label_out itself, and k_out_init is not needed
  const bool fused = direct && !r.d_minid;
  uint32_t *label0 = fused ? r.d_label : nullptr, *next0 = fused ? r.d_next : nullptr;

  Grid G;
  G.start = start;
  G.cell_of = label;  // sparse: the label buffer is free until k_label
  G.klo = B.cnt;      // sparse: the flags' buffer and the sizes' (cleared after linking)
  G.khi = gsize;
  G.ncell = small + kSmU;
  G.err = small + kSmErr;
  G.sparse = pl.sparse ? 1 : 0;
  G.volshift = pl.volshift;
  if (!pl.sparse) {
    // 1-3: counting sort by cell: partitions A (coarse) and B (fine), then C
    const uint32_t F = pl.F, Bc = pl.Bc, ntA = pl.ntA, ntBmax = pl.ntBmax;
    const uint64_t nA = pl.nA, nB = pl.nB;
    // pass A's histogram and its prefix in the fine-coordinate buffer (free
    // until k_subsort) where they fit
    const bool inf = pl.hist_in_fine;
    uint32_t *histA = inf ? reinterpret_cast<uint32_t *>(B.fine) : B.part;
    const uint64_t nA4 = (nA + 3) / 4 * 4 + 32;  // the scans' vector accesses stay aligned
    uint32_t *offA = histA + nA4;                 // nA + 1
    uint32_t *histB = inf ? B.part : offA + nA4;  // nB
    uint32_t *offB = histB + nB + 32;      // nB + 1
    uint32_t *cst = offB + nB + 32;        // Bc + 1
    uint32_t *t0 = cst + Bc + 32;          // Bc + 1
    uint32_t *tinfo = t0 + Bc + 32;        // ntBmax
    uint32_t *fst = tinfo + ntBmax + 32;   // F + 1
    uint32_t *k1 = gsize, *k2 = label;     // free until the union-find finish / k_label
    float4 *p1 = pos4;                     // pass A output, consumed before pass C writes
    float4 *p2 = reinterpret_cast<float4 *>(sk0);
    const uint32_t ptile = pl.ptile;
    const int fb = pl.fb, shift = pl.two_level ? fb + 8 : fb;
    if ((rc = tb(0))) return rc;
    k_pa_count<<<ntA, 256, 0, st>>>(dbase, stride, offpos, NN, dV, dVB, (int)nvol, Bc, ntA, ptile,
                                    shift, key, histA, label0, next0, small + kSmErr);
    FOF_HIP(hipGetLastError());
    if ((rc = te(0))) return rc;
    if ((rc = tb(1))) return rc;
    if ((rc = scan_u32(histA, offA, nA, B.tmp, st))) return rc;
    if (pl.two_level) {
      k_pa_starts<<<grid_for(Bc + 1), 256, 0, st>>>(Bc, ntA, offA, cst);
      FOF_HIP(hipGetLastError());
      k_pb_tiles<<<1, kMaxCoarse, 0, st>>>(Bc, ntBmax, ptile, cst, t0, tinfo, small + kSmNtB);
      FOF_HIP(hipGetLastError());
    }
    if ((rc = te(1))) return rc;
    if ((rc = tb(2))) return rc;
    // one level: straight to pass C's input
    uint32_t *ka = pl.two_level ? k1 : k2;
    float4 *pa = pl.two_level ? p1 : p2;
    k_pa_scatter<<<ntA, kPartNT, 0, st>>>(dbase, stride, offpos, NN, Bc, ntA, ptile, shift, key,
                                          offA, ka, pa);
    FOF_HIP(hipGetLastError());
    if (pl.two_level) {
      k_pb_count<<<ntBmax, 256, 0, st>>>(ptile, fb, tinfo, t0, cst, k1, histB);
      FOF_HIP(hipGetLastError());
      if ((rc = scan_u32(histB, offB, nB, B.tmp, st))) return rc;
      k_pb_scatter<<<ntBmax, kPartNT, 0, st>>>(ptile, fb, tinfo, t0, cst, offB, k1, p1, k2, p2);
      FOF_HIP(hipGetLastError());
      k_pb_starts<<<grid_for(F + 1), 256, 0, st>>>(F, t0, cst, offB, NN, fst);
      FOF_HIP(hipGetLastError());
    }
    k_pc_sort<<<F, kPcThreads, 0, st>>>((uint64_t)pl.C, fb, pl.two_level ? fst : offA,
                                        pl.two_level ? 1u : ntA, k2, p2, start, pos4, dV,
                                        (int)nvol, small + kSmErr, T, dense, small + kSmNDense, dbig,
                                        small + kSmNBig, par, runend, gsize);
    FOF_HIP(hipGetLastError());
    if ((rc = te(2))) return rc;
  } else {
    // 1-3: composite keys, LSD sort by (volume, cell), occupied cells
    uint32_t *cnt = B.cnt;
    if ((rc = tb(0))) return rc;
    k_keys_sparse<<<gN, 256, 0, st>>>(dbase, stride, offpos, NN, dV, dVB, (int)nvol, G, sk0, key,
                                      sv0, label0, next0, small + kSmErr);
    FOF_HIP(hipGetLastError());
    if ((rc = te(0))) return rc;
    if ((rc = tb(1))) return rc;
    if ((rc = radix_sort_u32(sk0, sv0, sk1, sv1, N, std::min(pl.key_bits, 32), B.tmp, st)))
      return rc;
    if (pl.key_bits > 32) {
      k_gather_u32<<<gN, 256, 0, st>>>(NN, key, sv0, gsize);
      FOF_HIP(hipGetLastError());
      if ((rc = radix_sort_u32(gsize, sv0, sk1, sv1, N, pl.key_bits - 32, B.tmp, st)))
        return rc;
    }
    if ((rc = te(1))) return rc;
    if ((rc = tb(2))) return rc;
    k_scatter_sparse<<<gN, 256, 0, st>>>(dbase, stride, offpos, NN, sv0, dV, dVB, (int)nvol, G,
                                         pos4, par, runend);
    FOF_HIP(hipGetLastError());
    if ((rc = te(2))) return rc;
    k_cell_flags<<<gN, 256, 0, st>>>(NN, par, runend, cnt);
    FOF_HIP(hipGetLastError());
    if ((rc = compact_flagged(cnt, N, kFlag, start, label, small + kSmU, B.tmp, st))) return rc;
    k_cells_finish<<<(uint32_t)((N + kCellTile - 1) / kCellTile), 256, 0, st>>>(
        small + kSmU, NN, start, par, runend, cnt, gsize, dV, dVB, (int)nvol, small + kSmErr, T, dense,
        small + kSmNDense, dbig, small + kSmNBig);
    FOF_HIP(hipGetLastError());
    if ((rc = tb(3))) return rc;
    k_init_uf<<<gN, 256, 0, st>>>(NN, par, runend);
    FOF_HIP(hipGetLastError());
    if ((rc = te(3))) return rc;
  }
  // 4: sub-cell sort of dense cells (tmp4 aliases the sort buffers s0..s3);
  // grids for the most dense cells there can be, the lists' lengths are read
  // on the device
  const uint32_t gsml = (uint32_t)std::min<uint64_t>(pl.ndense_cap, 65536);
  const uint32_t gbig = (uint32_t)std::min<uint64_t>(N / kBigCell + 1, pl.big_grid);
  bool any_sub = false;
  for (uint32_t v = 0; v < nvol; v++) any_sub = any_sub || pl.hv[v].d.m[0] > 0;
  // constant l on a dense grid: k_link_sparse skips every dense cell, so only
  // the cells k_link_dense links need runs; otherwise it scans dense forward
  // cells run by run, and the smaller dense cells are sub-sorted too
  bool fast = !pl.sparse;
  for (uint32_t v = 0; v < nvol; v++) fast = fast && pl.hv[v].d.vntab == 0 && pl.hv[v].d.m[0] > 0;
  if (any_sub) {
    if ((rc = tb(4))) return rc;
    if (!fast) {
      k_subsort<256><<<gsml, 256, 0, st>>>(dense, small + kSmNDense, start, dV, dVB, (int)nvol,
                                           pos4, reinterpret_cast<float4 *>(sk0), par, runend,
                                           fine, rtoff, rtab);
      FOF_HIP(hipGetLastError());
    }
    k_subsort<256><<<gbig, 256, 0, st>>>(dbig, small + kSmNBig, start, dV, dVB, (int)nvol,
                                                pos4, reinterpret_cast<float4 *>(sk0), par, runend,
                                                fine, rtoff, rtab);
    FOF_HIP(hipGetLastError());
    if ((rc = te(4))) return rc;
  }
  // 5-6: linking.  The three kernels unite particles of one shared union-find
  // and need nothing of each other, so in eager, untimed calls k_link_small
  // runs beside the other two: with few cells each waits for its largest one
  // (64^3 box: 264, 47 and 289 us; the call took 0.97 ms in one stream, 0.75 so;
  // 1024^3 in 64 volumes: no difference).  A captured call keeps to one stream
  // a pipeline.
  hipStream_t st15 = r.side ? pp.side : st;
  if (r.side) {
    FOF_HIP(hipEventRecord(pp.side_fork, st));
    FOF_HIP(hipStreamWaitEvent(pp.side, pp.side_fork, 0));
  }
  // the most sub-cells (so runs) a dense cell of the batch can have
  uint32_t maxbins = 1;
  for (uint32_t v = 0; v < nvol; v++)
    if (pl.hv[v].d.m[0] > 0)
      maxbins = std::max(maxbins, (uint32_t)(pl.hv[v].d.m[0] * pl.hv[v].d.m[1] * pl.hv[v].d.m[2]));
  // dense cells below kBigCell particles, with or without sub-cells
  if ((rc = tb(15))) return rc;
  k_link_small<<<(gsml + kSmallWaves - 1) / kSmallWaves, 64 * kSmallWaves, 0, st15>>>(
      dense, small + kSmNDense, pos4, G, T, par, dV, dVB, (int)nvol, ctr);
  FOF_HIP(hipGetLastError());
  if ((rc = te(15))) return rc;
  if (any_sub) {
    if ((rc = tb(6))) return rc;
    constexpr int kRB = 448;
    const uint32_t ra = std::min(maxbins, (uint32_t)kMaxRuns);
    // wider workgroups while there are too few cells to fill the chip and the
    // largest one's chain is what is waited for: 31^3, 64^3, 144^3, 192^3 and
    // 256^3 boxes 134, 249, 525, 530 and 777 us with 256 threads, 92, 203, 436,
    // 499 and 872 with 512, 74, 186, 420, - and 1418 with 1024 (with a division
    // a test of long pairs; without it 74, 160, 356, 490 and 738 as chosen here)
    auto link_dense = [&](auto kernel, int nt) {
      kernel<<<gbig, nt, dense_lds(ra, kRB), st>>>(dbig, small + kSmNBig, pos4, G, runend, fine,
                                                   rtoff, rtab, T, par, dV, dVB, (int)nvol, ctr, ra,
                                                   small + kSmDq);
    };
    if (N <= (1u << 20)) link_dense(k_link_dense<1024, 4, kMaxRuns, kRB>, 1024);
    else if (N <= (1u << 23)) link_dense(k_link_dense<512, 6, kMaxRuns, kRB>, 512);
    else link_dense(k_link_dense<256, 6, kMaxRuns, kRB>, 256);
    FOF_HIP(hipGetLastError());
    if ((rc = te(6))) return rc;
  }
  if ((rc = tb(5))) return rc;
  if (fast)
    k_link_sparse<true><<<gN, 256, 0, st>>>(NN, pos4, G, runend, fine, par, dV, dVB, (int)nvol, T, ctr);
  else if (pl.sparse)
    k_link_rows<<<(uint32_t)((N + 4 * kRowRun - 1) / (4 * kRowRun)), 256, 0, st>>>(
        NN, pos4, G, runend, fine, rtoff, rtab, par, dV, dVB, (int)nvol, T, ctr);
  else
    k_link_sparse<false><<<gN, 256, 0, st>>>(NN, pos4, G, runend, fine, par, dV, dVB, (int)nvol, T, ctr);
  FOF_HIP(hipGetLastError());
  if ((rc = te(5))) return rc;
  if (r.side) {
    FOF_HIP(hipEventRecord(pp.side_join, pp.side));
    FOF_HIP(hipStreamWaitEvent(st, pp.side_join, 0));
  }
  // 7: union-find finish (minorig reuses runend, hsize reuses key, the
  // members' minimum ID reuses fine)
  uint32_t *minorig = runend, *hsize = key;
  unsigned long long *idroot = pl.want_minid ? fine : nullptr;
  if ((rc = tb(7))) return rc;
  const uint64_t nw = (N + 31) / 32;
  uint32_t *gbits = key;  // the label bitmap (the head sizes follow in k_label)
  k_init_groups<<<gN, 256, 0, st>>>(NN, minorig, idroot, pl.sparse ? gsize : nullptr, (uint32_t)nw,
                                    gbits, pos4, par, dV, dVB, (int)nvol, ctr);
  FOF_HIP(hipGetLastError());
  k_flatten<<<gN, 256, 0, st>>>(NN, par, pos4, minorig, gsize, ctr, dbase, stride, offid, idroot);
  FOF_HIP(hipGetLastError());
  if ((rc = te(7))) return rc;
  // 8: the group list -- groups of two or more (and kept groups of one) in
  // label order, each group's first slot in the member list -- and the halo
  // list (first slots of the groups passing the size cut), then the labels,
  // which also fill the member list.  The sizes by label live in the label
  // array (before its defaults), the first slots in sk1 (and one word of sv1
  // behind it: there may be N + 1 of them); lists of larger groups go to the
  // cell-sorted positions once k_label has read them.
  const int single = pl.single_halos ? 1 : 0;
  const uint64_t rcap = std::max<uint64_t>(single ? N : N / 2, 1);
  uint32_t *lsize = label;
  uint32_t *offs = sk1;
  uint32_t *cursor = rtab;             // per label, from its group's first slot
  uint32_t *p32 = reinterpret_cast<uint32_t *>(pos4);
  // groups above kSegLds, kSegWave and four members (at most N / 4096,
  // N / 1024 and N / 5 of them)
  uint32_t *huge = p32 + 3 * N, *large = huge + N / kSegLds, *mid = large + N / kSegWave;
  uint32_t *hlist = pl.want_halos ? B.hhead : nullptr;
  if ((rc = tb(9))) return rc;
  k_group_bits<<<gN, 256, 0, st>>>(NN, par, gsize, minorig, pos4, gbits, lsize, single, dV, dVB,
                                   (int)nvol);
  FOF_HIP(hipGetLastError());
  const uint32_t runs = group_runs(nw), gb = (uint32_t)((nw + 256ull * runs - 1) / (256ull * runs));
  GroupTot *gtot = static_cast<GroupTot *>(B.tmp);
  k_group_sums<<<gb, 256, 0, st>>>(nw, runs, gbits, lsize, dV, dVB, (int)nvol, gtot);
  FOF_HIP(hipGetLastError());
  k_group_emit<<<gb, 256, 0, st>>>(nw, runs, gbits, lsize, dV, dVB, (int)nvol, gtot, offs, cursor,
                                   hlist, small);
  FOF_HIP(hipGetLastError());
  if (!fused) {
    k_label_init<<<tiles_for(N), 256, 0, st>>>(NN, dV, dVB, (int)nvol, label, hsize);
    FOF_HIP(hipGetLastError());
  }
  if ((rc = te(9))) return rc;
  if ((rc = tb(8))) return rc;
  const uint32_t glab = (uint32_t)((N + kLabTile - 1) / kLabTile);
  if (direct)
    k_label<true><<<glab, 256, 0, st>>>(NN, par, pos4, minorig, gsize, label, hsize, cursor, sk0,
                                        sv0, dbase, stride, offid, idroot, B.idhead, single, dV,
                                        dVB, (int)nvol, fused ? r.d_label : nullptr);
  else
    k_label<false><<<glab, 256, 0, st>>>(NN, par, pos4, minorig, gsize, label, hsize, cursor, sk0,
                                         sv0, dbase, stride, offid, idroot, B.idhead, single, dV,
                                         dVB, (int)nvol, nullptr);
  FOF_HIP(hipGetLastError());
  if (!direct && (rc = scatter_u32(sv0, sk0, p32, p32 + N, N, small + kSmM, N, label, kFlag,
                                   B.tmp, st)))
    return rc;
  if (!fused) {
    k_out_init<<<tiles_for(N), 256, 0, st>>>(NN, label, dVB, (int)nvol, r.d_label, r.d_next,
                                             hsize, dbase, stride, offid, B.idhead, r.d_minid);
    FOF_HIP(hipGetLastError());
  }
  if ((rc = te(8))) return rc;
  // members in index order inside each group (large groups through the
  // free cell-sorted positions)
  if ((rc = tb(10))) return rc;
  k_seg_sort<<<(uint32_t)std::min<uint64_t>((rcap + 255) / 256, 8192), 256, 0, st>>>(
      small + kSmR, offs, sv0, mid, small + kSmMid, large, small + kSmLarge, huge, small + kSmHuge);
  FOF_HIP(hipGetLastError());
  if (N > kSegLds) {
    k_seg_sort_list<1024, kSegLdsBig, false>
        <<<(uint32_t)std::min<uint64_t>(N / kSegLds, 512), 1024, 0, st>>>(
            small + kSmHuge, huge, nullptr, nullptr, offs, sv0, p32, bits_for(N));
    FOF_HIP(hipGetLastError());
  }
  k_seg_sort_list<256, kSegLds, true><<<(uint32_t)std::min<uint64_t>(N / 20 + 1, 8192), 256, 0, st>>>(
      small + kSmLarge, large, small + kSmMid, mid, offs, sv0, p32, bits_for(N));
  FOF_HIP(hipGetLastError());
  if ((rc = te(10))) return rc;
  // 9: the rings
  if ((rc = tb(11))) return rc;
  {
    // ring pairs (the partitioned way) in the free cell-sorted positions
    uint32_t *pidx = (r.d_next && !direct) ? p32 : nullptr;
    k_ring<<<tiles_for(N), 256, 0, st>>>(small + kSmM, sk0, sv0, dVB, (int)nvol, r.d_next, pidx,
                                        p32 + N);
    FOF_HIP(hipGetLastError());
    if (pidx && (rc = scatter_u32(p32, p32 + N, p32 + 2 * N, p32 + 3 * N, N, small + kSmM, N,
                                  r.d_next, 0u, B.tmp, st)))
      return rc;
  }
  if ((rc = te(11))) return rc;
  if (pl.want_halos) {
    if ((rc = tb(13))) return rc;
    const uint32_t gh = (uint32_t)std::min<uint64_t>((pl.Hbound * 64 + 255) / 256, 8192);
    if (r.d_mom)
      k_halo_sums<true><<<gh, 256, 0, st>>>(small + kSmH, hlist, sk0, sv0, hsize, dbase, stride,
                                            offpos, offvel, dV, dVB, (int)nvol, r.d_halo, r.d_mom,
                                            r.hcap, B.hoff, ctr);
    else
      k_halo_sums<false><<<gh, 256, 0, st>>>(small + kSmH, hlist, sk0, sv0, hsize, dbase, stride,
                                             offpos, offvel, dV, dVB, (int)nvol, r.d_halo, nullptr,
                                             r.hcap, B.hoff, ctr);
    FOF_HIP(hipGetLastError());
    if ((rc = te(13))) return rc;
  }
  return 0;
}

// Counts, flags, counters and halo offsets back to the host (after the
// pipeline's kernels, on the same stream).
static int readback_run(Run &r, hipStream_t st) {
  if (r.pl.N == 0) return 0;
  const HeadLayout hl(r.pl.nvol, r.pl.vt_entries);
  FOF_HIP(hipMemcpyAsync(r.pp->down.ptr, r.B.small, r.pl.want_halos ? hl.vols : kSmallBytes,
                         hipMemcpyDeviceToHost, st));
  return 0;
}

static uint32_t run_nhalos(const Run &r) {
  if (r.pl.N == 0 || !r.pl.want_halos) return 0;
  return static_cast<const uint32_t *>(r.pp->down.ptr)[kSmH];
}

// Staged halos (and moments) of the pipelines of a call into the output, at
// each pipeline's prefix of the halo counts (read on the device).
struct HaloParts {
  const fof_halo_v1 *src[kMaxPipes];
  const fof_moments_v1 *msrc[kMaxPipes];
  const uint32_t *cnt[kMaxPipes];
  uint64_t stage[kMaxPipes];
  int k;
};

__global__ __launch_bounds__(256) void k_gather_halos(HaloParts hp, fof_halo_v1 *__restrict__ out,
                                                      fof_moments_v1 *__restrict__ mout,
                                                      uint64_t cap) {
  uint64_t base = 0;
  for (int g = 0; g < hp.k; g++) {
    const uint64_t h = hp.cnt[g] ? min((uint64_t)*hp.cnt[g], hp.stage[g]) : 0;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < h; i += (uint64_t)gridDim.x * 256) {
      if (base + i >= cap) break;
      if (out) out[base + i] = hp.src[g][i];
      if (mout) mout[base + i] = hp.msrc[g][i];
    }
    base += hp.cnt[g] ? *hp.cnt[g] : 0u;
  }
}

// ---------------------------------------------------------------------------
// Autotuning: dense-cell threshold, concurrent pipelines and the grid of
// k_link_dense, per workload shape.
// ---------------------------------------------------------------------------
static uint32_t ilog2(uint64_t x) {
  uint32_t b = 0;
  while (x > 1) x >>= 1, b++;
  return b;
}

// Shape of a call: log2 of particles and volumes, addressing, variable l,
// particles per cell (x16, log2) and the linking length over the cell size
// (x64).  Calls with one key behave alike for the tuned parameters.
static TuneKey tune_key(const Plan &pl) {
  TuneKey k;
  k.lg_n = ilog2(pl.N);
  k.lg_nvol = ilog2(pl.nvol);
  k.sparse = pl.sparse ? 1 : 0;
  k.varlink = pl.varlink ? 1 : 0;
  k.ppc16 = ilog2((uint64_t)(16.0 * (double)pl.N / std::max(1.0, pl.Cd)) + 1);
  double b = 0;
  for (const HostVol &h : pl.hv) b += h.d.linklength / h.d.lcell[0];
  k.b64 = (uint32_t)std::lround(64.0 * b / std::max<size_t>(1, pl.hv.size()));
  return k;
}

static std::mutex g_tune_mu;

static const char *tune_path() {
  const char *p = getenv("FOF_TUNE_CACHE");
  return (p && *p) ? p : nullptr;
}

static bool tune_lookup(EngineState &S, const TuneKey &k, TuneVal &v) {
  for (auto &e : S.tuned)
    if (e.first == k) {
      v = e.second;
      return true;
    }
  const char *path = tune_path();
  if (!path) return false;
  std::lock_guard<std::mutex> lk(g_tune_mu);
  FILE *f = fopen(path, "r");
  if (!f) return false;
  char line[256];
  bool found = false;
  while (fgets(line, sizeof line, f)) {
    TuneKey q;
    TuneVal w;
    if (sscanf(line, "%u %u %u %u %u %u -> %u %u %u", &q.lg_n, &q.lg_nvol, &q.sparse, &q.varlink,
               &q.ppc16, &q.b64, &w.T, &w.pipes, &w.gbig) == 9 &&
        q == k) {
      v = w;  // the last entry for a key wins
      found = true;
    }
  }
  fclose(f);
  if (found) S.tuned.push_back({k, v});
  return found;
}

static void tune_store(EngineState &S, const TuneKey &k, const TuneVal &v) {
  S.tuned.push_back({k, v});
  const char *path = tune_path();
  if (!path) return;
  std::lock_guard<std::mutex> lk(g_tune_mu);
  FILE *f = fopen(path, "a");
  if (!f) return;
  fprintf(f, "%u %u %u %u %u %u -> %u %u %u\n", k.lg_n, k.lg_nvol, k.sparse, k.varlink, k.ppc16,
          k.b64, v.T, v.pipes, v.gbig);
  fclose(f);
}

}  // namespace fof

using namespace fof;

extern "C" int fof_engine_plan(const fof_particles_v1 *P, const fof_volume_v1 *vols,
                               uint32_t nvol, const fof_opts_v1 *opts, fof_plan_v1 *out) {
  Plan pl;
  fof_outputs_v1 o;
  memset(&o, 0, sizeof(o));
  o.location = FOF_MEM_DEVICE;
  o.label = reinterpret_cast<uint32_t *>(1);  // a typical call: ring, labels, halos
  o.next = reinterpret_cast<uint32_t *>(1);
  int rc = make_plan(P, vols, nvol, opts, &o, pl);
  if (rc) return rc;
  Bufs b;
  memset(out, 0, sizeof(*out));
  out->version = FOF_ABI_VERSION;
  out->sparse = pl.sparse ? 1u : 0u;
  out->n = pl.N;
  out->cells = pl.sparse ? 0 : pl.C;
  out->grid_cells = pl.Cd;
  out->workspace_bytes = layout(pl, nullptr, b);
  out->dense_threshold = pl.T;
  return 0;
}

namespace fof {

// FNV-1a over the bytes that fix a call's launch sequence.
struct Sig {
  uint64_t h = 1469598103934665603ull;
  void add(const void *p, size_t n) {
    const uint8_t *b = static_cast<const uint8_t *>(p);
    for (size_t i = 0; i < n; i++) h = (h ^ b[i]) * 1099511628211ull;
  }
  template <class T>
  void add(const T &x) {
    add(&x, sizeof(T));
  }
};

// Volumes split into k contiguous groups of about equal particle counts.
static std::vector<uint32_t> split_volumes(const fof_volume_v1 *vols, uint32_t nvol, uint32_t k) {
  uint64_t tot = 0;
  for (uint32_t v = 0; v < nvol; v++) tot += vols[v].n;
  std::vector<uint32_t> cut{0};
  uint64_t acc = 0;
  for (uint32_t v = 0; v < nvol; v++) {
    acc += vols[v].n;
    const uint32_t g = (uint32_t)cut.size();
    // cut after v when this group has its share, or when every later group
    // needs one of the remaining volumes
    if (g < k && v + 1 < nvol && (acc * k >= tot * g || nvol - (v + 1) <= k - g)) cut.push_back(v + 1);
  }
  cut.push_back(nvol);
  return cut;
}

// A pipeline's side stream: pipeline 0's is made at context set-up (0.2 ms),
// another's by its first eager call.
static int open_side(Pipe &pp) {
  if (!pp.side) FOF_HIP(hipStreamCreate(&pp.side));
  if (!pp.side_fork) FOF_HIP(hipEventCreateWithFlags(&pp.side_fork, hipEventDisableTiming));
  if (!pp.side_join) FOF_HIP(hipEventCreateWithFlags(&pp.side_join, hipEventDisableTiming));
  return 0;
}

// One call with a fixed configuration: pipelines `pipes`, graph replay when
// asked for and possible; with one_stream the link kernels of a pipeline one
// after the other, as in a captured or timed call.
static int run_call(fof_ctx *ctx, const fof_particles_v1 *P, const fof_volume_v1 *vols,
                    uint32_t nvol, const fof_opts_v1 *opts, fof_outputs_v1 *out, uint32_t pipes,
                    double *wall_ms, HostCheck *check, bool one_stream = false,
                    uint8_t *fixed = nullptr, size_t fixed_bytes = 0) {
  EngineState &S = ctx->st;
  const uint32_t flags = opts ? opts->flags : 0u;
  fof_stats_v1 *stats = out->stats;
  out->nhalos = 0;
  if (out->halo_offsets)
    for (uint32_t v = 0; v <= nvol; v++) out->halo_offsets[v] = 0;
  pipes = std::max(1u, std::min({pipes, nvol, (uint32_t)kMaxPipes}));
  const std::vector<uint32_t> cut = split_volumes(vols, nvol, pipes);
  const uint32_t K = (uint32_t)cut.size() - 1;
  int rc = 0;
  if (S.pipes.empty()) S.pipes.push_back(nullptr);  // pipeline 0 is S.main
  while (S.pipes.size() < K) {
    S.pipes.push_back(new Pipe);
    FOF_HIP(hipStreamCreate(&S.pipes.back()->stream));
  }
  if (!S.sync_events) {  // created at context set-up; kept for safety
    FOF_HIP(hipEventCreateWithFlags(&S.fork, hipEventDisableTiming));
    for (auto &e : S.join) FOF_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    FOF_HIP(hipEventCreate(&S.t0));
    FOF_HIP(hipEventCreate(&S.t1));
    S.sync_events = true;
  }
  std::vector<Run> runs(K);
  const bool timing = (flags & FOF_OPT_TIMING) != 0;
  for (uint32_t g = 0; g < K; g++) {
    Pipe &pp = g == 0 ? S.main : *S.pipes[g];
    if ((rc = prepare_run(runs[g], pp, P, vols, cut[g], cut[g + 1] - cut[g], opts, out, K > 1,
                          fixed, fixed_bytes)))
      return rc;
  }
  const Plan &pl0 = runs[0].pl;
  uint64_t Ntot = 0;
  bool varlink = false, sparse = false, host_io = false;
  for (auto &r : runs) {
    Ntot += r.pl.N;
    varlink = varlink || r.pl.varlink;
    sparse = sparse || r.pl.sparse;
    host_io = host_io || r.pl.host_input || r.pl.host_out;
  }
  if (stats) {
    memset(stats, 0, sizeof(*stats));
    stats->version = FOF_ABI_VERSION;
    stats->nvol = nvol;
    stats->n = Ntot;
    stats->dense_threshold = pl0.T;
    stats->big_grid = pl0.big_grid;
    stats->sparse = sparse ? 1u : 0u;
    stats->pipelines = K;
    for (auto &r : runs) stats->ncells += r.pl.sparse ? 0 : r.pl.C;
  }
  if (Ntot == 0) return 0;
  hipStream_t st = S.main.stream;
  const bool want_halos = pl0.want_halos;
  const bool gather = K > 1 && want_halos && !pl0.host_out && (out->halos || out->moments);
  const bool graph = (flags & FOF_OPT_GRAPH) && !varlink && !sparse && !host_io;
  // the pipelines' kernels, forked from and joined back to the main stream
  auto enqueue_all = [&](bool with_timing) -> int {
    for (uint32_t g = 0; g < K; g++) {
      runs[g].timing = with_timing && g == 0;
      runs[g].side = !graph && !with_timing && !one_stream;
      if (runs[g].side)
        if (int e = open_side(*runs[g].pp)) return e;
    }
    if (K > 1) FOF_HIP(hipEventRecord(S.fork, st));
    for (uint32_t g = 0; g < K; g++) {
      hipStream_t sg = runs[g].pp->stream;
      if (g > 0) FOF_HIP(hipStreamWaitEvent(sg, S.fork, 0));
      int e = enqueue_run(runs[g], sg);
      if (e) return e;
      if (g > 0) {
        FOF_HIP(hipEventRecord(S.join[g], sg));
        FOF_HIP(hipStreamWaitEvent(st, S.join[g], 0));
      }
    }
    if (gather) {
      HaloParts hp;
      memset(&hp, 0, sizeof(hp));
      hp.k = (int)K;
      for (uint32_t g = 0; g < K; g++) {
        hp.src[g] = runs[g].B.st_halo;
        hp.msrc[g] = runs[g].B.st_mom;
        hp.cnt[g] = runs[g].pl.N ? runs[g].B.small + kSmH : nullptr;
        hp.stage[g] = runs[g].pl.Hstage;
      }
      k_gather_halos<<<1024, 256, 0, st>>>(hp, out->halos, pl0.want_mom ? out->moments : nullptr,
                                           out->halo_cap);
      FOF_HIP(hipGetLastError());
    }
    return 0;
  };
  // uploads, on the main stream ahead of everything; they leave from the
  // pipelines' page-locked buffers, and kernels forked to other streams use
  // the workspaces, so an early return waits for all of them
  struct Settle {
    hipStream_t st;
    const std::vector<Run> &runs;
    bool on;
    ~Settle() {
      if (!on) return;
      (void)hipStreamSynchronize(st);
      for (const Run &r : runs) {
        if (r.pp->side) (void)hipStreamSynchronize(r.pp->side);
        if (r.pp->stream != st) (void)hipStreamSynchronize(r.pp->stream);
      }
    }
  } settle{st, runs, true};
  bool all_seen = pl0.host_input;
  for (auto &r : runs)
    if ((rc = upload_run(ctx, r, st, check, all_seen))) return rc;
  if (check) {  // no kernel sees a bad particle
    if (all_seen && check->state.load() == 0) check->state = 1;
    if ((rc = check->finish())) return rc;
  }
  const bool timed = timing || wall_ms;
  if (timed) FOF_HIP(hipEventRecord(S.t0, st));
  uint32_t graph_state = 0;
  if (graph) {
    Sig sig;
    sig.add(*P);
    sig.add(nvol);
    for (uint32_t v = 0; v < nvol; v++) sig.add(vols[v]);
    if (opts) sig.add(*opts);
    sig.add(out->location);
    sig.add(out->next), sig.add(out->label), sig.add(out->minid), sig.add(out->halos);
    sig.add(out->moments), sig.add(out->halo_cap);
    sig.add(K);
    for (auto &r : runs) sig.add(r.pp->arena.ptr);
    if (S.graph_exec && S.graph_sig == sig.h) {
      FOF_HIP(hipGraphLaunch(S.graph_exec, st));
      graph_state = 1;
    } else {
      if (S.graph_exec) (void)hipGraphExecDestroy(S.graph_exec);
      S.graph_exec = nullptr;
      FOF_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
      rc = enqueue_all(false);
      hipGraph_t gr = nullptr;
      hipError_t e = hipStreamEndCapture(st, &gr);
      if (rc) {
        if (gr) (void)hipGraphDestroy(gr);
        return rc;
      }
      if (e != hipSuccess) return fof_set_hip_error(e, "hipStreamEndCapture", __FILE__, __LINE__);
      e = hipGraphInstantiate(&S.graph_exec, gr, nullptr, nullptr, 0);
      (void)hipGraphDestroy(gr);
      if (e != hipSuccess) {
        S.graph_exec = nullptr;
        return fof_set_hip_error(e, "hipGraphInstantiate", __FILE__, __LINE__);
      }
      S.graph_sig = sig.h;
      FOF_HIP(hipGraphLaunch(S.graph_exec, st));
      graph_state = 2;
    }
  } else {
    if ((rc = enqueue_all(timing))) return rc;
  }
  if (timed) FOF_HIP(hipEventRecord(S.t1, st));
  for (auto &r : runs)
    if ((rc = readback_run(r, st))) return rc;
  FOF_HIP(hipStreamSynchronize(st));
  settle.on = false;
  float tot_ms = 0;
  if (timed) FOF_HIP(hipEventElapsedTime(&tot_ms, S.t0, S.t1));
  if (wall_ms) *wall_ms = tot_ms;

  // ---- results ----
  uint64_t H = 0;
  bool dom_err = false;
  for (auto &r : runs) {
    if (r.pl.N == 0) continue;
    const uint32_t *hsm = static_cast<const uint32_t *>(r.pp->down.ptr);
    dom_err = dom_err || hsm[kSmErr];
    H += run_nhalos(r);
  }
  out->nhalos = H;
  if (dom_err) return FOF_E_DOMAIN;
  if (want_halos && H > out->halo_cap && (out->halos || out->moments)) {
    if (out->halo_offsets) out->halo_offsets[nvol] = H;  // the capacity needed
    if (stats) stats->nhalos = H;
    return FOF_E_RANGE;
  }
  if (out->halo_offsets && want_halos) {
    uint64_t base = 0;
    for (auto &r : runs) {
      const uint64_t *ho = reinterpret_cast<const uint64_t *>(static_cast<const uint8_t *>(r.pp->down.ptr) + kSmallBytes);
      for (uint32_t v = 0; v < r.pl.nvol; v++) out->halo_offsets[r.v0 + v] = base + (r.pl.N ? ho[v] : 0);
      base += run_nhalos(r);
    }
    out->halo_offsets[nvol] = H;
  }
  // host outputs
  if (pl0.host_out) {
    uint64_t hb = 0;
    for (auto &r : runs) {
      const uint64_t n = r.pl.N, h = run_nhalos(r);
      if (n) {
        if (r.pl.want_ring && (rc = to_host(ctx, out->next + r.poff, r.B.st_next, n * 4, st))) return rc;
        if (r.pl.want_label && (rc = to_host(ctx, out->label + r.poff, r.B.st_label, n * 4, st))) return rc;
        if (r.pl.want_minid && (rc = to_host(ctx, out->minid + r.poff, r.B.st_minid, n * 8, st))) return rc;
        if (out->halos && h &&
            (rc = to_host(ctx, out->halos + hb, r.B.st_halo, h * sizeof(fof_halo_v1), st)))
          return rc;
        if (out->moments && h &&
            (rc = to_host(ctx, out->moments + hb, r.B.st_mom, h * sizeof(fof_moments_v1), st)))
          return rc;
      }
      hb += h;
    }
    FOF_HIP(hipStreamSynchronize(st));
  }
  if (stats) {
    unsigned long long hc[kCtrStride] = {};
    for (auto &r : runs) {
      if (r.pl.N == 0) continue;
      const uint32_t *hsm = static_cast<const uint32_t *>(r.pp->down.ptr);
      const unsigned long long *hcs = reinterpret_cast<const unsigned long long *>(hsm + kSmCtr);
      for (int q = 0; q < kCtrSlots; q++)
        for (int k = 0; k < kCtrStride; k++) hc[k] += hcs[q * kCtrStride + k];
      stats->ndense += (uint64_t)hsm[kSmNDense] + hsm[kSmNBig];
      stats->nmembers += hsm[kSmM];
      if (r.pl.sparse) stats->ncells += hsm[kSmU];
    }
    stats->pair_tests_kernel[0] = hc[kCtrTestsSparse];
    stats->pair_tests_kernel[1] = hc[kCtrTestsBig];
    stats->pair_tests_kernel[2] = hc[kCtrTestsSmall];
    stats->pair_tests = hc[kCtrTestsSparse] + hc[kCtrTestsBig] + hc[kCtrTestsSmall];
    stats->pairs_joined = hc[kCtrJoined];
    stats->rechecks = hc[kCtrRechecks];
    stats->ngroups = hc[kCtrGroups];
    stats->nhalos = H;
    stats->nhalos_owned = hc[kCtrOwned];
    stats->graph = graph_state;
    if (timing) {
      const Run &r = runs[0];
      Pipe &pp = *r.pp;
      float ms;
      if (!graph_state)
        for (int k = 0; k < FOF_NPHASE - 1; k++) {
          if (!(r.spans & (1u << k))) continue;
          FOF_HIP(hipEventElapsedTime(&ms, pp.ev[2 * k], pp.ev[2 * k + 1]));
          stats->phase_ms[k] = ms;
        }
      stats->phase_ms[FOF_NPHASE - 1] = tot_ms;
      stats->link_kernel_ms = stats->phase_ms[5] + stats->phase_ms[6] + stats->phase_ms[15];
    }
  }
  return 0;
}

}  // namespace fof

extern "C" int fof_engine_run(fof_ctx *ctx, const fof_particles_v1 *P, const fof_volume_v1 *vols,
                              uint32_t nvol, const fof_opts_v1 *opts, fof_outputs_v1 *out,
                              HostCheck *check) {
  EngineState &S = ctx->st;
  fof_opts_v1 o;
  memset(&o, 0, sizeof(o));
  o.version = FOF_ABI_VERSION;
  if (opts) o = *opts;
  uint32_t pipes = o.pipelines ? o.pipelines : 1u;
  if (!(o.flags & FOF_OPT_AUTOTUNE)) return run_call(ctx, P, vols, nvol, &o, out, pipes, nullptr, check);
  // Autotuned: the shape's cached choice, or a search on this call's own
  // input (every candidate links the same groups, so the last run's outputs
  // are the call's outputs).
  Plan pl;
  fof_outputs_v1 probe = *out;
  int rc = make_plan(P, vols, nvol, &o, &probe, pl);
  if (rc) return rc;
  const TuneKey key = tune_key(pl);
  TuneVal best;
  if (!tune_lookup(S, key, best)) {
    fof_stats_v1 *user_stats = out->stats;
    out->stats = nullptr;
    // the candidates run as the call itself will: eagerly, but with the link
    // kernels overlapped only where the call overlaps them
    const bool one_stream =
        (o.flags & FOF_OPT_TIMING) ||
        ((o.flags & FOF_OPT_GRAPH) && !pl.varlink && !pl.sparse && !pl.host_input && !pl.host_out);
    auto trial = [&](uint32_t T, uint32_t K, uint32_t gb, double &ms) -> int {
      fof_opts_v1 q = o;
      q.flags &= ~(FOF_OPT_TIMING | FOF_OPT_GRAPH);
      q.dense_threshold = T;
      q.big_grid = gb;
      double best_ms = 1e300;
      for (int rep = 0; rep < 2; rep++) {  // the first run also warms the workspace
        double w = 0;
        int e = run_call(ctx, P, vols, nvol, &q, out, K, &w, check, one_stream);
        if (e) return e;
        best_ms = std::min(best_ms, w);
      }
      ms = best_ms;
      return 0;
    };
    best = TuneVal{kDefaultT, 1, 0};
    double bms = 1e300, ms;
    for (uint32_t T : {16u, 24u, 32u}) {
      if ((rc = trial(T, 1, 0, ms))) break;
      if (ms < bms) bms = ms, best.T = T;
    }
    for (uint32_t gb : {2048u, 32768u}) {
      if (rc || (rc = trial(best.T, 1, gb, ms))) break;
      if (ms < bms * 0.99) bms = ms, best.gbig = gb;
    }
    for (uint32_t K : {2u, 3u, 4u}) {
      if (rc || K > nvol) break;
      if ((rc = trial(best.T, K, best.gbig, ms))) break;
      if (ms < bms * 0.99) bms = ms, best.pipes = K;
    }
    out->stats = user_stats;
    if (rc) return rc;
    tune_store(S, key, best);
  }
  o.dense_threshold = best.T;
  o.big_grid = best.gbig;
  return run_call(ctx, P, vols, nvol, &o, out, best.pipes, nullptr, check);
}

// ---------------------------------------------------------------------------
// Fixed workspace for callers that cannot allocate (fof_link_gpu_noalloc).
// Each device holds its own copy of the array from the time the library's
// code is loaded on it until the process ends; host code must use the
// address hipGetSymbolAddress returns for the device, never the array's name.
// ---------------------------------------------------------------------------
constexpr size_t kNoAllocBytes = (size_t)256 << 20;
static __device__ __align__(256) uint8_t scratch[kNoAllocBytes];

namespace {
std::mutex g_scratch_mu;
uint8_t *g_scratch[64];  // per device, from hipGetSymbolAddress
}  // namespace

extern "C" int fof_engine_init(fof_ctx *ctx) {
  EngineState &S = ctx->st;
  FOF_HIP(hipStreamCreate(&S.main.stream));
  // everything a later call on one pipeline may need besides workspace, so that
  // fof_link_gpu_noalloc makes and allocates nothing, on the device or
  // page-locked, from the first call on: the side stream, the head blocks of
  // one volume, the fork / join and timing events, and the fixed workspace's
  // address on this device
  const HeadLayout hl(1, 0);
  int rc;
  if ((rc = open_side(S.main)) || (rc = ensure_host(S.main.up, hl.bytes)) ||
      (rc = ensure_host(S.main.down, hl.vols)))
    return rc;
  FOF_HIP(hipEventCreateWithFlags(&S.fork, hipEventDisableTiming));
  for (auto &e : S.join) FOF_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  FOF_HIP(hipEventCreate(&S.t0));
  FOF_HIP(hipEventCreate(&S.t1));
  S.sync_events = true;
  if (ctx->device >= 0 && ctx->device < 64) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[ctx->device]) {
      void *ptr = nullptr;
      FOF_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
      g_scratch[ctx->device] = static_cast<uint8_t *>(ptr);
    }
  }
  return 0;
}

extern "C" int fof_engine_run_noalloc(fof_ctx *ctx, const fof_particles_v1 *P,
                                      const fof_volume_v1 *vol, const fof_opts_v1 *opts,
                                      fof_outputs_v1 *out) {
  if (ctx->device < 0 || ctx->device >= 64 || !g_scratch[ctx->device]) return FOF_E_NODEV;
  if (P->location != FOF_MEM_DEVICE || out->location != FOF_MEM_DEVICE) return FOF_E_ARG;
  if (vol->domain.varlink) return FOF_E_ARG;
  fof_opts_v1 o;
  memset(&o, 0, sizeof(o));
  o.version = FOF_ABI_VERSION;
  if (opts) o = *opts;
  // no graph (instantiation allocates), no events, one pipeline, no tuning
  o.flags &= ~(FOF_OPT_TIMING | FOF_OPT_GRAPH | FOF_OPT_AUTOTUNE);
  o.pipelines = 1;
  return run_call(ctx, P, vol, 1, &o, out, 1, nullptr, nullptr, false, g_scratch[ctx->device],
                  kNoAllocBytes);
}

extern "C" uint64_t fof_engine_noalloc_bytes(void) { return kNoAllocBytes; }

static void free_pipe(Pipe &pp) {
  release_host(pp.up);
  release_host(pp.down);
  release(pp.arena);
  if (pp.events)
    for (auto &e : pp.ev) (void)hipEventDestroy(e);
  pp.events = false;
  if (pp.side) (void)hipStreamDestroy(pp.side);
  if (pp.side_fork) (void)hipEventDestroy(pp.side_fork);
  if (pp.side_join) (void)hipEventDestroy(pp.side_join);
  pp.side = nullptr;
  pp.side_fork = pp.side_join = nullptr;
  if (pp.stream) (void)hipStreamDestroy(pp.stream);
  pp.stream = nullptr;
}

extern "C" void fof_engine_free(fof_ctx *ctx) {
  EngineState &S = ctx->st;
  release_host(S.pieces);
  for (auto &e : S.piece_ev)
    if (e) (void)hipEventDestroy(e);
  if (S.graph_exec) (void)hipGraphExecDestroy(S.graph_exec);
  S.graph_exec = nullptr;
  free_pipe(S.main);
  for (auto &p : S.pipes) {
    if (!p) continue;
    free_pipe(*p);
    delete p;
  }
  S.pipes.clear();
  if (S.sync_events) {
    (void)hipEventDestroy(S.fork);
    for (auto &e : S.join) (void)hipEventDestroy(e);
    (void)hipEventDestroy(S.t0);
    (void)hipEventDestroy(S.t1);
  }
  S.sync_events = false;
}
