// Droplet-droplet collision pairs (cell list) and coalescence events.
//
// No counterpart in the reference (its droplets only grow by collecting the
// continuum density, particles.py:828).  Specification, shared with the CPU
// brute-force checker bit for bit:
//   d = x_j - x_i per axis on wrapped positions, d -= L * rint(d / L),
//   d2 = (dx*dx + dy*dy) + dz*dz, pair iff d2 < (r_i + r_j)^2, i < j,
//   IEEE binary64 without fused multiply-add; pairs sorted by (i, j).
// Coalescence visits the sorted pairs once, merging (i, j) only if neither
// droplet merged earlier in the call: survivor i takes m = m_i + m_j, the
// mass-weighted velocity and x_i + (m_j/m) d; droplet j is left with zero
// mass and velocity.
#pragma once
#include "ld_particles.hpp"

namespace ld {

// Cell of a wrapped position on an nc^3 cell grid of side `cell`.
__device__ __forceinline__ int collCell(double x, double cell, int nc) {
  int c = (int)(x / cell);
  return c < 0 ? 0 : (c >= nc ? nc - 1 : c);
}

// The cells per side: nc, or fine (if set) when the droplets crowd in the nc^3
// cells (*same > many).  Read on the device, so that a call which has to choose
// neither waits nor differs under capture.
struct CellGrid {
  int nc, fine;
  unsigned long long *same, many;
  __device__ __forceinline__ bool crowd() const { return same && *same > many; }
  __device__ __forceinline__ int cells() const { return fine && crowd() ? fine : nc; }
};

// Count of the droplets per cell.  A droplet's rank is the number that its cell
// held before it, so the ranks add up to the pairs of droplets that share a cell
// (n / 2 of them for uniform droplets, one per cell).  *same += what they exceed
// two per droplet by, block by block: nothing, and no atomic, where droplets
// spread over the box (a pass of its own over 10^6 counts took 21 us).
// again: the second count, in the fine cells if those are taken.
static __global__ void __launch_bounds__(256)
k_coll_count(const double* __restrict__ rows, int np, double L, CellGrid G, bool again, int* __restrict__ key,
             int* __restrict__ rank, int* __restrict__ hist) {
  __shared__ unsigned long long sh[4];
  if (again && !G.crowd()) return;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long sum = 0;
  if (p < np) {
    const int nc = again ? G.fine : G.nc;
    const double cell = L / nc;
    const double* r = rows + (size_t)p * 7;
    const int cx = collCell(wrapL(r[0], L), cell, nc), cy = collCell(wrapL(r[1], L), cell, nc),
              cz = collCell(wrapL(r[2], L), cell, nc);
    const int k = (cx * nc + cy) * nc + cz;
    key[p] = k;
    const int before = atomicAdd(&hist[k], 1);
    rank[p] = before;
    sum = (unsigned long long)before;
  }
  if (again || !G.same) return;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    sum = sh[0] + sh[1] + sh[2] + sh[3];
    if (sum > 2 * 256) atomicAdd(G.same, sum - 2 * 256);
  }
}

// The fine cells' counts cleared, if those are taken; then the scans over the
// cells taken.  Their launches are of the size that the chip holds, whatever the
// cells.
static __global__ void __launch_bounds__(256) k_coll_clear(int* __restrict__ hist, CellGrid G) {
  if (!G.crowd()) return;
  const int n = G.fine * G.fine * G.fine;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) hist[i] = 0;
}
static __global__ void __launch_bounds__(1024)
k_coll_scan_local(int* __restrict__ hist, CellGrid G, int* __restrict__ bsum) {
  __shared__ int sh[32];
  const int nc = G.cells(), n = nc * nc * nc;
  for (int c = blockIdx.x; c * 4096 < n; c += gridDim.x) scanChunk(hist, n, bsum, c, sh);
}
static __global__ void __launch_bounds__(1024)
k_coll_scan_add(int* __restrict__ hist, CellGrid G, const int* __restrict__ bsum) {
  __shared__ int sh[16];
  const int nc = G.cells(), n = nc * nc * nc;
  for (int c = blockIdx.x; c * 4096 < n; c += gridDim.x) {
    if (c) scanAddChunk(hist, n, bsum, c, sh);
    __syncthreads();                     // sh, before the next chunk's sums
  }
}

// Droplets in cell order: wrapped position and radius, input row, and (for the
// statistics) velocity, so the pair search reads 32-byte records that its
// neighbours read too instead of 56-byte rows through an index.
static __global__ void __launch_bounds__(256)
k_coll_scatter(const double* __restrict__ rows, const double* __restrict__ rad, int np, double L,
               const int* __restrict__ key, const int* __restrict__ rank, const int* __restrict__ start,
               int* __restrict__ order, double4* __restrict__ pos, double4* __restrict__ vel) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const int s = start[key[p]] + rank[p];
  const double* r = rows + (size_t)p * 7;
  order[s] = p;
  double4 x;
  x.x = wrapL(r[0], L); x.y = wrapL(r[1], L); x.z = wrapL(r[2], L); x.w = rad ? rad[p] : 0.0;
  pos[s] = x;
  if (vel) {
    double4 v;
    v.x = r[3]; v.y = r[4]; v.z = r[5]; v.w = 0.0;
    vel[s] = v;
  }
}

// Minimum-image separation b - a of wrapped positions.  t / L of a wrapped
// difference lies in [-1, 1], so rint(t / L) is 1 above L/2, -1 below -L/2
// and 0 between: t > L/2 makes the quotient round above 1/2 (the distance
// from L/2 to the next double is more than half the quotient's spacing), and
// t <= L/2 makes it round to at most 1/2, which rint takes to 0.
__device__ __forceinline__ double minImage(double a, double b, double L) {
#pragma clang fp contract(off)
  const double t = b - a, h = 0.5 * L;
  return t > h ? t - L : (t < -h ? t + L : t);
}
__device__ __forceinline__ double separation(const double4& a, const double4& b, double L, double d[3]) {
#pragma clang fp contract(off)
  d[0] = minImage(a.x, b.x, L); d[1] = minImage(a.y, b.y, L); d[2] = minImage(a.z, b.z, L);
  return (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2];
}

// Pair search over the cell list, one thread per droplet in cell order.  Each
// unordered pair is met once: a droplet tests the slots after it in its own
// cell and every slot of the next z cell and of four of the eight neighbouring
// (x, y) columns (nc >= 3; one cell holding everything tests the slots after
// its own).  The cells along z are consecutive, so that is at most ten slot
// ranges, which a lane walks as one sequence: a wavefront's steps are its
// longest lane's candidates.  Pairs that pass the test go to a queue in LDS,
// and the wavefront works them off 64 at a time, so that the pair work (square
// root and divisions for the statistics) runs with full lanes.
//
// STATS = false: pairs with d2 < (r_i + r_j)^2, appended as (i << 32 | j), i < j
// the input rows, through one atomic per batch; the caller sorts them.
// STATS = true (no reference counterpart; the input of the radial
// distribution function and the kinematic collision kernel): for every pair
// with d2 < rmax^2: dist = sqrt(d2), bin k = min((int)(dist / dr), nbins - 1),
//   w_r = ((dv_x d_x + dv_y d_y) + dv_z d_z) / dist  (dv = v_j - v_i; 0 if dist == 0),
//   counts[k] += 1, wsum[k] += |w_r|, wneg[k] += max(-w_r, 0),
// in LDS histograms per block, then one global atomic per bin and block; counts
// are exact, the FP64 sums depend on the summation order.
//
// Bound by the candidates' 32-byte loads and FP64 tests.  10^6 droplets, rmax
// 0.1 (8.4 million pairs): 2590 us when each droplet read all 27 cells' rows
// through the index with a wrap and divisions per candidate and the pair work
// ran in the lanes that found a pair; 286 us now.  Collision pairs of the same
// droplets 522 -> 95 us.
struct NearArgs {
  const double4 *pos, *vel;
  const int *order, *start;
  int np;
  CellGrid grid;                       // crowded without fine cells: nothing is done (the caller searches finer ones)
  double L;
  unsigned long long *out, max_pairs, *count;                   // pairs
  double rmax, dr;                                               // statistics
  int nbins;
  unsigned long long* counts;
  double *wsum, *wneg;
};
template <bool STATS> struct NearHist { unsigned long long c[512]; double w[512], n[512]; };
template <> struct NearHist<false> {};
template <bool STATS>
__global__ void __launch_bounds__(256) k_near(NearArgs A) {
#pragma clang fp contract(off)
  __shared__ NearHist<STATS> H;
  __shared__ int2 queue[4][128];
  const bool crowd = A.grid.crowd();
  if (crowd && !A.grid.fine) return;
  const int nc = crowd ? A.grid.fine : A.grid.nc, np = A.np;
  const double cell = A.L / nc;
  if constexpr (STATS) {
    for (int k = threadIdx.x; k < A.nbins; k += 256) { H.c[k] = 0ull; H.w[k] = 0.0; H.n[k] = 0.0; }
    __syncthreads();
  }
  const int lane = threadIdx.x & 63;
  int2* q = queue[threadIdx.x >> 6];
  const int per = gridDim.x / 8, lb = (blockIdx.x % 8) * per + blockIdx.x / 8;   // XCD-aware: contiguous slots
  const uint32_t slot = (uint32_t)lb * 256u + threadIdx.x;
  bool run = slot < (uint32_t)np;
  const int s = run ? (int)slot : 0;
  double4 me = {0.0, 0.0, 0.0, 0.0};
  int cx = 0, cy = 0, cz = 0, t = 0, e = 0;
  if (run) {
    me = A.pos[s];
    cx = collCell(me.x, cell, nc); cy = collCell(me.y, cell, nc); cz = collCell(me.z, cell, nc);
    const int own = (cx * nc + cy) * nc + cz, last = (nc >= 3 && cz + 1 < nc) ? own + 1 : own;
    t = s + 1;
    e = last + 1 < nc * nc * nc ? A.start[last + 1] : np;
  }
  int r = 0;                         // range number: 0 done above, 1 own column's wrapped cell, 2.. columns
  const double r2max = A.rmax * A.rmax;
  int qn = 0;
  auto work = [&](int n) {           // the queue's first n (<= 64) pairs, one per lane
    int2 ij = {0, 0};
    if (lane < n) ij = q[lane];
    if constexpr (STATS) {
      if (lane < n) {
        double d[3];
        const double4 a = A.pos[ij.x], b = A.pos[ij.y], va = A.vel[ij.x], vb = A.vel[ij.y];
        const double dist = sqrt(separation(a, b, A.L, d));
        int k = (int)(dist / A.dr);
        k = k < A.nbins ? k : A.nbins - 1;
        double wr = 0.0;
        if (dist > 0.0) {
          const double dv0 = vb.x - va.x, dv1 = vb.y - va.y, dv2 = vb.z - va.z;
          wr = ((dv0 * d[0] + dv1 * d[1]) + dv2 * d[2]) / dist;
        }
        atomicAdd(&H.c[k], 1ull);
        atomicAdd(&H.w[k], fabs(wr));
        if (wr < 0.0) atomicAdd(&H.n[k], -wr);
      }
    } else {
      unsigned long long base = 0;
      if (lane == 0) base = atomicAdd(A.count, (unsigned long long)n);
      base = __shfl(base, 0, 64);
      if (lane < n && base + lane < A.max_pairs) {
        const int i = A.order[ij.x], j = A.order[ij.y];
        A.out[base + lane] = ((unsigned long long)(i < j ? i : j) << 32) | (unsigned long long)(unsigned)(i < j ? j : i);
      }
    }
  };
  while (__any(run)) {
    // the next non-empty range of a lane that has used up its own
    while (run && t >= e) {
      if (++r > 9 || nc < 3) { run = false; break; }
      // r = 1: cell 0 of the own column when the next z cell wraps; then per
      // column (0,1), (1,-1), (1,0), (1,1) the z-run cz-1..cz+1 as two pieces
      const int col = r >> 1, piece = r & 1;
      const int ox = col < 2 ? 0 : 1, oy = col == 0 ? 0 : col == 1 ? 1 : col - 3;
      int z0, z1;                    // cells [z0, z1) of the column
      if (col == 0) {
        if (cz + 1 < nc) continue;
        z0 = 0; z1 = 1;
      } else if (piece == 0) {
        z0 = cz > 0 ? cz - 1 : 0; z1 = cz + 2 < nc ? cz + 2 : nc;
      } else {
        if (cz > 0 && cz + 1 < nc) continue;
        z0 = cz == 0 ? nc - 1 : 0; z1 = z0 + 1;
      }
      const int x = cx + ox < nc ? cx + ox : 0, y = cy + oy < 0 ? nc - 1 : (cy + oy < nc ? cy + oy : 0);
      const int c0 = (x * nc + y) * nc;
      t = A.start[c0 + z0];
      e = c0 + z1 < nc * nc * nc ? A.start[c0 + z1] : np;
    }
    bool near = false;
    if (run) {
      double d[3];
      const double4 b = A.pos[t];
      const double d2 = separation(me, b, A.L, d);
      if constexpr (STATS) near = d2 < r2max;
      else { const double sr = me.w + b.w; near = d2 < sr * sr; }
    }
    const unsigned long long m = __ballot(near);
    if (m) {
      if (near) {
        const int at = qn + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
        q[at] = make_int2(s, t);
      }
      qn += __popcll(m);
      __builtin_amdgcn_wave_barrier();
      if (qn >= 64) {
        work(64);
        __builtin_amdgcn_wave_barrier();
        qn -= 64;
        int2 rest = {0, 0};
        if (lane < qn) rest = q[64 + lane];
        __builtin_amdgcn_wave_barrier();
        if (lane < qn) q[lane] = rest;
        __builtin_amdgcn_wave_barrier();
      }
    }
    ++t;
  }
  if (qn) work(qn);
  if constexpr (STATS) {
    __syncthreads();
    for (int k = threadIdx.x; k < A.nbins; k += 256)
      if (H.c[k]) {
        atomicAdd(&A.counts[k], H.c[k]);
        unsafeAtomicAdd(&A.wsum[k], H.w[k]);
        unsafeAtomicAdd(&A.wneg[k], H.n[k]);
      }
  }
}

// Bitonic sort of n = 2^m keys (the first cnt are given, the rest count as
// largest).  k_bitonic_block does every step whose partner lies in the same
// 2048-key chunk in LDS: with k = 0 it sorts each chunk from unsorted keys,
// else it finishes the merges of length k.  k_bitonic does one step across
// chunks.  116 pairs of 10^6 droplets: 28 launches of one step each before,
// one now, which also writes the pairs (`pairs` set: n <= 2048).
// Key numbers and merge lengths are 64-bit: 2^29 + 1 pairs (33000 droplets that
// all overlap) already sort 2^30 keys, whose last doubling of an int overflows.
constexpr int SORT_CHUNK = 2048;
static __global__ void __launch_bounds__(1024)
k_bitonic_block(unsigned long long* __restrict__ a, int64_t cnt, int64_t n, int64_t k, int64_t* __restrict__ pairs) {
  __shared__ unsigned long long sh[SORT_CHUNK];
  const int64_t base = (int64_t)blockIdx.x * SORT_CHUNK;
  const int len = n < SORT_CHUNK ? (int)n : SORT_CHUNK;
  for (int i = threadIdx.x; i < len; i += 1024) sh[i] = base + i < cnt ? a[base + i] : ~0ull;
  __syncthreads();
  // the steps of merges of length kk from partner distance j down
  auto merge = [&](int64_t kk, int j) {
    for (; j > 0; j >>= 1) {
      for (int p = threadIdx.x; p < len / 2; p += 1024) {
        const int i = 2 * p - (p & (j - 1));        // the pair's lower key: bit j clear
        const bool up = ((base + i) & kk) == 0;
        const unsigned long long x = sh[i], y = sh[i + j];
        if ((x > y) == up) { sh[i] = y; sh[i + j] = x; }
      }
      __syncthreads();
    }
  };
  if (k) merge(k, len / 2);
  else
    for (int kk = 2; kk <= len; kk <<= 1) merge(kk, kk / 2);
  if (pairs) {
    for (int i = threadIdx.x; i < cnt; i += 1024) {
      pairs[2 * i] = (int64_t)(sh[i] >> 32);
      pairs[2 * i + 1] = (int64_t)(sh[i] & 0xffffffffull);
    }
  } else {
    for (int i = threadIdx.x; i < len; i += 1024) a[base + i] = sh[i];
  }
}
static __global__ void __launch_bounds__(256)
k_bitonic(unsigned long long* __restrict__ a, int64_t n, int64_t j, int64_t k) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t ixj = i ^ j;
  if (ixj > i) {
    const bool up = (i & k) == 0;
    const unsigned long long x = a[i], y = a[ixj];
    if ((x > y) == up) { a[i] = y; a[ixj] = x; }
  }
}

static __global__ void __launch_bounds__(256)
k_pairs_out(const unsigned long long* __restrict__ keys, int64_t n, int64_t* __restrict__ pairs) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= n) return;
  pairs[2 * t] = (int64_t)(keys[t] >> 32);
  pairs[2 * t + 1] = (int64_t)(keys[t] & 0xffffffffull);
}

// Sequential greedy coalescence over the sorted pairs (one thread; the pair
// list is short).  used[] must be zero on entry.
static __global__ void k_coalesce(double* rows, const int64_t* __restrict__ pairs, int npairs, double L,
                                  int* __restrict__ used, int64_t* __restrict__ events, int* __restrict__ nevents) {
#pragma clang fp contract(off)
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  int ne = 0;
  for (int t = 0; t < npairs; ++t) {
    const int64_t i = pairs[2 * t], j = pairs[2 * t + 1];
    if (used[i] || used[j]) continue;
    double* a = rows + (size_t)i * 7;
    double* b = rows + (size_t)j * 7;
    const double mi = a[6], mj = b[6];
    const double m = mi + mj;
    const double w = mj / m;
    for (int c = 0; c < 3; ++c) {
      const double xi = wrapL(a[c], L), xj = wrapL(b[c], L);
      double d = xj - xi;
      d = d - L * rint(d / L);
      a[c] = wrapL(xi + w * d, L);
      a[3 + c] = (mi * a[3 + c] + mj * b[3 + c]) / m;
      b[3 + c] = 0.0;
    }
    a[6] = m;
    b[6] = 0.0;
    used[i] = 1;
    used[j] = 1;
    events[2 * ne] = i;
    events[2 * ne + 1] = j;
    ++ne;
  }
  *nevents = ne;
}

}  // namespace ld
