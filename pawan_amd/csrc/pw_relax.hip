// pw_relax.hip -- particle management of one wake on the device: split and
// merge (__wake::split / merge / relax, src/wake/wake.cpp:61-165), behind
// pw_wake_split and pw_wake_merge (include/pawan_gpu.h).
//
// Split.  Whether a particle splits depends on that particle alone, so every
// particle of the age prefix is tested at once; an exclusive scan of the
// decisions gives each new particle its row (new particles in the order of
// their parents, after the last particle, as the reference appends them).
//
// Merge.  The reference walks particle i over all later j, moving x_i and
// growing a_i as it merges, so later tests see the moved x_i: the result
// depends on the order.  It is reproduced exactly in two steps.
//  1. A cell list (cells of the largest merge distance, (sigma_i +
//     sigma_j)/8 <= sigma_max/4, keyed by cell and sorted) lets every i of the
//     age prefix test its later neighbours in parallel with the original
//     state.  The first merge of i needs such a neighbour (x_i is unmoved
//     until then, and strengths only ever drop to zero), so an i with none
//     does nothing and is left out.
//  2. The flagged i are visited in order and the reference's inner loop is
//     replayed: the next j > (last j seen) within the merge distance of the
//     current x_i, found among the 27 cells around x_i, with the current
//     strengths.  Later particles have not moved (only the outer particle of
//     an iteration moves), so the cell list of the original positions still
//     finds them.  Flagged particles far enough apart cannot touch the same
//     particles, so they are first gathered into groups (k_group_link) and
//     every group is replayed by a block of its own.
// The arithmetic is the reference's (GSL's dnrm2 and ddot, dscal by the
// reciprocal, no contraction), so the result is bit-for-bit the
// sequential one.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <string>
#include <utility>
#include <vector>

#include "pw_ctx.h"

namespace {

using pwi::fail;

constexpr int kB = 256;
constexpr int kExtentBlocks = 64;
constexpr int kCellBits = 21;  // cell coordinate bits per axis of a key
constexpr int64_t kCellMax = (int64_t(1) << kCellBits) - 1;
constexpr uint64_t kNoCell = ~uint64_t(0);

#pragma clang fp contract(off)

// gsl_blas_dnrm2 of a 3-vector: the netlib scaled sum of squares
__device__ double dnrm2_3(double x0, double x1, double x2) {
  double scale = 0.0, ssq = 1.0;
  const double x[3] = {x0, x1, x2};
  for (int i = 0; i < 3; ++i) {
    if (x[i] != 0.0) {
      const double ax = fabs(x[i]);
      if (scale < ax) {
        ssq = 1.0 + ssq * (scale / ax) * (scale / ax);
        scale = ax;
      } else {
        ssq += (ax / scale) * (ax / scale);
      }
    }
  }
  return scale * sqrt(ssq);
}

// the age test of both loops (wake.cpp:64, 115): stepnum - active > 45
__global__ void k_age_prefix(const double* __restrict__ active, int n, double stepnum, int* __restrict__ prefix) {
  const int i = blockIdx.x * kB + static_cast<int>(threadIdx.x);
  if (i < n && !(stepnum - active[i] > 45)) atomicMin(prefix, i);
}

// ---- split ----------------------------------------------------------------

__global__ void k_split_flags(int n, const int* __restrict__ prefix, const double* __restrict__ alpha,
                              const double* __restrict__ birth, int* __restrict__ flag) {
  const int i = blockIdx.x * kB + static_cast<int>(threadIdx.x);
  if (i >= n) return;
  int f = 0;
  if (i < *prefix) {
    const double ib = birth[i];
    const double m = dnrm2_3(alpha[3 * i], alpha[3 * i + 1], alpha[3 * i + 2]);
    f = (m >= 2 * ib && ib > 0.0001) ? 1 : 0;
  }
  flag[i] = f;
}

// parent i (flagged) and its new particle at row first + off[i]
__global__ void k_split_apply(int n, int64_t first, const int* __restrict__ flag, const int* __restrict__ off,
                              double* __restrict__ pos, double* __restrict__ alpha, double* __restrict__ radius,
                              double* __restrict__ volume, double* __restrict__ birth, double* __restrict__ active) {
  const int i = blockIdx.x * kB + static_cast<int>(threadIdx.x);
  if (i >= n || !flag[i]) return;
  const int64_t k = first + off[i];
  double* ip = pos + 3 * static_cast<int64_t>(i);
  double* iv = alpha + 3 * static_cast<int64_t>(i);
  const double im = dnrm2_3(iv[0], iv[1], iv[2]);
  const double ir = radius[i];
  const double sc = 0.25 * ir / im;  // gsl_blas_dscal(0.25*iradius/ivormag, deltapos)
  double dp[3], x[3], a[3];
  for (int c = 0; c < 3; ++c) {
    dp[c] = iv[c] * sc;
    x[c] = ip[c];
    a[c] = iv[c];
  }
  for (int c = 0; c < 3; ++c) {
    pos[3 * k + c] = x[c] + dp[c];
    alpha[3 * k + c] = a[c] * 0.5;
    ip[c] = x[c] - dp[c];
    iv[c] = a[c] * 0.5;
  }
  radius[k] = ir;
  volume[k] = volume[i];
  birth[k] = 0.5 * im;
  active[k] = active[i];
  birth[i] = 0.5 * im;
}

// ---- merge ----------------------------------------------------------------

// bounding box and largest radius, a row of seven per block (the host takes
// the rest; one block of 1,024 threads read 98,304 particles in 67 us, 64 blocks
// in 9)
__global__ __launch_bounds__(kB) void k_extent(const double* __restrict__ pos, const double* __restrict__ radius,
                                               int n, double* __restrict__ out) {
  __shared__ double red[7][kB];
  double v[7] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, 0.0};
  for (int64_t i = blockIdx.x * kB + threadIdx.x; i < n; i += kExtentBlocks * kB) {
    for (int c = 0; c < 3; ++c) {
      const double x = pos[3 * i + c];
      if (isfinite(x)) {
        v[c] = fmin(v[c], x);
        v[3 + c] = fmax(v[3 + c], x);
      }
    }
    const double r = radius[i];
    if (isfinite(r)) v[6] = fmax(v[6], r);
  }
  for (int k = 0; k < 7; ++k) red[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int s = kB / 2; s > 0; s >>= 1) {
    if (static_cast<int>(threadIdx.x) < s)
      for (int k = 0; k < 7; ++k)
        red[k][threadIdx.x] = k < 3 ? fmin(red[k][threadIdx.x], red[k][threadIdx.x + s])
                                    : fmax(red[k][threadIdx.x], red[k][threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x < 7) out[7 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

struct Grid {
  double x0, y0, z0, h;  // origin and cell size
};

__device__ __forceinline__ uint64_t cell_key(int64_t ix, int64_t iy, int64_t iz) {
  return (static_cast<uint64_t>(iz) << (2 * kCellBits)) | (static_cast<uint64_t>(iy) << kCellBits) |
         static_cast<uint64_t>(ix);
}

__device__ __forceinline__ bool cell_of(const Grid& g, double x, double y, double z, int64_t* c) {
  if (!(isfinite(x) && isfinite(y) && isfinite(z))) return false;
  c[0] = static_cast<int64_t>(floor((x - g.x0) / g.h));
  c[1] = static_cast<int64_t>(floor((y - g.y0) / g.h));
  c[2] = static_cast<int64_t>(floor((z - g.z0) / g.h));
  for (int k = 0; k < 3; ++k) c[k] = min(max(c[k], int64_t(0)), kCellMax);
  return true;
}

__global__ void k_cell_keys(const double* __restrict__ pos, int n, Grid g, uint64_t* __restrict__ key,
                            int* __restrict__ idx) {
  const int i = blockIdx.x * kB + static_cast<int>(threadIdx.x);
  if (i >= n) return;
  int64_t c[3];
  const double* x = pos + 3 * static_cast<int64_t>(i);
  key[i] = cell_of(g, x[0], x[1], x[2], c) ? cell_key(c[0], c[1], c[2]) : kNoCell;
  idx[i] = i;
}

// [lo, hi) of the sorted keys equal to k
__device__ __forceinline__ void equal_range(const uint64_t* __restrict__ keys, int n, uint64_t k, int* lo, int* hi) {
  int a = 0, b = n;
  while (a < b) {
    const int m = (a + b) >> 1;
    if (keys[m] < k) a = m + 1;
    else b = m;
  }
  int c = a, d = n;
  while (c < d) {
    const int m = (c + d) >> 1;
    if (keys[m] <= k) c = m + 1;
    else d = m;
  }
  *lo = a;
  *hi = c;
}

// first of the sorted keys not below k (upper: above k)
__device__ __forceinline__ int bound_of(const uint64_t* __restrict__ keys, int n, uint64_t k, bool upper) {
  int a = 0, b = n;
  while (a < b) {
    const int m = (a + b) >> 1;
    if (upper ? keys[m] <= k : keys[m] < k) a = m + 1;
    else b = m;
  }
  return a;
}

// the cells of row r = 0 .. 8 about cell c (y, z offsets r % 3 - 1, r / 3 - 1):
// x is the lowest part of a key, so its three cells are one range of the
// sorted keys, from the first not below `first` to the first above `last`;
// false if the row is outside the grid
__device__ __forceinline__ bool cell_row(const int64_t* c, int r, uint64_t* first, uint64_t* last) {
  const int64_t y = c[1] + r % 3 - 1, z = c[2] + r / 3 - 1;
  if (y < 0 || z < 0 || y > kCellMax || z > kCellMax) return false;
  *first = cell_key(max(c[0] - 1, int64_t(0)), y, z);
  *last = cell_key(min(c[0] + 1, kCellMax), y, z);
  return true;
}

// can pair (i, j) merge (wake.cpp:129-135), for positions xi, xj and
// strengths ai, aj with norms mi, mj
__device__ __forceinline__ bool in_reach(const double* xi, const double* xj, double ri, double rj) {
  const double rho = dnrm2_3(xi[0] - xj[0], xi[1] - xj[1], xi[2] - xj[2]);
  return rho < 0.125 * (ri + rj);
}
__device__ __forceinline__ double misalignment(const double* ai, const double* aj, double mi, double mj) {
  double al = 0.0;  // gsl_blas_ddot
  al += ai[0] * aj[0];
  al += ai[1] * aj[1];
  al += ai[2] * aj[2];
  return 1 - al / mi / mj;
}

// step 1: particles of the age prefix that have a later neighbour they
// would merge with in the original state.  One thread per particle and row of
// cells (a search is a chain of 17 reads; nine rows of two searches one after
// another took 81 us for 98,304 particles, this 39); flag is zero before.
__global__ void k_merge_flags(int n, const int* __restrict__ prefix, Grid g, const uint64_t* __restrict__ keys,
                              const int* __restrict__ sidx, const double* __restrict__ pos,
                              const double* __restrict__ alpha, const double* __restrict__ radius,
                              int* __restrict__ flag) {
  const int64_t t = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x;
  const int i = static_cast<int>(t / 9), r = static_cast<int>(t % 9);
  if (i >= n || i >= *prefix) return;
  const double* xi = pos + 3 * static_cast<int64_t>(i);
  const double* ai = alpha + 3 * static_cast<int64_t>(i);
  int64_t c[3];
  uint64_t first, last;
  if (!cell_of(g, xi[0], xi[1], xi[2], c) || !cell_row(c, r, &first, &last)) return;
  const double mi = dnrm2_3(ai[0], ai[1], ai[2]);
  if (mi == 0.0) return;
  const double ri = radius[i];
  for (int e = bound_of(keys, n, first, false); e < n && keys[e] <= last; ++e) {
    const int j = sidx[e];
    if (j <= i) continue;
    const double* aj = alpha + 3 * static_cast<int64_t>(j);
    const double mj = dnrm2_3(aj[0], aj[1], aj[2]);
    if (mj == 0.0 || !in_reach(xi, pos + 3 * static_cast<int64_t>(j), ri, radius[j])) continue;
    if (misalignment(ai, aj, mi, mj) >= 0.0001) {
      flag[i] = 1;  // (any row's thread may store it)
      return;
    }
  }
}

// ---- groups of flagged particles ------------------------------------------
// While x_i stays within kTravel cells' width h of where it started, iteration
// i touches (merges, or tests as in reach) only particles within (kTravel + 1)
// h of that point: a merge distance is at most h.  Another group's flagged
// particle p stays as near to its own start, so at any time (its coordinates
// read one by one, each old or new: at most sqrt(3) kTravel h from the start)
// it is out of reach of x_i if the starts are more than
//   (1 + kTravel + sqrt(3) kTravel) h = 5.1 h
// apart, and so are the particles it absorbs ((2 kTravel + 2) h = 5 h).
// Particles within kLink h are put into one group; an x_i that leaves its range
// stops the replay, which then starts over with everything in one group.
constexpr double kTravel = 1.5, kLink = 6.25;
constexpr int kExactLinks = 32;  // cells with more flagged particles are linked whole

__device__ __forceinline__ int group_root(int* parent, int x) {
  for (;;) {
    const int p = __hip_atomic_load(parent + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (p == x) return x;
    x = p;  // parents only decrease: the walk ends
  }
}

__device__ __forceinline__ void group_unite(int* parent, int a, int b) {
  for (;;) {
    a = group_root(parent, a);
    b = group_root(parent, b);
    if (a == b) return;
    if (a < b) {
      const int t = a;
      a = b;
      b = t;
    }
    // the larger root under the smaller; if a got a parent meanwhile, again
    // from there (a strictly smaller index)
    const int old = atomicCAS(parent + a, a, b);
    if (old == a) return;
    a = old;
  }
}

// coarse cells (width kLink h) of the flagged particles
__global__ void k_group_keys(const double* __restrict__ pos, const int* __restrict__ list, int count, Grid g,
                             uint64_t* __restrict__ key, int* __restrict__ idx, int* __restrict__ parent) {
  const int k = blockIdx.x * kB + static_cast<int>(threadIdx.x);
  if (k >= count) return;
  int64_t c[3];
  const double* x = pos + 3 * static_cast<int64_t>(list[k]);
  g.h *= kLink;
  key[k] = cell_of(g, x[0], x[1], x[2], c) ? cell_key(c[0], c[1], c[2]) : kNoCell;
  idx[k] = k;
  parent[k] = k;
}

// flagged particle e (in the order of the coarse cells) with those within
// kLink h in its own cell and in the 13 neighbour cells after it; one thread per
// particle and cell (one per particle: 67 us for 930 of them, this 11)
__global__ void k_group_link(const double* __restrict__ pos, const int* __restrict__ list,
                             const uint64_t* __restrict__ keys, const int* __restrict__ sidx, int count, Grid g,
                             int* parent) {
  const int64_t t = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x;
  const int e = static_cast<int>(t / 14);
  const int q = 13 + static_cast<int>(t % 14);  // the cell itself, then the 13 after it in z, y, x order
  if (e >= count || keys[e] == kNoCell) return;
  const double* x = pos + 3 * static_cast<int64_t>(list[sidx[e]]);
  const double reach = kLink * g.h;
  const uint64_t key = keys[e], mask = static_cast<uint64_t>(kCellMax);
  const int64_t nx = static_cast<int64_t>(key & mask) + q % 3 - 1,
                ny = static_cast<int64_t>((key >> kCellBits) & mask) + (q / 3) % 3 - 1,
                nz = static_cast<int64_t>(key >> (2 * kCellBits)) + q / 9 - 1;
  if (nx < 0 || ny < 0 || nz < 0 || nx > kCellMax || ny > kCellMax || nz > kCellMax) return;
  int lo, hi;
  equal_range(keys, count, cell_key(nx, ny, nz), &lo, &hi);
  if (lo == hi) return;
  if (hi - lo > kExactLinks) {
    // a crowded cell is one group: each of its particles joins the first
    group_unite(parent, sidx[e], sidx[lo]);
    return;
  }
  for (int f = lo; f < hi; ++f) {
    if (q == 13 && f >= e) break;
    const double* y = pos + 3 * static_cast<int64_t>(list[sidx[f]]);
    const double dx = x[0] - y[0], dy = x[1] - y[1], dz = x[2] - y[2];
    if (dx * dx + dy * dy + dz * dz <= reach * reach) group_unite(parent, sidx[e], sidx[f]);
  }
}

__global__ void k_group_roots(int count, int* parent, int* __restrict__ root) {
  const int k = blockIdx.x * kB + static_cast<int>(threadIdx.x);
  if (k < count) root[k] = group_root(parent, k);
}

// ---- replay ----------------------------------------------------------------
constexpr int kRT = 64;     // threads of a replaying block: one wave, no other to wait for
constexpr int kCap = 1024;  // later neighbours of one outer particle kept in LDS

__device__ __forceinline__ int wave_min_int(int v) {
  for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
  return v;
}

// step 2: a block replays the reference's loops over one group: the particles
// list[k] of one root (consecutive, ascending particles), the block of the
// first of them doing the work.  For the current outer particle the later
// particles of the 27 cells around it (index, position, radius) are gathered
// into LDS, again when x_i moves to another cell; each step then takes the
// smallest j past the last one seen that is within reach of the current x_i.
// More than kCap of them: the step scans the cells in memory instead.
//
// A replay is a chain of dependent memory reads, so it is bound by latency:
// one block over all flagged particles took 9.2 ms for a 98,304-particle wake
// with one particle in 200 turned; by groups the same replay takes 0.09 ms,
// the linking 0.01.
__global__ __launch_bounds__(kRT) void k_merge_resolve(int n, const int* __restrict__ list,
                                                       const int* __restrict__ root, int count, Grid g,
                                                       const uint64_t* __restrict__ keys,
                                                       const int* __restrict__ sidx, double* pos, double* alpha,
                                                       const double* __restrict__ radius, double* volume,
                                                       unsigned long long* merges, int* left) {
  const int k0 = static_cast<int>(blockIdx.x);
  if (k0 > 0 && (!root || root[k0] == root[k0 - 1])) return;
  const int group = root ? root[k0] : 0;
  __shared__ int s_lo[9], s_hi[9];
  __shared__ int s_cnt;
  __shared__ int s_j[kCap];
  __shared__ double s_x[3 * kCap];
  __shared__ double s_r[kCap];
  const int tid = static_cast<int>(threadIdx.x);
  unsigned long long done = 0;
  for (int k = k0; k < count && (!root || root[k] == group); ++k) {
    const int i = list[k];
    double xi[3], x0[3], ai[3];
    for (int c = 0; c < 3; ++c) {
      xi[c] = x0[c] = pos[3 * static_cast<int64_t>(i) + c];
      ai[c] = alpha[3 * static_cast<int64_t>(i) + c];
    }
    const double mi = dnrm2_3(ai[0], ai[1], ai[2]);  // once per i, as the reference takes it
    if (mi == 0.0) continue;
    const double ri = radius[i];
    int jlast = i;
    int64_t cur[3] = {-1, -1, -1};
    bool have = false;
    for (;;) {
      int64_t c[3];
      const bool in_grid = cell_of(g, xi[0], xi[1], xi[2], c);
      if (!in_grid) break;  // a non-finite position reaches nothing
      if (!have || c[0] != cur[0] || c[1] != cur[1] || c[2] != cur[2]) {
        // the ranges of the 27 cells, then the later particles in them
        __syncthreads();
        int edge = 0;  // lanes 0-8: first entries of the nine rows, 9-17: their ends
        if (tid < 18) {
          uint64_t first, last;
          if (cell_row(c, tid % 9, &first, &last)) edge = bound_of(keys, n, tid < 9 ? first : last, tid >= 9);
        }
        const int end = __shfl(edge, tid + 9, 64);
        if (tid < 9) {
          s_lo[tid] = edge;
          s_hi[tid] = end;
        }
        if (tid == 0) s_cnt = 0;
        __syncthreads();
        int total = 0;
        for (int q = 0; q < 9; ++q) total += s_hi[q] - s_lo[q];
        for (int f = tid; f < total; f += kRT) {
          int e = f, q = 0;  // entry f of the nine rows together
          while (e >= s_hi[q] - s_lo[q]) e -= s_hi[q] - s_lo[q], ++q;
          const int j = sidx[s_lo[q] + e];
          if (j <= jlast) continue;
          const int slot = atomicAdd(&s_cnt, 1);
          if (slot < kCap) {
            s_j[slot] = j;
            for (int c2 = 0; c2 < 3; ++c2) s_x[3 * slot + c2] = pos[3 * static_cast<int64_t>(j) + c2];
            s_r[slot] = radius[j];
          }
        }
        __syncthreads();
        for (int c2 = 0; c2 < 3; ++c2) cur[c2] = c[c2];
        have = true;
      }
      // the smallest j > jlast within reach of the current x_i, with a
      // non-zero strength
      int best = INT_MAX;
      const int cnt = s_cnt;
      if (cnt <= kCap) {
        for (int e = tid; e < cnt; e += kRT) {
          const int j = s_j[e];
          if (j <= jlast || j >= best) continue;
          if (!in_reach(xi, &s_x[3 * e], ri, s_r[e])) continue;
          const double* aj = alpha + 3 * static_cast<int64_t>(j);
          if (dnrm2_3(aj[0], aj[1], aj[2]) != 0.0) best = j;
        }
      } else {
        for (int q = 0; q < 9; ++q)
          for (int e = s_lo[q] + tid; e < s_hi[q]; e += kRT) {
            const int j = sidx[e];
            if (j <= jlast || j >= best) continue;
            if (!in_reach(xi, pos + 3 * static_cast<int64_t>(j), ri, radius[j])) continue;
            const double* aj = alpha + 3 * static_cast<int64_t>(j);
            if (dnrm2_3(aj[0], aj[1], aj[2]) != 0.0) best = j;
          }
      }
      const int j = wave_min_int(best);
      if (j == INT_MAX) break;
      double xj[3], aj[3];
      for (int c2 = 0; c2 < 3; ++c2) {
        xj[c2] = pos[3 * static_cast<int64_t>(j) + c2];
        aj[c2] = alpha[3 * static_cast<int64_t>(j) + c2];
      }
      const double mj = dnrm2_3(aj[0], aj[1], aj[2]);
      if (misalignment(ai, aj, mi, mj) >= 0.0001) {
        const double sc = 1 / (mi + mj);
        for (int c2 = 0; c2 < 3; ++c2) {
          xi[c2] = (xi[c2] * mi + xj[c2] * mj) * sc;
          ai[c2] = ai[c2] + aj[c2];
        }
        __syncthreads();  // every thread has read a_j
        if (tid == 0) {
          for (int c2 = 0; c2 < 3; ++c2) alpha[3 * static_cast<int64_t>(j) + c2] = 0.0;
          volume[j] = 0.0;
        }
        __threadfence_block();
        __syncthreads();
        ++done;
        if (root) {
          // out of the range that keeps the groups apart (or not a number):
          // the caller starts over with one group
          const double dx = xi[0] - x0[0], dy = xi[1] - x0[1], dz = xi[2] - x0[2];
          const double t = kTravel * g.h;
          if (!(dx * dx + dy * dy + dz * dz <= t * t)) {
            if (tid == 0) *left = 1;
            return;  // the same for every thread
          }
        }
      }
      jlast = j;
    }
    __syncthreads();
    if (tid == 0)
      for (int c2 = 0; c2 < 3; ++c2) {
        pos[3 * static_cast<int64_t>(i) + c2] = xi[c2];
        alpha[3 * static_cast<int64_t>(i) + c2] = ai[c2];
      }
    __threadfence_block();
    __syncthreads();
  }
  if (tid == 0 && done) atomicAdd(merges, done);
}

#pragma clang fp contract(on)

// device buffers of one call, parts of one allocation, freed on every path
struct Buffers {
  std::vector<void*> p;
  hipStream_t st = nullptr;
  std::vector<std::pair<void**, size_t>> parts;
  // `count` elements at *out once allocate() has run
  template <typename T>
  void add(T** out, size_t count) {
    *out = nullptr;
    parts.emplace_back(reinterpret_cast<void**>(out), std::max<size_t>(count, 1) * sizeof(T));
  }
  bool allocate() {
    size_t total = 0;
    for (const auto& q : parts) total += (q.second + 255) / 256 * 256;
    char* base = nullptr;
    if (pwi::dalloc(&base, total) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    p.push_back(base);
    for (const auto& q : parts) {
      *q.first = base;
      base += (q.second + 255) / 256 * 256;
    }
    parts.clear();
    return true;
  }
  ~Buffers() {
    if (st) (void)hipStreamSynchronize(st);
    for (void* q : p) (void)hipFree(q);
    if (st) (void)hipStreamDestroy(st);
  }
};

int open_device(int device, Buffers& b) {
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(PW_ERR_HIP, "no HIP device available");
  if (device < 0 || device >= ndev) return fail(PW_ERR_ARG, "device index out of range");
  if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&b.st, hipStreamNonBlocking) != hipSuccess)
    return fail(PW_ERR_HIP, "stream creation failed");
  return PW_OK;
}

#define RX_HIP(call)                                                                      \
  do {                                                                                    \
    hipError_t e_ = (call);                                                               \
    if (e_ != hipSuccess) return fail(PW_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

template <typename T>
hipError_t up(T* d, const T* h, size_t count, hipStream_t st) {
  return hipMemcpyAsync(d, h, count * sizeof(T), hipMemcpyHostToDevice, st);
}
template <typename T>
hipError_t down(T* h, const T* d, size_t count, hipStream_t st) {
  return hipMemcpyAsync(h, d, count * sizeof(T), hipMemcpyDeviceToHost, st);
}

}  // namespace

extern "C" {

int pw_wake_split(int device, double stepnum, int64_t maxn, int64_t* num_particles, int64_t* npidx, double* pos,
                  double* alpha, double* radius, double* volume, double* birthstrength, double* active,
                  int64_t* nsplit) {
  if (!num_particles || !npidx || !pos || !alpha || !radius || !volume || !birthstrength || !active)
    return fail(PW_ERR_ARG, "null argument");
  const int64_t n = *num_particles;
  if (n < 0 || maxn < n || maxn > INT32_MAX / 2) return fail(PW_ERR_ARG, "need 0 <= num_particles <= maxn < 2^30");
  if (*npidx != n)
    return fail(PW_ERR_UNSUPPORTED, "new particles are appended after the last one: npidx must equal "
                                    "num_particles (the reference writes them at npidx, wake.cpp:81-99)");
  if (nsplit) *nsplit = 0;
  if (n == 0) return PW_OK;
  Buffers b;
  PW_TRY(open_device(device, b));
  const size_t m = static_cast<size_t>(maxn);
  double *d_pos, *d_alpha, *d_rad, *d_vol, *d_birth, *d_act;
  int *d_prefix, *d_flag, *d_off;
  const int ni = static_cast<int>(n);
  size_t tb = 0;
  RX_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, static_cast<int*>(nullptr), static_cast<int*>(nullptr), ni, b.st));
  char* d_temp;
  b.add(&d_pos, 3 * m);
  b.add(&d_alpha, 3 * m);
  b.add(&d_rad, m);
  b.add(&d_vol, m);
  b.add(&d_birth, m);
  b.add(&d_act, m);
  b.add(&d_prefix, 1);
  b.add(&d_flag, n);
  b.add(&d_off, n);
  b.add(&d_temp, tb);
  if (!b.allocate()) return fail(PW_ERR_NOMEM, "device buffers");
  const size_t nn = static_cast<size_t>(n);
  RX_HIP(up(d_pos, pos, 3 * nn, b.st));
  RX_HIP(up(d_alpha, alpha, 3 * nn, b.st));
  RX_HIP(up(d_rad, radius, nn, b.st));
  RX_HIP(up(d_vol, volume, nn, b.st));
  RX_HIP(up(d_birth, birthstrength, nn, b.st));
  RX_HIP(up(d_act, active, nn, b.st));
  const dim3 grid((ni + kB - 1) / kB);
  RX_HIP(pw::launch_fill_int(d_prefix, 1, ni, b.st));
  hipLaunchKernelGGL(k_age_prefix, grid, dim3(kB), 0, b.st, d_act, ni, stepnum, d_prefix);
  RX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_split_flags, grid, dim3(kB), 0, b.st, ni, d_prefix, d_alpha, d_birth, d_flag);
  RX_HIP(hipGetLastError());
  RX_HIP(hipcub::DeviceScan::ExclusiveSum(d_temp, tb, d_flag, d_off, ni, b.st));
  int last_off = 0, last_flag = 0;
  RX_HIP(down(&last_off, d_off + (ni - 1), 1, b.st));
  RX_HIP(down(&last_flag, d_flag + (ni - 1), 1, b.st));
  RX_HIP(hipStreamSynchronize(b.st));
  const int64_t s = static_cast<int64_t>(last_off) + last_flag;
  if (n + s > maxn)
    return fail(PW_ERR_UNSUPPORTED, "the new particles would not fit in maxn rows (the reference then wraps "
                                    "and overwrites its first particles, wake.cpp:96-99)");
  if (s > 0) {
    hipLaunchKernelGGL(k_split_apply, grid, dim3(kB), 0, b.st, ni, n, d_flag, d_off, d_pos, d_alpha, d_rad, d_vol,
                       d_birth, d_act);
    RX_HIP(hipGetLastError());
    const size_t nt = static_cast<size_t>(n + s);
    RX_HIP(down(pos, d_pos, 3 * nt, b.st));
    RX_HIP(down(alpha, d_alpha, 3 * nt, b.st));
    RX_HIP(down(radius, d_rad, nt, b.st));
    RX_HIP(down(volume, d_vol, nt, b.st));
    RX_HIP(down(birthstrength, d_birth, nt, b.st));
    RX_HIP(down(active, d_act, nt, b.st));
    RX_HIP(hipStreamSynchronize(b.st));
  }
  *num_particles = n + s;
  *npidx = n + s;
  if (nsplit) *nsplit = s;
  return PW_OK;
}

int pw_wake_merge(int device, double stepnum, int64_t num_particles, double* pos, double* alpha,
                  const double* radius, double* volume, const double* active, int64_t* nmerged) {
  if (!pos || !alpha || !radius || !volume || !active) return fail(PW_ERR_ARG, "null argument");
  if (num_particles < 0 || num_particles > INT32_MAX / 2) return fail(PW_ERR_ARG, "need 0 <= num_particles < 2^30");
  if (nmerged) *nmerged = 0;
  const int64_t n = num_particles;
  if (n < 2) return PW_OK;
  Buffers b;
  PW_TRY(open_device(device, b));
  const size_t nn = static_cast<size_t>(n);
  const int ni = static_cast<int>(n);
  double *d_pos, *d_alpha, *d_rad, *d_vol, *d_act, *d_ext;
  int *d_prefix, *d_flag, *d_idx, *d_sidx, *d_list, *d_count;
  int *d_parent, *d_root, *d_sroot, *d_slist, *d_left;
  uint64_t *d_key, *d_skey, *d_gkey, *d_sgkey;
  unsigned long long* d_merges;
  char* d_temp;
  size_t t1 = 0, t2 = 0;
  {
    uint64_t* k0 = nullptr;
    int* i0 = nullptr;
    RX_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, t1, k0, k0, i0, i0, ni, 0, 64, b.st));
    RX_HIP(hipcub::DeviceSelect::Flagged(nullptr, t2, i0, i0, i0, i0, ni, b.st));
  }
  b.add(&d_pos, 3 * nn);
  b.add(&d_alpha, 3 * nn);
  b.add(&d_rad, nn);
  b.add(&d_vol, nn);
  b.add(&d_act, nn);
  b.add(&d_ext, 7 * kExtentBlocks);
  b.add(&d_prefix, 1);
  b.add(&d_flag, nn);
  b.add(&d_idx, nn);
  b.add(&d_sidx, nn);
  b.add(&d_list, nn);
  b.add(&d_count, 1);
  b.add(&d_key, nn);
  b.add(&d_skey, nn);
  b.add(&d_merges, 1);
  b.add(&d_left, 1);
  b.add(&d_temp, std::max(t1, t2));
  if (!b.allocate()) return fail(PW_ERR_NOMEM, "device buffers");
  RX_HIP(up(d_pos, pos, 3 * nn, b.st));
  RX_HIP(up(d_alpha, alpha, 3 * nn, b.st));
  RX_HIP(up(d_rad, radius, nn, b.st));
  RX_HIP(up(d_vol, volume, nn, b.st));
  RX_HIP(up(d_act, active, nn, b.st));
  // the cell size: the largest merge distance, with room for rounding
  hipLaunchKernelGGL(k_extent, dim3(kExtentBlocks), dim3(kB), 0, b.st, d_pos, d_rad, ni, d_ext);
  RX_HIP(hipGetLastError());
  double ext[7 * kExtentBlocks];
  RX_HIP(down(ext, d_ext, 7 * kExtentBlocks, b.st));
  RX_HIP(hipStreamSynchronize(b.st));
  for (int k = 7; k < 7 * kExtentBlocks; ++k)
    ext[k % 7] = k % 7 < 3 ? std::min(ext[k % 7], ext[k]) : std::max(ext[k % 7], ext[k]);
  if (!(ext[6] > 0.0)) return PW_OK;  // no radius: nothing is within reach
  Grid g;
  g.x0 = std::isfinite(ext[0]) ? ext[0] : 0.0;
  g.y0 = std::isfinite(ext[1]) ? ext[1] : 0.0;
  g.z0 = std::isfinite(ext[2]) ? ext[2] : 0.0;
  double span = 0.0;
  for (int c = 0; c < 3; ++c)
    if (std::isfinite(ext[c]) && std::isfinite(ext[3 + c])) span = std::max(span, ext[3 + c] - ext[c]);
  g.h = std::max(0.25 * ext[6] * (1.0 + 1e-6), span / static_cast<double>(kCellMax - 1));
  const dim3 grid((ni + kB - 1) / kB);
  RX_HIP(pw::launch_fill_int(d_prefix, 1, ni, b.st));
  hipLaunchKernelGGL(k_age_prefix, grid, dim3(kB), 0, b.st, d_act, ni, stepnum, d_prefix);
  RX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_cell_keys, grid, dim3(kB), 0, b.st, d_pos, ni, g, d_key, d_idx);
  RX_HIP(hipGetLastError());
  RX_HIP(hipcub::DeviceRadixSort::SortPairs(d_temp, t1, d_key, d_skey, d_idx, d_sidx, ni, 0, 64, b.st));
  RX_HIP(pw::launch_fill_int(d_flag, ni, 0, b.st));
  const dim3 rgrid(static_cast<unsigned>((9 * static_cast<int64_t>(ni) + kB - 1) / kB));
  hipLaunchKernelGGL(k_merge_flags, rgrid, dim3(kB), 0, b.st, ni, d_prefix, g, d_skey, d_sidx, d_pos, d_alpha, d_rad,
                     d_flag);
  RX_HIP(hipGetLastError());
  // the flagged particles in ascending order (the sort left d_idx = 0..n-1)
  RX_HIP(hipcub::DeviceSelect::Flagged(d_temp, t2, d_idx, d_flag, d_list, d_count, ni, b.st));
  int count = 0;
  RX_HIP(down(&count, d_count, 1, b.st));
  RX_HIP(hipStreamSynchronize(b.st));
  if (count == 0) return PW_OK;
  // groups of flagged particles that cannot reach each other's, each
  // replayed by a block of its own
  b.add(&d_parent, count);
  b.add(&d_root, count);
  b.add(&d_sroot, count);
  b.add(&d_slist, count);
  b.add(&d_gkey, count);
  b.add(&d_sgkey, count);
  char* d_temp2;
  size_t t4 = 0, t5 = 0;
  RX_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, t4, d_key, d_skey, d_flag, d_sidx, count, 0, 64, b.st));
  RX_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, t5, d_flag, d_sidx, d_flag, d_sidx, count, 0, 32, b.st));
  b.add(&d_temp2, std::max(t4, t5));
  if (!b.allocate()) return fail(PW_ERR_NOMEM, "merge groups");
  const dim3 lgrid((count + kB - 1) / kB);
  RX_HIP(pw::launch_fill_int(reinterpret_cast<int*>(d_merges), 2, 0, b.st));
  RX_HIP(pw::launch_fill_int(d_left, 1, 0, b.st));
  hipLaunchKernelGGL(k_group_keys, lgrid, dim3(kB), 0, b.st, d_pos, d_list, count, g, d_gkey, d_flag, d_parent);
  RX_HIP(hipGetLastError());
  // (d_flag and d_slist are free: indices before and after the sort)
  RX_HIP(hipcub::DeviceRadixSort::SortPairs(d_temp2, t4, d_gkey, d_sgkey, d_flag, d_slist, count, 0, 64, b.st));
  const dim3 cgrid(static_cast<unsigned>((14 * static_cast<int64_t>(count) + kB - 1) / kB));
  hipLaunchKernelGGL(k_group_link, cgrid, dim3(kB), 0, b.st, d_pos, d_list, d_sgkey, d_slist, count, g, d_parent);
  RX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_group_roots, lgrid, dim3(kB), 0, b.st, count, d_parent, d_root);
  RX_HIP(hipGetLastError());
  // a stable sort: ascending particles within a group
  RX_HIP(hipcub::DeviceRadixSort::SortPairs(d_temp2, t5, d_root, d_sroot, d_list, d_slist, count, 0, 32, b.st));
  hipLaunchKernelGGL(k_merge_resolve, dim3(count), dim3(kRT), 0, b.st, ni, d_slist, d_sroot, count, g, d_skey, d_sidx,
                     d_pos, d_alpha, d_rad, d_vol, d_merges, d_left);
  RX_HIP(hipGetLastError());
  unsigned long long merges = 0;
  int left = 0;
  RX_HIP(down(&merges, d_merges, 1, b.st));
  RX_HIP(down(&left, d_left, 1, b.st));
  RX_HIP(hipStreamSynchronize(b.st));
  if (left) {
    // a particle travelled further than the groups are apart: from the start,
    // one block over all of them
    RX_HIP(up(d_pos, pos, 3 * nn, b.st));
    RX_HIP(up(d_alpha, alpha, 3 * nn, b.st));
    RX_HIP(up(d_vol, volume, nn, b.st));
    RX_HIP(pw::launch_fill_int(reinterpret_cast<int*>(d_merges), 2, 0, b.st));
    hipLaunchKernelGGL(k_merge_resolve, dim3(1), dim3(kRT), 0, b.st, ni, d_list, static_cast<const int*>(nullptr), count,
                       g, d_skey, d_sidx, d_pos, d_alpha, d_rad, d_vol, d_merges, d_left);
    RX_HIP(hipGetLastError());
    RX_HIP(down(&merges, d_merges, 1, b.st));
    RX_HIP(hipStreamSynchronize(b.st));
  }
  if (merges > 0) {
    RX_HIP(down(pos, d_pos, 3 * nn, b.st));
    RX_HIP(down(alpha, d_alpha, 3 * nn, b.st));
    RX_HIP(down(volume, d_vol, nn, b.st));
    RX_HIP(hipStreamSynchronize(b.st));
  }
  if (nmerged) *nmerged = static_cast<int64_t>(merges);
  return PW_OK;
}

}  // extern "C"
