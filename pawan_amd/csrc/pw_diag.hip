// pw_diag.hip -- FP64 conserved-quantity diagnostics on the device.
//
// __interaction::diagnose (src/interaction/interaction.cpp:64-194) has two
// kinds of sums:
//   * O(N), per wake: total vorticity sum(a), linear impulse sum(x x a)/2,
//     angular impulse sum(x x (x x a))/3 and the centroid sums
//     |a| z (x^2+y^2) and |a| (x^2+y^2)  (interaction.cpp:489-527, 135-157);
//   * O(N^2), over every unordered pair counted twice plus self terms:
//     helicity, kinetic energy and its div-free variant, enstrophy and its
//     div-free variant (interaction_utils.h:107-331; the enstrophies are
//     identically zero for the Gaussian kernel, gaussian.h:69-92, and
//     nonzero for the high-order algebraic one, highorder.h:77-106).
// Both are computed here as per-block partial sums in a fixed tree order, and
// the partials are added in a fixed order, so results are deterministic.
// Pair terms are symmetric in the two particles: each unordered pair of a
// system is evaluated once, with the weight 2 of the reference's sums.
#include <hip/hip_runtime.h>

#include "pw_core64.h"
#include "pw_internal.h"

namespace pw {
namespace {

constexpr int kTB = 256;
constexpr double kPi = 3.14159265358979323846;
constexpr double k1Pi = 0.31830988618379067154;  // M_1_PI
constexpr double kQ = 0x1.45f306dc9c883p-4;      // 0.25 * M_1_PI
constexpr double kFar64 = 90.0;                  // beyond 90 sigma^2 the Gaussian terms are below FP64 rounding

// Sum of v over the block, exact same tree every call: butterfly within
// each 64-lane wavefront, then the four wave totals in wave order.
template <int M>
__device__ __forceinline__ void block_sum(double (&v)[M], double* red) {
  for (int off = 32; off > 0; off >>= 1)
    for (int m = 0; m < M; ++m) v[m] += __shfl_xor(v[m], off, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0)
    for (int m = 0; m < M; ++m) red[wave * M + m] = v[m];
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int m = 0; m < M; ++m) {
      double s = red[m];
      for (int w = 1; w < kTB / 64; ++w) s += red[w * M + m];
      v[m] = s;
    }
  }
}

// Linear sums over blocks of up to kTB particles of one wake.
// items[b] = {first, last, wake, 0}; out[b * 11 + m].
__global__ __launch_bounds__(kTB) void k_diag_linear(
    const Rec64* __restrict__ y, const WorkItem* __restrict__ items,
    double* __restrict__ out) {
  __shared__ double red[(kTB / 64) * 11];
  const WorkItem it = items[blockIdx.x];
  const int i = it.t0 + static_cast<int>(threadIdx.x);
  double v[11];
  for (int m = 0; m < 11; ++m) v[m] = 0.0;
  if (i < it.t1) {
    const Rec64 p = y[i];
    // x x a
    const double rx = p.y * p.az - p.z * p.ay;
    const double ry = p.z * p.ax - p.x * p.az;
    const double rz = p.x * p.ay - p.y * p.ax;
    v[0] = p.ax; v[1] = p.ay; v[2] = p.az;
    v[3] = rx; v[4] = ry; v[5] = rz;
    // x x (x x a)
    v[6] = p.y * rz - p.z * ry;
    v[7] = p.z * rx - p.x * rz;
    v[8] = p.x * ry - p.y * rx;
    const double oy = sqrt(p.ax * p.ax + p.ay * p.ay + p.az * p.az);
    const double rr = p.x * p.x + p.y * p.y;
    v[9] = oy * p.z * rr;
    v[10] = oy * rr;
  }
  block_sum<11>(v, red);
  if (threadIdx.x == 0)
    for (int m = 0; m < 11; ++m) out[blockIdx.x * 11 + m] = v[m];
}

// 1/sqrt(x) for positive finite x: the hardware estimate and one third-order
// correction (relative error below 2^-52)
__device__ __forceinline__ double rsqrt_pos(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// Sums of one target's pairs, the constants of the energies factored out.
struct DiagSum {
  double h = 0.0, ke = 0.0, kef = 0.0, en = 0.0, enf = 0.0;
};

// helicity, KE, KEF (and, for the high-order kernel, the two enstrophies) of
// one pair (interaction_utils.h:141-331), I = target, J = source
template <bool HighOrder>
__device__ __forceinline__ void diag_pair(const Rec64& me, const Rec64& s, const double* __restrict__ tab,
                                          DiagSum& d) {
  const double x0 = s.x - me.x, x1 = s.y - me.y, x2 = s.z - me.z;  // x12 = x_J - x_I
  const double rho2 = x0 * x0 + x1 * x1 + x2 * x2;
  const double sigma2 = 0.5 * (me.s2 + s.s2);
  const double ib = rsqrt_pos(rho2 + sigma2);
  const double ib2 = ib * ib, ib3 = ib2 * ib;
  double q;
  if (HighOrder) {
    // QSIG (highorder.h:31-39) in closed form; 0/0 for coincident particles
    q = kQ * fma(2.5, sigma2, rho2) * (ib3 * ib2);
    if (rho2 == 0.0) q = __builtin_nan("");
  } else {
    const double ir = rsqrt_pos(rho2);
    q = kQ * (ir * (ir * ir));
    if (rho2 <= kFar64 * sigma2) {
      const double isg = rsqrt_pos(sigma2);
      const double isg2 = isg * isg;
      double e, g;
      const double sb = fma(ir, 0.0, rho2 * isg2);  // not finite for coincident particles, as in the reference
      core64(sb, tab, e, g);
      q = kCore64K * (isg2 * isg) * fma(sb, g, e * (1.0 / 3.0));
    }
  }
  const double c0 = me.ay * s.az - me.az * s.ay;
  const double c1 = me.az * s.ax - me.ax * s.az;
  const double c2 = me.ax * s.ay - me.ay * s.ax;
  d.h = fma(q, x0 * c0 + x1 * c1 + x2 * c2, d.h);
  const double a1a2 = me.ax * s.ax + me.ay * s.ay + me.az * s.az;
  const double xx = (x0 * me.ax + x1 * me.ay + x2 * me.az) * (x0 * s.ax + x1 * s.ay + x2 * s.az);
  // ((rho^2 + 2 sigma^2) a1.a2 + (x12.a1)(x12.a2)) / b^1.5 / 16 pi and
  // (rho^2 + 1.5 sigma^2) a1.a2 / b^1.5 / 8 pi (:278-331)
  const double a3 = a1a2 * ib3;
  d.ke = fma(ib3, xx, fma(fma(2.0, sigma2, rho2), a3, d.ke));
  d.kef = fma(fma(1.5, sigma2, rho2), a3, d.kef);
  if (HighOrder) {
    // ENST / ENSTF (highorder.h:77-96): F1 a1.a2 + F2 (x12.a1)(x12.a2), b^3.5 below
    const double ib7 = ib3 * (ib2 * ib2);
    const double r4 = rho2 * rho2, rs = rho2 * sigma2, s4 = sigma2 * sigma2;
    const double f1 = 2.0 * r4 + 7.0 * rs + 20.0 * s4;
    const double f2 = 6.0 * r4 + 27.0 * rs + 21.0 * s4;
    d.en = fma(ib7, fma(f1, a1a2, -(f2 * ib2) * xx), d.en);
    d.enf = fma(s4 * ib7, a1a2, d.enf);
  }
}

// One item: its targets [t0, t1) (at most 64, one per lane of each of the
// block's four waves) against its sources [s0, s1), a quarter of each
// 256-source tile per wave.  nself = 0: a range of the targets' own system,
// of which only the sources before the target count, twice, and the item
// whose range ends with the targets adds their self terms; nself = 1: a
// cross-wake block, every source once, no self terms.  The block total goes
// to out[kDiagQuad * b].
//
// The ordered pairs of 94 blocks, each with an exp, an erf, two square roots
// and seven divisions, took 18.7 ms for 24,000 particles; unordered, split
// over 4,600 blocks and with the divisions taken out (about 60 instructions a
// pair, the core from pw_core64.h) FP64 issue bounds it.
template <bool HighOrder>
__global__ __launch_bounds__(kTB) void k_diag_pairs(
    const Rec64* __restrict__ y, const double* __restrict__ radius,
    const WorkItem* __restrict__ items, double* __restrict__ out) {
  constexpr int kWaves = kTB / 64;
  __shared__ Rec64 tile[kTB];
  __shared__ double red[kWaves * kDiagQuad];
  __shared__ __align__(16) double tab[HighOrder ? 2 : kCore64Pieces * kCore64Row];
  if (!HighOrder) stage_core64<kTB>(tab);  // (synchronised with the first tile)
  const WorkItem it = items[blockIdx.x];
  const int lane = static_cast<int>(threadIdx.x) & 63, wave = static_cast<int>(threadIdx.x) >> 6;
  const int t = it.t0 + lane;
  const bool active = t < it.t1;
  const bool cross = it.nself != 0;
  const Rec64 me = y[active ? t : it.t0];
  DiagSum d;
  for (int base = it.s0; base < it.s1; base += kTB) {
    const int cnt = min(kTB, it.s1 - base);
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < cnt) tile[threadIdx.x] = y[base + threadIdx.x];
    __syncthreads();
    const int l0 = cnt * wave / kWaves, l1 = cnt * (wave + 1) / kWaves;
    if (cross || base + l1 <= it.t0) {
#pragma unroll 2
      for (int l = l0; l < l1; ++l) diag_pair<HighOrder>(me, tile[l], tab, d);
    } else {
      for (int l = l0; l < l1; ++l)
        if (base + l < t) diag_pair<HighOrder>(me, tile[l], tab, d);
    }
  }
  const double f = cross ? 1.0 : 2.0;
  double v[kDiagQuad] = {active ? f * d.h : 0.0, active ? f * d.ke / 16.0 / kPi : 0.0,
                         active ? f * d.kef / 8.0 / kPi : 0.0, active ? f * d.en * (k1Pi / 8.0) : 0.0,
                         active ? f * d.enf * (15.0 * k1Pi / 8.0) : 0.0};
  if (active && !cross && wave == 0 && it.s1 == it.t1) {
    // self terms (interaction_utils.h:249-267)
    const double sg = radius[t];
    const double a2 = me.ax * me.ax + me.ay * me.ay + me.az * me.az;
    v[1] += k1Pi * a2 / sg / 8.0;
    v[2] += 3 * k1Pi * a2 / (sg * 16.0);
    if (HighOrder) {
      // ENST(sigma), ENSTF(sigma) (highorder.h:98-106)
      v[3] += 5.0 * k1Pi / 2.0 / (sg * sg * sg) * a2;
      v[4] += 15.0 * k1Pi / 8.0 / (sg * sg * sg) * a2;
    }
  }
  block_sum<kDiagQuad>(v, red);
  if (threadIdx.x == 0)
    for (int m = 0; m < kDiagQuad; ++m) out[kDiagQuad * blockIdx.x + m] = v[m];
}

// out[kDiagQuad * s + m] = sum of the items [first[s], first[s + 1]): one
// block per system, lanes over the items, then the fixed tree
__global__ __launch_bounds__(kTB) void k_diag_sum(const double* __restrict__ items, const int* __restrict__ first,
                                                  double* __restrict__ out) {
  __shared__ double red[(kTB / 64) * kDiagQuad];
  double v[kDiagQuad] = {0.0, 0.0, 0.0, 0.0, 0.0};
  for (int i = first[blockIdx.x] + static_cast<int>(threadIdx.x); i < first[blockIdx.x + 1]; i += kTB)
    for (int m = 0; m < kDiagQuad; ++m) v[m] += items[static_cast<size_t>(kDiagQuad) * i + m];
  block_sum<kDiagQuad>(v, red);
  if (threadIdx.x == 0)
    for (int m = 0; m < kDiagQuad; ++m) out[kDiagQuad * blockIdx.x + m] = v[m];
}

}  // namespace

hipError_t launch_diag_linear(const Rec64* y, const WorkItem* items,
                              int nitems, double* out, hipStream_t st) {
  if (nitems <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_diag_linear, dim3(nitems), dim3(kTB), 0, st, y, items, out);
  return hipGetLastError();
}

hipError_t launch_diag_pairs(const Rec64* y, const double* radius,
                             const WorkItem* items, int nitems, double* out,
                             bool high_order, hipStream_t st) {
  if (nitems <= 0) return hipSuccess;
  if (high_order)
    hipLaunchKernelGGL(k_diag_pairs<true>, dim3(nitems), dim3(kTB), 0, st, y, radius, items, out);
  else
    hipLaunchKernelGGL(k_diag_pairs<false>, dim3(nitems), dim3(kTB), 0, st, y, radius, items, out);
  return hipGetLastError();
}

hipError_t launch_diag_sum(const double* items, const int* first, int nsys, double* out, hipStream_t st) {
  if (nsys <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_diag_sum, dim3(nsys), dim3(kTB), 0, st, items, first, out);
  return hipGetLastError();
}

}  // namespace pw
