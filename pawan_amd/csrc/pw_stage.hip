// pw_stage.hip -- stage arithmetic of the time integrators (FP64).
//
// The reference advances the concatenated state vector with GSL BLAS-1
// calls (src/integration/rk4.cpp:12-77, rk3.cpp:12-65,
// integration.cpp:126-136); these kernels do the same element-wise
// operations in the same order, with multiply and add kept separate
// (contraction off), on the device-resident particle records.
#include <hip/hip_runtime.h>

#include "pw_internal.h"

namespace pw {
namespace {

constexpr int kEW = 256;

// One right-hand side's tail: the sum of its partial rates, the finite check
// and the stage arithmetic, one thread per rate component (component c of
// particle t is double 6 t + c of the rates, so every partial slice or slab is
// read coalesced).  A small wake's step is bound by its launches: 3 kernels
// per right-hand side became 1, and by the latency of the partial loads, which
// the unrolled loop keeps several in flight of.
//
// The partial rates are summed in order (deterministic).  Sum: 0 none, 1
// slices of n rows, 2 slabs of 64 rows (k_pair_split).
constexpr int kGroupThreads = 6 * 64;  // a group's 64 rows
// Loads of the split sum in flight at a time.  The kernel is a chain of memory
// latencies (a group's slabs were written through other XCDs' caches): with 8,
// and the stage's own inputs loaded after the sum, a right-hand side of 1,000
// particles took 14.5 us (FP64), with 8 and the inputs loaded first 13.1, with
// 16 12.4, with 32 12.5 (and 200 particles 9.0, 8.8, 9.6).
constexpr int kSumUnroll = 16;

struct FinishArgs {
  const double* partial;
  int parts;
  const SplitGroup* groups;
  double* rates;
  int n;
  int* flag;
  StageOp op;
};

// What a component's stage arithmetic reads besides the rate; loaded before the
// partial rates are summed, so that the two waits overlap.
struct StageIn {
  double y = 0, next = 0, k1 = 0, k2 = 0, k3 = 0;
};

// the component's place in Rec64: x y z s2 ax ay az vol
__device__ __forceinline__ int64_t stage_at(int64_t e) {
  const int64_t t = e / 6;
  const int c = static_cast<int>(e - 6 * t);
  return 8 * t + c + (c >= 3 ? 1 : 0);
}

template <int Op>
__device__ __forceinline__ StageIn stage_in(const StageOp& op, int64_t e) {
  StageIn in;
  if (Op == kStageNone) return in;
  const int64_t at = stage_at(e);
  const double* y = reinterpret_cast<const double*>(op.y);
  in.y = y[at];
  if ((Op == kStageLin || Op == kStageRk3Mid) && e % 3 == 2) in.next = y[at + 1];  // s2, vol
  if (Op == kStageRk3Mid || Op == kStageRk4 || Op == kStageRk3) in.k1 = reinterpret_cast<const double*>(op.k1)[e];
  if (Op == kStageRk4 || Op == kStageRk3) in.k2 = reinterpret_cast<const double*>(op.k2)[e];
  if (Op == kStageRk4) in.k3 = reinterpret_cast<const double*>(op.k3)[e];
  return in;
}

template <int Op>
__device__ __forceinline__ void stage_component(const StageOp& op, const StageIn& in, int64_t e, double k) {
#pragma clang fp contract(off)
  if (Op == kStageNone) return;
  const int64_t at = stage_at(e);
  if (Op == kStageLin || Op == kStageRk3Mid) {
    double* out = reinterpret_cast<double*>(op.out);
    if (Op == kStageLin) {
      out[at] = k * op.a + in.y;
    } else {
      const double b1 = in.k1 * op.a;
      out[at] = (k * op.b + in.y) - b1;
      reinterpret_cast<double*>(op.k1)[e] = b1;
    }
    if (e % 3 == 2) out[at + 1] = in.next;
    return;
  }
  double* y = reinterpret_cast<double*>(op.y);
  if (Op == kStageRk4)
    y[at] = in.y + ((in.k1 + k) * op.a + (in.k2 + in.k3) * op.b);
  else if (Op == kStageRk3)
    y[at] = in.y + ((in.k1 * (1.0 / 6.0) + k * op.a) + in.k2 * op.b);
  else
    y[at] = in.y + k * op.a;
}

// p[0] + p[stride] + ... in that order, UNROLL loads in flight at a time
template <int kUnroll>
__device__ __forceinline__ double sum_slices(const double* __restrict__ p, size_t stride, int count) {
  double k = p[0];
  int i = 1;
  for (; i + kUnroll <= count; i += kUnroll) {
    double v[kUnroll];
#pragma unroll
    for (int j = 0; j < kUnroll; ++j) v[j] = p[(i + j) * stride];
#pragma unroll
    for (int j = 0; j < kUnroll; ++j) k += v[j];
  }
  if (i < count) {
    double v[kUnroll];  // the rest: loads past the end repeat the last slice and are not added
#pragma unroll
    for (int j = 0; j < kUnroll; ++j) v[j] = p[min(i + j, count - 1) * stride];
#pragma unroll
    for (int j = 0; j < kUnroll; ++j)
      if (i + j < count) k += v[j];
  }
  return k;
}

template <int Sum, int Op>
__global__ __launch_bounds__(Sum == 2 ? kGroupThreads : kEW) void k_finish(FinishArgs f) {
  int64_t e;
  double k;
  StageIn in;
  if (Sum == 2) {
    const SplitGroup g = f.groups[blockIdx.x];
    if (static_cast<int>(threadIdx.x) >= 6 * (g.t1 - g.t0)) return;
    e = 6 * static_cast<int64_t>(g.t0) + threadIdx.x;
    in = stage_in<Op>(f.op, e);
    k = sum_slices<kSumUnroll>(f.partial + static_cast<size_t>(g.first) * kGroupThreads + threadIdx.x, kGroupThreads, g.count);
    f.rates[e] = k;
  } else {
    e = static_cast<int64_t>(blockIdx.x) * kEW + threadIdx.x;
    const int64_t total = 6 * static_cast<int64_t>(f.n);
    if (e >= total) return;
    in = stage_in<Op>(f.op, e);
    if (Sum == 1) {
      k = f.partial[e];
#pragma unroll 8
      for (int i = 1; i < f.parts; ++i) k += f.partial[static_cast<size_t>(i) * total + e];
      f.rates[e] = k;
    } else {
      k = f.rates[e];
    }
  }
  if (!isfinite(k)) *f.flag = 1;  // (host memory: every writer stores the same word)
  stage_component<Op>(f.op, in, e, k);
}

__global__ __launch_bounds__(kEW) void k_check_finite(
    const Rate64* __restrict__ k, int n, int* __restrict__ flag) {
  const int i = blockIdx.x * kEW + threadIdx.x;
  if (i >= n) return;
  const Rate64 r = k[i];
  const double s = r.ux + r.uy + r.uz + r.wx + r.wy + r.wz;
  if (!isfinite(s) || !isfinite(r.ux) || !isfinite(r.wx)) *flag = 1;
}

__global__ void k_fill_int(int* __restrict__ p, int n, int value) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

__global__ void k_zero_doubles(double* __restrict__ p, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0;
}

__global__ __launch_bounds__(kEW) void k_add_rates(Rate64* __restrict__ acc, const Rate64* __restrict__ add,
                                                   int first, int last) {
  const int i = first + blockIdx.x * kEW + static_cast<int>(threadIdx.x);
  if (i >= last) return;
  Rate64 a = acc[i];
  const Rate64 b = add[i];
  a.ux += b.ux; a.uy += b.uy; a.uz += b.uz;
  a.wx += b.wx; a.wy += b.wy; a.wz += b.wz;
  acc[i] = a;
}

// Particles [first, first + count) of the state or the rates to and from the
// two 3-vectors per particle that callers hold: xyz and alpha (or u and dalpha)
// of all the particles, one after the other, one thread per double.  The
// packed side is pinned host memory, read and written by the kernel itself
// (coalesced 8-byte accesses over the bus), so a transfer is one launch and
// moves 48 bytes per particle; copying the records both ways and converting
// them on one host thread took 20 ms of a 1M right-hand side.
template <bool State, bool Store>
__global__ __launch_bounds__(kEW) void k_pack(double* __restrict__ dev, int64_t first, int64_t count,
                                              double* __restrict__ host) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * kEW + threadIdx.x;
  if (e >= 6 * count) return;
  const int half = e >= 3 * count ? 1 : 0;
  const int64_t v = e - 3 * count * half;
  const int64_t i = v / 3;
  const int c = static_cast<int>(v - 3 * i);
  double* d = dev + (State ? 8 * (first + i) + 4 * half : 6 * (first + i) + 3 * half) + c;
  if (Store) *d = host[e];
  else host[e] = *d;
}

inline int ew_blocks(int n) { return (n + kEW - 1) / kEW; }

}  // namespace

hipError_t launch_zero_doubles(double* p, int64_t n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_doubles, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, p, n);
  return hipGetLastError();
}

hipError_t launch_add_rates(Rate64* acc, const Rate64* add, int first, int last, hipStream_t st) {
  if (last <= first) return hipSuccess;
  hipLaunchKernelGGL(k_add_rates, dim3(ew_blocks(last - first)), dim3(kEW), 0, st, acc, add, first, last);
  return hipGetLastError();
}

namespace {
template <int Op>
void finish_kernel(const SumForm& sum, const FinishArgs& f, hipStream_t st) {
  const dim3 flat(static_cast<unsigned>((6 * static_cast<int64_t>(f.n) + kEW - 1) / kEW));
  if (sum.groups) hipLaunchKernelGGL((k_finish<2, Op>), dim3(sum.ngroups), dim3(kGroupThreads), 0, st, f);
  else if (sum.parts > 1) hipLaunchKernelGGL((k_finish<1, Op>), flat, dim3(kEW), 0, st, f);
  else hipLaunchKernelGGL((k_finish<0, Op>), flat, dim3(kEW), 0, st, f);
}
}  // namespace

hipError_t launch_finish(const SumForm& sum, Rate64* rates, int n, int* flag, const StageOp& op, hipStream_t st) {
  static_assert(sizeof(Rate64) == 6 * sizeof(double) && sizeof(Rec64) == 8 * sizeof(double), "flat components");
  if (n <= 0) return hipSuccess;
  const FinishArgs f{reinterpret_cast<const double*>(sum.partial), sum.parts, sum.groups,
                     reinterpret_cast<double*>(rates), n, flag, op};
  switch (op.kind) {
    case kStageNone: finish_kernel<kStageNone>(sum, f, st); break;
    case kStageLin: finish_kernel<kStageLin>(sum, f, st); break;
    case kStageRk4: finish_kernel<kStageRk4>(sum, f, st); break;
    case kStageRk3Mid: finish_kernel<kStageRk3Mid>(sum, f, st); break;
    case kStageRk3: finish_kernel<kStageRk3>(sum, f, st); break;
    case kStageEuler: finish_kernel<kStageEuler>(sum, f, st); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_pack_state(Rec64* y, int64_t first, int64_t count, double* host, bool store, hipStream_t st) {
  if (count <= 0) return hipSuccess;
  const dim3 g(static_cast<unsigned>((6 * count + kEW - 1) / kEW)), b(kEW);
  double* d = reinterpret_cast<double*>(y);
  if (store) hipLaunchKernelGGL((k_pack<true, true>), g, b, 0, st, d, first, count, host);
  else hipLaunchKernelGGL((k_pack<true, false>), g, b, 0, st, d, first, count, host);
  return hipGetLastError();
}

hipError_t launch_pack_rates(const Rate64* k, int64_t first, int64_t count, double* host, hipStream_t st) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL((k_pack<false, false>), dim3(static_cast<unsigned>((6 * count + kEW - 1) / kEW)), dim3(kEW), 0, st,
                     reinterpret_cast<double*>(const_cast<Rate64*>(k)), first, count, host);
  return hipGetLastError();
}

hipError_t launch_fill_int(int* p, int n, int value, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_int, dim3((n + 63) / 64), dim3(64), 0, st, p, n, value);
  return hipGetLastError();
}

hipError_t launch_check_finite(const Rate64* k, int n, int* flag,
                               hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_check_finite, dim3(ew_blocks(n)), dim3(kEW), 0, st, k, n, flag);
  return hipGetLastError();
}

}  // namespace pw
