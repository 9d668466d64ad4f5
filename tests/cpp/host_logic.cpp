// Host side of the C API on a stand-in for the HIP runtime: device memory is
// host memory, allocations can be made to fail, and the kernel launchers check
// the buffers they are given instead of launching.  Built from pw_capi.hip and
// pw_ff.hip with the host compiler by tests/test_host_logic.py; runs without a
// GPU.  Usage: host_logic CHECK
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <map>
#include <string>
#include <vector>

#include "pw_ctx.h"
#include "pw_mlp.h"

// ---- the stand-in runtime ---------------------------------------------------
namespace {

size_t g_device_limit = std::numeric_limits<size_t>::max();  // bytes of device memory
size_t g_pinned_limit = std::numeric_limits<size_t>::max();  // bytes of pinned memory
size_t g_device_used = 0;
std::map<const void*, size_t> g_device, g_pinned;
std::vector<std::string> g_calls;  // launches and event records, in order
std::vector<pw::WorkItem> g_diag;  // the last diagnostics launch
int g_failures = 0;

void expect(bool ok, const std::string& what) {
  if (!ok) {
    ++g_failures;
    std::printf("FAILED: %s\n", what.c_str());
  }
}

// bytes from p to the end of the device allocation that holds it
size_t room(const void* p) {
  auto it = g_device.upper_bound(p);
  if (!p || it == g_device.begin()) return 0;
  --it;
  const char *at = static_cast<const char*>(p), *from = static_cast<const char*>(it->first);
  return at < from + it->second ? static_cast<size_t>(from + it->second - at) : 0;
}

size_t pinned_used() {
  size_t s = 0;
  for (const auto& a : g_pinned) s += a.second;
  return s;
}

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  *p = nullptr;
  if (bytes > g_device_limit || g_device_used > g_device_limit - bytes) return hipErrorOutOfMemory;
  *p = std::malloc(bytes ? bytes : 1);
  if (!*p) return hipErrorOutOfMemory;
  g_device[*p] = bytes;
  g_device_used += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  const auto it = g_device.find(p);
  if (it == g_device.end()) return hipErrorInvalidValue;
  g_device_used -= it->second;
  g_device.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = nullptr;
  if (bytes > g_pinned_limit || pinned_used() > g_pinned_limit - bytes) return hipErrorOutOfMemory;
  *p = std::malloc(bytes ? bytes : 1);
  g_pinned[*p] = bytes;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  if (p && g_pinned.erase(p)) std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t bytes, hipMemcpyKind) {
  std::memcpy(d, s, bytes);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t bytes, hipMemcpyKind k, hipStream_t) {
  return hipMemcpy(d, s, bytes, k);
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) {
  *p = const_cast<void*>(s);
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(1);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(1);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) {
  g_calls.push_back("event");
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

// ---- the launchers ----------------------------------------------------------
namespace pw {

int pair_kernel_waves(int, const PairConfig&) { return 8; }

hipError_t launch_pair(int, const PairConfig& cfg, const PairArgs& a, int, hipStream_t) {
  g_calls.push_back("pair");
  expect(room(a.items) >= a.nitems * sizeof(WorkItem), "pair items hold the launch");
  const size_t rows = cfg.split > 0 ? 64 * static_cast<size_t>(a.nitems)
                                    : cfg.parts > 1 ? static_cast<size_t>(cfg.parts) * a.n : 0;
  bool chunks = true;
  for (int b = 0; b < a.nitems; ++b) {
    const WorkItem& it = a.items[b];
    const auto holds = [&](int32_t chunk, int32_t s) {
      return chunk >= 0 && chunk < a.nchunks && a.chunks[chunk].first <= s && s < a.chunks[chunk].first + a.chunks[chunk].count;
    };
    chunks = chunks && holds(it.chunk0, it.s0) && (cfg.split == 0 || holds(it.tchunk, it.t0));
  }
  expect(chunks, "the items name their chunks");
  expect(room(a.partial) >= rows * sizeof(Rate64), "the partial rows hold the launch");
  return hipSuccess;
}
hipError_t launch_finish(const SumForm&, Rate64*, int, int*, const StageOp&, hipStream_t) {
  g_calls.push_back("finish");
  return hipSuccess;
}
hipError_t launch_zero_doubles(double*, int64_t, hipStream_t) { return hipSuccess; }
hipError_t launch_diag_linear(const Rec64*, const WorkItem*, int nitems, double* out, hipStream_t) {
  for (int k = 0; k < 11 * nitems; ++k) out[k] = 0.0;
  return hipSuccess;
}
// every item's sums are its number of pairs
hipError_t launch_diag_pairs(const Rec64*, const double*, const WorkItem* items, int nitems, double* out, bool,
                             hipStream_t) {
  g_diag.assign(items, items + nitems);
  expect(room(out) >= kDiagQuad * sizeof(double) * nitems, "the sums hold the items");
  for (int b = 0; b < nitems; ++b)
    for (int m = 0; m < kDiagQuad; ++m)
      out[kDiagQuad * b + m] =
          static_cast<double>(items[b].t1 - items[b].t0) * static_cast<double>(items[b].s1 - items[b].s0);
  return hipSuccess;
}
hipError_t launch_diag_sum(const double* items, const int* first, int nsys, double* out, hipStream_t) {
  for (int s = 0; s < nsys; ++s)
    for (int m = 0; m < kDiagQuad; ++m) {
      double v = 0.0;
      for (int b = first[s]; b < first[s + 1]; ++b) v += items[kDiagQuad * b + m];
      out[kDiagQuad * s + m] = v;
    }
  return hipSuccess;
}
hipError_t launch_pack_state(Rec64* y, int64_t first, int64_t count, double* host, bool store, hipStream_t) {
  g_calls.push_back("pack");
  expect(g_pinned.count(host) && g_pinned[host] >= 48 * static_cast<size_t>(count), "staging holds the piece");
  for (int64_t i = 0; i < count; ++i) {
    Rec64& r = y[first + i];
    double *x = host + 3 * i, *a = host + 3 * (count + i);
    if (store) {
      r.x = x[0]; r.y = x[1]; r.z = x[2];
      r.ax = a[0]; r.ay = a[1]; r.az = a[2];
    } else {
      x[0] = r.x; x[1] = r.y; x[2] = r.z;
      a[0] = r.ax; a[1] = r.ay; a[2] = r.az;
    }
  }
  return hipSuccess;
}

hipError_t launch_pack_rates(const Rate64* k, int64_t first, int64_t count, double* host, hipStream_t) {
  g_calls.push_back("pack");
  expect(g_pinned.count(host) && g_pinned[host] >= 48 * static_cast<size_t>(count), "staging holds the piece");
  for (int64_t i = 0; i < count; ++i) {
    std::memcpy(host + 3 * i, &k[first + i].ux, 24);
    std::memcpy(host + 3 * (count + i), &k[first + i].wx, 24);
  }
  return hipSuccess;
}
int train_blocks(int) { return 256; }
void pack_mlp(const float*, std::vector<uint16_t>& frag, std::vector<float>& bias) {
  frag.assign(kMlpFragElems, 0);
  bias.assign(kMlpBiasLen, 0.0f);
}
// the gradient is the sum of the inputs, the loss that of the targets
hipError_t launch_mlp_grad(const float*, const float* X, const float* Y, const int*, int n, float*, float*, float* grad,
                           float* loss, hipStream_t) {
  float x = 0.0f, y = 0.0f;
  for (int i = 0; i < 16 * n; ++i) x += X[i];
  for (int i = 0; i < 12 * n; ++i) y += Y[i];
  for (int p = 0; p < kMlpParams; ++p) grad[p] = x;
  *loss = y;
  return hipSuccess;
}

}  // namespace pw

// ---- the checks -------------------------------------------------------------
namespace {

pw_ctx* context(const std::vector<int64_t>& wakes, bool coupled = true) {
  pw_ctx* c = nullptr;
  expect(pw_create(&c, 0) == PW_OK, "create");
  expect(pw_set_coupled(c, coupled) == PW_OK, "set_coupled");
  int64_t base = 0;
  for (const int64_t n : wakes) {
    std::vector<double> x(3 * n), a(3 * n), r(n, 0.1), v(n, 1.0);
    for (int64_t i = 0; i < 3 * n; ++i) {
      x[i] = base + i;
      a[i] = -(base + i) - 0.5;
    }
    base += 3 * n;
    expect(pw_add_wake(c, n, n, x.data(), a.data(), r.data(), v.data(), nullptr) == PW_OK, "add_wake");
  }
  return c;
}

// One precision's larger partial-sum buffer does not fit: it runs in one part,
// and what other precisions had built must not be launched without rows.
void partial_buffer() {
  for (const size_t left : {size_t(100) << 20, size_t(8) << 20, size_t(1) << 20}) {
    pw_ctx* c = context({60000});
    g_device_limit = std::numeric_limits<size_t>::max();
    expect(pw_solve(c, PW_FP64) == PW_OK, "fp64");  // 64 parts: 184 MB of rows
    g_device_limit = g_device_used + left;
    expect(pw_solve(c, PW_FP32C) == PW_OK, "fp32c");  // split: more than that
    expect(pw_solve(c, PW_FP64) == PW_OK, "fp64 again");
    expect(pw_step(c, PW_RK4, 1e-3, PW_FP32C, 1) == PW_OK, "fp32c step");
    expect(pw_step(c, PW_RK4, 1e-3, PW_FP64, 1) == PW_OK, "fp64 step");
    pw_destroy(c);
  }
  // a number of parts that was asked for and does not fit is an error, and
  // leaves the other precision a launch that has its rows
  pw_ctx* c = context({60000});
  g_device_limit = std::numeric_limits<size_t>::max();
  expect(pw_set_pair_config(c, PW_FP64, 16, 1, 0) == PW_OK, "16 parts");
  expect(pw_set_pair_config(c, PW_FP32C, 256, 1, 0) == PW_OK, "256 parts");
  expect(pw_solve(c, PW_FP64) == PW_OK, "fp64 in 16 parts");
  g_device_limit = g_device_used + (size_t(64) << 20);
  expect(pw_solve(c, PW_FP32C) == PW_ERR_NOMEM, "256 parts do not fit");
  expect(pw_solve(c, PW_FP32C) == PW_ERR_NOMEM, "nor the second time");
  expect(pw_solve(c, PW_FP64) == PW_OK, "fp64 in 16 parts again");
  pw_destroy(c);
}

// Wake blocks of the diagnostics: at most 131,072 items whatever the sizes, at
// most 64 targets each, which together cover the block.
void diagnose_items() {
  const std::vector<std::vector<int64_t>> sizes = {{500000, 500000}, {1100000, 900000}, {65, 70000}, {70000, 65}, {1, 1}};
  for (const auto& n : sizes) {
    pw_ctx* c = context(n);
    double out[16];
    expect(pw_diagnose_wakes(c, 0, 1, out, 16) == PW_OK, "cross block");
    expect(g_diag.size() <= 131072, "items of a cross block: " + std::to_string(g_diag.size()));
    double pairs = 0.0;
    for (const auto& it : g_diag) {
      expect(it.nself == 1 && it.t0 >= 0 && it.t1 <= n[0] && it.s0 >= n[0] && it.s1 <= n[0] + n[1] && it.t0 < it.t1 &&
                 it.t1 - it.t0 <= 64 && it.s0 < it.s1,
             "an item of a cross block");
      pairs += static_cast<double>(it.t1 - it.t0) * static_cast<double>(it.s1 - it.s0);
    }
    const double all = static_cast<double>(n[0]) * static_cast<double>(n[1]);
    expect(pairs == all, "a cross block is covered");
    expect(out[9] == 2.0 * all, "the sum of a cross block");
    expect(pw_diagnose_wakes(c, 1, 1, out, 16) == PW_OK && g_diag.size() <= 131072, "a wake's own block");
    for (const auto& it : g_diag) expect(it.nself == 0 && it.s0 >= n[0] && it.s1 <= it.t1, "an item of a wake");
    pw_destroy(c);
  }
}

// With little pinned memory to be had, transfers go in smaller pieces and the
// training samples straight from the caller's memory.
void little_pinned_memory() {
  g_pinned_limit = 100000;  // 2,083 particles
  const std::vector<int64_t> n = {30000, 7, 4001};
  pw_ctx* c = context(n, false);
  expect(pw_diagnose_wakes(c, 1, 1, std::vector<double>(16).data(), 16) == PW_OK, "build");
  const int64_t all = 30000 + 7 + 4001;
  std::vector<double> x(3 * all), a(3 * all);
  const auto is = [&](const std::vector<double>& v, int64_t from, int64_t m, double sign, double shift) {
    for (int64_t i = 0; i < m; ++i)
      if (v[i] != sign * (from + i) + shift) return false;
    return true;
  };
  expect(pw_get_all_state(c, x.data(), a.data()) == PW_OK, "all state");
  expect(is(x, 0, 3 * all, 1.0, 0.0) && is(a, 0, 3 * all, -1.0, -0.5), "the state of all wakes");
  expect(pw_get_wake_state(c, 2, x.data(), a.data()) == PW_OK, "a wake's state");
  expect(is(x, 3 * 30007, 3 * 4001, 1.0, 0.0) && is(a, 3 * 30007, 3 * 4001, -1.0, -0.5), "the state of a wake");
  std::vector<double> x0(3 * 30000), a0(3 * 30000);
  for (size_t i = 0; i < x0.size(); ++i) {
    x0[i] = i + 0.25;
    a0[i] = 2.0 - i;
  }
  expect(pw_set_wake_state(c, 0, x0.data(), a0.data()) == PW_OK, "set a wake's state");
  expect(pw_get_all_state(c, x.data(), a.data()) == PW_OK, "all state");
  expect(is(x, 0, 3 * 30000, 1.0, 0.25) && is(a, 0, 3 * 30000, -1.0, 2.0), "the state that was set");
  expect(pw_get_all_rates(c, x.data(), a.data()) == PW_OK, "all rates");
  const int64_t batch = 5000;  // 560 kB of samples
  std::vector<float> w(pw::kMlpParams, 0.5f), X(16 * batch, 1.0f), Y(12 * batch, 2.0f), grad(pw::kMlpParams);
  double loss = 0.0;
  expect(pw_ff_set_weights(c, w.data(), pw::kMlpParams) == PW_OK, "weights");
  expect(pw_ff_mlp_grad(c, X.data(), Y.data(), batch, grad.data(), &loss) == PW_OK, "gradient");
  expect(grad[0] == 16.0f * batch && grad[pw::kMlpParams - 1] == 16.0f * batch && loss == 24.0f * batch,
         "the gradient's result");
  pw_destroy(c);
  expect(g_pinned.empty() && g_device.empty(), "everything is given back");
  g_pinned_limit = std::numeric_limits<size_t>::max();
}

// The pair timing holds the sum of the partial rates, where there are any.
void timed_launches() {
  using Calls = std::vector<std::string>;
  const Calls summed = {"event", "pair", "finish", "event"}, whole = {"event", "pair", "event", "finish"};
  pw_ctx* c = context({5000});
  expect(pw_set_profiling(c, 1) == PW_OK, "profiling");
  const auto solve = [&](int precision, const Calls& order, const char* what) {
    g_calls.clear();
    expect(pw_solve(c, precision) == PW_OK && g_calls == order, what);
  };
  solve(PW_FP64, summed, "the default launch of a small system");
  expect(pw_set_pair_config(c, PW_FP32C, 8, 1, 0) == PW_OK, "8 parts");
  solve(PW_FP32C, summed, "8 parts");
  solve(PW_FP64_REF, whole, "one part");
  expect(pw_set_pair_config(c, PW_FP32C, 1, 1, 0) == PW_OK, "1 part");
  solve(PW_FP32C, whole, "one part, persistent");
  double ms = 0.0;
  int64_t launches = 0;
  expect(pw_get_pair_timing(c, &ms, &launches) == PW_OK && launches == 4 && ms == 4.0, "totals");
  pw_destroy(c);
}

// Every launch's items name the chunks that hold their sources (and targets).
void item_chunks() {
  const std::vector<std::vector<int64_t>> sizes = {{1}, {64}, {65}, {1000}, {5000, 0, 777}, {63, 64, 65, 300, 1, 9001}, {41000}, {70001, 3}};
  for (const auto& n : sizes)
    for (const bool coupled : {false, true}) {
      pw_ctx* c = context(n, coupled);
      for (const int precision : {PW_FP64, PW_FP32C, PW_FP64_REF}) {
        expect(pw_solve(c, precision) == PW_OK, "the default launch");
        for (const int parts : {1, 2, 7}) {
          expect(pw_set_pair_config(c, precision, parts, 1, PW_VARIANT_SCALAR_FEED) == PW_OK, "parts");
          expect(pw_solve(c, precision) == PW_OK, "a launch in parts");
        }
      }
      pw_destroy(c);
    }
}

// The reference's state and rate vectors (per wake maxn rows twice) pass in one
// launch whatever the number of wakes, or one per piece of the staging.
void state_vectors() {
  for (const size_t pinned : {std::numeric_limits<size_t>::max(), size_t(30000)}) {
    g_pinned_limit = pinned;  // 625 particles a piece
    pw_ctx* c = nullptr;
    expect(pw_create(&c, 0) == PW_OK && pw_set_coupled(c, 0) == PW_OK, "create");
    const int wakes = 500;
    std::vector<int64_t> n(wakes), maxn(wakes);
    std::vector<double> state;
    int64_t all = 0;
    for (int w = 0; w < wakes; ++w) {
      n[w] = w % 7 == 3 ? 0 : 1 + w % 13;
      maxn[w] = n[w] + w % 3;
      all += n[w];
      std::vector<double> x(3 * n[w] + 1, 0.0), r(n[w] + 1, 0.1), v(n[w] + 1, 1.0);
      expect(pw_add_wake(c, n[w], maxn[w], x.data(), x.data(), r.data(), v.data(), nullptr) == PW_OK, "add_wake");
      for (int64_t i = 0; i < 6 * maxn[w]; ++i) state.push_back(i % (3 * maxn[w]) < 3 * n[w] ? 1.0 + state.size() : 0.0);
    }
    std::vector<double> out16(16), back(state.size(), -1.0);
    expect(pw_diagnose_wakes(c, 0, 0, out16.data(), 16) == PW_OK, "build");
    const size_t pieces = pinned < 40000 ? (all + 299) / 300 + 1 : 1;
    const int64_t len = static_cast<int64_t>(state.size());
    const auto calls = [&](const char* what) {
      expect(g_calls.size() <= pieces, std::string(what) + ": " + std::to_string(g_calls.size()) + " launches");
      g_calls.clear();
    };
    g_calls.clear();
    expect(pw_set_states(c, state.data(), len) == PW_OK, "set_states");
    calls("set_states");
    expect(pw_get_states(c, back.data(), len) == PW_OK && back == state, "get_states returns what was set");
    calls("get_states");
    for (int64_t i = 0; i < all; ++i) {
      std::memcpy(&c->rates[i].ux, &c->y[i].x, 24);
      std::memcpy(&c->rates[i].wx, &c->y[i].ax, 24);
    }
    std::fill(back.begin(), back.end(), -1.0);
    expect(pw_get_rates(c, back.data(), len) == PW_OK && back == state, "get_rates");
    calls("get_rates");
    pw_destroy(c);
  }
  g_pinned_limit = std::numeric_limits<size_t>::max();
}

}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> checks = {{"partial_buffer", partial_buffer},
                                                      {"diagnose_items", diagnose_items},
                                                      {"little_pinned_memory", little_pinned_memory},
                                                      {"timed_launches", timed_launches},
                                                      {"item_chunks", item_chunks},
                                                      {"state_vectors", state_vectors}};
  if (argc != 2 || !checks.count(argv[1])) {
    std::fprintf(stderr, "usage: host_logic CHECK\n");
    return 2;
  }
  checks.at(argv[1])();
  if (g_failures) std::printf("last error: %s\n", pw_last_error());
  std::printf("%s: %d failures\n", argv[1], g_failures);
  return g_failures ? 1 : 0;
}
