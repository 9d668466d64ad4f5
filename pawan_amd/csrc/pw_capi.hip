// pw_capi.hip -- solver context and the extern "C" entry points declared in
// include/pawan_gpu.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <tuple>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "pw_ctx.h"

using pw::Rate64;
using pw::Rec64;
using pw::WorkItem;
using pwi::dalloc;
using pwi::fail;
using pwi::kKindLearned;
using pwi::kTargetsPerItem;

namespace pwi {

namespace {
thread_local std::string g_error;
}  // namespace

int fail(int code, const std::string& msg) {
  g_error = msg;
  return code;
}

}  // namespace pwi

// Staging of pw_velocity_at_noalloc: the points, then their velocities, for
// at most kNoAllocPoints points (3 MiB).  Every GPU the library runs on holds
// its own copy until the process ends; host code reaches it only through the
// per-device address that hipGetSymbolAddress gives (noalloc_staging).
constexpr int64_t kNoAllocPoints = 65536;
static __device__ __align__(256) double scratch[2 * 3 * kNoAllocPoints];

namespace {

// Device address of scratch on each device, resolved by pw_create with the
// device current, once per device.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

int resolve_noalloc_staging(int device) {
  if (device < 0 || device >= kMaxDevices) return fail(PW_ERR_UNSUPPORTED, "device index beyond 63");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return PW_OK;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p)
    return fail(PW_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_scratch_ptr[device] = static_cast<double*>(p);
  return PW_OK;
}

double* noalloc_staging(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_ptr[device];
}

// Device buffers of the context.  Captured step graphs hold kernel nodes
// whose arguments point into these buffers, so they are destroyed first,
// after the stream has drained.
void free_buffers(pw_ctx* c) {
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto& g : c->graphs) (void)hipGraphExecDestroy(g.second);
  c->graphs.clear();
  (void)hipFree(c->y);
  (void)hipFree(c->ys);
  for (auto& p : c->k) (void)hipFree(p);
  (void)hipFree(c->d_radius);
  (void)hipFree(c->pair_items);
  (void)hipFree(c->lin_items);
  (void)hipFree(c->d_lin);
  (void)hipFree(c->d_quad);
  (void)hipFree(c->diag_items);
  (void)hipFree(c->d_diag_first);
  c->diag_items = nullptr;
  c->d_diag_first = nullptr;
  c->ndiag = 0;
  (void)hipHostFree(c->h_flag);
  (void)hipHostFree(c->h_stage);
  c->h_flag = nullptr;
  c->h_stage = nullptr;
  c->stage_particles = 0;
  for (auto& k : c->ks) {
    (void)hipFree(k.d_items);
    (void)hipFree(k.d_groups);
  }
  (void)hipFree(c->partial);
  (void)hipFree(c->d_queue);
  (void)hipFree(c->d_points);
  c->d_points = nullptr;
  c->points_len = 0;
  (void)hipFree(c->d_chunks);
  (void)hipFree(c->d_src32);
  (void)hipFree(c->d_src64);
  c->d_chunks = nullptr;
  c->d_src32 = nullptr;
  c->d_src64 = nullptr;
  c->y = c->ys = nullptr;
  for (auto& p : c->k) p = nullptr;
  c->rates = nullptr;
  c->d_radius = nullptr;
  c->pair_items = c->lin_items = nullptr;
  c->d_lin = c->d_quad = nullptr;
  c->d_queue = nullptr;
  for (auto& k : c->ks) {
    k.d_items = nullptr;
    k.d_groups = nullptr;
    k.nitems = k.ngroups = 0;
    k.built_parts = k.built_split = 0;
    k.rows = 0;
    k.lean = false;
  }
  c->partial = nullptr;
  c->partial_rows = 0;
  pwi::ff_release(c);
}

// Everything the context holds on the device: buffers, events, stream.
void release(pw_ctx* c) {
  free_buffers(c);
  for (auto& e : c->ev_used) {
    (void)hipEventDestroy(e.first);
    (void)hipEventDestroy(e.second);
  }
  for (auto& e : c->ev_free) {
    (void)hipEventDestroy(e.first);
    (void)hipEventDestroy(e.second);
  }
  if (c->stream) (void)hipStreamDestroy(c->stream);
}

// index of the source chunk holding particle s (chunk_first is ascending)
int32_t chunk_of(const pw_ctx* c, int64_t s) {
  const auto it = std::upper_bound(c->chunk_first.begin(), c->chunk_first.end(), static_cast<int32_t>(s));
  return static_cast<int32_t>(it - c->chunk_first.begin()) - 1;
}

// Work items: blocks of up to 256 consecutive targets of one system, each
// against all sources of that system.  For independent wakes the largest
// systems come first (longest-processing-time order), so the tail of the
// grid is made of short blocks.
void build_items(pw_ctx* c) {
  c->h_pair_items.clear();
  c->h_lin_items.clear();
  c->lin_wake.clear();
  const int nw = static_cast<int>(c->wn.size());
  // source chunks of the scalar-fed and split kernels: runs of up to 64
  // particles of one system, in particle order
  c->systems.clear();
  c->chunk_first.clear();
  const auto add_system = [&](int64_t a, int64_t b, int id) {
    c->systems.push_back({a, b, id, static_cast<int32_t>(c->chunk_first.size())});
    for (int64_t i = a; i < b; i += 64) c->chunk_first.push_back(static_cast<int32_t>(i));
  };
  if (c->coupled)
    add_system(0, c->n, 0);
  else
    for (int w = 0; w < nw; ++w) add_system(c->woff[w], c->woff[w + 1], w);
  c->nchunks = static_cast<int>(c->chunk_first.size());
  std::stable_sort(c->systems.begin(), c->systems.end(),
                   [](const pw_ctx::SysRange& p, const pw_ctx::SysRange& q) { return (p.b - p.a) > (q.b - q.a); });
  for (const auto& s : c->systems)
    for (int64_t t0 = s.a; t0 < s.b; t0 += kTargetsPerItem) {
      c->h_pair_items.push_back({static_cast<int32_t>(t0),
                                 static_cast<int32_t>(std::min<int64_t>(t0 + kTargetsPerItem, s.b)),
                                 static_cast<int32_t>(s.a), static_cast<int32_t>(s.b), -1, 0, s.chunk, 0});
    }
  for (int w = 0; w < nw; ++w)
    for (int64_t t0 = c->woff[w]; t0 < c->woff[w + 1]; t0 += kTargetsPerItem) {
      c->h_lin_items.push_back(
          {static_cast<int32_t>(t0),
           static_cast<int32_t>(std::min<int64_t>(t0 + kTargetsPerItem, c->woff[w + 1])), w, 0,
           0, 0, 0, 0});
      c->lin_wake.push_back(w);
    }
  c->npair = static_cast<int>(c->h_pair_items.size());
  c->nlin = static_cast<int>(c->h_lin_items.size());
}

int ensure_built(pw_ctx* c) {
  if (c->built) return PW_OK;
  if (c->n <= 0) return fail(PW_ERR_STATE, "context has no particles (add a wake first)");
  if (c->n > INT32_MAX / 2) return fail(PW_ERR_UNSUPPORTED, "too many particles");
  PW_HIP(hipSetDevice(c->device));
  build_items(c);
  const size_t n = static_cast<size_t>(c->n);
  if (dalloc(&c->y, n) != hipSuccess || dalloc(&c->ys, n) != hipSuccess ||
      dalloc(&c->k[0], n) != hipSuccess || dalloc(&c->k[1], std::max<size_t>(n, pw::kPointScratchRows)) != hipSuccess ||
      dalloc(&c->k[2], n) != hipSuccess || dalloc(&c->k[3], n) != hipSuccess ||
      dalloc(&c->d_radius, n) != hipSuccess ||
      dalloc(&c->pair_items, c->h_pair_items.size()) != hipSuccess ||
      dalloc(&c->lin_items, c->h_lin_items.size()) != hipSuccess ||
      dalloc(&c->d_lin, 11 * c->h_lin_items.size()) != hipSuccess ||
      hipHostMalloc(reinterpret_cast<void**>(&c->h_flag), sizeof(int), hipHostMallocCoherent) != hipSuccess ||
      dalloc(&c->d_queue, 1) != hipSuccess ||
      dalloc(&c->d_chunks, static_cast<size_t>(c->nchunks)) != hipSuccess ||
      dalloc(&c->d_src32, n) != hipSuccess) {
    free_buffers(c);  // the stream stays: the context remains usable
    (void)hipGetLastError();
    return fail(PW_ERR_NOMEM, "device allocation failed");
  }
  PW_HIP(hipMemcpyAsync(c->y, c->pending.data(), n * sizeof(Rec64), hipMemcpyHostToDevice,
                        c->stream));
  PW_HIP(hipMemcpyAsync(c->d_radius, c->radius.data(), n * sizeof(double),
                        hipMemcpyHostToDevice, c->stream));
  PW_HIP(hipMemcpyAsync(c->pair_items, c->h_pair_items.data(),
                        c->h_pair_items.size() * sizeof(WorkItem), hipMemcpyHostToDevice,
                        c->stream));
  {
    // chunk extents now; their spheres are rebuilt before every launch
    std::vector<pw::Chunk32> ch(static_cast<size_t>(c->nchunks));
    for (int k = 0; k < c->nchunks; ++k) {
      std::memset(&ch[k], 0, sizeof(pw::Chunk32));
      ch[k].first = c->chunk_first[k];
      const int64_t end = k + 1 < c->nchunks ? c->chunk_first[k + 1] : c->n;
      ch[k].count = static_cast<int32_t>(std::min<int64_t>(64, end - c->chunk_first[k]));
    }
    PW_HIP(hipMemcpy(c->d_chunks, ch.data(), ch.size() * sizeof(pw::Chunk32), hipMemcpyHostToDevice));
  }
  PW_HIP(hipMemcpyAsync(c->lin_items, c->h_lin_items.data(),
                        c->h_lin_items.size() * sizeof(WorkItem), hipMemcpyHostToDevice,
                        c->stream));
  // rates start at zero (a calloc'd rate vector in the reference)
  PW_HIP(pw::launch_zero_doubles(reinterpret_cast<double*>(c->k[0]), 6 * c->n, c->stream));
  PW_HIP(hipStreamSynchronize(c->stream));
  c->rates = c->k[0];
  c->zc.assign(c->nsys(), 0.0);
  {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, c->device) == hipSuccess && prop.multiProcessorCount > 0)
      c->num_cus = prop.multiProcessorCount;
  }
  c->pending.clear();
  c->pending.shrink_to_fit();
  c->built = true;
  return PW_OK;
}

int kind_of(int precision, int* kind) {
  switch (precision) {
    case PW_FP64: *kind = pw::kPairFP64; return PW_OK;
    case PW_FP64_REF: *kind = pw::kPairFP64Exact; return PW_OK;
    case PW_FP32C: *kind = pw::kPairFP32C; return PW_OK;
    case PW_LEARNED: *kind = kKindLearned; return PW_OK;
    default:
      return fail(PW_ERR_ARG, "unknown precision " + std::to_string(precision));
  }
}

// Work items for a launch split into `parts` source ranges per target
// block (parts == 1: one item per block writing its rates directly).
// Split points fall on tile boundaries of the block's system, so the
// diagonal tile (and its self pairs) stays inside one part.  Items are
// ordered by cost, largest first, and among equal costs part by part: the
// items in flight at any time then read one source range, which the L2 of
// every XCD holds (a part of a 1M-particle wake split 16 ways is 3 MB of
// FP32 source records), instead of every range at once.
std::vector<WorkItem> make_items(const pw_ctx* c, int parts) {
  std::vector<WorkItem> items;
  items.reserve(c->h_pair_items.size() * static_cast<size_t>(parts));
  for (const auto& s : c->systems) {
    const int64_t ntile = (s.b - s.a + kTargetsPerItem - 1) / kTargetsPerItem;
    for (int p = 0; p < parts; ++p) {
      const int64_t a = s.a + kTargetsPerItem * (ntile * p / parts);
      const int64_t b = std::min<int64_t>(s.b, s.a + kTargetsPerItem * (ntile * (p + 1) / parts));
      for (int64_t t0 = s.a; t0 < s.b; t0 += kTargetsPerItem) {
        const int32_t t1 = static_cast<int32_t>(std::min<int64_t>(t0 + kTargetsPerItem, s.b));
        items.push_back({static_cast<int32_t>(t0), t1, static_cast<int32_t>(a),
                         static_cast<int32_t>(std::max(a, b)), parts == 1 ? -1 : p, 0,
                         s.chunk + static_cast<int32_t>((a - s.a) / 64), 0});
      }
    }
  }
  std::stable_sort(items.begin(), items.end(), [](const WorkItem& x, const WorkItem& y) {
    return int64_t(x.s1 - x.s0) * (x.t1 - x.t0) > int64_t(y.s1 - y.s0) * (y.t1 - y.t0);
  });
  return items;
}

// Captured steps are replayed only while nothing they were captured with
// has changed; the stream drains first, so no replay is in flight.
void drop_graphs(pw_ctx* c) {
  if (c->graphs.empty()) return;
  (void)hipStreamSynchronize(c->stream);
  for (auto& g : c->graphs) (void)hipGraphExecDestroy(g.second);
  c->graphs.clear();
}

// the pair-kernel kind a precision launches under the context's kernel and
// summation settings
int launch_kind_of(const pw_ctx* c, int kind) {
  if (c->smoothing == PW_KERNEL_HIGHORDER) return kind == pw::kPairFP32C ? pw::kPairFP32CHO : pw::kPairFP64HO;
  if (kind == pw::kPairFP32C && !c->compensated) return pw::kPairFP32CPlain;
  return kind;
}

bool is_default(const pw::PairConfig& p) {
  return p.parts == 1 && !p.persistent && !p.waves8 && !p.scalar_feed && !p.two_per_lane && p.split == 0;
}

int64_t split_items(const pw_ctx* c, int split) {
  int64_t items = 0;
  for (const auto& s : c->systems) items += ((s.b - s.a + 63) / 64) * ((s.b - s.a + split - 1) / split);
  return items;
}

// Items and groups of a split launch: every system's targets in groups of 64,
// each against source ranges of `split` particles, items group by group.  Built
// on the first launch, so counted first and without a search per item (48 rings
// of 512-16,384, 105,000 items: 2.3 -> 0.12 ms).
void make_split(const pw_ctx* c, int split, std::vector<WorkItem>& items, std::vector<pw::SplitGroup>& groups) {
  items.reserve(static_cast<size_t>(split_items(c, split)));
  for (const auto& s : c->systems)
    for (int64_t t0 = s.a; t0 < s.b; t0 += 64) {
      const int32_t t1 = static_cast<int32_t>(std::min<int64_t>(t0 + 64, s.b));
      pw::SplitGroup g{static_cast<int32_t>(t0), t1, static_cast<int32_t>(items.size()), 0};
      for (int64_t a = s.a; a < s.b; a += split, ++g.count)
        items.push_back({static_cast<int32_t>(t0), t1, static_cast<int32_t>(a),
                         static_cast<int32_t>(std::min<int64_t>(a + split, s.b)),
                         static_cast<int32_t>(items.size()), 0,
                         s.chunk + static_cast<int32_t>((a - s.a) / 64), s.chunk + static_cast<int32_t>((t0 - s.a) / 64)});
      groups.push_back(g);
    }
}

// The launch of a kind whose configuration is the default (one part, grid, LDS
// tiles, as set by nobody or set again).  Two launches cover the sizes; times
// are one right-hand side in microseconds, leapfrogging rings or helix:
//
// * The split kernel while the largest system has at most kSplitUpTo*
//   particles.  Its source ranges are the longest of 64, 128 and 256 that
//   leave kSplitItems items, ten blocks per CU: shorter ones add partial sums
//   (N = 10,000 FP64: 247 at 64, 238 at 128, 248 at 256, 301 at 1,024), longer
//   ones leave the chip idle (N = 1,000: 15.7 at 64, 21 at 128, 96 at 1,024,
//   347 in one part).  Where that is 64 and half of it leaves no more than
//   kSplitItemsFew items, the chain of a wave is what is left to cut: 32 and
//   16 (N = 1,000: 14.3 at 32, 17.0 at 16; N = 400: 14.5 at 64, 11.5, 10.0;
//   N = 2,000: 23.9 at 64, 27.8 at 32).  Beyond kSplitItemsMax items (403 MB
//   of partial rates) the ranges double.  From kSplitSepItems items of whole
//   256-source tiles, the 64-particle chunks' spheres are formed first (one
//   launch, about 5 us) and chunks separated from an item's targets take the
//   separated sums: two rings of 32,000 FP64 2,100 -> 1,825, FP32C 947 -> 757;
//   48 rings of 512-16,384 FP64 4,158 -> 3,650, FP32C 1,807 -> 1,485; helix
//   16,384 FP64 563 -> 534, FP32C 265 -> 257; at 6,400 items a coarse helix,
//   which separates little, is still up to 4% slower with them.
// * Beyond, the scalar-fed kernels, one persistent wave per 64 targets, over 64
//   source parts (32 from 196,608 particles: there 32 are 3% faster in FP64 and
//   level in FP32C at half the partial rates).  Split against scalar-fed, rings
//   and helix: FP64 32,000 1,825 and 1,997 against 2,059 and 2,007, 48,000
//   3,945 and 4,090 against 4,324 and 3,995, 64,000 7,465 and 6,632 against
//   7,370 and 6,596; FP32C 64,000 2,862 and 3,087 against 3,393 and 3,267,
//   96,000 7,232 and 6,940 against 7,155 and 6,627.  The high-order FP64 kernel
//   has no scalar-fed form: split at every size (131,072: 33.8 ms against 34.7
//   LDS-tiled in 16 parts, 39.7 in one).
//
// Systems of a batch are far below these sizes: split wins there by the same
// rule (48 rings of 512-16,384, FP64 3.65 ms against 5.4 over 64 parts).
constexpr int64_t kSplitUpTo64 = 40960, kSplitUpTo32 = 65536;
constexpr int64_t kSplitItems = 2560, kSplitItemsFew = 640, kSplitItemsMax = 131072, kSplitSepItems = 8192;

pw::PairConfig auto_config(const pw_ctx* c, int launch_kind) {
  pw::PairConfig p;
  const bool f32 = launch_kind == pw::kPairFP32C || launch_kind == pw::kPairFP32CHO;
  if (!f32 && launch_kind != pw::kPairFP64 && launch_kind != pw::kPairFP64HO) return p;
  const int64_t largest = c->systems.empty() ? 0 : c->systems.front().b - c->systems.front().a;
  if (launch_kind == pw::kPairFP64HO || largest <= (f32 ? kSplitUpTo32 : kSplitUpTo64)) {
    p.split = 64;
    while (p.split < 256 && split_items(c, 2 * p.split) >= kSplitItems) p.split *= 2;
    while (p.split > 16 && p.split <= 64 && split_items(c, p.split / 2) <= kSplitItemsFew) p.split /= 2;
    while (split_items(c, p.split) > kSplitItemsMax && p.split < largest) p.split *= 2;
    p.split_sep = launch_kind != pw::kPairFP64HO && p.split >= 256 && split_items(c, p.split) >= kSplitSepItems;
    return p;
  }
  p.parts = c->n < 196608 ? 64 : 32;
  p.persistent = true;
  p.waves8 = f32;
  p.scalar_feed = true;
  return p;
}

// The buffer is shared by all kinds and freed before a larger one is tried (both
// need not fit at once): when that fails there is none, and a kind built earlier
// is built again before its next launch (ensure_kind compares its rows).
int ensure_partial(pw_ctx* c, size_t rows) {
  if (rows <= c->partial_rows) return PW_OK;
  (void)hipFree(c->partial);
  c->partial = nullptr;
  c->partial_rows = 0;
  if (dalloc(&c->partial, rows) != hipSuccess) {
    (void)hipGetLastError();
    return fail(PW_ERR_NOMEM, "partial-sum buffer");
  }
  c->partial_rows = rows;
  return PW_OK;
}

// Work items of cfg on the device, and the partial buffer they need.
int build_kind(pw_ctx* c, int kind, const pw::PairConfig& cfg) {
  auto& k = c->ks[kind];
  std::vector<WorkItem> items;
  std::vector<pw::SplitGroup> groups;
  if (cfg.split > 0) make_split(c, cfg.split, items, groups);
  else items = make_items(c, cfg.parts);
  PW_HIP(hipStreamSynchronize(c->stream));
  drop_graphs(c);  // captured steps point at the buffers replaced here
  (void)hipFree(k.d_items);
  (void)hipFree(k.d_groups);
  k.d_items = nullptr;
  k.d_groups = nullptr;
  k.built_parts = k.built_split = 0;
  k.rows = 0;
  if (dalloc(&k.d_items, items.size()) != hipSuccess ||
      (!groups.empty() && dalloc(&k.d_groups, groups.size()) != hipSuccess)) {
    (void)hipGetLastError();
    return fail(PW_ERR_NOMEM, "work items");
  }
  PW_HIP(hipMemcpy(k.d_items, items.data(), items.size() * sizeof(WorkItem), hipMemcpyHostToDevice));
  if (!groups.empty())
    PW_HIP(hipMemcpy(k.d_groups, groups.data(), groups.size() * sizeof(pw::SplitGroup), hipMemcpyHostToDevice));
  const size_t rows =
      cfg.split > 0 ? 64 * items.size() : cfg.parts > 1 ? static_cast<size_t>(cfg.parts) * static_cast<size_t>(c->n) : 0;
  PW_TRY(ensure_partial(c, rows));
  k.rows = rows;
  k.nitems = static_cast<int>(items.size());
  k.ngroups = static_cast<int>(groups.size());
  k.built_parts = cfg.parts;
  k.built_split = cfg.split;
  return PW_OK;
}

int ensure_kind(pw_ctx* c, int kind) {
  if (kind == kKindLearned) return PW_OK;  // the tree path sets itself up
  auto& k = c->ks[kind];
  const bool chosen = is_default(k.cfg) && !k.lean;
  k.run = chosen ? auto_config(c, launch_kind_of(c, kind)) : k.cfg;
  for (;;) {
    // the scalar-fed FP64 kernel's source records, allocated before any
    // step is captured (no allocation may happen inside a capture)
    int rc = PW_OK;
    if ((k.run.scalar_feed || k.run.split_sep) && kind == pw::kPairFP64 && !c->d_src64 &&
        dalloc(&c->d_src64, c->n) != hipSuccess) {
      (void)hipGetLastError();
      rc = fail(PW_ERR_NOMEM, "scalar-fed FP64 source records");
    }
    // (the rows too: another kind's larger buffer may have replaced them by none)
    if (rc == PW_OK && k.d_items && k.built_parts == k.run.parts && k.built_split == k.run.split &&
        c->partial_rows >= k.rows)
      return PW_OK;
    if (rc == PW_OK) rc = build_kind(c, kind, k.run);
    // a launch chosen here that does not fit in memory: the one that needs none
    if (rc != PW_ERR_NOMEM || !chosen || is_default(k.run)) return rc;
    k.run = pw::PairConfig{};
    k.lean = true;
  }
}

// Blocks of wake pairs for the per-wake hooks: pairs (a, b) with a <= b,
// a == b the self pairs of wake a, a < b the cross pairs of a and b.
int check_blocks(const pw_ctx* c, const int* pairs, int npairs) {
  if (npairs < 0 || (npairs > 0 && !pairs)) return fail(PW_ERR_ARG, "null or negative wake-pair list");
  const int nw = static_cast<int>(c->wn.size());
  for (int k = 0; k < npairs; ++k) {
    const int a = pairs[2 * k], b = pairs[2 * k + 1];
    if (a < 0 || b < a || b >= nw) return fail(PW_ERR_ARG, "wake pairs need 0 <= a <= b < wakes");
    if (a != b && !c->coupled) return fail(PW_ERR_STATE, "cross-wake pairs need a coupled context");
  }
  return PW_OK;
}

// targets of wake a (256 at a time) against the sources of wake b
void append_items(const pw_ctx* c, int a, int b, int nself, std::vector<WorkItem>& out) {
  for (int64_t t0 = c->woff[a]; t0 < c->woff[a + 1]; t0 += kTargetsPerItem)
    out.push_back({static_cast<int32_t>(t0), static_cast<int32_t>(std::min<int64_t>(t0 + kTargetsPerItem, c->woff[a + 1])),
                   static_cast<int32_t>(c->woff[b]), static_cast<int32_t>(c->woff[b + 1]), -1, nself,
                   chunk_of(c, c->woff[b]), 0});
}

// Source range of the diagnostics' pair items, count(range) of them: the longest
// of 64 ... 1,024 particles that leaves ten blocks per CU (short ranges cost the
// staging of a block's tiles and table per few pairs), longer where the items
// would exceed 131,072.
template <typename Count>
int diag_range(const Count& count) {
  int range = 64;
  while (range < 1024 && count(2 * range) >= 2560) range *= 2;
  while (range < (1 << 28) && count(range) > 131072) range *= 2;
  return range;
}

// over the unordered pairs of `systems` ([a, b) each)
int diag_range(const std::vector<std::pair<int64_t, int64_t>>& systems) {
  return diag_range([&](int64_t range) {
    int64_t items = 0;
    for (const auto& s : systems) {
      const int64_t len = s.second - s.first;
      items += (len + 63) / 64 * ((len + range - 1) / range + 1) / 2;
    }
    return items;
  });
}

// over na x nb pairs of two wakes
int diag_range(int64_t na, int64_t nb) {
  return diag_range([=](int64_t range) { return (na + 63) / 64 * ((nb + range - 1) / range); });
}

// pair items of one system's unordered pairs
void append_diag_items(int64_t a, int64_t b, int range, std::vector<WorkItem>& out) {
  for (int64_t t0 = a; t0 < b; t0 += 64) {
    const int64_t t1 = std::min<int64_t>(t0 + 64, b);
    for (int64_t s0 = a; s0 < t1; s0 += range)
      out.push_back({static_cast<int32_t>(t0), static_cast<int32_t>(t1), static_cast<int32_t>(s0),
                     static_cast<int32_t>(std::min<int64_t>(s0 + range, t1)), -1, 0, 0, 0});
  }
}

int ensure_diag(pw_ctx* c) {
  if (c->diag_items) return PW_OK;
  // systems in their own order (c->systems is sorted by size)
  std::vector<std::pair<int64_t, int64_t>> sys(c->nsys());
  for (const auto& s : c->systems) sys[s.id] = {s.a, s.b};
  std::vector<WorkItem> items;
  std::vector<int> first{0};
  const int range = diag_range(sys);
  for (const auto& s : sys) {
    append_diag_items(s.first, s.second, range, items);
    first.push_back(static_cast<int>(items.size()));
  }
  // each item's sums, then each system's
  const size_t rows = items.size() + sys.size();
  if (dalloc(&c->diag_items, items.size()) != hipSuccess || dalloc(&c->d_diag_first, first.size()) != hipSuccess ||
      dalloc(&c->d_quad, pw::kDiagQuad * rows) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipFree(c->diag_items);
    (void)hipFree(c->d_diag_first);
    c->diag_items = nullptr;
    c->d_diag_first = nullptr;
    return fail(PW_ERR_NOMEM, "diagnostic buffers");
  }
  PW_HIP(hipMemcpy(c->diag_items, items.data(), items.size() * sizeof(WorkItem), hipMemcpyHostToDevice));
  PW_HIP(hipMemcpy(c->d_diag_first, first.data(), first.size() * sizeof(int), hipMemcpyHostToDevice));
  c->ndiag = static_cast<int>(items.size());
  return PW_OK;
}

// One right-hand side f(state) -> out, with optional event timing, and the
// stage arithmetic that follows it.
int rhs(pw_ctx* c, int kind, const Rec64* state, Rate64* out, const pw::StageOp& op = pw::StageOp{}) {
  const int n = static_cast<int>(c->n);
  if (kind == kKindLearned) {
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (c->profiling) {
      PW_TRY(pwi::prof_begin(c, &e0, &e1));
      PW_HIP(hipEventRecord(e0, c->stream));
    }
    PW_TRY(pwi::ff_rhs(c, state, out));
    if (c->profiling) {
      PW_HIP(hipEventRecord(e1, c->stream));
      c->ev_used.emplace_back(e0, e1);
    }
    PW_HIP(pw::launch_finish(pw::SumForm{}, out, n, c->h_flag, op, c->stream));
    return PW_OK;
  }
  if (kind == pw::kPairFP32C && !c->compensated && c->smoothing == PW_KERNEL_GAUSSIAN) {
    // plain FP32 sums: one item per 256-target block over all its sources
    pw::PairArgs args{state, c->pair_items, c->npair, n, out, nullptr, c->d_queue, c->nu,
                      c->d_chunks, c->d_src32, nullptr, c->nchunks};
    PW_HIP(pw::launch_pair(pw::kPairFP32CPlain, pw::PairConfig{}, args, c->npair, c->stream));
    PW_HIP(pw::launch_finish(pw::SumForm{}, out, n, c->h_flag, op, c->stream));
    return PW_OK;
  }
  PW_TRY(ensure_kind(c, kind));
  const auto& k = c->ks[kind];
  pw::PairArgs args;
  args.state = state;
  args.items = k.d_items;
  args.nitems = k.nitems;
  args.n = n;
  args.rates = out;
  args.partial = c->partial;
  args.queue = c->d_queue;
  args.nu = c->nu;
  args.chunks = c->d_chunks;
  args.src = c->d_src32;
  args.src64 = nullptr;
  args.nchunks = c->nchunks;
  // the high-order kernel replaces the Gaussian kinds (pw_set_kernel)
  const int launch_kind = launch_kind_of(c, kind);
  if ((k.run.scalar_feed || k.run.split_sep) && launch_kind == pw::kPairFP64)
    args.src64 = c->d_src64;  // ensure_kind made it
  const int grid = c->num_cus * pw::pair_kernel_waves(launch_kind, k.run);
  pw::SumForm sum;
  sum.partial = c->partial;
  sum.parts = k.run.parts;
  if (k.run.split > 0) {
    sum.groups = k.d_groups;
    sum.ngroups = k.ngroups;
  }
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (c->profiling) {
    PW_TRY(pwi::prof_begin(c, &e0, &e1));
    PW_HIP(hipEventRecord(e0, c->stream));
  }
  PW_HIP(pw::launch_pair(launch_kind, k.run, args, grid, c->stream));
  // the timing holds the sum of the partial rates (and the stage arithmetic that
  // goes with it), but no pass of its own over finished rates
  const bool summed = sum.groups || sum.parts > 1;
  if (c->profiling && !summed) PW_HIP(hipEventRecord(e1, c->stream));
  PW_HIP(pw::launch_finish(sum, out, n, c->h_flag, op, c->stream));
  if (c->profiling) {
    if (summed) PW_HIP(hipEventRecord(e1, c->stream));
    c->ev_used.emplace_back(e0, e1);
  }
  return PW_OK;
}

// The flag is host memory the kernels write: cleared once nothing queued can
// still write it.
int clear_flag(pw_ctx* c) {
  PW_HIP(hipStreamSynchronize(c->stream));
  *static_cast<volatile int*>(c->h_flag) = 0;
  return PW_OK;
}

int check_flag(pw_ctx* c, const char* what) {
  PW_TRY(pwi::ff_check(c));
  PW_HIP(hipStreamSynchronize(c->stream));
  if (*static_cast<volatile int*>(c->h_flag)) return fail(PW_ERR_NONFINITE, std::string(what) + ": non-finite rate (coincident particles?)");
  return PW_OK;
}

int collect_profile(pw_ctx* c) {
  if (c->ev_used.empty()) return PW_OK;
  PW_HIP(hipStreamSynchronize(c->stream));
  for (auto& e : c->ev_used) {
    float ms = 0.0f;
    PW_HIP(hipEventElapsedTime(&ms, e.first, e.second));
    c->prof_ms += ms;
    c->prof_launches += 1;
    c->ev_free.push_back(e);
  }
  c->ev_used.clear();
  return PW_OK;
}

int64_t total_maxsize(const pw_ctx* c) {
  int64_t s = 0;
  for (int64_t m : c->wmax) s += 6 * m;
  return s;
}

int download_state(pw_ctx* c, std::vector<Rec64>& h) {
  h.resize(static_cast<size_t>(c->n));
  if (!c->built) {
    h = c->pending;
    return PW_OK;
  }
  PW_HIP(hipMemcpyAsync(h.data(), c->y, h.size() * sizeof(Rec64), hipMemcpyDeviceToHost,
                        c->stream));
  PW_HIP(hipStreamSynchronize(c->stream));
  return PW_OK;
}

int upload_state(pw_ctx* c, const std::vector<Rec64>& h) {
  if (!c->built) {
    c->pending = h;
    return PW_OK;
  }
  PW_HIP(hipMemcpyAsync(c->y, h.data(), h.size() * sizeof(Rec64), hipMemcpyHostToDevice,
                        c->stream));
  PW_HIP(hipStreamSynchronize(c->stream));
  return PW_OK;
}

// Copies between caller memory and the pinned staging.  A caller's fresh pages
// fault on their first write, which bounds one thread at 5 GB/s (8 threads: 17
// GB/s), so large copies are spread over threads.
struct Segment {
  void* dst;
  const void* src;
  size_t bytes;
};

void copy_range(const std::vector<Segment>& segs, size_t from, size_t to) {
  size_t at = 0;
  for (const Segment& s : segs) {
    const size_t a = std::max(from, at), b = std::min(to, at + s.bytes);
    if (a < b) std::memcpy(static_cast<char*>(s.dst) + (a - at), static_cast<const char*>(s.src) + (a - at), b - a);
    at += s.bytes;
  }
}

void copy_segments(const std::vector<Segment>& segs) {
  size_t total = 0;
  for (const Segment& s : segs) total += s.bytes;
  constexpr size_t kPerThread = size_t(1) << 20;  // a thread costs about what it copies in 30 us
  const size_t nt = std::min<size_t>(8, total / kPerThread);
  if (nt < 2) {
    copy_range(segs, 0, total);
    return;
  }
  const size_t step = (total / nt + 4095) / 4096 * 4096;
  std::vector<std::thread> th;
  size_t done = step;  // this thread takes the first range
  try {
    th.reserve(nt);
    for (; done < total; done += step) th.emplace_back(copy_range, std::cref(segs), done, std::min(total, done + step));
  } catch (...) {  // no more threads: the rest here
    copy_range(segs, done, total);
  }
  copy_range(segs, 0, std::min(step, total));
  for (auto& t : th) t.join();
}

// Pinned staging for up to `count` particles (6 doubles each, 256 MB at most:
// longer transfers go in pieces, and so do those that pinned memory cannot be had
// for).  The stream is idle when it returns, so the staging is free.
int ensure_stage(pw_ctx* c, int64_t count) {
  constexpr int64_t kMaxParticles = (int64_t(256) << 20) / 48;
  const int64_t want = std::min(count, kMaxParticles);
  PW_HIP(hipStreamSynchronize(c->stream));
  for (int64_t m = want; m > static_cast<int64_t>(c->stage_particles); m /= 2) {
    double* fresh = nullptr;
    if (hipHostMalloc(reinterpret_cast<void**>(&fresh), 48 * static_cast<size_t>(m), hipHostMallocCoherent) != hipSuccess) {
      (void)hipGetLastError();
      continue;
    }
    (void)hipHostFree(c->h_stage);
    c->h_stage = fresh;
    c->stage_particles = static_cast<size_t>(m);
    return PW_OK;
  }
  return c->stage_particles > 0 ? PW_OK : fail(PW_ERR_NOMEM, "pinned staging");
}

// Where the caller's rows of particles [first, first + count) are: positions and
// strengths (or velocities and vorticity rates), 3 doubles each.  A transfer takes
// a list of consecutive ones, one per wake, in one launch per piece of the staging
// (one per wake cost 12 us each: the state vector of 20,000 wakes 245 ms).
template <typename T>
struct Rows {
  int64_t first, count;
  T *a, *b;
};

// f(row, from, to) for the parts of the rows in particles [p, end); rows before
// `at` are done with
template <typename T, typename F>
void each_part(const std::vector<Rows<T>>& rows, size_t& at, int64_t p, int64_t end, F f) {
  while (at < rows.size() && rows[at].first + rows[at].count <= p) ++at;
  for (size_t r = at; r < rows.size() && rows[r].first < end; ++r) {
    const int64_t from = std::max(p, rows[r].first), to = std::min(end, rows[r].first + rows[r].count);
    if (from < to) f(rows[r], from, to);
  }
}

// the device's rows into the caller's (a or b may be null)
int read_particles(pw_ctx* c, bool rates, const std::vector<Rows<double>>& rows) {
  if (rows.empty()) return PW_OK;
  const int64_t first = rows.front().first, last = rows.back().first + rows.back().count;
  if (last <= first) return PW_OK;
  PW_TRY(ensure_stage(c, last - first));
  size_t at = 0;
  for (int64_t p = first; p < last; p += static_cast<int64_t>(c->stage_particles)) {
    const int64_t m = std::min<int64_t>(last - p, static_cast<int64_t>(c->stage_particles));
    if (rates) PW_HIP(pw::launch_pack_rates(c->rates, p, m, c->h_stage, c->stream));
    else PW_HIP(pw::launch_pack_state(c->y, p, m, c->h_stage, false, c->stream));
    PW_HIP(hipStreamSynchronize(c->stream));
    std::vector<Segment> segs;
    each_part(rows, at, p, p + m, [&](const Rows<double>& r, int64_t from, int64_t to) {
      const size_t bytes = 24 * static_cast<size_t>(to - from);
      if (r.a) segs.push_back({r.a + 3 * (from - r.first), c->h_stage + 3 * (from - p), bytes});
      if (r.b) segs.push_back({r.b + 3 * (from - r.first), c->h_stage + 3 * (m + from - p), bytes});
    });
    copy_segments(segs);
  }
  return PW_OK;
}

// the caller's positions and strengths into the state
int write_particles(pw_ctx* c, const std::vector<Rows<const double>>& rows) {
  if (rows.empty()) return PW_OK;
  const int64_t first = rows.front().first, last = rows.back().first + rows.back().count;
  if (last <= first) return PW_OK;
  PW_TRY(ensure_stage(c, last - first));
  size_t at = 0;
  for (int64_t p = first; p < last; p += static_cast<int64_t>(c->stage_particles)) {
    const int64_t m = std::min<int64_t>(last - p, static_cast<int64_t>(c->stage_particles));
    if (p > first) PW_HIP(hipStreamSynchronize(c->stream));  // the previous piece has been read
    std::vector<Segment> segs;
    each_part(rows, at, p, p + m, [&](const Rows<const double>& r, int64_t from, int64_t to) {
      const size_t bytes = 24 * static_cast<size_t>(to - from);
      segs.push_back({c->h_stage + 3 * (from - p), r.a + 3 * (from - r.first), bytes});
      segs.push_back({c->h_stage + 3 * (m + from - p), r.b + 3 * (from - r.first), bytes});
    });
    copy_segments(segs);
    PW_HIP(pw::launch_pack_state(c->y, p, m, c->h_stage, true, c->stream));
  }
  return PW_OK;
}

// the rows of a state or rate vector in the reference's layout: per wake the
// first 3-vectors of maxn particles, then the second ones (wake.cpp:860-866, :876)
template <typename T>
std::vector<Rows<T>> vector_rows(const pw_ctx* c, T* v) {
  std::vector<Rows<T>> rows;
  rows.reserve(c->wn.size());
  for (size_t w = 0; w < c->wn.size(); ++w) {
    rows.push_back({c->woff[w], c->wn[w], v, v + 3 * c->wmax[w]});
    v += 6 * c->wmax[w];
  }
  return rows;
}

// zeros in the rows of such a vector that hold no particle
void clear_unused_rows(const pw_ctx* c, double* v) {
  for (size_t w = 0; w < c->wn.size(); ++w) {
    const size_t pad = 24 * static_cast<size_t>(c->wmax[w] - c->wn[w]);
    std::memset(v + 3 * c->wn[w], 0, pad);
    std::memset(v + 3 * (c->wmax[w] + c->wn[w]), 0, pad);
    v += 6 * c->wmax[w];
  }
}

// velocities at m points on the device; the partial sums go to the second
// rate array, which holds no result between calls (and has room for every
// split of up to kPointBlocks blocks, however few particles there are)
hipError_t point_velocity(pw_ctx* c, const double* d_pts, int m, double* d_u) {
  return pw::launch_point_velocity(c->y, static_cast<int>(c->n), d_pts, m, d_u, reinterpret_cast<double*>(c->k[1]),
                                   6 * std::max(static_cast<size_t>(c->n), pw::kPointScratchRows),
                                   c->smoothing == PW_KERNEL_HIGHORDER, c->stream);
}

}  // namespace

namespace pwi {

int ensure_built(pw_ctx* c) { return ::ensure_built(c); }

int staging(pw_ctx* c, size_t bytes, void** out) {
  PW_TRY(ensure_stage(c, static_cast<int64_t>((bytes + 47) / 48)));
  if (bytes > 48 * c->stage_particles) return fail(PW_ERR_NOMEM, "pinned staging");
  *out = c->h_stage;
  return PW_OK;
}

int prof_begin(pw_ctx* c, hipEvent_t* e0, hipEvent_t* e1) {
  if (c->ev_free.empty()) {
    PW_HIP(hipEventCreate(e0));
    PW_HIP(hipEventCreate(e1));
  } else {
    *e0 = c->ev_free.back().first;
    *e1 = c->ev_free.back().second;
    c->ev_free.pop_back();
  }
  return PW_OK;
}

}  // namespace pwi

extern "C" {

const char* pw_version(void) { return "pawan-mi355x 0.1 (gfx950)"; }

const char* pw_last_error(void) { return pwi::g_error.c_str(); }

int pw_device_count(int* count) {
  if (!count) return fail(PW_ERR_ARG, "null count");
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) {
    *count = 0;
    return fail(PW_ERR_HIP, std::string("hipGetDeviceCount: ") + hipGetErrorString(e));
  }
  *count = n;
  return PW_OK;
}

int pw_create(pw_ctx** out, int device) {
  if (!out) return fail(PW_ERR_ARG, "null output pointer");
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    return fail(PW_ERR_HIP, "no HIP device available");
  if (device < 0 || device >= ndev)
    return fail(PW_ERR_ARG, "device index out of range");
  pw_ctx* c = new (std::nothrow) pw_ctx();
  if (!c) return fail(PW_ERR_NOMEM, "host allocation failed");
  c->device = device;
  if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return fail(PW_ERR_HIP, "stream creation failed");
  }
  const int rc = resolve_noalloc_staging(device);
  if (rc != PW_OK) {
    (void)hipStreamDestroy(c->stream);
    delete c;
    return rc;
  }
  *out = c;
  return PW_OK;
}

int pw_destroy(pw_ctx* c) {
  if (!c) return PW_OK;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  release(c);
  delete c;
  return PW_OK;
}

int pw_add_wake(pw_ctx* c, int64_t n, int64_t maxn, const double* pos, const double* alpha,
                const double* radius, const double* volume, int* wake) {
  PW_CTX(c);
  if (c->built) return fail(PW_ERR_STATE, "wakes must be added before the first solve/step");
  if (n < 0 || maxn < n) return fail(PW_ERR_ARG, "need 0 <= n <= maxn");
  if (n > 0 && (!pos || !alpha || !radius || !volume))
    return fail(PW_ERR_ARG, "null particle array");
  if (c->n + n > INT32_MAX / 2) return fail(PW_ERR_UNSUPPORTED, "too many particles");
  for (int64_t i = 0; i < n; ++i) {
    Rec64 r;
    r.x = pos[3 * i];
    r.y = pos[3 * i + 1];
    r.z = pos[3 * i + 2];
    r.s2 = radius[i] * radius[i];  // gsl_pow_2(s), interaction_utils.h:476
    r.ax = alpha[3 * i];
    r.ay = alpha[3 * i + 1];
    r.az = alpha[3 * i + 2];
    r.vol = volume[i];
    c->pending.push_back(r);
    c->radius.push_back(radius[i]);
    c->volume.push_back(volume[i]);
  }
  c->wn.push_back(n);
  c->wmax.push_back(maxn);
  c->n += n;
  c->woff.push_back(c->n);
  if (wake) *wake = static_cast<int>(c->wn.size()) - 1;
  return PW_OK;
}

int pw_set_nu(pw_ctx* c, double nu) {
  PW_CTX(c);
  if (!std::isfinite(nu) || nu < 0) return fail(PW_ERR_ARG, "nu must be finite and >= 0");
  if (nu != c->nu) {
    drop_graphs(c);  // captured steps carry nu in their kernel arguments
    c->nu = nu;
  }
  return PW_OK;
}

int pw_get_nu(pw_ctx* c, double* nu) {
  PW_CTX(c);
  if (!nu) return fail(PW_ERR_ARG, "null output");
  *nu = c->nu;
  return PW_OK;
}

int pw_set_coupled(pw_ctx* c, int coupled) {
  PW_CTX(c);
  if (c->built) return fail(PW_ERR_STATE, "coupling must be set before the first solve/step");
  c->coupled = coupled != 0;
  return PW_OK;
}

int pw_set_kernel(pw_ctx* c, int kernel) {
  PW_CTX(c);
  if (kernel != PW_KERNEL_GAUSSIAN && kernel != PW_KERNEL_HIGHORDER)
    return fail(PW_ERR_ARG, "kernel must be PW_KERNEL_GAUSSIAN or PW_KERNEL_HIGHORDER");
  if (kernel != c->smoothing) {
    drop_graphs(c);  // captured steps hold the other kernel's launches
    c->smoothing = kernel;
  }
  return PW_OK;
}

int pw_set_compensation(pw_ctx* c, int enable) {
  PW_CTX(c);
  if ((enable != 0) != c->compensated) {
    drop_graphs(c);  // captured steps hold the other summation's launches
    c->compensated = enable != 0;
  }
  return PW_OK;
}

int pw_get_kernel(pw_ctx* c, int* kernel) {
  PW_CTX(c);
  if (!kernel) return fail(PW_ERR_ARG, "null output");
  *kernel = c->smoothing;
  return PW_OK;
}

int pw_get_size(pw_ctx* c, int64_t* num_particles, int* num_wakes) {
  PW_CTX(c);
  if (num_particles) *num_particles = c->n;
  if (num_wakes) *num_wakes = static_cast<int>(c->wn.size());
  return PW_OK;
}

int pw_set_wake_state(pw_ctx* c, int w, const double* pos, const double* alpha) {
  PW_CTX(c);
  if (w < 0 || w >= static_cast<int>(c->wn.size())) return fail(PW_ERR_ARG, "wake index out of range");
  if (c->wn[w] > 0 && (!pos || !alpha)) return fail(PW_ERR_ARG, "null array");
  if (c->built) return write_particles(c, {{c->woff[w], c->wn[w], pos, alpha}});
  for (int64_t i = 0; i < c->wn[w]; ++i) {
    Rec64& r = c->pending[c->woff[w] + i];
    r.x = pos[3 * i]; r.y = pos[3 * i + 1]; r.z = pos[3 * i + 2];
    r.ax = alpha[3 * i]; r.ay = alpha[3 * i + 1]; r.az = alpha[3 * i + 2];
  }
  return PW_OK;
}

int pw_set_wake_volume(pw_ctx* c, int w, const double* volume) {
  PW_CTX(c);
  if (w < 0 || w >= static_cast<int>(c->wn.size())) return fail(PW_ERR_ARG, "wake index out of range");
  if (c->wn[w] > 0 && !volume) return fail(PW_ERR_ARG, "null array");
  std::vector<Rec64> h;
  PW_TRY(download_state(c, h));
  for (int64_t i = 0; i < c->wn[w]; ++i) {
    h[c->woff[w] + i].vol = volume[i];
    c->volume[c->woff[w] + i] = volume[i];
  }
  return upload_state(c, h);
}

int pw_get_wake_state(pw_ctx* c, int w, double* pos, double* alpha) {
  PW_CTX(c);
  if (w < 0 || w >= static_cast<int>(c->wn.size())) return fail(PW_ERR_ARG, "wake index out of range");
  if (c->built) return read_particles(c, false, {{c->woff[w], c->wn[w], pos, alpha}});
  for (int64_t i = 0; i < c->wn[w]; ++i) {
    const Rec64& r = c->pending[c->woff[w] + i];
    if (pos) { pos[3 * i] = r.x; pos[3 * i + 1] = r.y; pos[3 * i + 2] = r.z; }
    if (alpha) { alpha[3 * i] = r.ax; alpha[3 * i + 1] = r.ay; alpha[3 * i + 2] = r.az; }
  }
  return PW_OK;
}

int pw_get_wake_rates(pw_ctx* c, int w, double* vel, double* retvor) {
  PW_CTX(c);
  if (w < 0 || w >= static_cast<int>(c->wn.size())) return fail(PW_ERR_ARG, "wake index out of range");
  if (c->built) return read_particles(c, true, {{c->woff[w], c->wn[w], vel, retvor}});
  const size_t bytes = 24 * static_cast<size_t>(c->wn[w]);
  if (vel) std::memset(vel, 0, bytes);
  if (retvor) std::memset(retvor, 0, bytes);
  return PW_OK;
}

// Every wake's rows at once: one launch and one wait instead of one of each per
// wake (the rates of 48 rings, 167,000 particles: a solve 5.35 -> 4.34 ms).
int pw_get_all_state(pw_ctx* c, double* pos, double* alpha) {
  PW_CTX(c);
  if (c->built) return read_particles(c, false, {{0, c->n, pos, alpha}});
  for (size_t w = 0; w < c->wn.size(); ++w)
    PW_TRY(pw_get_wake_state(c, static_cast<int>(w), pos ? pos + 3 * c->woff[w] : nullptr,
                             alpha ? alpha + 3 * c->woff[w] : nullptr));
  return PW_OK;
}

int pw_get_all_rates(pw_ctx* c, double* vel, double* retvor) {
  PW_CTX(c);
  if (c->built) return read_particles(c, true, {{0, c->n, vel, retvor}});
  const size_t bytes = 24 * static_cast<size_t>(c->n);
  if (vel) std::memset(vel, 0, bytes);
  if (retvor) std::memset(retvor, 0, bytes);
  return PW_OK;
}

int pw_set_states(pw_ctx* c, const double* state, int64_t len) {
  PW_CTX(c);
  if (!state) return fail(PW_ERR_ARG, "null state");
  if (len != total_maxsize(c)) return fail(PW_ERR_ARG, "state length != sum of 6*maxn");
  const auto rows = vector_rows(c, state);
  if (c->built) return write_particles(c, rows);
  for (size_t w = 0; w < rows.size(); ++w) PW_TRY(pw_set_wake_state(c, static_cast<int>(w), rows[w].a, rows[w].b));
  return PW_OK;
}

int pw_get_states(pw_ctx* c, double* state, int64_t len) {
  PW_CTX(c);
  if (!state) return fail(PW_ERR_ARG, "null state");
  if (len != total_maxsize(c)) return fail(PW_ERR_ARG, "state length != sum of 6*maxn");
  const auto rows = vector_rows(c, state);
  clear_unused_rows(c, state);
  if (c->built) return read_particles(c, false, rows);
  for (size_t w = 0; w < rows.size(); ++w) PW_TRY(pw_get_wake_state(c, static_cast<int>(w), rows[w].a, rows[w].b));
  return PW_OK;
}

int pw_get_rates(pw_ctx* c, double* rate, int64_t len) {
  PW_CTX(c);
  if (!rate) return fail(PW_ERR_ARG, "null rate");
  if (len != total_maxsize(c)) return fail(PW_ERR_ARG, "rate length != sum of 6*maxn");
  if (!c->built) {
    std::memset(rate, 0, sizeof(double) * static_cast<size_t>(len));
    return PW_OK;
  }
  clear_unused_rows(c, rate);
  return read_particles(c, true, vector_rows(c, rate));
}

int pw_velocity_at(pw_ctx* c, const double* points, int64_t m, double* u) {
  PW_CTX(c);
  if (m < 0 || m > (int64_t(1) << 28)) return fail(PW_ERR_ARG, "m must be in [0, 2^28]");
  if (m == 0) return PW_OK;
  if (!points || !u) return fail(PW_ERR_ARG, "null points or output");
  PW_TRY(ensure_built(c));
  const size_t len = 3 * static_cast<size_t>(m);
  // the points and their velocities pass through a buffer the context keeps
  // (bounded: larger sets get one of their own)
  constexpr size_t kKeepPoints = size_t(1) << 20;
  double* own = nullptr;
  double* d_pts = c->d_points;
  if (2 * len > c->points_len) {
    double* fresh = nullptr;
    if (dalloc(&fresh, 2 * len) != hipSuccess) {
      (void)hipGetLastError();
      return fail(PW_ERR_NOMEM, "point buffers");
    }
    d_pts = fresh;
    if (static_cast<size_t>(m) <= kKeepPoints) {
      (void)hipFree(c->d_points);
      c->d_points = fresh;
      c->points_len = 2 * len;
    } else {
      own = fresh;
    }
  }
  double* d_u = d_pts + len;
  hipError_t e = hipMemcpyAsync(d_pts, points, len * sizeof(double), hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) e = point_velocity(c, d_pts, static_cast<int>(m), d_u);
  if (e == hipSuccess) e = hipMemcpyAsync(u, d_u, len * sizeof(double), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  else (void)hipStreamSynchronize(c->stream);  // nothing queued may still use the buffers
  (void)hipFree(own);
  if (e != hipSuccess) return fail(PW_ERR_HIP, std::string("pw_velocity_at: ") + hipGetErrorString(e));
  return PW_OK;
}

// pw_velocity_at without its per-call buffers: the points and velocities
// pass through the device's static staging array.  Calls on one GPU share
// that array, so calls that overlap on one GPU (several host threads) race.
int pw_velocity_at_noalloc(pw_ctx* c, const double* points, int64_t m, double* u) {
  PW_CTX(c);
  if (m < 0 || m > kNoAllocPoints)
    return fail(PW_ERR_ARG, "m must be in [0, " + std::to_string(kNoAllocPoints) +
                                "], the capacity of the static staging buffer");
  if (m == 0) return PW_OK;
  if (!points || !u) return fail(PW_ERR_ARG, "null points or output");
  if (!c->built)
    return fail(PW_ERR_STATE, "the context's particles are not on the device yet: its first pw_solve, pw_step "
                              "or pw_velocity_at puts them there (and allocates)");
  double* st = noalloc_staging(c->device);
  if (!st) return fail(PW_ERR_STATE, "staging buffer of this device not resolved");
  double *d_pts = st, *d_u = st + 3 * kNoAllocPoints;
  const size_t bytes = 3 * static_cast<size_t>(m) * sizeof(double);
  hipError_t e = hipMemcpyAsync(d_pts, points, bytes, hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) e = point_velocity(c, d_pts, static_cast<int>(m), d_u);
  if (e == hipSuccess) e = hipMemcpyAsync(u, d_u, bytes, hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  else (void)hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return fail(PW_ERR_HIP, std::string("pw_velocity_at_noalloc: ") + hipGetErrorString(e));
  return PW_OK;
}

int pw_vring_particles(double R, double core, int nlayers, int nazi, double sig, double* pos,
                       double* radius, double* volume) {
  (void)core;  // sets only the ideal profile (pw_vring_resolve)
  if (nlayers < 0 || nazi < 1 || (2 * nlayers + 1) * (2 * nlayers + 1) > pw::kVringMaxCells)
    return fail(PW_ERR_ARG, "nlayers must be in [0, 15] and nazi >= 1");
  if (!(std::isfinite(R) && R > 0.0) || !(std::isfinite(sig) && sig > 0.0))
    return fail(PW_ERR_ARG, "ring radius and smoothing radius must be finite and positive");
  if (!pos || !radius || !volume) return fail(PW_ERR_ARG, "null output");
  // the particle layout of __vring (vring.cpp:50-100): one centre particle
  // and layers of 8j particles per station, the cell volumes of its
  // annular sectors
  const double r0 = 0.35 / (2 * nlayers + 1);
  const double dpsi = 2.0 * M_PI / nazi;
  int64_t q = 0;
  for (int a = 0; a < nazi; ++a) {
    const double psi = a * dpsi, sp = std::sin(psi), cp = std::cos(psi);
    pos[3 * q] = R * cp;
    pos[3 * q + 1] = R * sp;
    pos[3 * q + 2] = 0.0;
    radius[q] = sig;
    volume[q] = M_PI * (r0 * r0) * R * dpsi;
    ++q;
    for (int j = 1; j <= nlayers; ++j) {
      const double jj = static_cast<double>(j) * j;
      const double r = r0 * (12. * jj + 1.0) / (6. * j);
      const int ncell = 8 * j;
      const double dth = 2. * M_PI / ncell;
      for (int k = 0; k < ncell; ++k) {
        const double th = k * dth;
        pos[3 * q] = (R + r * std::cos(th)) * cp;
        pos[3 * q + 1] = (R + r * std::cos(th)) * sp;
        pos[3 * q + 2] = r * std::sin(th);
        radius[q] = sig;
        volume[q] = 2.0 * r0 * dpsi * (2.0 * dth * j * R * r0 + (12.0 * jj + 1.0) * (r0 * r0) *
                                                                    (std::sin(th + dth) - std::sin(th)) / 3.0);
        ++q;
      }
    }
  }
  return PW_OK;
}

int pw_vring_resolve(pw_ctx* c, int wake, int nlayers, int nazi, double R, double core, double* strength,
                     double* influence) {
  PW_CTX(c);
  if (wake < 0 || wake >= static_cast<int>(c->wn.size())) return fail(PW_ERR_ARG, "wake index out of range");
  if (nlayers < 0 || nazi < 1 || (2 * nlayers + 1) * (2 * nlayers + 1) > pw::kVringMaxCells)
    return fail(PW_ERR_ARG, "nlayers must be in [0, 15] and nazi >= 1");
  if (!(std::isfinite(core) && core > 0.0) || !(std::isfinite(R) && R > 0.0))
    return fail(PW_ERR_ARG, "radius and core must be finite and positive");
  const int m = (2 * nlayers + 1) * (2 * nlayers + 1);
  if (c->wn[wake] != static_cast<int64_t>(m) * nazi)
    return fail(PW_ERR_ARG, "the wake does not hold nazi (2 nlayers + 1)^2 particles");
  // a zero or non-finite smoothing radius makes every influence entry 0/0
  for (int64_t q = c->woff[wake]; q < c->woff[wake + 1]; ++q)
    if (!(std::isfinite(c->radius[q]) && c->radius[q] > 0.0))
      return fail(PW_ERR_ARG, "the ring's smoothing radii must be finite and positive");
  PW_TRY(ensure_built(c));
  // __vring::getIdealRates (vring.cpp:223-242): the Gaussian core profile
  std::vector<double> ideal(m);
  {
    const double mag0 = 0.5 / (M_PI * core * core), r0 = 0.35 / (2 * nlayers + 1);
    int idx = 0;
    ideal[idx++] = mag0;
    for (int j = 1; j <= nlayers; ++j) {
      const double r = r0 * (12. * (static_cast<double>(j) * j) + 1.0) / (6. * j);
      const int ncell = 8 * j;
      const double dth = 2. * M_PI / ncell, decay = std::exp(-0.5 * r * r / (core * core));
      for (int k = 0; k < ncell; ++k) ideal[idx++] = mag0 * (1.0 + r * std::cos(k * dth) / R) * decay;
    }
  }
  double *d_M = nullptr, *d_lu = nullptr, *d_b = nullptr, *d_s = nullptr;
  int* d_flag = nullptr;
  const size_t mm = static_cast<size_t>(m) * m;
  if (dalloc(&d_M, mm) != hipSuccess || dalloc(&d_lu, mm) != hipSuccess || dalloc(&d_b, m) != hipSuccess ||
      dalloc(&d_s, m) != hipSuccess || dalloc(&d_flag, 1 + static_cast<size_t>(m)) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipFree(d_M); (void)hipFree(d_lu); (void)hipFree(d_b); (void)hipFree(d_s); (void)hipFree(d_flag);
    return fail(PW_ERR_NOMEM, "resolve buffers");
  }
  int flag = 0;
  hipError_t e = hipMemcpyAsync(d_b, ideal.data(), m * sizeof(double), hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess)
    e = pw::launch_vring_resolve(c->y, static_cast<int>(c->woff[wake]), m, nazi,
                                 c->smoothing == PW_KERNEL_HIGHORDER, d_M, d_lu, d_b, d_s, d_flag, c->stream);
  if (e == hipSuccess && strength)
    e = hipMemcpyAsync(strength, d_s, m * sizeof(double), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess && influence)
    e = hipMemcpyAsync(influence, d_M, mm * sizeof(double), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(&flag, d_flag, sizeof(int), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  else (void)hipStreamSynchronize(c->stream);  // nothing queued may still use the buffers
  (void)hipFree(d_M); (void)hipFree(d_lu); (void)hipFree(d_b); (void)hipFree(d_s); (void)hipFree(d_flag);
  if (e != hipSuccess) return fail(PW_ERR_HIP, std::string("pw_vring_resolve: ") + hipGetErrorString(e));
  if (flag) return fail(PW_ERR_NONFINITE, "pw_vring_resolve: singular influence matrix");
  return PW_OK;
}

int pw_solve(pw_ctx* c, int precision) {
  PW_CTX(c);
  int kind = 0;
  PW_TRY(kind_of(precision, &kind));
  PW_TRY(ensure_built(c));
  PW_TRY(clear_flag(c));
  PW_TRY(rhs(c, kind, c->y, c->k[0]));
  c->rates = c->k[0];
  return check_flag(c, "pw_solve");
}

}  // extern "C"

namespace {

// The kernels of one step of `scheme` on the context stream; each right-hand
// side carries the stage arithmetic that uses it.
int enqueue_step(pw_ctx* c, int scheme, int kind, double dt) {
  Rate64** k = c->k;
  pw::StageOp op;
  op.y = c->y;
  op.out = c->ys;
  if (scheme == PW_RK4) {
    // rk4.cpp:20-66
    op.kind = pw::kStageLin;
    op.a = 0.5 * dt;
    PW_TRY(rhs(c, kind, c->y, k[0], op));
    PW_TRY(rhs(c, kind, c->ys, k[1], op));
    op.a = dt;
    PW_TRY(rhs(c, kind, c->ys, k[2], op));
    op.kind = pw::kStageRk4;
    op.k1 = k[0];
    op.k2 = k[1];
    op.k3 = k[2];
    op.a = dt / 6.;
    op.b = dt / 3.;
    PW_TRY(rhs(c, kind, c->ys, k[3], op));
  } else if (scheme == PW_RK3) {
    // rk3.cpp:20-55
    op.kind = pw::kStageLin;
    op.a = 0.5 * dt;
    PW_TRY(rhs(c, kind, c->y, k[0], op));
    op.kind = pw::kStageRk3Mid;
    op.k1 = k[0];
    op.a = dt;
    op.b = 2. * dt;
    PW_TRY(rhs(c, kind, c->ys, k[1], op));
    op.kind = pw::kStageRk3;
    op.k2 = k[1];
    op.a = dt / 6.0;
    op.b = dt * 2.0 / 3.0;
    PW_TRY(rhs(c, kind, c->ys, k[2], op));
  } else {
    // integration.cpp:126-136
    op.kind = pw::kStageEuler;
    op.a = dt;
    PW_TRY(rhs(c, kind, c->y, k[0], op));
  }
  return PW_OK;
}

Rate64* last_rates(pw_ctx* c, int scheme) {
  return scheme == PW_RK4 ? c->k[3] : scheme == PW_RK3 ? c->k[2] : c->k[0];
}

// One step captured as a HIP graph (per scheme, kind and dt), replayed for
// every step: one launch instead of up to 13.
int step_graph(pw_ctx* c, int scheme, int kind, double dt, hipGraphExec_t* out) {
  uint64_t bits;
  std::memcpy(&bits, &dt, sizeof bits);
  const auto key = std::make_tuple(scheme, kind, bits);
  auto it = c->graphs.find(key);
  if (it != c->graphs.end()) {
    *out = it->second;
    return PW_OK;
  }
  PW_TRY(ensure_kind(c, kind));  // allocations happen outside the capture
  hipGraph_t g = nullptr;
  PW_HIP(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  const int rc = enqueue_step(c, scheme, kind, dt);
  hipGraph_t captured = nullptr;
  const hipError_t ec = hipStreamEndCapture(c->stream, &captured);
  if (rc != PW_OK || ec != hipSuccess) {
    // a failed capture leaves its error as the thread's last error: clear
    // it, so that the next launch's check does not report it again
    (void)hipGetLastError();
    if (captured) (void)hipGraphDestroy(captured);
    if (rc != PW_OK) return rc;
    return fail(PW_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(ec));
  }
  g = captured;
  hipGraphExec_t exec = nullptr;
  const hipError_t ei = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (ei != hipSuccess) return fail(PW_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(ei));
  c->graphs[key] = exec;
  *out = exec;
  return PW_OK;
}

}  // namespace

extern "C" {

int pw_step(pw_ctx* c, int scheme, double dt, int precision, int64_t nsteps) {
  PW_CTX(c);
  int kind = 0;
  PW_TRY(kind_of(precision, &kind));
  if (scheme != PW_EULER && scheme != PW_RK3 && scheme != PW_RK4)
    return fail(PW_ERR_ARG, "scheme must be PW_EULER, PW_RK3 or PW_RK4");
  if (!std::isfinite(dt)) return fail(PW_ERR_ARG, "dt must be finite");
  if (nsteps < 0) return fail(PW_ERR_ARG, "nsteps must be >= 0");
  PW_TRY(ensure_built(c));
  PW_TRY(ensure_kind(c, kind));
  PW_TRY(clear_flag(c));
  // the tree path re-sorts the particles every stage (host-side sort
  // set-up), so its steps are launched eagerly
  if (c->use_graph && !c->profiling && nsteps > 0 && kind != kKindLearned) {
    hipGraphExec_t exec = nullptr;
    PW_TRY(step_graph(c, scheme, kind, dt, &exec));
    for (int64_t it = 0; it < nsteps; ++it) PW_HIP(hipGraphLaunch(exec, c->stream));
  } else {
    for (int64_t it = 0; it < nsteps; ++it) PW_TRY(enqueue_step(c, scheme, kind, dt));
  }
  if (nsteps > 0) c->rates = last_rates(c, scheme);
  return check_flag(c, "pw_step");
}

int pw_interact_wakes(pw_ctx* c, int precision, const int* pairs, int npairs) {
  PW_CTX(c);
  int kind = 0;
  PW_TRY(kind_of(precision, &kind));
  if (kind == kKindLearned) return fail(PW_ERR_UNSUPPORTED, "the tree path evaluates the whole system at once");
  PW_TRY(check_blocks(c, pairs, npairs));
  PW_TRY(ensure_built(c));
  std::vector<WorkItem> items;
  std::vector<int> first(npairs + 1, 0);
  for (int k = 0; k < npairs; ++k) {
    const int a = pairs[2 * k], b = pairs[2 * k + 1];
    append_items(c, a, b, 0, items);
    if (a != b) append_items(c, b, a, 0, items);
    first[k + 1] = static_cast<int>(items.size());
  }
  const int n = static_cast<int>(c->n);
  Rate64* acc = c->k[0];
  Rate64* blk = c->k[1];
  PW_TRY(clear_flag(c));
  PW_HIP(pw::launch_zero_doubles(reinterpret_cast<double*>(acc), 6 * static_cast<int64_t>(n), c->stream));
  WorkItem* d_items = nullptr;
  if (!items.empty() && dalloc(&d_items, items.size()) != hipSuccess) {
    (void)hipGetLastError();
    return fail(PW_ERR_NOMEM, "work items");
  }
  hipError_t e = items.empty() ? hipSuccess
                               : hipMemcpyAsync(d_items, items.data(), items.size() * sizeof(WorkItem),
                                                hipMemcpyHostToDevice, c->stream);
  const int lk = launch_kind_of(c, kind);
  for (int k = 0; k < npairs && e == hipSuccess; ++k) {
    // one block at a time: its items have distinct targets and write their
    // rates into blk, which is then added to the targets' totals
    pw::PairArgs args{c->y,     d_items + first[k], first[k + 1] - first[k], n, blk, nullptr, c->d_queue, c->nu,
                      c->d_chunks, c->d_src32,        nullptr, c->nchunks};
    e = pw::launch_pair(lk, pw::PairConfig{}, args, args.nitems, c->stream);
    const int a = pairs[2 * k], b = pairs[2 * k + 1];
    if (e == hipSuccess)
      e = pw::launch_add_rates(acc, blk, static_cast<int>(c->woff[a]), static_cast<int>(c->woff[a + 1]), c->stream);
    if (e == hipSuccess && a != b)
      e = pw::launch_add_rates(acc, blk, static_cast<int>(c->woff[b]), static_cast<int>(c->woff[b + 1]), c->stream);
  }
  if (e == hipSuccess) e = pw::launch_check_finite(acc, n, c->h_flag, c->stream);
  (void)hipStreamSynchronize(c->stream);  // the items are freed below
  (void)hipFree(d_items);
  if (e != hipSuccess) return fail(PW_ERR_HIP, std::string("pw_interact_wakes: ") + hipGetErrorString(e));
  c->rates = acc;
  return check_flag(c, "pw_interact_wakes");
}

int pw_vorticity_field(pw_ctx* c, const int* pairs, int npairs, double* field, int64_t len) {
  PW_CTX(c);
  if (!field) return fail(PW_ERR_ARG, "null output");
  if (pairs) PW_TRY(check_blocks(c, pairs, npairs));
  PW_TRY(ensure_built(c));
  const int n = static_cast<int>(c->n);
  if (len != 3 * static_cast<int64_t>(n)) return fail(PW_ERR_ARG, "field needs 3 doubles per particle");
  // launch groups whose items have distinct targets: the whole system at
  // once, or one block of wake pairs at a time
  std::vector<WorkItem> items;
  std::vector<int> first{0};
  if (!pairs) {
    items = c->h_pair_items;
    first.push_back(static_cast<int>(items.size()));
  } else {
    for (int k = 0; k < npairs; ++k) {
      const int a = pairs[2 * k], b = pairs[2 * k + 1];
      append_items(c, a, b, 0, items);
      if (a != b) append_items(c, b, a, 0, items);
      first.push_back(static_cast<int>(items.size()));
    }
  }
  double* d_field = reinterpret_cast<double*>(c->k[1]);  // 6 doubles per particle
  WorkItem* d_items = nullptr;
  if (!items.empty() && dalloc(&d_items, items.size()) != hipSuccess) {
    (void)hipGetLastError();
    return fail(PW_ERR_NOMEM, "work items");
  }
  hipError_t e = pw::launch_zero_doubles(d_field, 3 * static_cast<int64_t>(n), c->stream);
  if (e == hipSuccess && !items.empty())
    e = hipMemcpyAsync(d_items, items.data(), items.size() * sizeof(WorkItem), hipMemcpyHostToDevice, c->stream);
  const bool ho = c->smoothing == PW_KERNEL_HIGHORDER;
  for (size_t g = 0; g + 1 < first.size() && e == hipSuccess; ++g)
    e = pw::launch_vorticity_field(c->y, d_items + first[g], first[g + 1] - first[g], ho, d_field, c->stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(field, d_field, sizeof(double) * 3 * static_cast<size_t>(n), hipMemcpyDeviceToHost,
                       c->stream);
  (void)hipStreamSynchronize(c->stream);
  (void)hipFree(d_items);
  if (e != hipSuccess) return fail(PW_ERR_HIP, std::string("pw_vorticity_field: ") + hipGetErrorString(e));
  return PW_OK;
}

int pw_diagnose_wakes(pw_ctx* c, int wa, int wb, double* out, int64_t out_len) {
  PW_CTX(c);
  if (!out || out_len < 16) return fail(PW_ERR_ARG, "output needs 16 doubles");
  const int pair[2] = {wa, wb};
  PW_TRY(check_blocks(c, pair, 1));
  PW_TRY(ensure_built(c));
  std::vector<WorkItem> items;
  if (wa == wb) {
    append_diag_items(c->woff[wa], c->woff[wa + 1], diag_range({{c->woff[wa], c->woff[wa + 1]}}), items);
  } else {
    // every source of wake b, a range at a time, for each 64 targets of wake a
    const int range = diag_range(c->wn[wa], c->wn[wb]);
    for (int64_t t0 = c->woff[wa]; t0 < c->woff[wa + 1]; t0 += 64)
      for (int64_t s0 = c->woff[wb]; s0 < c->woff[wb + 1]; s0 += range)
        items.push_back({static_cast<int32_t>(t0), static_cast<int32_t>(std::min<int64_t>(t0 + 64, c->woff[wa + 1])),
                         static_cast<int32_t>(s0), static_cast<int32_t>(std::min<int64_t>(s0 + range, c->woff[wb + 1])),
                         -1, 1, 0, 0});
  }
  constexpr size_t Q = pw::kDiagQuad;
  const int ni = static_cast<int>(items.size());
  // the wake's linear-sum items are contiguous in the context's list
  int l0 = 0, nl = 0;
  for (int b = 0; b < c->nlin; ++b)
    if (c->lin_wake[b] == wa) {
      if (nl == 0) l0 = b;
      ++nl;
    }
  WorkItem* d_items = nullptr;
  double* d_q = nullptr;
  // each item's sums, the block's, and the items of the block: [0, ni)
  if (ni > 0 && (dalloc(&d_items, items.size()) != hipSuccess || dalloc(&d_q, Q * (items.size() + 1) + 1) != hipSuccess)) {
    (void)hipGetLastError();
    (void)hipFree(d_items);
    return fail(PW_ERR_NOMEM, "diagnostic buffers");
  }
  double q[Q] = {0.0};
  const int first[2] = {0, ni};
  std::vector<double> lin(11 * static_cast<size_t>(nl));
  hipError_t e = hipSuccess;
  if (ni > 0) {
    double* d_sum = d_q + Q * items.size();
    int* d_first = reinterpret_cast<int*>(d_sum + Q);
    e = hipMemcpyAsync(d_items, items.data(), items.size() * sizeof(WorkItem), hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(d_first, first, sizeof first, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess)
      e = pw::launch_diag_pairs(c->y, c->d_radius, d_items, ni, d_q, c->smoothing == PW_KERNEL_HIGHORDER,
                                c->stream);
    if (e == hipSuccess) e = pw::launch_diag_sum(d_q, d_first, 1, d_sum, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(q, d_sum, sizeof q, hipMemcpyDeviceToHost, c->stream);
  }
  if (e == hipSuccess && wa == wb && nl > 0) {
    e = pw::launch_diag_linear(c->y, c->lin_items + l0, nl, c->d_lin + 11 * static_cast<size_t>(l0), c->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync(lin.data(), c->d_lin + 11 * static_cast<size_t>(l0), lin.size() * sizeof(double),
                         hipMemcpyDeviceToHost, c->stream);
  }
  (void)hipStreamSynchronize(c->stream);
  (void)hipFree(d_items);
  (void)hipFree(d_q);
  if (e != hipSuccess) return fail(PW_ERR_HIP, std::string("pw_diagnose_wakes: ") + hipGetErrorString(e));
  for (int m = 0; m < 16; ++m) out[m] = 0.0;
  if (wa == wb) {
    double v[11] = {0};
    for (int b = 0; b < nl; ++b)
      for (int m = 0; m < 11; ++m) v[m] += lin[11 * b + m];
    for (int m = 0; m < 3; ++m) {
      out[m] = v[m];                       // calculateTotalVorticity
      out[3 + m] = v[3 + m] * 0.5;         // calculateLinearImpulse
      out[6 + m] = v[6 + m] * (1.0 / 3.0); // calculateAngularImpulse
    }
    out[14] = v[9];
    out[15] = v[10];
  }
  // within a wake 2 sum_{i<j} plus the self terms; across wakes one
  // direction, doubled as in calculate*(W1, W2) (interaction.cpp:551-718)
  const double f = wa == wb ? 1.0 : 2.0;
  out[9] = f * q[0];   // helicity
  out[10] = f * q[3];  // enstrophy
  out[11] = f * q[4];  // div-free enstrophy
  out[12] = f * q[1];  // kinetic energy
  out[13] = f * q[2];  // div-free kinetic energy
  return PW_OK;
}

int pw_diagnose(pw_ctx* c, double* out, int64_t out_len) {
  PW_CTX(c);
  if (!out) return fail(PW_ERR_ARG, "null output");
  PW_TRY(ensure_built(c));
  const int ns = c->nsys();
  if (out_len < 15 * static_cast<int64_t>(ns))
    return fail(PW_ERR_ARG, "output needs 15 doubles per system");
  PW_TRY(ensure_diag(c));
  PW_HIP(pw::launch_diag_linear(c->y, c->lin_items, c->nlin, c->d_lin, c->stream));
  const bool ho = c->smoothing == PW_KERNEL_HIGHORDER;
  constexpr int Q = pw::kDiagQuad;
  double* d_sys = c->d_quad + Q * static_cast<size_t>(c->ndiag);
  PW_HIP(pw::launch_diag_pairs(c->y, c->d_radius, c->diag_items, c->ndiag, c->d_quad, ho, c->stream));
  PW_HIP(pw::launch_diag_sum(c->d_quad, c->d_diag_first, ns, d_sys, c->stream));
  std::vector<double> lin(11 * static_cast<size_t>(c->nlin)), sq(Q * static_cast<size_t>(ns));
  PW_HIP(hipMemcpyAsync(lin.data(), c->d_lin, lin.size() * sizeof(double), hipMemcpyDeviceToHost,
                        c->stream));
  PW_HIP(hipMemcpyAsync(sq.data(), d_sys, sq.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  PW_HIP(hipStreamSynchronize(c->stream));
  const int nw = static_cast<int>(c->wn.size());
  // per-wake linear sums in block order
  std::vector<double> wl(11 * static_cast<size_t>(nw), 0.0);
  for (int b = 0; b < c->nlin; ++b)
    for (int m = 0; m < 11; ++m) wl[11 * c->lin_wake[b] + m] += lin[11 * b + m];
  for (int s = 0; s < ns; ++s) {
    double* o = out + 15 * s;
    for (int m = 0; m < 9; ++m) o[m] = 0.0;
    const int w0 = c->coupled ? 0 : s, w1 = c->coupled ? nw : s + 1;
    for (int w = w0; w < w1; ++w) {
      const double* v = &wl[11 * w];
      // calculateTotalVorticity / LinearImpulse (* 0.5) / AngularImpulse
      // (* 1/3), interaction.cpp:489-527, summed over wakes (:74-84)
      for (int m = 0; m < 3; ++m) {
        o[m] += v[m];
        o[3 + m] += v[3 + m] * 0.5;
        o[6 + m] += v[6 + m] * (1.0 / 3.0);
      }
      if (v[10] != 0.0) c->zc[s] = v[9] / v[10];  // interaction.cpp:153-155
    }
    o[9] = sq[Q * s + 0];   // helicity
    o[10] = sq[Q * s + 3];  // enstrophy (ENST == 0 for the Gaussian kernel)
    o[11] = sq[Q * s + 4];  // div-free enstrophy (ENSTF == 0 likewise)
    o[12] = sq[Q * s + 1];  // kinetic energy
    o[13] = sq[Q * s + 2];  // div-free kinetic energy
    o[14] = c->zc[s];
  }
  return PW_OK;
}

int pw_synchronize(pw_ctx* c) {
  PW_CTX(c);
  PW_HIP(hipStreamSynchronize(c->stream));
  return PW_OK;
}

int pw_set_profiling(pw_ctx* c, int enable) {
  PW_CTX(c);
  PW_TRY(collect_profile(c));
  PW_TRY(pwi::ff_collect_stages(c));
  c->profiling = enable != 0;
  c->prof_ms = 0.0;
  c->prof_launches = 0;
  pwi::ff_reset_stages(c);
  return PW_OK;
}

int pw_get_pair_timing(pw_ctx* c, double* total_ms, int64_t* launches) {
  PW_CTX(c);
  PW_TRY(collect_profile(c));
  if (total_ms) *total_ms = c->prof_ms;
  if (launches) *launches = c->prof_launches;
  return PW_OK;
}

int pw_set_pair_config(pw_ctx* c, int precision, int parts, int persistent, int variant) {
  PW_CTX(c);
  int kind = 0;
  PW_TRY(kind_of(precision, &kind));
  if (kind == kKindLearned) return fail(PW_ERR_UNSUPPORTED, "launch configuration applies to the direct-sum kinds");
  if (parts < 1 || parts > 256) return fail(PW_ERR_ARG, "parts must be in [1, 256]");
  auto& k = c->ks[kind];
  if (variant < 0 || variant > (PW_VARIANT_WAVES8 | PW_VARIANT_SCALAR_FEED | PW_VARIANT_TWO_PER_LANE))
    return fail(PW_ERR_ARG, "variant must be a combination of the PW_VARIANT_* bits");
  k.cfg.parts = parts;
  k.cfg.persistent = persistent != 0;
  k.cfg.scalar_feed = (variant & PW_VARIANT_SCALAR_FEED) != 0 && (kind == pw::kPairFP32C || kind == pw::kPairFP64);
  k.cfg.two_per_lane = (variant & PW_VARIANT_TWO_PER_LANE) != 0 && k.cfg.scalar_feed && kind == pw::kPairFP32C;
  k.cfg.waves8 = (variant & PW_VARIANT_WAVES8) != 0 && kind == pw::kPairFP32C && !k.cfg.two_per_lane;
  k.tuned = true;
  drop_graphs(c);
  return PW_OK;
}

int pw_get_pair_config(pw_ctx* c, int precision, int* parts, int* persistent, int* variant) {
  PW_CTX(c);
  int kind = 0;
  PW_TRY(kind_of(precision, &kind));
  if (kind == kKindLearned) return fail(PW_ERR_UNSUPPORTED, "launch configuration applies to the direct-sum kinds");
  const auto& k = c->ks[kind];
  if (parts) *parts = k.cfg.parts;
  if (persistent) *persistent = k.cfg.persistent ? 1 : 0;
  if (variant)
    *variant = (k.cfg.waves8 ? PW_VARIANT_WAVES8 : 0) | (k.cfg.scalar_feed ? PW_VARIANT_SCALAR_FEED : 0) |
               (k.cfg.two_per_lane ? PW_VARIANT_TWO_PER_LANE : 0);
  return PW_OK;
}

int pw_set_graph(pw_ctx* c, int enable) {
  PW_CTX(c);
  c->use_graph = enable != 0;
  if (!c->use_graph) drop_graphs(c);
  return PW_OK;
}

}  // extern "C"

namespace {

// Tuning results shared by every context of the process, keyed by the
// problem's shape; optionally also appended to / read from the text file
// named by $PAWAN_TUNE_CACHE ("kind n nsys largest parts persistent variant",
// kind the pair-kernel family: 0-2 for the Gaussian precisions, 4 and 5
// for the high-order FP64 and FP32C kernels; variant the PW_VARIANT_* bits;
// 1 0 0 leaves the launch to auto_config).
using TuneKey = std::tuple<int, int64_t, int, int64_t>;
std::map<TuneKey, pw::PairConfig>& tune_cache() {
  static std::map<TuneKey, pw::PairConfig> m;
  return m;
}
// guards the cache and its file (contexts may be driven from several threads)
std::mutex& tune_mutex() {
  static std::mutex m;
  return m;
}

void load_tune_file() {
  static bool loaded = false;
  if (loaded) return;
  loaded = true;
  const char* path = std::getenv("PAWAN_TUNE_CACHE");
  if (!path) return;
  FILE* f = std::fopen(path, "r");
  if (!f) return;
  int kind, nsys, parts, pers, w8;
  long long n, largest;
  while (std::fscanf(f, "%d %lld %d %lld %d %d %d", &kind, &n, &nsys, &largest, &parts, &pers, &w8) == 7) {
    // the ranges pw_set_pair_config accepts; other lines are skipped
    if (kind < 0 || kind > pw::kPairFP32CHO || kind == kKindLearned || parts < 1 || parts > 256) continue;
    pw::PairConfig cfg;
    cfg.parts = parts;
    cfg.persistent = pers != 0;
    if (w8 < 0 || w8 > (PW_VARIANT_WAVES8 | PW_VARIANT_SCALAR_FEED | PW_VARIANT_TWO_PER_LANE)) continue;
    const bool f32 = kind == pw::kPairFP32C || kind == pw::kPairFP32CHO;
    cfg.scalar_feed = (w8 & PW_VARIANT_SCALAR_FEED) != 0 && (f32 || kind == pw::kPairFP64);
    cfg.two_per_lane = (w8 & PW_VARIANT_TWO_PER_LANE) != 0 && cfg.scalar_feed && f32;
    cfg.waves8 = (w8 & PW_VARIANT_WAVES8) != 0 && f32 && !cfg.two_per_lane;
    tune_cache()[TuneKey(kind, n, nsys, largest)] = cfg;
  }
  std::fclose(f);
}

void save_tune_file(const TuneKey& key, const pw::PairConfig& cfg) {
  const char* path = std::getenv("PAWAN_TUNE_CACHE");
  if (!path) return;
  FILE* f = std::fopen(path, "a");
  if (!f) return;
  std::fprintf(f, "%d %lld %d %lld %d %d %d\n", std::get<0>(key), static_cast<long long>(std::get<1>(key)),
               std::get<2>(key), static_cast<long long>(std::get<3>(key)), cfg.parts,
               cfg.persistent ? 1 : 0,
               (cfg.waves8 ? PW_VARIANT_WAVES8 : 0) | (cfg.scalar_feed ? PW_VARIANT_SCALAR_FEED : 0) |
                   (cfg.two_per_lane ? PW_VARIANT_TWO_PER_LANE : 0));
  std::fclose(f);
}

int time_rhs(pw_ctx* c, int kind, double* ms, int reps = 4) {
  hipEvent_t e0, e1;
  PW_HIP(hipEventCreate(&e0));
  PW_HIP(hipEventCreate(&e1));
  float best = 1e30f;
  for (int rep = 0; rep < reps; ++rep) {
    PW_HIP(hipEventRecord(e0, c->stream));
    const int rc = rhs(c, kind, c->y, c->k[0]);
    if (rc != PW_OK) {
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
      return rc;
    }
    PW_HIP(hipEventRecord(e1, c->stream));
    PW_HIP(hipEventSynchronize(e1));
    float t = 0.0f;
    PW_HIP(hipEventElapsedTime(&t, e0, e1));
    best = std::min(best, t);
    if (t > 50.0f) break;  // long enough that the first-launch cost is noise
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  *ms = best;
  return PW_OK;
}

}  // namespace

extern "C" {

int pw_autotune(pw_ctx* c, int precision, double* best_ms) {
  PW_CTX(c);
  int kind = 0;
  PW_TRY(kind_of(precision, &kind));
  if (kind == kKindLearned) return fail(PW_ERR_UNSUPPORTED, "launch configuration applies to the direct-sum kinds");
  PW_TRY(ensure_built(c));
  const int64_t largest = c->systems.empty() ? 0 : c->systems.front().b - c->systems.front().a;
  // keyed by the kernel family the launches run (the high-order kernels
  // have their own best shapes)
  const int family = c->smoothing == PW_KERNEL_HIGHORDER ? launch_kind_of(c, kind) : kind;
  const TuneKey key(family, c->n, c->nsys(), largest);
  auto& k = c->ks[kind];
  const bool was_profiling = c->profiling;
  c->profiling = false;
  bool found = false;
  pw::PairConfig cached;
  {
    std::lock_guard<std::mutex> lock(tune_mutex());
    load_tune_file();
    auto hit = tune_cache().find(key);
    if (hit != tune_cache().end()) {
      found = true;
      cached = hit->second;
    }
  }
  if (found) {
    k.cfg = cached;
    k.tuned = true;
    drop_graphs(c);
    // one timed right-hand side (or more, when the time is asked for), so
    // that the rates of the current state are on the device as after a
    // search
    double ms = 0.0;
    const int rc = time_rhs(c, kind, &ms, best_ms ? 4 : 1);
    c->profiling = was_profiling;
    if (rc != PW_OK) return rc;
    if (best_ms) *best_ms = ms;
    c->rates = c->k[0];
    return PW_OK;
  }
  // candidates: split the sources (fills the GPU for few target blocks and
  // cuts the tail of the last block wave), keep blocks resident, and for
  // FP32C the 8-wave register budget
  int64_t blocks = 0, max_tiles = 1;
  for (const auto& sr : c->systems) {
    const int64_t nt = (sr.b - sr.a + kTargetsPerItem - 1) / kTargetsPerItem;
    blocks += nt;
    max_tiles = std::max(max_tiles, nt);
  }
  std::vector<pw::PairConfig> cands;
  auto add = [&](int parts, bool pers, bool w8, bool sf = false, bool t2 = false) {
    if (parts > max_tiles) return;
    pw::PairConfig p;
    p.parts = parts;
    p.persistent = pers;
    p.waves8 = w8 && !t2;
    p.scalar_feed = sf;
    p.two_per_lane = t2;
    cands.push_back(p);
  };
  const bool f32 = kind == pw::kPairFP32C;
  add(1, false, false);
  add(1, true, false);
  add(2, false, false);
  add(4, true, false);
  add(8, true, false);
  if (f32) {
    add(1, false, true);
    add(4, true, true);
    add(8, true, true);
    // sources through scalar loads, one wave per 64 targets
    add(1, false, true, true);
    add(1, true, true, true);
    add(4, true, true, true);
    add(8, true, true, true);
    add(4, true, false, true);
  }
  const int64_t resident = static_cast<int64_t>(c->num_cus) * 8;
  for (int parts = 16; parts <= 64; parts *= 2)
    if (blocks * parts <= 8 * resident) add(parts, true, f32);
  // finer source ranges at any size: with the items ordered part by part,
  // a part of 1/16 or 1/32 of a large system stays in every XCD's L2 while
  // its items run
  for (int parts = 16; parts <= 32; parts *= 2) {
    if (blocks * parts > 8 * resident) add(parts, true, f32);
    if (f32) add(parts, true, true, true);
  }
  // two targets per lane (particles per thread): each scalar source record
  // feeds two pairs, at half the waves
  if (f32) {
    add(8, true, false, true, true);
    add(16, true, false, true, true);
    add(32, true, false, true, true);
  }
  // the scalar-fed FP64 kernel (Gaussian FP64 only)
  if (kind == pw::kPairFP64 && c->smoothing == PW_KERNEL_GAUSSIAN) {
    add(1, false, false, true);
    add(8, true, false, true);
    add(16, true, false, true);
    add(32, true, false, true);
  }
  pw::PairConfig best_cfg = cands.front();
  double best = 1e300;
  for (const auto& cand : cands) {
    k.cfg = cand;
    double ms = 0.0;
    const int rc = time_rhs(c, kind, &ms);
    if (rc != PW_OK) {
      c->profiling = was_profiling;
      return rc;
    }
    if (ms < best) {
      best = ms;
      best_cfg = cand;
    }
  }
  k.cfg = best_cfg;
  k.tuned = true;
  drop_graphs(c);
  {
    std::lock_guard<std::mutex> lock(tune_mutex());
    tune_cache()[key] = best_cfg;
    save_tune_file(key, best_cfg);
  }
  // the rates of the chosen configuration (the candidates' reductions of
  // source-split partial sums differ in rounding)
  {
    const int rc = rhs(c, kind, c->y, c->k[0]);
    c->profiling = was_profiling;
    if (rc != PW_OK) return rc;
  }
  c->rates = c->k[0];
  if (best_ms) *best_ms = best;
  return PW_OK;
}

}  // extern "C"
