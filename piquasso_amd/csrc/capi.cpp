// C ABI of the permanent engine (include/pqp_permanent.h).
//
// Host side of every call: plan (plan.cpp), copy the arena to the device,
// launch the sweep kernels (perm_fwd.hip) and the finalize kernel on a HIP
// stream, copy the results back.  Errors become status codes plus a
// thread-local message; nothing throws across the ABI.
#include "pqp_permanent.h"

#include <hip/hip_runtime.h>
#include <rocprofiler-sdk-roctx/roctx.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "capi_internal.hpp"
#include "perm_kernels.hpp"
#include "plan.hpp"
#include "poly_plan.hpp"
#include "pqp_types.hpp"

namespace {

using namespace pqp;

thread_local std::string g_error;
thread_local double g_last_bound = std::numeric_limits<double>::quiet_NaN();

int fail(int code, const std::string &msg) {
  g_error = msg;
  return code;
}

// Allocation-failure test hook (pqp_debug_fail_allocation): -1 = off; k >= 0
// lets k more device or pinned-host allocations through, fails the next one
// with PQP_ERR_NOMEM, and switches itself off.
std::atomic<int64_t> g_alloc_countdown{-1};

bool forced_alloc_failure() {
  int64_t c = g_alloc_countdown.load();
  while (c >= 0) {
    if (g_alloc_countdown.compare_exchange_weak(c, c - 1)) return c == 0;
  }
  return false;
}

// One roctx range per compute call, named after the entry point: under
// rocprofv3 --marker-trace the kernels and copies of a call fall inside it.
struct CallRange {
  explicit CallRange(const char *name) { roctxRangePushA(name); }
  ~CallRange() { roctxRangePop(); }
  CallRange(const CallRange &) = delete;
  CallRange &operator=(const CallRange &) = delete;
};

#define PQP_HIP(expr)                                                               \
  do {                                                                              \
    hipError_t e_ = (expr);                                                         \
    if (e_ != hipSuccess)                                                           \
      return fail(PQP_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

// ---------------------------------------------------------------- device --

struct DeviceState {
  bool ok = false;
  int n_devices = 0;
  int device = 0;
  int cus = 0;
  std::string name;
  std::string error;
  // occupancy cache: [bucket][fp32][comp][persistent], -1 = not queried
  int occ[kBuckets][2][2][2];
};

DeviceState &device_state() {
  static DeviceState st;
  static std::once_flag once;
  std::call_once(once, [] {
    std::memset(st.occ, 0xff, sizeof(st.occ));
    const char *force = std::getenv("PQP_FORCE_NO_DEVICE");
    if (force && *force && std::strcmp(force, "0") != 0) {
      // decided before any HIP call, so the runtime is never initialised
      st.error = "no HIP device available (PQP_FORCE_NO_DEVICE is set)";
      return;
    }
    hipError_t e = hipGetDeviceCount(&st.n_devices);
    if (e != hipSuccess || st.n_devices < 1) {
      st.error = std::string("no HIP device available (") +
                 (e != hipSuccess ? hipGetErrorString(e) : "device count is 0") + ")";
      st.n_devices = 0;
      return;
    }
    if (hipGetDevice(&st.device) != hipSuccess) st.device = 0;
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, st.device);
    if (e != hipSuccess) {
      st.error = std::string("hipGetDeviceProperties: ") + hipGetErrorString(e);
      return;
    }
    st.cus = prop.multiProcessorCount;
    st.name = prop.gcnArchName;
    st.ok = true;
  });
  return st;
}

// Work units a launch is split into (measured on MI355X, 256 CUs): one
// permanent of T Gray terms runs best with about 1.4 sqrt(T) units (n = 20:
// 1024, n = 24: 4096, n = 28: 16384), capped at 128 per CU (n = 32: 32768);
// a batch of uneven permanents with 32 per CU over the whole batch (4096
// items of n = 8..24: 8192 units; finer splits add per-unit start cost).
constexpr int64_t kSingleUnitsPerCu = 128;
constexpr int64_t kBatchUnitsPerCu = 32;
// Gradient sweeps write every row's gradient per unit and run two waves per
// SIMD: about 8 units per CU over the batch measured best (256 gradients of
// n = 12..20: 0.74 ms at 8 or 16 per CU, 0.91 ms at 32).
constexpr int64_t kGradUnitsPerCu = 8;
// Waves a lone column-minor problem is spread over before its waves sweep
// more than one state a lane: two per SIMD of 256 CUs.
constexpr int64_t kLaplaceWaves = 2048;
// Shots of one pass of the sampler (its buffers: 64 partials of 48
// components and 24 columns of 64 modes each, 200 MB at most).
constexpr int64_t kSampleShots = 2048;
// Waves of an exact permanent before its lanes sweep more states, and inner
// digits at most.
constexpr int64_t kIntWaves = 4096;
constexpr int kIntInnerDigits = 7;
// Bytes of a polynomial permanent's exponent rows that are compared with the
// kept plan's before anything runs (3 us).
constexpr size_t kPolyCompareFirst = size_t{64} << 10;
// Outputs up to which 6 and 7 particles take the subset sum.
constexpr size_t kPolyFew6 = 64, kPolyFew7 = 4;
// Device buffers one-shot batches may leave for the next ones, and how many
// calls' worth: as many threads find theirs ready.
constexpr size_t kKeptBytes = size_t{256} << 20;
constexpr size_t kKeptExecs = 4;

// Permanents without tables: one block up to kOneBlockTerms Gray terms (the
// blocks' meeting costs about 3 us: 13 particles 17.0 us a call in one block
// and 16.5 in four), else blocks for about kOneStates states a lane, up
// to a wave per SIMD, and two above kOneManyTerms terms (2^23 terms: 85 us
// at one, 61 at two).  Above kOneMaxTerms the planned sweep, whose units
// walk longer, is as fast.
constexpr double kOneBlockTerms = 2048.0;
constexpr double kOneStates = 4.0;
constexpr int kOneBlockWaves = 4;  // one per SIMD
constexpr double kOneManyTerms = 2097152.0;
constexpr double kOneMaxTerms = 16777216.0;

int expand_mode(uint32_t flags) {
  if (flags & PQP_FLAG_EXPAND_COLS) return 1;
  if (flags & PQP_FLAG_KEEP_COLS) return 0;
  return 2;
}

int require_device() {
  DeviceState &d = device_state();
  if (!d.ok) return fail(PQP_ERR_DEVICE, d.error);
  return PQP_OK;
}

int blocks_per_cu(int bucket, bool fp32, bool comp, bool persistent) {
  DeviceState &d = device_state();
  int &slot = d.occ[bucket][fp32][comp][persistent];
  if (slot < 0) {
    int b = 0;
    if (occupancy_fwd(bucket, persistent, fp32, comp, &b) != hipSuccess || b < 1) b = 1;
    slot = b;
  }
  return slot;
}

// -------------------------------------------------------- device buffers --

struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
  int ensure(size_t n) {
    if (n <= bytes) return PQP_OK;
    if (p) {
      (void)hipFree(p);
      p = nullptr;
      bytes = 0;
    }
    size_t alloc = std::max<size_t>(n, 4096);
    if (forced_alloc_failure()) return fail(PQP_ERR_NOMEM, "hipMalloc: forced failure (test hook)");
    hipError_t e = hipMalloc(&p, alloc);
    if (e != hipSuccess) return fail(PQP_ERR_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    bytes = alloc;
    return PQP_OK;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
};

// Pinned host staging buffer (hipHostMalloc): uploads and result downloads
// go through it as true asynchronous DMA instead of pageable-memory copies.
struct HostBuf {
  void *p = nullptr;
  size_t bytes = 0;
  int ensure(size_t n) {
    if (n <= bytes) return PQP_OK;
    if (p) {
      (void)hipHostFree(p);
      p = nullptr;
      bytes = 0;
    }
    size_t alloc = std::max<size_t>(n, 65536);
    if (forced_alloc_failure()) return fail(PQP_ERR_NOMEM, "hipHostMalloc: forced failure (test hook)");
    hipError_t e = hipHostMalloc(&p, alloc, hipHostMallocDefault);
    if (e != hipSuccess)
      return fail(PQP_ERR_NOMEM, std::string("hipHostMalloc: ") + hipGetErrorString(e));
    bytes = alloc;
    return PQP_OK;
  }
  void release() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
    bytes = 0;
  }
};

// Pinned host memory mapped into the device's address space: kernels write
// small results straight into it, so a call needs no device-to-host copy
// (the stream synchronisation makes the writes visible).
struct MappedBuf {
  void *host = nullptr;
  void *dev = nullptr;
  size_t bytes = 0;
  int ensure(size_t n) {
    if (n <= bytes) return PQP_OK;
    release();
    size_t alloc = std::max<size_t>(n, 4096);
    if (forced_alloc_failure()) return fail(PQP_ERR_NOMEM, "hipHostMalloc: forced failure (test hook)");
    hipError_t e = hipHostMalloc(&host, alloc, hipHostMallocMapped | hipHostMallocCoherent);
    if (e != hipSuccess) {
      host = nullptr;
      return fail(PQP_ERR_NOMEM, std::string("hipHostMalloc: ") + hipGetErrorString(e));
    }
    e = hipHostGetDevicePointer(&dev, host, 0);
    if (e != hipSuccess) {
      release();
      return fail(PQP_ERR_DEVICE, std::string("hipHostGetDevicePointer: ") + hipGetErrorString(e));
    }
    bytes = alloc;
    return PQP_OK;
  }
  void release() {
    if (host) (void)hipHostFree(host);
    host = dev = nullptr;
    bytes = 0;
  }
};

// A stream that is created once, also when what follows its creation fails.
int ensure_stream(hipStream_t &stream) {
  if (!stream) PQP_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
  return PQP_OK;
}

// Device image of one plan plus the stream it runs on.
struct Exec {
  Plan plan;
  std::vector<int32_t> item_first_unit;  // first unit of each item in plan.units
  DevBuf arena, partials, heads;
  DevBuf results;   // 2 doubles per result, 4 (dd parts) per result, 1 (term magnitudes) per result
  bool mapped_results = false;  // results in results_m (host memory) instead
  MappedBuf results_m;
  HostBuf stage;    // pinned staging for the arena upload and result downloads
  size_t n_results = 0;
  bool heads_clean = false;  // queue heads zeroed since (re)allocation
  bool abs_valid = false;    // the last evaluation left term magnitudes
  hipStream_t stream = nullptr;
  uint32_t flags = 0;
  // side streams and events for running several width buckets concurrently
  hipStream_t side[kMaxRanges] = {};
  hipEvent_t ev_fork = nullptr;
  hipEvent_t ev_join[kMaxRanges] = {};

  LaunchArgs args() const {
    LaunchArgs a;
    a.arena = static_cast<const char *>(arena.p);
    a.items = reinterpret_cast<const ItemDesc *>(static_cast<const char *>(arena.p) + plan.items_off);
    a.units = reinterpret_cast<const WorkUnit *>(static_cast<const char *>(arena.p) + plan.units_off);
    a.partials = static_cast<double *>(partials.p);
    double *r = static_cast<double *>(mapped_results ? results_m.dev : results.p);
    a.out = r;
    a.out_dd = r + 2 * n_results;
    a.out_abs = r + 6 * n_results;
    a.part_abs = static_cast<double *>(partials.p) + 4 * std::max<int64_t>(plan.n_partials, 1);
    a.queue_head = static_cast<int *>(heads.p);
    a.n_units = static_cast<int32_t>(plan.units.size());
    a.n_items = static_cast<int32_t>(plan.items.size());
    return a;
  }
};

void index_units(Exec &x) {
  x.item_first_unit.assign(x.plan.items.size(), -1);
  for (size_t u = 0; u < x.plan.units.size(); ++u) {
    const WorkUnit &w = x.plan.units[u];
    if (x.item_first_unit[w.item] < 0) x.item_first_unit[w.item] = static_cast<int32_t>(u);
  }
}

// Upload the plan (allocating device buffers as needed).
int upload(Exec &x) {
  const Plan &p = x.plan;
  const size_t n_out = static_cast<size_t>(std::max<int64_t>(p.n_out, 1));
  int st;
  if ((st = x.arena.ensure(p.arena.size())) != PQP_OK) return st;
  // partials: 4 doubles per slot, then 1 (term magnitudes) per slot
  if ((st = x.partials.ensure(std::max<int64_t>(p.n_partials, 1) * 5 * sizeof(double))) != PQP_OK) return st;
  if (x.mapped_results) {
    if ((st = x.results_m.ensure(n_out * 7 * sizeof(double))) != PQP_OK) return st;
  } else if ((st = x.results.ensure(n_out * 7 * sizeof(double))) != PQP_OK) {
    return st;
  }
  x.n_results = n_out;
  const void *heads_before = x.heads.p;
  if ((st = x.heads.ensure(64 * sizeof(int))) != PQP_OK) return st;
  if (x.heads.p != heads_before) x.heads_clean = false;
  // the previous use of the staging buffer (an upload or a download on this
  // stream) has completed: every entry point synchronises before returning
  if ((st = x.stage.ensure(p.arena.size())) != PQP_OK) return st;
  std::memcpy(x.stage.p, p.arena.data(), p.arena.size());
  PQP_HIP(hipMemcpyAsync(x.arena.p, x.stage.p, p.arena.size(), hipMemcpyHostToDevice, x.stream));
  if (!x.heads_clean) {
    // queue heads start at zero; the finalize kernel rewinds them after
    // every launch that uses them
    PQP_HIP(hipMemsetAsync(x.heads.p, 0, 64 * sizeof(int), x.stream));
    x.heads_clean = true;
  }
  return PQP_OK;
}

// Side streams (default priority) and fork/join events, created once per Exec.
int ensure_side_streams(Exec &x) {
  if (x.ev_fork) return PQP_OK;
  int st;
  for (int i = 1; i < kMaxRanges; ++i) {
    if ((st = ensure_stream(x.side[i])) != PQP_OK) return st;
    if (!x.ev_join[i]) PQP_HIP(hipEventCreateWithFlags(&x.ev_join[i], hipEventDisableTiming));
  }
  PQP_HIP(hipEventCreateWithFlags(&x.ev_fork, hipEventDisableTiming));
  return PQP_OK;
}

// Everything an Exec holds, its stream too where it is the Exec's own.
void release_exec(Exec &x, bool stream) {
  x.arena.release();
  x.partials.release();
  x.results.release();
  x.results_m.release();
  x.stage.release();
  x.heads.release();
  for (int i = 1; i < kMaxRanges; ++i) {
    if (x.side[i]) (void)hipStreamDestroy(x.side[i]);
    if (x.ev_join[i]) (void)hipEventDestroy(x.ev_join[i]);
  }
  if (x.ev_fork) (void)hipEventDestroy(x.ev_fork);
  if (stream && x.stream) (void)hipStreamDestroy(x.stream);
}

// Enqueue one evaluation.  ev_begin / ev_end (optional) bracket the sweep
// kernels only when kernel_only is set, the whole evaluation otherwise.
int enqueue(Exec &x, int mode, hipEvent_t ev_begin, hipEvent_t ev_end) {
  const Plan &p = x.plan;
  const LaunchArgs a = x.args();
  const int n_items = static_cast<int>(p.items.size());
  const bool kernel_only = (mode == PQP_RUN_KERNEL);
  if (ev_begin) PQP_HIP(hipEventRecord(ev_begin, x.stream));
  if ((p.minors || p.grad) && mode == PQP_RUN_PLAIN)
    return fail(PQP_ERR_INVALID, "no plain mode for column minors or gradients");
  // compensated static forward launches also leave the term magnitudes
  x.abs_valid = !p.minors && !p.grad &&
                (mode == PQP_RUN_PLAIN ? p.fp32
                                       : ((x.flags & PQP_FLAG_STATIC) &&
                                          (!(x.flags & PQP_FLAG_PLAIN) || p.fp32)));
  if (mode == PQP_RUN_PLAIN) {
    for (int k = 0; k < n_items; ++k) {
      const ItemDesc &d = p.items[k];
      if (d.units > 0) {
        FwdLaunch l;
        l.args = a;
        l.first_unit = x.item_first_unit[k];
        l.n_units = d.units;
        l.persistent = false;
        l.fp32 = p.fp32;
        l.comp = p.fp32;  // FP32 products always accumulate in dd
        l.stream = x.stream;
        int b = 0, mcp = 0;
        b = bucket_for_width(d.mcp, p.fp32, &mcp);
        PQP_HIP(launch_fwd(b, l));
      }
      PQP_HIP(launch_finalize(p.fp32, a, k, 1, 0, d.units, x.stream));
    }
  } else {
    const bool fixed = (x.flags & PQP_FLAG_STATIC) != 0;
    const DeviceState &dev = device_state();
    // Width buckets run concurrently: the costliest range launches first on
    // the main stream, the others on side streams forked from it, so their
    // waves fill the slots the first one's tail leaves idle.
    std::vector<int> order(p.ranges.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = static_cast<int>(i);
    std::stable_sort(order.begin(), order.end(),
                     [&](int u, int v) { return p.ranges[u].cost > p.ranges[v].cost; });
    const bool fork = order.size() > 1;
    double total_cost = 0.0;
    for (const Plan::Range &r : p.ranges) total_cost += r.cost;
    if (fork) {
      int st = ensure_side_streams(x);
      if (st != PQP_OK) return st;
      PQP_HIP(hipEventRecord(x.ev_fork, x.stream));
    }
    for (size_t i = 0; i < order.size(); ++i) {
      const int ri = order[i];
      const Plan::Range &r = p.ranges[ri];
      hipStream_t s = (i == 0) ? x.stream : x.side[i];
      if (i > 0) PQP_HIP(hipStreamWaitEvent(s, x.ev_fork, 0));
      FwdLaunch l;
      l.args = a;
      l.first_unit = r.first;
      l.n_units = r.count;
      l.head_slot = ri;
      l.persistent = !fixed;
      l.fp32 = p.fp32;
      l.comp = !(x.flags & PQP_FLAG_PLAIN) || p.fp32;
      l.stream = s;
      if (l.persistent && !p.minors && !p.grad) {
        // resident waves in proportion to the range's share of the work, so
        // concurrent ranges run side by side instead of one after another
        const int per_cu = blocks_per_cu(r.bucket, l.fp32, l.comp, true);
        const double share = total_cost > 0.0 ? r.cost / total_cost : 1.0;
        const int slots = static_cast<int>(std::ceil(share * dev.cus * per_cu));
        l.grid = std::max(1, std::min(r.count, std::max(slots, dev.cus / 4)));
      }
      if (p.grad)
        PQP_HIP(launch_grad(r.bucket, a, r.first, r.count, s));
      else if (p.minors)
        PQP_HIP(launch_minors(r.bucket, a, r.first, r.count, s));
      else
        PQP_HIP(launch_fwd(r.bucket, l));
      if (i > 0) {
        PQP_HIP(hipEventRecord(x.ev_join[i], s));
        PQP_HIP(hipStreamWaitEvent(x.stream, x.ev_join[i], 0));
      }
    }
    if (kernel_only && ev_end) PQP_HIP(hipEventRecord(ev_end, x.stream));
    const bool comp = !(x.flags & PQP_FLAG_PLAIN) || p.fp32;
    if (p.grad) {
      int max_values = 1;
      for (const ItemDesc &d : p.items)
        if (d.n > 0) max_values = std::max(max_values, 1 + (1 + d.L + d.Dt) * d.mc);
      PQP_HIP(launch_grad_finalize(a, n_items, max_values, x.stream));
    } else if (p.all_direct && !p.minors) {
      // every item was a single unit that wrote its own result
    } else if (p.minors)
      PQP_HIP(launch_minors_finalize(a, n_items, p.max_units, x.stream));
    else
      PQP_HIP(launch_finalize(comp, a, 0, n_items, static_cast<int>(p.ranges.size()),
                              p.max_units, x.stream));
  }
  if (ev_end && !kernel_only) PQP_HIP(hipEventRecord(ev_end, x.stream));
  return PQP_OK;
}

}  // namespace

struct pqp_batch {
  Exec x;
  // gradient batches: x runs the gradient plan (the permanent and its
  // gradient of every item from one sweep); with grad_minors (permanents
  // above 32 particles) x runs the permanents and xm the column minors
  bool grad = false;
  bool grad_minors = false;
  Exec xm;
  std::vector<std::vector<int32_t>> minor_rows;  // r - e_i of every minor item
  std::vector<int64_t> minor_item, minor_row;    // (permanent, row) of each minor item
  std::vector<std::vector<int64_t>> minor_slot;  // output slot of each minor (per column)
  std::vector<int64_t> m_r, m_c;                 // shapes of the permanents
  std::vector<std::vector<int32_t>> rows, cols;  // multiplicities of the permanents
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  bool ran = false;
};

namespace {

// Shared state of the single-permanent entry points: buffers grow and are
// reused across calls; calls serialise on a mutex.
struct SingleState {
  std::mutex mu;
  Exec x;       // column minors, gradients, tensor permanents
  Exec xs;      // single permanents: results in mapped host memory
  // the plan resident in xs and its key (shape, multiplicities, flags)
  std::vector<int64_t> xs_key;
  bool xs_planned = false;
  // permanents without tables (perm_one.hip)
  bool init_one = false;
  hipStream_t one_stream = nullptr;
  DevBuf one_work;
  MappedBuf one_res;
  uint64_t one_seq = 0;
};

SingleState &single_state() {
  static SingleState *s = new SingleState();  // never destroyed: outlives atexit HIP teardown
  return *s;
}

// One-shot batches: each call has an Exec (buffers and streams) to itself, so
// calls of several threads run side by side.  What a call leaves is kept for
// the next one, up to kKeptExecs of them and kKeptBytes in all.
struct OneShotPool {
  std::mutex mu;
  std::vector<std::unique_ptr<Exec>> idle;
};

OneShotPool &one_shot_pool() {
  static OneShotPool *p = new OneShotPool();  // never destroyed: outlives atexit HIP teardown
  return *p;
}

struct OneShotLease {
  std::unique_ptr<Exec> x;
  bool finished = false;  // the call's work on the stream is done

  OneShotLease() {
    OneShotPool &pool = one_shot_pool();
    std::lock_guard<std::mutex> lock(pool.mu);
    if (pool.idle.empty()) {
      x.reset(new Exec());
    } else {
      x = std::move(pool.idle.back());
      pool.idle.pop_back();
    }
  }
  ~OneShotLease() {
    auto bytes = [](const Exec &e) { return e.arena.bytes + e.partials.bytes + e.results.bytes; };
    x->plan = Plan();
    if (finished) {
      OneShotPool &pool = one_shot_pool();
      std::lock_guard<std::mutex> lock(pool.mu);
      size_t held = bytes(*x);
      for (const auto &e : pool.idle) held += bytes(*e);
      if (pool.idle.size() < kKeptExecs && held <= kKeptBytes) {
        pool.idle.push_back(std::move(x));
        return;
      }
    }
    if (x->stream) (void)hipStreamSynchronize(x->stream);
    release_exec(*x, true);
  }
  OneShotLease(const OneShotLease &) = delete;
  OneShotLease &operator=(const OneShotLease &) = delete;
};

// ---------------------------------------------------- exact integers --

// The eight largest primes below 2^49 (moduli of perm_int.hip).
constexpr uint64_t kIntPrimes[kIntMaxPrimes] = {
    562949953421231ull, 562949953421201ull, 562949953421189ull, 562949953421173ull,
    562949953421131ull, 562949953421111ull, 562949953421099ull, 562949953421047ull};

using u128 = unsigned __int128;

uint64_t pow_mod(uint64_t b, uint64_t e, uint64_t m) {
  u128 r = 1, x = b % m;
  while (e) {
    if (e & 1) r = r * x % m;
    x = x * x % m;
    e >>= 1;
  }
  return static_cast<uint64_t>(r);
}

// x (kIntLimbs little-endian 64-bit words) = x * m + add
constexpr int kIntLimbs = 8;
void limbs_mul_add(uint64_t *x, uint64_t m, uint64_t add) {
  u128 carry = add;
  for (int k = 0; k < kIntLimbs; ++k) {
    const u128 t = static_cast<u128>(x[k]) * m + carry;
    x[k] = static_cast<uint64_t>(t);
    carry = t >> 64;
  }
}

// Garner's mixed-radix reconstruction of the residues r[k] (in [0, p_k)),
// then the symmetric range (-M/2, M/2], as two's complement limbs.
void crt_limbs(const double *res, int K, uint64_t *x) {
  uint64_t v[kIntMaxPrimes];
  for (int k = 0; k < K; ++k) {
    const uint64_t p = kIntPrimes[k];
    // value of v_0 + v_1 p_0 + ... + v_{k-1} p_0..p_{k-2} modulo p, and p_0..p_{k-1} mod p
    u128 acc = 0, prod = 1;
    for (int i = 0; i < k; ++i) {
      acc = (acc + static_cast<u128>(v[i]) * prod) % p;
      prod = prod * (kIntPrimes[i] % p) % p;
    }
    const uint64_t r = static_cast<uint64_t>(res[k]);
    const uint64_t diff = static_cast<uint64_t>((static_cast<u128>(r) + p - acc) % p);
    v[k] = static_cast<uint64_t>(static_cast<u128>(diff) * pow_mod(static_cast<uint64_t>(prod), p - 2, p) % p);
  }
  std::memset(x, 0, kIntLimbs * sizeof(uint64_t));
  for (int k = K - 1; k >= 0; --k) limbs_mul_add(x, k == K - 1 ? 0 : kIntPrimes[k], v[k]);
  // M = prod p_k; values at or above M / 2 are negative: x - M
  uint64_t M[kIntLimbs] = {1};
  for (int k = 0; k < K; ++k) limbs_mul_add(M, kIntPrimes[k], 0);
  uint64_t half[kIntLimbs];
  for (int k = 0; k < kIntLimbs; ++k)
    half[k] = (M[k] >> 1) | (k + 1 < kIntLimbs ? M[k + 1] << 63 : 0);
  bool ge = true;  // x >= half ?
  for (int k = kIntLimbs - 1; k >= 0; --k)
    if (x[k] != half[k]) {
      ge = x[k] > half[k];
      break;
    }
  if (ge) {
    uint64_t borrow = 0;
    for (int k = 0; k < kIntLimbs; ++k) {
      const uint64_t a = x[k], b = M[k];
      x[k] = a - b - borrow;
      borrow = (a < b) || (a - b < borrow);
    }
  }
}

// x (two's complement limbs) rounded to `bits` <= 53 significant bits, ties
// to even, as a double.
double limbs_round(const uint64_t *x, int bits) {
  uint64_t m[kIntLimbs];
  const bool neg = (x[kIntLimbs - 1] >> 63) != 0;
  if (neg) {
    uint64_t carry = 1;
    for (int k = 0; k < kIntLimbs; ++k) {
      m[k] = ~x[k] + carry;
      carry = (carry && m[k] == 0) ? 1 : 0;
    }
  } else {
    std::memcpy(m, x, sizeof(m));
  }
  int top = -1;
  for (int k = kIntLimbs - 1; k >= 0 && top < 0; --k)
    if (m[k]) top = 64 * k + 63 - __builtin_clzll(m[k]);
  if (top < 0) return 0.0;
  const int lo = top - bits + 1;  // lowest kept bit
  double v;
  if (lo <= 0) {
    v = static_cast<double>(m[0]);  // fewer than `bits` bits: exact
  } else {
    auto bit = [&](int pos) -> uint64_t { return (m[pos / 64] >> (pos % 64)) & 1u; };
    uint64_t keep = 0;
    for (int pos = top; pos >= lo; --pos) keep = (keep << 1) | bit(pos);
    const bool half = bit(lo - 1) != 0;
    bool sticky = false;  // any bit below lo - 1
    for (int k = 0; k * 64 < lo - 1 && !sticky; ++k) {
      const int nb = std::min(lo - 1, 64 * (k + 1)) - 64 * k;
      const uint64_t mask = nb >= 64 ? ~0ull : ((1ull << nb) - 1);
      sticky = (m[k] & mask) != 0;
    }
    if (half && (sticky || (keep & 1))) ++keep;
    v = std::ldexp(static_cast<double>(keep), lo);
  }
  return neg ? -v : v;
}

// x -= d for an integer-valued double d (two's complement limbs).
void limbs_sub_double(uint64_t *x, double d) {
  if (d == 0.0) return;
  int e = 0;
  const double f = std::frexp(std::fabs(d), &e);  // |d| = f 2^e, f in [0.5, 1)
  const uint64_t mant = static_cast<uint64_t>(std::ldexp(f, 53));
  const int shift = e - 53;  // |d| = mant 2^shift, shift >= 0 or mant has trailing zeros
  uint64_t y[kIntLimbs] = {};
  if (shift >= 0) {
    y[shift / 64] = mant << (shift % 64);
    if (shift % 64 && shift / 64 + 1 < kIntLimbs) y[shift / 64 + 1] = mant >> (64 - shift % 64);
  } else {
    y[0] = mant >> (-shift);
  }
  if (d < 0.0) {  // x += |d|
    u128 carry = 0;
    for (int k = 0; k < kIntLimbs; ++k) {
      const u128 s = static_cast<u128>(x[k]) + y[k] + carry;
      x[k] = static_cast<uint64_t>(s);
      carry = s >> 64;
    }
  } else {
    uint64_t borrow = 0;
    for (int k = 0; k < kIntLimbs; ++k) {
      const uint64_t a = x[k], b = y[k];
      x[k] = a - b - borrow;
      borrow = (a < b) || (a - b < borrow);
    }
  }
}

// What the exact path needs to know about a matrix: whether every selected
// entry is an integer of magnitude <= 2^47 with zero imaginary part, the
// largest column bound R_j = sum_i r_i |a_ij| (every Glynn row sum
// |cs_j| <= R_j), log2 of a bound on every Glynn term (the binomial weights
// prod_i C(r_i, r_i / 2) times prod_j R_j^{c_j}) and log2 of the bound
// prod_i (sum_j c_j |a_ij|)^{r_i} >= |perm| (the permanent of the expanded
// matrix is at most the product of its absolute row sums).
struct IntScan {
  bool integral = false;
  double rmax = 0.0, log2_weight = 0.0, log2_term = 0.0, log2_perm = 0.0;
};

IntScan int_scan(const PermInput &in) {
  IntScan sc;
  auto entry = [&](int64_t i, int64_t j, double &re, double &im) {
    const int64_t o = 2 * (i * in.ld + j);
    if (in.a_is_float) {
      re = static_cast<const float *>(in.a)[o];
      im = static_cast<const float *>(in.a)[o + 1];
    } else {
      re = static_cast<const double *>(in.a)[o];
      im = static_cast<const double *>(in.a)[o + 1];
    }
  };
  const double lim = std::ldexp(1.0, 47);
  for (int64_t i = 0; i < in.m_r; ++i) {  // usually ends at the first entry
    if (in.rows[i] <= 0) continue;
    for (int64_t j = 0; j < in.m_c; ++j) {
      if (in.cols[j] <= 0) continue;
      double re, im;
      entry(i, j, re, im);
      if (im != 0.0 || !(std::fabs(re) <= lim) || re != std::nearbyint(re)) return sc;
    }
  }
  std::vector<double> rsum(static_cast<size_t>(std::max<int64_t>(in.m_r, 1)), 0.0);
  double log2_cols = 0.0;
  for (int64_t j = 0; j < in.m_c; ++j) {
    if (in.cols[j] <= 0) continue;
    double rj = 0.0;
    for (int64_t i = 0; i < in.m_r; ++i) {
      if (in.rows[i] <= 0) continue;
      double re, im;
      entry(i, j, re, im);
      rj += in.rows[i] * std::fabs(re);
      rsum[static_cast<size_t>(i)] += in.cols[j] * std::fabs(re);
    }
    sc.rmax = std::max(sc.rmax, rj);
    log2_cols += in.cols[j] * (rj > 0.0 ? std::log2(rj) : -1e9);
  }
  for (int64_t i = 0; i < in.m_r; ++i) {
    if (in.rows[i] <= 0) continue;
    const double s = rsum[static_cast<size_t>(i)];
    sc.log2_perm += in.rows[i] * (s > 0.0 ? std::log2(s) : -1e9);
    const int r = in.rows[i];
    sc.log2_weight += (std::lgamma(r + 1.0) - std::lgamma(r / 2 + 1.0) - std::lgamma(r - r / 2 + 1.0)) /
                      std::log(2.0);
  }
  sc.log2_term = sc.log2_weight + log2_cols;
  sc.integral = true;
  return sc;
}

// Wait for `seq` in the host-visible done slot a launch publishes.
// A kernel that never signals (a device error) is caught by synchronising
// the stream after 10 s of polling.
int wait_done(hipStream_t stream, volatile uint64_t *done, uint64_t seq) {
  const auto t0 = std::chrono::steady_clock::now();
  for (uint32_t spin = 1; *done != seq; ++spin) {
    if ((spin & 4095u) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::seconds(10)) {
      PQP_HIP(hipStreamSynchronize(stream));
      if (*done != seq) return fail(PQP_ERR_DEVICE, "kernel did not signal completion");
      break;
    }
    __builtin_ia32_pause();
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  return PQP_OK;
}

// Buffers of exact integer permanents: `in` the moduli and rows, `work` the
// waves' residues, `res` the permanent's and the done slot.
struct IntState {
  std::mutex mu;
  hipStream_t stream = nullptr;
  DevBuf in, work;
  HostBuf stage;
  MappedBuf res;
  uint64_t seq = 0;
};

IntState &int_state() {
  static IntState *s = new IntState();  // never destroyed: outlives atexit HIP teardown
  return *s;
}

// The exact permanent of an integral matrix (int_scan(in).integral) as
// two's complement limbs: the multi-modular Glynn sweep of perm_int.hip and
// Garner's reconstruction.  PQP_ERR_RANGE when the row sums or binomial
// weights leave FP64's exact integers or the permanent may exceed the
// product of the moduli / 4.
int run_int(const PermInput &in, const IntScan &sc, uint64_t *v) {
  if (in.m_r < 0 || in.m_c < 0 || (in.m_r * in.m_c > 0 && !in.a) || (in.m_r > 0 && !in.rows) ||
      (in.m_c > 0 && !in.cols) || (in.m_r > 0 && in.ld < in.m_c))
    return fail(PQP_ERR_INVALID, "item 0: invalid shape or null pointer");
  int64_t sr = 0, sum_c = 0;
  for (int64_t i = 0; i < in.m_r; ++i) {
    if (in.rows[i] < 0) return fail(PQP_ERR_INVALID, "item 0: negative row multiplicity");
    sr += in.rows[i];
  }
  for (int64_t j = 0; j < in.m_c; ++j) {
    if (in.cols[j] < 0) return fail(PQP_ERR_INVALID, "item 0: negative column multiplicity");
    sum_c += in.cols[j];
  }
  if (sr != sum_c) return fail(PQP_ERR_SUM_MISMATCH, "Number of input and output states should be equal");
  if (sr > kMaxCols) return fail(PQP_ERR_RANGE, "item 0: more than 64 particles");
  const int n = static_cast<int>(sr);
  if (!sc.integral)
    return fail(PQP_ERR_RANGE, "matrix entries are not all integers of magnitude <= 2^47");
  if (sc.rmax > std::ldexp(1.0, 48)) return fail(PQP_ERR_RANGE, "row sums of the matrix exceed 2^48");
  if (sc.log2_weight > 52.0)
    return fail(PQP_ERR_RANGE, "binomial weights of the row multiplicities exceed 2^52");
  // products of G row sums stay below 2^49: exact in FP64 and valid
  // inputs of the modular multiply
  const double lr = sc.rmax > 1.0 ? std::log2(sc.rmax) : 0.0;
  int group = 1;
  for (int g : {12, 8, 4, 2})
    if (group == 1 && g * lr <= 49.0) group = g;
  // moduli: their product (each prime > 2^48.99) must exceed 4 |perm|
  const int K = std::max(1, static_cast<int>(std::ceil((std::max(sc.log2_perm, 0.0) + 2.0) / 48.99)));
  if (K > kIntMaxPrimes)
    return fail(PQP_ERR_RANGE, "the permanent may exceed 2^390 in magnitude: beyond the eight moduli");
  if (n == 0) {  // empty selection: 1 (src/permanent.cpp:106-108)
    std::memset(v, 0, kIntLimbs * sizeof(uint64_t));
    v[0] = 1;
    return PQP_OK;
  }
  // Gray terms, with the first smallest row one lower
  int least = 0;
  int64_t i0 = 0;
  for (int64_t i = 0; i < in.m_r; ++i)
    if (in.rows[i] > 0 && (!least || in.rows[i] < least)) {
      least = in.rows[i];
      i0 = i;
    }
  double states = 1.0;  // of the digits of larger radix
  int nb = 0, m = 0;
  for (int64_t i = 0; i < in.m_r; ++i) {
    const int rho = in.rows[i] - (i == i0 ? 1 : 0);
    m += in.rows[i] > 0;
    if (rho == 1) ++nb;
    if (rho > 1) states *= rho + 1;
  }
  const double terms = std::ldexp(states, nb);
  if (terms > 0x1p62) return fail(PQP_ERR_RANGE, "item 0: Gray term count exceeds 2^62");
  IntArgs a;
  a.k_max = 0;
  while (a.k_max < kIntInnerDigits && terms / 64.0 / (1 << a.k_max) > static_cast<double>(kIntWaves)) ++a.k_max;
  int k = 0;
  while (k < a.k_max && k < nb && std::ldexp(states, nb - k - 1) >= 64.0) ++k;
  const double top = std::ldexp(states, nb - k);
  if (top >= 0x1p50) return fail(PQP_ERR_RANGE, "item 0: too many top states");
  a.waves = static_cast<int32_t>(std::min(std::ceil(top / 64.0), 8.0 * static_cast<double>(kIntWaves)));
  int st;
  if ((st = require_device()) != PQP_OK) return st;
  IntState &S = int_state();
  std::lock_guard<std::mutex> lock(S.mu);
  if ((st = ensure_stream(S.stream)) != PQP_OK) return st;
  // the moduli table: p, 1/p, 2^-(n-1) mod p; then the rows with each column
  // repeated by its multiplicity, and their multiplicities
  const int W = n <= 32 ? (n + 3) / 4 * 4 : (n + 7) / 8 * 8;
  const size_t o_rows = 3 * kIntMaxPrimes * sizeof(double);
  const size_t o_occ = o_rows + static_cast<size_t>(m + 1) * W * sizeof(double);
  const size_t in_bytes = o_occ + static_cast<size_t>(m);
  if ((st = S.in.ensure(in_bytes)) != PQP_OK) return st;
  if ((st = S.stage.ensure(in_bytes)) != PQP_OK) return st;
  if ((st = S.work.ensure(static_cast<size_t>(K) * a.waves * sizeof(double))) != PQP_OK) return st;
  if ((st = S.res.ensure((kIntMaxPrimes + 1) * sizeof(double))) != PQP_OK) return st;
  char *h = static_cast<char *>(S.stage.p);
  double *mt = reinterpret_cast<double *>(h);
  for (int q = 0; q < kIntMaxPrimes; ++q) {
    const uint64_t p = kIntPrimes[q];
    mt[q] = static_cast<double>(p);
    mt[kIntMaxPrimes + q] = 1.0 / static_cast<double>(p);
    mt[2 * kIntMaxPrimes + q] = q < K ? static_cast<double>(pow_mod((p + 1) / 2, static_cast<uint64_t>(n - 1), p)) : 0.0;
  }
  double *rows = reinterpret_cast<double *>(h + o_rows);
  auto fill = [&](int64_t i, double *dst, double pad) {
    int at = 0;
    for (int64_t j = 0; j < in.m_c; ++j) {
      if (in.cols[j] == 0) continue;
      const int64_t e = 2 * (i * in.ld + j);
      const double x = in.a_is_float ? static_cast<const float *>(in.a)[e] : static_cast<const double *>(in.a)[e];
      for (int32_t q = 0; q < in.cols[j]; ++q) dst[at++] = x;
    }
    while (at < W) dst[at++] = pad;
  };
  int at = 0;
  for (int64_t i = 0; i < in.m_r; ++i) {
    if (in.rows[i] == 0) continue;
    fill(i, rows + static_cast<size_t>(at) * W, 0.0);
    h[o_occ + at] = static_cast<char>(in.rows[i]);
    ++at;
  }
  fill(i0, rows + static_cast<size_t>(m) * W, 1.0);
  PQP_HIP(hipMemcpyAsync(S.in.p, h, in_bytes, hipMemcpyHostToDevice, S.stream));
  const char *d = static_cast<const char *>(S.in.p);
  a.mod = reinterpret_cast<const double *>(d);
  a.rows = reinterpret_cast<const double *>(d + o_rows);
  a.occ = reinterpret_cast<const uint8_t *>(d + o_occ);
  a.partials = static_cast<double *>(S.work.p);
  a.out = static_cast<double *>(S.res.dev);
  a.modes = m;
  a.n = n;
  a.n_primes = K;
  a.group = group;
  a.done = static_cast<uint64_t *>(S.res.dev) + kIntMaxPrimes;
  a.seq = ++S.seq;
  volatile uint64_t *done = static_cast<uint64_t *>(S.res.host) + kIntMaxPrimes;
  *done = 0;
  PQP_HIP(launch_int(W, a, S.stream));
  PQP_HIP(launch_int_sum(a, S.stream));
  if ((st = wait_done(S.stream, done, a.seq)) != PQP_OK) return st;
  crt_limbs(static_cast<const double *>(S.res.host), K, v);
  return PQP_OK;
}

// Key of a single-permanent plan: everything the plan's tables depend on
// (shape, multiplicities, flags, input precision); the matrix values only
// fill the rows of B.
void single_key(const PermInput &in, uint32_t flags, std::vector<int64_t> &key) {
  key.clear();
  key.push_back(in.m_r);
  key.push_back(in.m_c);
  key.push_back(static_cast<int64_t>(flags));
  key.push_back(in.a_is_float ? 1 : 0);
  for (int64_t i = 0; i < in.m_r; ++i) key.push_back(in.rows[i]);
  for (int64_t j = 0; j < in.m_c; ++j) key.push_back(in.cols[j]);
}

// A single permanent on perm_one.hip: one launch, polled.
int run_one(OnePlan &p, double *out2, double *out_dd4) {
  int st;
  if ((st = require_device()) != PQP_OK) return st;
  SingleState &S = single_state();
  std::lock_guard<std::mutex> lock(S.mu);
  constexpr size_t kPartials = 256;  // after the counter
  if (!S.init_one) {
    if ((st = ensure_stream(S.one_stream)) != PQP_OK) return st;
    if ((st = S.one_res.ensure(8 * sizeof(double))) != PQP_OK) return st;
    if ((st = S.one_work.ensure(kPartials + static_cast<size_t>(kOneMaxBlocks) * 5 * sizeof(double))) != PQP_OK)
      return st;
    PQP_HIP(hipMemsetAsync(S.one_work.p, 0, kPartials, S.one_stream));
    S.init_one = true;
  }
  thread_local OneArgs a;
  one_fill(p, a);
  char *work = static_cast<char *>(S.one_work.p);
  OneHead &h = a.rows.h;
  h.counter = reinterpret_cast<int *>(work);
  h.partials = reinterpret_cast<double *>(work + kPartials);
  h.out = static_cast<double *>(S.one_res.dev);
  h.done = reinterpret_cast<uint64_t *>(h.out + 7);
  h.seq = ++S.one_seq;
  const double *res = static_cast<const double *>(S.one_res.host);
  volatile uint64_t *done = static_cast<uint64_t *>(S.one_res.host) + 7;
  *done = 0;
  PQP_HIP(p.fp32 ? launch_one_f(p.width, p.kind, a, p.blocks, p.waves, S.one_stream)
                 : launch_one_d(p.width, p.kind, a, p.blocks, p.waves, S.one_stream));
  if ((st = wait_done(S.one_stream, done, h.seq)) != PQP_OK) {
    // a launch that did not finish its count leaves it behind
    (void)hipMemsetAsync(h.counter, 0, sizeof(int), S.one_stream);
    (void)hipStreamSynchronize(S.one_stream);
    return st;
  }
  out2[0] = res[0];
  out2[1] = res[1];
  if (out_dd4) std::memcpy(out_dd4, res + 2, 4 * sizeof(double));
  g_last_bound = sweep_error_bound(p.n, p.fp32, res[6], res[0], res[1]);
  return PQP_OK;
}

int run_single(const PermInput &in, uint32_t flags, double *out2, double *out_dd4) {
  const bool args_ok = in.m_r >= 0 && in.m_c >= 0 && (in.m_r * in.m_c == 0 || in.a) &&
                       (in.m_r == 0 || in.rows) && (in.m_c == 0 || in.cols) &&
                       (in.m_r == 0 || in.ld >= in.m_c);
  int st;
  if (args_ok && !(flags & PQP_FLAG_PLAIN)) {
    // Integer matrices whose Glynn terms may leave the exact integers of
    // the floating-point sweep (FP32 products: 2^24; FP64 products summed
    // in runs of kDdFold before the double-double fold: 2^53 / kDdFold)
    // take the multi-modular path: the exact permanent, rounded once.  The
    // scan stops at the first entry that is not an integer.
    const IntScan sc = int_scan(in);
    const bool fp32 = in.a_is_float || (flags & PQP_FLAG_FP32);
    if (sc.integral && sc.log2_term >= (fp32 ? 24.0 : 53.0 - std::log2(double(kDdFold)))) {
      uint64_t v[kIntLimbs];
      st = run_int(in, sc, v);
      if (st == PQP_OK) {
        out2[0] = limbs_round(v, fp32 ? 24 : 53);
        out2[1] = 0.0;
        g_last_bound = std::fabs(out2[0]) * (fp32 ? 0x1p-24 : 0x1p-53);  // one rounding
        if (out_dd4) {
          const double hi = limbs_round(v, 53);
          limbs_sub_double(v, hi);
          out_dd4[0] = hi;
          out_dd4[1] = limbs_round(v, 53);
          out_dd4[2] = out_dd4[3] = 0.0;
        }
        return PQP_OK;
      }
      if (st != PQP_ERR_RANGE) return st;
      // beyond the moduli or the weight bound: the floating-point sweep
      g_error.clear();
    }
  }
  OnePlan one;
  if (args_ok && one_plan(in, flags, one)) return run_one(one, out2, out_dd4);
  SingleState &S = single_state();
  std::unique_lock<std::mutex> lock(S.mu);
  Exec &x = S.xs;
  // A call with the plan key of the previous one (same shape, multiplicities
  // and flags) reuses its plan and device tables and refreshes only the
  // rows of B.  Planning validates the arguments first, so argument errors
  // are reported the same way with or without a device.
  thread_local std::vector<int64_t> key;
  if (args_ok) single_key(in, flags, key);
  const bool hit = args_ok && S.xs_planned && key == S.xs_key;
  if (!hit) {
    Plan plan;
    std::string err;
    S.xs_planned = false;
    st = plan_build(std::vector<PermInput>{in}, single_plan_options(flags, in), plan, err);
    if (st != PQP_OK) return fail(st, err);
    if ((st = require_device()) != PQP_OK) return st;
    if ((st = ensure_stream(x.stream)) != PQP_OK) return st;
    x.mapped_results = true;
    x.plan = std::move(plan);
    index_units(x);
    x.flags = (flags & PQP_FLAG_PLAIN) | PQP_FLAG_STATIC;
    if ((st = upload(x)) != PQP_OK) return st;
    S.xs_key = key;
    S.xs_planned = args_ok;
  }
  const ItemDesc &d = x.plan.items[0];
  const int n = d.n;
  const bool fp32 = x.plan.fp32;
  double *res = static_cast<double *>(x.results_m.host);
  const size_t b_bytes = x.plan.info[0].rowsrc.size() * static_cast<size_t>(d.mcp) * 2 *
                         (fp32 ? sizeof(float) : sizeof(double));
  if (hit) {
    plan_refresh_matrix(x.plan, std::vector<PermInput>{in});
    if (!x.plan.info[0].trivial_one) {
      const size_t off = static_cast<size_t>(d.b_off);
      std::memcpy(static_cast<char *>(x.stage.p) + off, x.plan.arena.data() + off, b_bytes);
      PQP_HIP(hipMemcpyAsync(static_cast<char *>(x.arena.p) + off, static_cast<char *>(x.stage.p) + off,
                             b_bytes, hipMemcpyHostToDevice, x.stream));
    }
  }
  if ((st = enqueue(x, (flags & PQP_FLAG_PLAIN) ? PQP_RUN_PLAIN : PQP_RUN_EAGER, nullptr, nullptr)) != PQP_OK)
    return st;
  PQP_HIP(hipStreamSynchronize(x.stream));
  // one item: results = [out (2)][out_dd (4)][term magnitudes (1)],
  // written by the kernels into mapped host memory
  out2[0] = res[0];
  out2[1] = res[1];
  if (out_dd4) std::memcpy(out_dd4, res + 2, 4 * sizeof(double));
  // (the plain baseline runs the non-compensated kernel, which keeps no
  // term magnitudes)
  g_last_bound = n == 0 ? 0.0
                 : x.abs_valid ? sweep_error_bound(n, fp32, res[6], res[0], res[1])
                               : std::numeric_limits<double>::quiet_NaN();
  return PQP_OK;
}

// Gradients beyond the single-sweep kernel (more than 32 particles): the
// column-minor inputs, one item per row with
// non-zero multiplicity, rows r - e_i, columns c.
void minor_inputs(const std::vector<PermInput> &inputs, std::vector<std::vector<int32_t>> &rows,
                  std::vector<int64_t> &item, std::vector<int64_t> &row,
                  std::vector<PermInput> &out) {
  rows.clear();
  item.clear();
  row.clear();
  out.clear();
  for (size_t k = 0; k < inputs.size(); ++k) {
    const PermInput &in = inputs[k];
    for (int64_t i = 0; i < in.m_r; ++i)
      if (in.rows[i] > 0) {
        rows.emplace_back(in.rows, in.rows + in.m_r);
        rows.back()[i] -= 1;
        item.push_back(static_cast<int64_t>(k));
        row.push_back(i);
      }
  }
  for (size_t q = 0; q < rows.size(); ++q) {
    const PermInput &in = inputs[item[q]];
    out.push_back(PermInput{in.a, in.a_is_float, in.m_r, in.m_c, in.ld, rows[q].data(), in.cols});
  }
}

// Complex results of the column-minor plan of x (host copy of x.out).
int fetch_out(Exec &x, std::vector<double> &res) {
  res.assign(static_cast<size_t>(std::max<int64_t>(x.plan.n_out, 1)) * 2, 0.0);
  PQP_HIP(hipMemcpyAsync(res.data(), x.results.p, res.size() * sizeof(double),
                         hipMemcpyDeviceToHost, x.stream));
  PQP_HIP(hipStreamSynchronize(x.stream));
  return PQP_OK;
}

// grad[i, j] = r_i c_j perm(A; r - e_i, c - e_j) from the column-minor results.
// Column minors perm(A; r, c - e_l), l < m_c, of problems with
// sum c = sum r + 1, as one plan, and where each lands in its output:
// slot[q][l] is the complex output index of problem q's minor l.  Problems
// with at most 32 columns of non-zero multiplicity run on the column-minor
// kernels (one sweep for all of a problem's minors).  If any problem is
// wider, every problem runs as forward items instead, one per column: rows
// r and columns c - e_l, or for c_l = 0 columns c with one column to spare
// (the uncut product the reference's loop gives such a column,
// src/permanent_laplace.cpp:168-172); the forward kernels take every width
// up to 64.
struct MinorsPlan {
  Plan plan;
  std::vector<std::vector<int64_t>> slot;
};

constexpr int64_t kMinorsMaxCols = 32;

int build_minors_plan(const std::vector<PermInput> &probs, PlanOptions opt, MinorsPlan &mp,
                      std::string &err) {
  bool wide = false;
  for (const PermInput &in : probs) {
    int64_t nz = 0;
    if (in.cols)
      for (int64_t j = 0; j < in.m_c; ++j) nz += in.cols[j] > 0;
    wide = wide || nz > kMinorsMaxCols;
  }
  mp.slot.assign(probs.size(), {});
  if (!wide) {
    opt.minors = true;
    const int st = plan_build(probs, opt, mp.plan, err);
    if (st != PQP_OK) return st;
    for (size_t q = 0; q < probs.size(); ++q) {
      const ItemInfo &inf = mp.plan.info[q];
      const int64_t mc = static_cast<int64_t>(inf.colsrc.size());
      // columns of zero multiplicity get the uncut product (slot mc)
      mp.slot[q].assign(static_cast<size_t>(std::max<int64_t>(probs[q].m_c, 0)), inf.out_offset + mc);
      for (int64_t l = 0; l < mc; ++l) mp.slot[q][static_cast<size_t>(inf.colsrc[l])] = inf.out_offset + l;
    }
    return PQP_OK;
  }
  // validate as the minors planner does before expanding into items
  for (size_t q = 0; q < probs.size(); ++q) {
    const PermInput &in = probs[q];
    if (in.m_r < 0 || in.m_c < 0 || (in.m_r * in.m_c > 0 && !in.a) || (in.m_r > 0 && !in.rows) ||
        (in.m_c > 0 && !in.cols) || (in.m_r > 0 && in.ld < in.m_c)) {
      err = "item " + std::to_string(q) + ": invalid shape or null pointer";
      return PQP_ERR_INVALID;
    }
    int64_t sr = 0, sc = 0;
    for (int64_t i = 0; i < in.m_r; ++i) {
      if (in.rows[i] < 0) {
        err = "item " + std::to_string(q) + ": negative row multiplicity";
        return PQP_ERR_INVALID;
      }
      sr += in.rows[i];
    }
    for (int64_t j = 0; j < in.m_c; ++j) {
      if (in.cols[j] < 0) {
        err = "item " + std::to_string(q) + ": negative column multiplicity";
        return PQP_ERR_INVALID;
      }
      sc += in.cols[j];
    }
    if (sr + 1 != sc) {
      err = "column multiplicities must sum to one more than the row multiplicities";
      return PQP_ERR_SUM_MISMATCH;
    }
  }
  size_t n_items = 0;
  for (const PermInput &in : probs) n_items += static_cast<size_t>(in.m_c);
  std::vector<std::vector<int32_t>> cols(n_items);
  std::vector<PermInput> items;
  items.reserve(n_items);
  for (size_t q = 0; q < probs.size(); ++q) {
    const PermInput &in = probs[q];
    for (int64_t l = 0; l < in.m_c; ++l) {
      std::vector<int32_t> &c = cols[items.size()];
      c.assign(in.cols, in.cols + in.m_c);
      PermInput it = in;
      if (c[static_cast<size_t>(l)] > 0) {
        c[static_cast<size_t>(l)] -= 1;
        it.col_excess = 0;
      } else {
        it.col_excess = 1;
      }
      it.cols = c.data();
      mp.slot[q].push_back(static_cast<int64_t>(items.size()));
      items.push_back(it);
    }
  }
  opt.minors = false;
  const int st = plan_build(items, opt, mp.plan, err);
  if (st != PQP_OK) return st;
  for (size_t q = 0; q < probs.size(); ++q)
    for (int64_t &s : mp.slot[q]) s = mp.plan.info[static_cast<size_t>(s)].out_offset;
  return PQP_OK;
}

// grad[i, j] = r_i c_j perm(A; r - e_i, c - e_j) from the column minors of
// the problems (rows r - e_i, columns c), minor q of permanent mitem[q].
void scatter_gradients(const std::vector<std::vector<int64_t>> &slot, const std::vector<double> &res,
                       const std::vector<int64_t> &mitem, const std::vector<int64_t> &mrow,
                       const std::vector<PermInput> &inputs, double *const *grads) {
  for (size_t k = 0; k < inputs.size(); ++k)
    if (grads[k])
      std::memset(grads[k], 0, static_cast<size_t>(inputs[k].m_r * inputs[k].m_c) * 2 * sizeof(double));
  for (size_t q = 0; q < mitem.size(); ++q) {
    const PermInput &in = inputs[mitem[q]];
    double *g = grads[mitem[q]];
    if (!g) continue;
    const int64_t i = mrow[q];
    const double ri = static_cast<double>(in.rows[i]);
    for (int64_t j = 0; j < in.m_c; ++j) {
      if (in.cols[j] <= 0) continue;
      const double f = ri * static_cast<double>(in.cols[j]);
      const double *m = res.data() + 2 * slot[q][static_cast<size_t>(j)];
      g[2 * (i * in.m_c + j)] = f * m[0];
      g[2 * (i * in.m_c + j) + 1] = f * m[1];
    }
  }
}

// The single-sweep gradient kernels keep up to 32 row sums per lane, and a
// gradient item's columns of multiplicity c are expanded into c columns, so
// they take permanents of at most 32 particles; larger ones (up to 64, with
// at most 32 distinct columns) run as one column-minor sweep per row.
constexpr int64_t kGradSweepMaxN = 32;

bool gradients_fit_single_sweep(const std::vector<PermInput> &inputs) {
  for (const PermInput &in : inputs) {
    int64_t n = 0;
    for (int64_t i = 0; i < in.m_r; ++i) n += std::max(in.rows[i], 0);
    if (n > kGradSweepMaxN) return false;
  }
  return true;
}

// Results of a gradient plan: perms[k] (2 doubles, may be null) and
// grads[k][i, j] = d perm / d A_ij = the sum of G_B[b, j'] over the rows b
// of B that copy row i of A (the prepended row and row i0's digit row both
// copy A's row i0) and the kernel columns j' that copy column j (c_j of
// them); rows or columns of multiplicity 0 get 0.  This equals
// r_i c_j perm(A; r - e_i, c - e_j) (src/permanent.cpp:271-300).
void scatter_grad_items(const Plan &p, const std::vector<double> &res,
                        const std::vector<PermInput> &inputs, double *perms, double *const *grads) {
  for (size_t k = 0; k < inputs.size(); ++k) {
    const ItemInfo &inf = p.info[k];
    const ItemDesc &d = p.items[k];
    const double *r = res.data() + 2 * inf.out_offset;
    if (perms) {
      perms[2 * k] = r[0];
      perms[2 * k + 1] = r[1];
    }
    double *g = grads ? grads[k] : nullptr;
    if (!g) continue;
    const PermInput &in = inputs[k];
    std::memset(g, 0, static_cast<size_t>(in.m_r * in.m_c) * 2 * sizeof(double));
    if (inf.trivial_one) continue;
    const int rows_B = 1 + d.L + d.Dt;
    for (int b = 0; b < rows_B; ++b) {
      const int64_t i = inf.rowsrc[b];
      for (int j = 0; j < d.mc; ++j) {
        // kernel columns have unit multiplicity: a column of multiplicity c
        // was planned as c copies, whose entries add up here
        const int64_t col = inf.colsrc[j];
        const double *v = r + 2 * (1 + static_cast<int64_t>(b) * d.mc + j);
        g[2 * (i * in.m_c + col)] += v[0];
        g[2 * (i * in.m_c + col) + 1] += v[1];
      }
    }
  }
}

// pqp_grad_batch_c128 for permanents above 32 particles: the permanents,
// then one column-minor sweep per row of non-zero multiplicity.
int grad_batch_minors(const std::vector<PermInput> &inputs, double *perms, double *const *grads);

}  // namespace

namespace {

// ------------------------------------------------------- tensor permanents --

// Buffers of tensor permanents, kept across calls (grown on demand): `in`
// the work units and what the host sends, `work` the matrices, sign rows and
// partials of a pass (kTensorBytes of sign rows, or one item's), `out` the
// results.
struct TensorState {
  std::mutex mu;
  hipStream_t stream = nullptr;
  DevBuf in, work, out;
  HostBuf stage;
  MappedBuf res;  // results of few items
};

// Items whose results the kernel writes to host memory (a copy of a few would
// cost a launch more than it moves: 5 us a call).
constexpr size_t kTensorMapped = 4096;

TensorState &tensor_state() {
  static TensorState *s = new TensorState();  // never destroyed: outlives atexit HIP teardown
  return *s;
}

constexpr size_t kTensorBytes = size_t{512} << 20;

// Steps per unit 2^kt for sign vectors of nb free signs, the same whatever
// the number of items (a value does not depend on its company): at most 512
// steps, or as many as keep the units near 2^20 (large n), fewer where that
// leaves less than about 8192 units, at least 16 (a unit's start costs about
// four), or 8 up to 9 particles, whose few units one output would wait for
// (9 particles, one output 40 -> 38 us, 300 108; 10 particles, 2000 outputs
// 1232 us by 16, 1460 by 8).  Against 4096 units of up to 1024 steps: 15
// particles, two outputs 1468 -> 1330 us, 16 particles 3041 -> 2780 us (the
// last waves run alone for less time); 32768 units cost one output of 14
// particles 351 us instead of 237.
int tensor_walk_bits(int nb, int ls) {
  auto units = [&](int kt) {
    return std::ldexp(1.0, (nb - ls) + (nb - kt)) / 2.0;
  };
  int kt = std::min(nb, 9);
  while (kt < nb && units(kt) > 1048576.0) ++kt;
  while (kt > 4 && units(kt) < 8192.0) --kt;
  if (kt == 4 && units(kt) <= 32.0) kt = 3;
  return kt;
}

// The work units of one item of order n >= 1, by eps block: neighbouring
// units then read the same sign rows.
void tensor_units(int n, int *ls, int *kt, std::vector<TensorUnit> &units) {
  const int nb = n - 1;  // free signs of a sign vector
  *ls = std::min(nb, 6);
  *kt = tensor_walk_bits(nb, *ls);
  const uint32_t n_s = 1u << (nb - *ls);
  const uint32_t n_t = 1u << (nb - *kt);
  units.clear();
  for (uint32_t tb = 0; tb < n_t; ++tb)
    for (uint32_t sh = 0; sh < n_s; ++sh) {
      const uint64_t lo = static_cast<uint64_t>(tb) << *kt;
      const uint64_t hi = lo + (1ull << *kt) - 1;
      if ((hi >> *ls) < sh) continue;  // every pair below the diagonal block
      units.push_back(TensorUnit{static_cast<int32_t>(sh), static_cast<int32_t>(tb), (lo >> *ls) <= sh ? 1 : 0});
    }
}

// Items per pass, and the layout of the work buffer for them: matrices, (1 -
// x)|A|^2, sign rows, partials.
struct TensorPass {
  int64_t items;
  size_t pw, signs, partials, bytes;
};

TensorPass tensor_pass(int n, int64_t count, size_t n_units) {
  TensorPass t;
  const size_t sign_bytes = (static_cast<size_t>(n) << (n - 1)) * 16;
  t.items = std::min<int64_t>(std::min<int64_t>(count, 32768),
                              std::max<int64_t>(1, static_cast<int64_t>(kTensorBytes / sign_bytes)));
  const size_t m = static_cast<size_t>(t.items), nn = static_cast<size_t>(n) * n;
  auto align = [](size_t v) { return (v + 255) & ~size_t{255}; };
  t.pw = align(m * nn * 16);
  t.signs = align(t.pw + m * nn * 8);
  t.partials = align(t.signs + m * sign_bytes);
  t.bytes = t.partials + m * n_units * 3 * sizeof(double);
  return t;
}

void tensor_buffers(TensorArgs &a, const TensorPass &t, char *work) {
  a.cols = reinterpret_cast<double *>(work);
  a.pw = reinterpret_cast<double *>(work + t.pw);
  a.signs = reinterpret_cast<double *>(work + t.signs);
  a.partials = reinterpret_cast<double *>(work + t.partials);
}

// One evaluation of a batch (gradient batches have no plain mode: their
// one sweep gives the permanents and the gradients).
int enqueue_all(pqp_batch *b, int mode, hipEvent_t ev_begin, hipEvent_t ev_end) {
  if (b->grad_minors) {
    int st = enqueue(b->x, mode, ev_begin, nullptr);
    if (st != PQP_OK) return st;
    return enqueue(b->xm, mode == PQP_RUN_PLAIN ? PQP_RUN_EAGER : mode, nullptr, ev_end);
  }
  if (b->grad && mode == PQP_RUN_PLAIN) mode = PQP_RUN_EAGER;
  return enqueue(b->x, mode, ev_begin, ev_end);
}
}  // namespace

namespace {

// Device buffers of the matrix-polynomial permanent entry point, kept across
// calls (grown on demand), with their own stream and lock.
struct PolyState {
  std::mutex mu;
  hipStream_t stream = nullptr;
  DevBuf arena, scratch, acc, out;
  HostBuf stage;
  // the last plan and the exponent rows it was built for
  bool have_plan = false;
  bool tables_on_device = false;  // the plan's tables are in `arena`
  int64_t key_n = 0, key_vars = 0, key_out = 0;
  std::vector<int32_t> key_exps;
  PolyPlan plan;
  std::vector<int16_t> subsets;        // poly_subsets of the plan's order (layer path)
  std::vector<uint16_t> subset_bits;
  std::vector<int64_t> subset_first;
};

PolyState &poly_state() {
  static PolyState *s = new PolyState();  // never destroyed: outlives atexit HIP teardown
  return *s;
}

size_t align256(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }

// The layer path's subset tables for matrices of order n: the subsets of
// 0 .. n - 1 columns by size, each size in increasing order of their bits
// (`bits`), and for each subset and column j the place of the subset
// without j in the next smaller size (`sub`; -1 when it does not hold j).
// first[i]: subsets of sizes 0 .. i - 1.
void poly_subsets(int n, std::vector<int16_t> &sub, std::vector<uint16_t> &bits,
                  std::vector<int64_t> &first) {
  std::vector<int16_t> place(size_t{1} << n, 0);
  sub.clear();
  bits.clear();
  first.assign(static_cast<size_t>(n) + 1, 0);
  for (int i = 0; i < n; ++i) {
    int16_t at = 0;
    first[i] = static_cast<int64_t>(bits.size());
    for (uint32_t s = 0; s < (1u << n); ++s) {
      if (__builtin_popcount(s) != i) continue;
      place[s] = at++;
      bits.push_back(static_cast<uint16_t>(s));
      for (int j = 0; j < n; ++j)
        sub.push_back((s >> j & 1u) ? place[s & ~(1u << j)] : static_cast<int16_t>(-1));
    }
  }
}

// Whether a polynomial permanent takes the layer path: the subsets of one
// size fit a block's threads, a row's coefficients its LDS, and the two
// largest layers 8 GiB.  Few outputs of 6 or 7 particles do not: their
// layers are as many kernels one after another, where the subset sum is one
// kernel and a reduction over outputs and workgroups (a call, layers against
// subsets: 6 particles in 4 modes, one output 61 and 50 us, 64 outputs 61 and
// 59, 210 outputs 57 and 61; 7 particles 62 and 59, 4 outputs 63 and 66; at 5
// particles the layers take 41 against 41 or less, at 8 67 against 85).
// `bytes` receives the size of one layer buffer.
bool poly_layers_fit(const PolyPlan &p, size_t *bytes) {
  if (p.out_index.empty()) return false;  // nothing to evaluate, no levels
  if (p.n > kPolyLayerMaxN || static_cast<size_t>(p.n) * (p.M + 1) * sizeof(double2) > 16384) return false;
  if ((p.n == 6 && p.out_index.size() <= kPolyFew6) || (p.n == 7 && p.out_index.size() <= kPolyFew7)) return false;
  double most = 1.0, choose = 1.0;
  for (int i = 1; i < p.n; ++i) {
    choose = choose * (p.n - i + 1) / i;
    most = std::max(most, choose * p.lvl_off[std::min(i, p.L) + 1]);
  }
  *bytes = static_cast<size_t>(most) * sizeof(double2);
  return *bytes <= (size_t{4} << 30);
}

// Buffers of the device-planned column minors: a lone problem (`res` holds
// its results and the done slot) and the sampler's steps, each with its own
// stream, kept across calls.
struct MinorsState {
  std::mutex mu;
  bool init = false;
  hipStream_t stream = nullptr;
  DevBuf in, work, counter;
  HostBuf stage;
  MappedBuf res;
  uint64_t seq = 0;
};

MinorsState &laplace_state() {
  static MinorsState *s = new MinorsState();  // never destroyed: outlives atexit HIP teardown
  return *s;
}

MinorsState &sample_state() {
  static MinorsState *s = new MinorsState();
  return *s;
}

// Column minors of one problem whose columns all hold one particle, planned
// by the kernel's waves: no tables, one copy (rows of non-zero multiplicity,
// compacted), two launches, the result polled.  Other problems (columns of
// other multiplicities, or wider) return false.
bool laplace_wave_fits(const PermInput &in) {
  if (in.m_r < 1 || in.m_c < 2 || in.m_c > kMinorsWaveMaxCols || !in.a || !in.rows || !in.cols || in.ld < in.m_c)
    return false;
  int64_t sr = 0;
  for (int64_t i = 0; i < in.m_r; ++i) {
    if (in.rows[i] < 0) return false;
    sr += in.rows[i];
  }
  for (int64_t j = 0; j < in.m_c; ++j)
    if (in.cols[j] != 1) return false;
  return sr + 1 == in.m_c;
}

int laplace_wave(const PermInput &in, double *out) {
  int st;
  if ((st = require_device()) != PQP_OK) return st;
  const int W = static_cast<int>(in.m_c);
  MinorsState &S = laplace_state();
  std::lock_guard<std::mutex> lock(S.mu);
  if (!S.init) {
    if ((st = ensure_stream(S.stream)) != PQP_OK) return st;
    if ((st = S.counter.ensure(sizeof(int))) != PQP_OK) return st;
    PQP_HIP(hipMemsetAsync(S.counter.p, 0, sizeof(int), S.stream));
    S.init = true;
  }
  // the occupied rows, and the digits the waves will find in them
  const size_t row_bytes = static_cast<size_t>(W) * 2 * sizeof(double);
  const size_t o_occ = static_cast<size_t>(W - 1) * row_bytes;  // at most W - 1 occupied rows
  const size_t in_bytes = o_occ + static_cast<size_t>(W);
  if ((st = S.stage.ensure(in_bytes)) != PQP_OK) return st;
  if ((st = S.in.ensure(in_bytes)) != PQP_OK) return st;
  char *h = static_cast<char *>(S.stage.p);
  int m = 0, least = 0, ones = 0;
  for (int64_t i = 0; i < in.m_r; ++i) {
    const int r = in.rows[i];
    if (r == 0) continue;
    std::memcpy(h + m * row_bytes, static_cast<const double *>(in.a) + 2 * i * in.ld, row_bytes);
    h[o_occ + m] = static_cast<char>(r);
    if (!least || r < least) least = r;
    ones += r == 1;
    ++m;
  }
  int64_t states = 1;  // of the digits of larger radix
  bool prepended = false;
  int nb = ones;
  for (int i = 0; i < m; ++i) {
    int rho = h[o_occ + i];
    if (!prepended && rho == least) {
      prepended = true;
      if (rho == 1) --nb;
      --rho;
      if (rho == 1) ++nb;
    }
    if (rho > 1) states *= rho + 1;
  }
  // Waves of one state per lane up to kLaplaceWaves of them (two per SIMD,
  // what the widest kernels hold), longer ones beyond: a lone call waits for
  // its slowest wave, and a state costs a fifth of the start and the sums.
  MinorsWaveArgs a;
  const int64_t terms = states << nb;
  a.k_max = 0;
  while (a.k_max < 7 && terms >> (6 + a.k_max) > kLaplaceWaves) ++a.k_max;
  int k = 0;
  while (k < a.k_max && k < nb && (states << (nb - k - 1)) >= 64) ++k;
  a.waves = static_cast<int32_t>(std::min<int64_t>(((terms >> k) + 63) / 64, 16 * kLaplaceWaves));
  if ((st = S.work.ensure(static_cast<size_t>(a.waves) * 4 * W * sizeof(double))) != PQP_OK) return st;
  const size_t res_bytes = static_cast<size_t>(kMinorsWaveMaxCols) * 2 * sizeof(double);
  if ((st = S.res.ensure(res_bytes + sizeof(uint64_t))) != PQP_OK) return st;
  PQP_HIP(hipMemcpyAsync(S.in.p, h, in_bytes, hipMemcpyHostToDevice, S.stream));
  a.rows = static_cast<const double *>(S.in.p);
  a.occ = static_cast<const uint8_t *>(S.in.p) + o_occ;
  a.units = nullptr;
  a.partials = static_cast<double *>(S.work.p);
  a.out = static_cast<double *>(S.res.dev);
  a.item_stride = 0;
  a.ld = W;
  a.modes = m;
  a.last_counter = static_cast<int *>(S.counter.p);
  a.done = reinterpret_cast<uint64_t *>(static_cast<char *>(S.res.dev) + res_bytes);
  a.seq = ++S.seq;
  volatile uint64_t *done = reinterpret_cast<volatile uint64_t *>(static_cast<char *>(S.res.host) + res_bytes);
  *done = 0;
  PQP_HIP(launch_minors_wave(W, a, 1, S.stream));
  PQP_HIP(launch_minors_sum(W, a, S.stream));
  if ((st = wait_done(S.stream, done, a.seq)) != PQP_OK) {
    // a launch that did not finish its count leaves it behind
    (void)hipMemsetAsync(S.counter.p, 0, sizeof(int), S.stream);
    (void)hipStreamSynchronize(S.stream);
    return st;
  }
  std::memcpy(out, S.res.host, static_cast<size_t>(W) * 2 * sizeof(double));
  return PQP_OK;
}

// Sizes of the sampler's passes over a call's shots.  Every pass, the short
// last one too, takes the same inner digits and waves per shot at a step, so
// the partials, sized for the longest pass, hold any of them.
struct SamplePasses {
  int64_t most;                       // shots of a pass at most
  int32_t digits[kMinorsWaveMaxCols + 1], waves[kMinorsWaveMaxCols + 1];  // of each step's minors
  size_t partials;                    // bytes
};

SamplePasses sample_passes(int64_t shots, int64_t photons) {
  SamplePasses p;
  const int64_t passes = std::max<int64_t>(1, (shots + kSampleShots - 1) / kSampleShots);
  p.most = (shots + passes - 1) / passes;
  p.partials = 0;
  p.digits[0] = p.waves[0] = 0;  // no minors before the first photon
  // Most shots have bunched outputs and need fewer waves than 2^(step - 1)
  // terms would; those left over end at once.  8 states a lane at least (the
  // start and the sums cost as much as a handful of states), 64 where that
  // leaves 8192 waves.
  for (int64_t step = 1; step <= photons; ++step) {
    int k = 3;
    while (k < 6 && p.most * (int64_t{1} << (step - 1)) >= (int64_t{64} * 8192) << (k + 1)) ++k;
    p.digits[step] = k;
    p.waves[step] = static_cast<int32_t>(
        std::min<int64_t>(64, std::max<int64_t>(1, (int64_t{1} << (step - 1)) >> (6 + k))));
    if (step < photons)
      p.partials = std::max(p.partials, static_cast<size_t>(p.most) * p.waves[step] * 4 * (step + 1) * sizeof(double));
  }
  return p;
}

// Buffers of the probability-table entry point, kept across calls (grown on
// demand, bounded by kTableSegment rows), with their own stream and lock.
struct TableState {
  std::mutex mu;
  hipStream_t stream = nullptr;
  DevBuf in, out, states;
  HostBuf stage;
};

TableState &table_state() {
  static TableState *s = new TableState();  // never destroyed: outlives atexit HIP teardown
  return *s;
}

// Rows of a table in one pass over the buffers (64 modes: 64 MiB of
// occupations), and rows packed before their copy and launch are issued: the
// device works on a chunk while the host packs the next.
constexpr int64_t kTableSegment = int64_t{1} << 20;
constexpr int64_t kTableChunk = int64_t{1} << 14;

// Occupations as bytes; values above 127 stay above every particle number.
// Returns false if one is negative.
bool pack_occupations(const int64_t *src, int64_t count, uint8_t *dst) {
  int64_t all = 0;
  for (int64_t k = 0; k < count; ++k) {
    const int64_t v = src[k];
    all |= v;
    dst[k] = static_cast<uint8_t>(v > 127 ? 127 : v);
  }
  return all >= 0;
}

// The coefficients by the plan in S (PolyState::plan).  same(): whether the
// plan belongs to the call's exponent rows; asked once, when the device has
// its work.  If not, nothing is written to `out`.
template <typename Same>
int poly_run(PolyState &S, const double *b0, const double *bm, int64_t n_out, double *out, int64_t *info,
             Same same) {
  const PolyPlan &p = S.plan;
  const int64_t n_keep = static_cast<int64_t>(p.out_index.size());
  const int64_t n_subsets = (int64_t{1} << p.n) - 1;
  if (info) {
    info[0] = p.n_mono;
    info[1] = static_cast<int64_t>(p.links.size());
    info[2] = 0;
    info[3] = 0;
    info[4] = p.flops_per_subset;
    info[5] = n_subsets;
  }
  if (n_keep == 0) {
    std::fill(out, out + 2 * n_out, 0.0);
    return PQP_OK;
  }
  if (n_keep > INT32_MAX / 2)
    return fail(PQP_ERR_RANGE, std::to_string(n_keep) + " requested coefficients exceed the kernel's index range");
  int st;
  if ((st = require_device()) != PQP_OK) return st;
  const DeviceState &dev = device_state();
  const int cus = std::max(dev.cus, 1);
  const int nn = p.n, M = p.M;
  const size_t rs_bytes = static_cast<size_t>(nn) * (M + 1) * sizeof(double2);
  const size_t poly_bytes = static_cast<size_t>(p.n_mono) * sizeof(double2);
  // the polynomial stays in LDS up to 64 KiB per workgroup (two or more
  // workgroups per CU), else in a global-memory slice per workgroup
  if (rs_bytes > 49152)
    return fail(PQP_ERR_RANGE, "n x (variables + 1) = " + std::to_string(nn * (M + 1)) +
                                   " row sums exceed the 3072 kept in LDS");
  const bool lds = rs_bytes + poly_bytes <= 65536;
  if (!lds && poly_bytes > (size_t{8} << 30))
    return fail(PQP_ERR_RANGE, "polynomial of " + std::to_string(p.n_mono) + " monomials is too large");
  // in global memory, kPolyGroup subsets share a workgroup (coefficients
  // interleaved) when their row sums fit in LDS and their slice in 8 GiB
  const int group = (!lds && kPolyGroup * rs_bytes <= 49152 &&
                     kPolyGroup * poly_bytes <= (size_t{8} << 30)) ? kPolyGroup : 1;
  const size_t slice_bytes = poly_bytes * static_cast<size_t>(group);
  const size_t lds_bytes = lds ? rs_bytes + poly_bytes : rs_bytes * static_cast<size_t>(group);
  // global memory: two 1024-thread workgroups per CU (32 waves) hide the
  // gather latency best (measured against one per CU and other groupings)
  int64_t per_cu = lds ? std::min<int64_t>(8, std::max<int64_t>(1, 163840 / static_cast<int64_t>(lds_bytes))) : 2;
  const int64_t n_groups = (n_subsets + group - 1) / group;
  int64_t n_wg = std::min<int64_t>(n_groups, cus * per_cu);
  // bound the per-workgroup slices: polynomials <= 8 GiB, accumulators <= 4 GiB
  if (!lds) n_wg = std::min<int64_t>(n_wg, std::max<int64_t>(1, (int64_t{8} << 30) / static_cast<int64_t>(slice_bytes)));
  n_wg = std::min<int64_t>(n_wg, std::max<int64_t>(1, (int64_t{4} << 30) / (n_keep * 16)));
  if (info) {
    info[2] = n_wg;
    info[3] = lds ? 1 : 0;
  }
  size_t layer_bytes = 0;
  const bool layers = poly_layers_fit(p, &layer_bytes);
  // arena: the plan's tables (link_ptr, links, lvl_off, out_mono, subsets),
  // then B_0 and the kept B_m (uploaded on every call)
  const size_t mat = static_cast<size_t>(nn) * nn * sizeof(double2);
  size_t off = 0;
  const size_t o_lp = off;
  off = align256(off + p.link_ptr.size() * sizeof(int32_t));
  const size_t o_ln = off;
  off = align256(off + std::max<size_t>(p.links.size(), 1) * sizeof(int32_t));
  const size_t o_lv = off;
  off = align256(off + p.lvl_off.size() * sizeof(int32_t));
  const size_t o_om = off;
  off = align256(off + p.out_mono.size() * sizeof(int32_t));
  const size_t o_sb = off;
  off = align256(off + S.subsets.size() * sizeof(int16_t));
  const size_t o_bits = off;
  off = align256(off + S.subset_bits.size() * sizeof(uint16_t));
  const size_t o_b0 = off;
  off = align256(off + mat);
  const size_t o_bm = off;
  off = align256(off + mat * static_cast<size_t>(M));
  const size_t arena_bytes = off;
  if ((st = ensure_stream(S.stream)) != PQP_OK) return st;
  const void *arena_before = S.arena.p;
  if ((st = S.arena.ensure(arena_bytes)) != PQP_OK) return st;
  if (S.arena.p != arena_before) S.tables_on_device = false;
  if ((st = S.stage.ensure(std::max(arena_bytes, static_cast<size_t>(n_keep) * 2 * sizeof(double)))) != PQP_OK)
    return st;
  if (layers) {
    // layers alternate between the two halves
    if ((st = S.scratch.ensure(2 * align256(layer_bytes))) != PQP_OK) return st;
  } else if ((st = S.acc.ensure(static_cast<size_t>(n_wg) * static_cast<size_t>(n_keep) * sizeof(double2))) != PQP_OK) {
    return st;
  }
  if ((st = S.out.ensure(static_cast<size_t>(n_keep) * 2 * sizeof(double))) != PQP_OK) return st;
  if (!layers && !lds && (st = S.scratch.ensure(static_cast<size_t>(n_wg) * slice_bytes)) != PQP_OK) return st;
  char *h = static_cast<char *>(S.stage.p);
  const size_t first = S.tables_on_device ? o_b0 : 0;
  if (!S.tables_on_device) {
    std::memcpy(h + o_lp, p.link_ptr.data(), p.link_ptr.size() * sizeof(int32_t));
    if (!p.links.empty()) std::memcpy(h + o_ln, p.links.data(), p.links.size() * sizeof(int32_t));
    std::memcpy(h + o_lv, p.lvl_off.data(), p.lvl_off.size() * sizeof(int32_t));
    std::memcpy(h + o_om, p.out_mono.data(), p.out_mono.size() * sizeof(int32_t));
    if (!S.subsets.empty()) {
      std::memcpy(h + o_sb, S.subsets.data(), S.subsets.size() * sizeof(int16_t));
      std::memcpy(h + o_bits, S.subset_bits.data(), S.subset_bits.size() * sizeof(uint16_t));
    }
  }
  std::memcpy(h + o_b0, b0, mat);
  for (int v = 0; v < M; ++v)
    std::memcpy(h + o_bm + mat * v, bm + static_cast<size_t>(p.vars[v]) * nn * nn * 2, mat);
  PQP_HIP(hipMemcpyAsync(static_cast<char *>(S.arena.p) + first, h + first, arena_bytes - first,
                         hipMemcpyHostToDevice, S.stream));
  const char *d = static_cast<const char *>(S.arena.p);
  if (layers) {
    PolyLayerArgs la;
    la.b0 = reinterpret_cast<const double2 *>(d + o_b0);
    la.bm = reinterpret_cast<const double2 *>(d + o_bm);
    la.link_ptr = reinterpret_cast<const int32_t *>(d + o_lp);
    la.links = reinterpret_cast<const int32_t *>(d + o_ln);
    la.out_mono = reinterpret_cast<const int32_t *>(d + o_om);
    la.out = static_cast<double *>(S.out.p);
    la.n = nn;
    la.M = M;
    la.n_out = static_cast<int32_t>(n_keep);
    double2 *buf[2] = {static_cast<double2 *>(S.scratch.p),
                       reinterpret_cast<double2 *>(static_cast<char *>(S.scratch.p) + align256(layer_bytes))};
    la.n_dst = 1;
    for (int i = 0; i < nn; ++i) {
      la.row = i;
      la.n_src = la.n_dst;
      la.n_dst = la.n_src * (nn - i) / (i + 1);
      la.n_src_mono = p.lvl_off[std::min(i, p.L) + 1];
      la.n_dst_mono = p.lvl_off[std::min(i + 1, p.L) + 1];
      la.src = i == 0 ? nullptr : buf[(i - 1) & 1];
      la.dst = buf[i & 1];
      const int64_t at = i + 1 < nn ? S.subset_first[i + 1] : 0;  // the last row reads no table
      la.sub = reinterpret_cast<const int16_t *>(d + o_sb) + at * nn;
      la.dst_bits = reinterpret_cast<const uint16_t *>(d + o_bits) + at;
      la.src_bits = reinterpret_cast<const uint16_t *>(d + o_bits) + S.subset_first[i];
      PQP_HIP(launch_poly_layer(la, S.stream));
    }
  } else {
    PolyArgs a;
    a.b0 = reinterpret_cast<const double2 *>(d + o_b0);
    a.bm = reinterpret_cast<const double2 *>(d + o_bm);
    a.link_ptr = reinterpret_cast<const int32_t *>(d + o_lp);
    a.links = reinterpret_cast<const int32_t *>(d + o_ln);
    a.lvl_off = reinterpret_cast<const int32_t *>(d + o_lv);
    a.out_mono = reinterpret_cast<const int32_t *>(d + o_om);
    a.scratch = lds ? nullptr : static_cast<double2 *>(S.scratch.p);
    a.acc = static_cast<double2 *>(S.acc.p);
    a.out = static_cast<double *>(S.out.p);
    a.n = nn;
    a.M = M;
    a.L = p.L;
    a.n_mono = static_cast<int32_t>(p.n_mono);
    a.n_out = static_cast<int32_t>(n_keep);
    a.n_wg = static_cast<int32_t>(n_wg);
    PQP_HIP(launch_perm_poly(a, lds, group, lds_bytes, S.stream));
  }
  PQP_HIP(hipMemcpyAsync(S.stage.p, S.out.p, static_cast<size_t>(n_keep) * 2 * sizeof(double),
                         hipMemcpyDeviceToHost, S.stream));
  // a plan taken on trust is compared while the device works
  const bool fresh = same();
  PQP_HIP(hipStreamSynchronize(S.stream));
  if (!fresh) return PQP_OK;
  // the tables stay in the device arena for the next call with these rows
  S.tables_on_device = true;
  const double *r = static_cast<const double *>(S.stage.p);
  if (n_keep == n_out) {  // every row kept, in order
    std::memcpy(out, r, static_cast<size_t>(n_out) * 2 * sizeof(double));
    return PQP_OK;
  }
  std::fill(out, out + 2 * n_out, 0.0);
  for (int64_t q = 0; q < n_keep; ++q) {
    out[2 * p.out_index[q]] = r[2 * q];
    out[2 * p.out_index[q] + 1] = r[2 * q + 1];
  }
  return PQP_OK;
}

}  // namespace


namespace {

// All column minors of the problems (sum c = sum r + 1) into outs[q]
// (2 m_c doubles each, column order), from the single-call state's stream.
int run_minors(const std::vector<PermInput> &probs, const PlanOptions &opt, double *const *outs) {
  MinorsPlan mp;
  std::string err;
  int st = build_minors_plan(probs, opt, mp, err);
  if (st != PQP_OK) return fail(st, err);
  if ((st = require_device()) != PQP_OK) return st;
  SingleState &S = single_state();
  std::lock_guard<std::mutex> lock(S.mu);
  Exec &x = S.x;
  if ((st = ensure_stream(x.stream)) != PQP_OK) return st;
  x.plan = std::move(mp.plan);
  index_units(x);
  x.flags = PQP_FLAG_STATIC;
  if ((st = upload(x)) != PQP_OK) return st;
  if ((st = enqueue(x, PQP_RUN_EAGER, nullptr, nullptr)) != PQP_OK) return st;
  std::vector<double> res;
  if ((st = fetch_out(x, res)) != PQP_OK) return st;
  for (size_t q = 0; q < probs.size(); ++q)
    for (int64_t j = 0; j < probs[q].m_c; ++j) {
      const double *v = res.data() + 2 * mp.slot[q][static_cast<size_t>(j)];
      outs[q][2 * j] = v[0];
      outs[q][2 * j + 1] = v[1];
    }
  return PQP_OK;
}

int grad_batch_minors(const std::vector<PermInput> &inputs, double *perms, double *const *grads) {
  Plan fwd;
  std::string err;
  PlanOptions fopt;
  fopt.total_units = static_cast<int64_t>(std::max(device_state().cus, 1)) * kBatchUnitsPerCu;
  int st = plan_build(inputs, fopt, fwd, err);
  if (st != PQP_OK) return fail(st, err);
  std::vector<std::vector<int32_t>> mrows;
  std::vector<int64_t> mitem, mrow;
  std::vector<PermInput> minputs;
  minor_inputs(inputs, mrows, mitem, mrow, minputs);
  PlanOptions mopt;
  mopt.total_units = fopt.total_units;
  MinorsPlan mplan;
  st = build_minors_plan(minputs, mopt, mplan, err);
  if (st != PQP_OK) return fail(st, err);
  if ((st = require_device()) != PQP_OK) return st;
  SingleState &S = single_state();
  std::lock_guard<std::mutex> lock(S.mu);
  Exec &x = S.x;
  if ((st = ensure_stream(x.stream)) != PQP_OK) return st;
  std::vector<double> res;
  if (perms && !inputs.empty()) {
    x.plan = std::move(fwd);
    index_units(x);
    x.flags = PQP_FLAG_STATIC;
    if ((st = upload(x)) != PQP_OK) return st;
    if ((st = enqueue(x, PQP_RUN_EAGER, nullptr, nullptr)) != PQP_OK) return st;
    if ((st = fetch_out(x, res)) != PQP_OK) return st;
    std::memcpy(perms, res.data(), inputs.size() * 2 * sizeof(double));
  }
  if (!minputs.empty()) {
    x.plan = std::move(mplan.plan);
    index_units(x);
    x.flags = PQP_FLAG_STATIC;
    if ((st = upload(x)) != PQP_OK) return st;
    if ((st = enqueue(x, PQP_RUN_EAGER, nullptr, nullptr)) != PQP_OK) return st;
    if ((st = fetch_out(x, res)) != PQP_OK) return st;
  }
  scatter_gradients(mplan.slot, res, mitem, mrow, inputs, grads);
  return PQP_OK;
}

}  // namespace

namespace pqp {

int capi_fail(int code, const std::string &msg) { return fail(code, msg); }

double sweep_error_bound(int n, bool fp32, double m, double re, double im) {
  const double u = fp32 ? 0x1p-24 : 0x1p-53;
  return 4.0 * (std::max(n, 0) + 2) * u * m + 0x1p-53 * std::hypot(re, im);
}

void capi_set_last_bound(double bound) { g_last_bound = bound; }

int capi_require_device() { return require_device(); }

double gray_terms(const PermInput &in) {
  int minelem = 0;
  int64_t i0 = -1;
  for (int64_t i = 0; i < in.m_r; ++i)
    if (in.rows[i] > 0 && (minelem == 0 || in.rows[i] < minelem)) {
      minelem = in.rows[i];
      i0 = i;
    }
  double T = 1.0;
  for (int64_t i = 0; i < in.m_r; ++i) {
    const int rho = in.rows[i] - (i == i0 ? 1 : 0);
    if (rho > 0) T *= rho + 1;
  }
  return T;
}

namespace {
int64_t first_smallest(const PermInput &in) {  // the prepended row
  int64_t i0 = -1;
  for (int64_t i = 0; i < in.m_r; ++i)
    if (in.rows[i] > 0 && (i0 < 0 || in.rows[i] < in.rows[i0])) i0 = i;
  return i0;
}
}  // namespace

bool one_plan(const PermInput &given, uint32_t flags, OnePlan &p) {
  if (flags & PQP_FLAG_PLAIN) return false;
  const bool expand = (flags & PQP_FLAG_EXPAND_COLS) != 0;  // a column per particle
  PermInput in = given;
  if (in.m_r <= 0 || in.m_c <= 0 || !in.a || !in.rows || !in.cols || in.ld < in.m_c) return false;
  if (!(flags & PQP_FLAG_AS_GIVEN)) plan_orient(in);
  int64_t sr = 0, sc = 0;
  int width = 0, cmax = 0;
  for (int64_t i = 0; i < in.m_r; ++i) {
    if (in.rows[i] < 0) return false;
    sr += in.rows[i];
  }
  for (int64_t j = 0; j < in.m_c; ++j) {
    if (in.cols[j] < 0) return false;
    sc += in.cols[j];
    width += expand ? std::min(in.cols[j], kOneMaxWidth + 1) : in.cols[j] > 0;
    if (width > kOneMaxWidth) return false;
    cmax = std::max(cmax, static_cast<int>(in.cols[j]));
  }
  if (sr != sc || sr < 1 || sr > kMaxCols) return false;
  int rmax = 0;
  for (int64_t i = 0; i < in.m_r; ++i) rmax = std::max(rmax, static_cast<int>(in.rows[i]));
  const double terms = gray_terms(in);
  if (terms > kOneMaxTerms) return false;
  p.in = in;
  p.n = static_cast<int>(sr);
  p.width = width;
  const bool ones = expand || cmax <= 1;
  p.kind = !ones ? kOneAny : rmax <= 1 ? kOneUnit : kOneOnes;
  p.fp32 = (flags & PQP_FLAG_FP32) != 0;
  p.terms = terms;
  return true;
}

namespace {

// The lanes' digits: those whose states fill whole sets of 64 lanes best, few
// of them (each is a row that every lane adds; the other digits' rows are
// added once per wave).  radix[0 .. digits), equal ones side by side; the
// search ends with the first set of digits that fills kOneFill of its lanes.
struct LaneDigits {
  const int *radix;
  int digits;
  uint32_t best;
  int best_states;
  double best_score;
  int visits;
};

constexpr double kOneFill = 0.95;
constexpr int kOneVisits = 400;

OneDigit one_digit(int rho) {
  OneDigit d{1.0 / (rho + 1), 0, rho, 0};
  if (rho > 10) return d;
  uint64_t c = 1;
  for (int g = 0; g <= rho / 2; ++g) {
    d.choose |= c << (8 * g);
    c = c * static_cast<uint64_t>(rho - g) / static_cast<uint64_t>(g + 1);
  }
  return d;
}

bool lane_search(LaneDigits &s, int from, int used, uint32_t set, int states) {
  const double fill = states / (64.0 * ((states + 63) / 64));
  const double score = fill - 0.02 * used;
  if (score > s.best_score) {
    s.best = set;
    s.best_states = states;
    s.best_score = score;
  }
  if (fill >= kOneFill || ++s.visits > kOneVisits) return true;
  for (int d = from; d < s.digits && used < kOneLaneDigits; ++d) {
    if (d > from && s.radix[d] == s.radix[d - 1]) continue;  // one of equal digits is as good as another
    if (states * s.radix[d] > kOneLaneStates) continue;
    if (lane_search(s, d + 1, used + 1, set | 1u << d, states * s.radix[d])) return true;
  }
  return false;
}

}  // namespace

void one_fill(OnePlan &p, OneArgs &args) {
  OneTables &t = args.tables;
  OneHead &a = args.rows.h;
  const PermInput &in = p.in;
  int64_t cols[kOneMaxWidth];
  int width = 0;
  if (p.kind == kOneAny) std::memset(t.more, 0, sizeof(t.more));
  for (int64_t j = 0; j < in.m_c; ++j) {
    if (in.cols[j] == 0) continue;
    const int64_t at = in.transposed ? j * in.ld : j;
    if (p.kind != kOneAny) {
      for (int r = 0; r < in.cols[j]; ++r) cols[width++] = at;
      continue;
    }
    t.more[width / 4] |= static_cast<uint32_t>(in.cols[j] - 1) << (8 * (width % 4));
    cols[width++] = at;
  }
  // the digits: every row, the first smallest one lower; binary ones first,
  // the others by radix
  const int64_t i0 = first_smallest(in);
  auto rho = [&](int64_t i) { return in.rows[i] - (i == i0 ? 1 : 0); };
  a.n = p.n;
  int64_t digit[kOneMaxRows];
  int radix[kOneMaxRows];
  int digits = 0, binary = 0;
  for (int64_t i = 0; i < in.m_r; ++i)
    if (rho(i) == 1) digit[digits++] = i;
  binary = digits;
  for (int64_t i = 0; i < in.m_r; ++i)
    if (rho(i) > 1) digit[digits++] = i;
  std::stable_sort(digit + binary, digit + digits, [&](int64_t x, int64_t y) { return rho(x) < rho(y); });
  for (int d = 0; d < digits; ++d) radix[d] = static_cast<int>(rho(digit[d])) + 1;
  uint32_t lane = (1u << std::min(binary, kOneLaneDigits)) - 1;
  a.lanes = 1 << std::min(binary, kOneLaneDigits);
  t.lane_binary = 1;
  if (binary < kOneLaneDigits && binary < digits) {
    LaneDigits s{radix, digits, 0, 1, -1.0, 0};
    lane_search(s, 0, 0, 0, 1);
    lane = s.best;
    a.lanes = s.best_states;
    t.lane_binary = (lane >> binary) == 0;
  }
  t.lane_chunks = (a.lanes + kWave - 1) / kWave;
  t.lane_inv = 1.0 / t.lane_chunks;
  // One block's waves, for two states a lane of single photons, one where a
  // state is a longer product; or as many blocks as keep about kOneStates
  // states a lane.  Inner digits as long as every wave keeps a chunk.
  double chunks = p.terms / a.lanes;  // of the other digits
  const double all = chunks * t.lane_chunks;
  double waves;
  if (p.terms > kOneBlockTerms) {
    p.waves = kOneBlockWaves;
    waves = std::min(all / kOneStates,
                     static_cast<double>(kOneBlockWaves * (p.terms > kOneManyTerms ? kOneMaxBlocks : kOneMaxBlocks / 2)));
  } else {
    p.blocks = 1;
    const double most = p.kind == kOneUnit ? std::min(all / 2.0, static_cast<double>(kOneBlockWaves))
                                           : std::min(all, static_cast<double>(kOneWaves));
    p.waves = std::max(1, static_cast<int>(most));
    waves = p.waves;
  }
  uint32_t inner = 0;
  a.S = 1;
  t.binary = 1;
  for (int d = 0; d < digits; ++d) {
    if ((lane >> d & 1u) || a.S * radix[d] > kOneMaxStates || chunks * t.lane_chunks < waves * radix[d]) continue;
    inner |= 1u << d;
    a.S *= radix[d];
    chunks /= radix[d];
    if (d >= binary) t.binary = 0;
  }
  a.chunks = static_cast<int32_t>(std::llround(chunks)) * t.lane_chunks;
  if (p.terms > kOneBlockTerms) p.blocks = std::min((a.chunks + p.waves - 1) / p.waves, kOneMaxBlocks);
  int64_t order[kOneMaxRows];
  int rows = 0;
  a.lane_digits = a.inner = a.rest = 0;
  for (int d = 0; d < digits; ++d)
    if (lane >> d & 1u) {
      t.lane[a.lane_digits++] = one_digit(radix[d] - 1);
      order[rows++] = digit[d];
    }
  order[rows++] = i0;
  for (int d = 0; d < digits; ++d)
    if (inner >> d & 1u) {
      t.digit[a.inner++] = one_digit(radix[d] - 1);
      order[rows++] = digit[d];
    }
  for (int d = 0; d < digits; ++d)
    if (!((lane | inner) >> d & 1u)) {
      t.digit[a.inner + a.rest++] = one_digit(radix[d] - 1);
      order[rows++] = digit[d];
    }
  if (!t.binary) {
    // reflected mixed-radix Gray code of the inner digits
    int g[kOneMaxRows] = {}, dir[kOneMaxRows];
    double coef = 1.0;
    std::fill(dir, dir + a.inner, 1);
    for (int v = 0; v < a.S; ++v) {
      t.step[v] = OneStep{coef, 0, 0};
      if (v + 1 == a.S) break;
      int i = 0;
      for (; g[i] + dir[i] < 0 || g[i] + dir[i] > t.digit[i].rho; ++i) dir[i] = -dir[i];
      // C(rho, g +- 1) from C(rho, g), exact
      coef = dir[i] > 0 ? -coef * (t.digit[i].rho - g[i]) / (g[i] + 1) : -coef * g[i] / (t.digit[i].rho - g[i] + 1);
      g[i] += dir[i];
      t.step[v].factor = dir[i] > 0 ? -2 : 2;
      t.step[v].row = 1 + i;
    }
  }
  const int64_t step = in.transposed ? 1 : in.ld;
  auto fill = [&](auto *dst, const auto *src) {
    using R = std::remove_reference_t<decltype(*dst)>;
    for (int r = 0; r < rows; ++r)
      for (int j = 0; j < width; ++j, dst += 2) {
        const auto *e = src + 2 * (order[r] * step + cols[j]);
        dst[0] = static_cast<R>(e[0]);
        dst[1] = static_cast<R>(e[1]);
      }
  };
  if (in.a_is_float) {
    if (p.fp32)
      fill(reinterpret_cast<float *>(args.rows.b), static_cast<const float *>(in.a));
    else
      fill(reinterpret_cast<double *>(args.rows.b), static_cast<const float *>(in.a));
  } else {
    if (p.fp32)
      fill(reinterpret_cast<float *>(args.rows.b), static_cast<const double *>(in.a));
    else
      fill(reinterpret_cast<double *>(args.rows.b), static_cast<const double *>(in.a));
  }
}

PlanOptions single_plan_options(uint32_t flags, const PermInput &in) {
  PlanOptions opt;
  opt.fp32_products = (flags & PQP_FLAG_FP32) != 0;
  opt.expand_cols = expand_mode(flags);
  opt.orient = (flags & PQP_FLAG_AS_GIVEN) == 0;
  const DeviceState &dev = device_state();
  // waves per permanent: ~1.4 sqrt(T), at most kSingleUnitsPerCu per CU; a permanent of one wave writes its result
  // from the sweep kernel
  opt.auto_units_cap = static_cast<int64_t>(std::max(dev.cus, 1)) * kSingleUnitsPerCu;
  const bool rows_ok = in.m_r == 0 || (in.m_r > 0 && in.rows);
  if (!(flags & PQP_FLAG_PLAIN) && rows_ok) {
    const double t = gray_terms(in);
    if (t <= kSingleFewTerms)
      opt.auto_units_cap = t <= kSingleFewestTerms ? kSingleFewestUnits : kSingleFewUnits;
  }
  opt.direct_out = (flags & PQP_FLAG_PLAIN) == 0;
  return opt;
}

}  // namespace pqp

extern "C" {

const char *pqp_version(void) { return "pqp-permanent 0.1.0 (gfx950)"; }

const char *pqp_last_error(void) { return g_error.c_str(); }

double pqp_last_error_bound(void) { return g_last_bound; }

int pqp_device_info(int *n_devices, int *cu_count, char *name, int name_len) {
  DeviceState &d = device_state();
  if (n_devices) *n_devices = d.n_devices;
  if (!d.ok) return fail(PQP_ERR_DEVICE, d.error);
  if (cu_count) *cu_count = d.cus;
  if (name && name_len > 0) {
    std::strncpy(name, d.name.c_str(), static_cast<size_t>(name_len) - 1);
    name[name_len - 1] = '\0';
  }
  return PQP_OK;
}

int pqp_debug_fail_allocation(int64_t after) {
  g_alloc_countdown.store(after < 0 ? -1 : after);
  return PQP_OK;
}

int pqp_permanent_c128(const double *matrix, int64_t m_r, int64_t m_c, int64_t ld,
                       const int32_t *rows, const int32_t *cols, uint32_t flags, double *out,
                       double *out_dd) {
  CallRange range_("pqp_permanent_c128");
  if (!out) return fail(PQP_ERR_INVALID, "out is null");
  PermInput in{matrix, false, m_r, m_c, ld, rows, cols};
  return run_single(in, flags, out, out_dd);
}

int pqp_permanent_c64(const float *matrix, int64_t m_r, int64_t m_c, int64_t ld,
                      const int32_t *rows, const int32_t *cols, uint32_t flags, float *out,
                      double *out_dd) {
  CallRange range_("pqp_permanent_c64");
  if (!out) return fail(PQP_ERR_INVALID, "out is null");
  PermInput in{matrix, true, m_r, m_c, ld, rows, cols};
  double o[2];
  const int st =
      run_single(in, PQP_FLAG_FP32 | (flags & (PQP_FLAG_EXPAND_COLS | PQP_FLAG_KEEP_COLS | PQP_FLAG_AS_GIVEN)),
                 o, out_dd);
  if (st != PQP_OK) return st;
  out[0] = static_cast<float>(o[0]);
  out[1] = static_cast<float>(o[1]);
  g_last_bound += 0x1p-24 * std::hypot(static_cast<double>(out[0]), static_cast<double>(out[1]));
  return PQP_OK;
}

int pqp_permanent_int64(const int64_t *matrix, int64_t m_r, int64_t m_c, int64_t ld,
                        const int32_t *rows, const int32_t *cols, double *out, uint64_t *limbs,
                        int32_t n_limbs) {
  CallRange range_("pqp_permanent_int64");
  if (!out) return fail(PQP_ERR_INVALID, "out is null");
  if (limbs && n_limbs < kIntLimbs)
    return fail(PQP_ERR_INVALID, "limbs needs room for 8 words (512 bits)");
  if (m_r < 0 || m_c < 0 || (m_r * m_c > 0 && !matrix) || (m_r > 0 && !rows) ||
      (m_c > 0 && !cols) || (m_r > 0 && ld < m_c))
    return fail(PQP_ERR_INVALID, "invalid shape or null pointer");
  for (int64_t i = 0; i < m_r; ++i)
    if (rows[i] < 0) return fail(PQP_ERR_INVALID, "negative row multiplicity");
  for (int64_t j = 0; j < m_c; ++j)
    if (cols[j] < 0) return fail(PQP_ERR_INVALID, "negative column multiplicity");
  // the matrix as complex128 with zero imaginary parts; entries beyond
  // 2^47 (which a double may not hold exactly) are refused by the scan when
  // they are selected
  std::vector<double> a(static_cast<size_t>(std::max<int64_t>(m_r * m_c, 1)) * 2, 0.0);
  for (int64_t i = 0; i < m_r; ++i)
    for (int64_t j = 0; j < m_c; ++j) {
      const int64_t e = matrix[i * ld + j];
      const int64_t lim = int64_t(1) << 47;
      a[static_cast<size_t>(2 * (i * m_c + j))] =
          static_cast<double>(e > lim ? lim + 1 : (e < -lim ? -lim - 1 : e));
    }
  const PermInput in{a.data(), false, m_r, m_c, m_c, rows, cols};
  uint64_t v[kIntLimbs];
  const int st = run_int(in, int_scan(in), v);
  if (st != PQP_OK) return st;
  out[0] = limbs_round(v, 53);
  if (limbs) std::memcpy(limbs, v, sizeof(v));
  return PQP_OK;
}

int pqp_laplace_c128(const double *matrix, int64_t m_r, int64_t m_c, int64_t ld,
                     const int32_t *rows, const int32_t *cols, double *out) {
  CallRange range_("pqp_laplace_c128");
  if (!out && m_c > 0) return fail(PQP_ERR_INVALID, "out is null");
  PermInput in{matrix, false, m_r, m_c, ld, rows, cols};
  if (laplace_wave_fits(in)) return laplace_wave(in, out);
  PlanOptions opt;
  const DeviceState &dev = device_state();
  opt.auto_units_cap = static_cast<int64_t>(std::max(dev.cus, 1)) * kSingleUnitsPerCu;
  return run_minors(std::vector<PermInput>{in}, opt, &out);
}

int pqp_laplace_batch_c128(int64_t count, const double *const *matrices, const int64_t *m_r,
                           const int64_t *m_c, const int64_t *ld, const int32_t *const *rows,
                           const int32_t *const *cols, double *const *outs) {
  CallRange range_("pqp_laplace_batch_c128");
  if (count < 0 || (count > 0 && (!matrices || !m_r || !m_c || !ld || !rows || !cols || !outs)))
    return fail(PQP_ERR_INVALID, "invalid laplace batch arguments");
  if (count > INT32_MAX) return fail(PQP_ERR_RANGE, "too many items");
  std::vector<PermInput> inputs;
  inputs.reserve(static_cast<size_t>(count));
  for (int64_t k = 0; k < count; ++k) {
    if (!outs[k] && m_c[k] > 0) return fail(PQP_ERR_INVALID, "item " + std::to_string(k) + ": out is null");
    inputs.push_back(PermInput{matrices[k], false, m_r[k], m_c[k], ld[k], rows[k], cols[k]});
  }
  if (count == 0) return PQP_OK;
  PlanOptions opt;
  const DeviceState &dev = device_state();
  // about kBatchUnitsPerCu waves per CU, shared in proportion to cost
  opt.total_units = static_cast<int64_t>(std::max(dev.cus, 1)) * kBatchUnitsPerCu;
  return run_minors(inputs, opt, outs);
}

int pqp_tensor_permanent_batch_c128(int64_t count, const double *const *matrices, const int64_t *n,
                                    const int64_t *ld, const double *overlap, double *out,
                                    double *abs_sum) {
  CallRange range_("pqp_tensor_permanent_batch_c128");
  if (count < 0 || (count > 0 && (!matrices || !n || !ld || !overlap || !out)))
    return fail(PQP_ERR_INVALID, "invalid tensor permanent arguments");
  if (count > INT32_MAX) return fail(PQP_ERR_RANGE, "too many items");
  if (count == 0) return PQP_OK;
  std::vector<int64_t> order;  // items by matrix order, empty matrices left out
  for (int64_t k = 0; k < count; ++k) {
    const std::string item = "item " + std::to_string(k);
    if (n[k] < 0 || n[k] > kTensorMaxN)
      return fail(n[k] < 0 ? PQP_ERR_INVALID : PQP_ERR_RANGE,
                  item + ": tensor permanents support matrices of order 0.." + std::to_string(kTensorMaxN));
    if (n[k] > 0 && (!matrices[k] || ld[k] < n[k]))
      return fail(PQP_ERR_INVALID, item + ": invalid matrix pointer or leading dimension");
    if (!std::isfinite(overlap[k])) return fail(PQP_ERR_INVALID, item + ": particle overlap is not finite");
    if (n[k] > 0) order.push_back(k);
  }
  std::stable_sort(order.begin(), order.end(), [&](int64_t a, int64_t b) { return n[a] < n[b]; });
  int st;
  if ((st = require_device()) != PQP_OK) return st;
  TensorState &S = tensor_state();
  std::lock_guard<std::mutex> lock(S.mu);
  if ((st = ensure_stream(S.stream)) != PQP_OK) return st;
  for (int64_t k = 0; k < count; ++k)
    if (n[k] == 0) {  // the empty product (probabilities.py:197-198)
      out[k] = 1.0;
      if (abs_sum) abs_sum[k] = 1.0;
    }
  // Passes of one order each, and flights of passes that fit the work buffer
  // together: one copy in, one wait.
  struct Pass {
    TensorArgs a;
    TensorPass t;
    const std::vector<TensorUnit> *units;
    size_t first, items;               // in `order`
    size_t o_units, o_x, o_cols, work, result;  // offsets of the flight's buffers (results in items)
  };
  std::vector<TensorUnit> units[kTensorMaxN + 1];
  std::vector<Pass> flight;
  size_t in_bytes = 0, work_bytes = 0, items = 0;
  auto run = [&]() -> int {
    if (flight.empty()) return PQP_OK;
    const size_t out_bytes = items * 2 * sizeof(double);
    const bool mapped = items <= kTensorMapped;
    int st;
    if ((st = S.in.ensure(in_bytes)) != PQP_OK) return st;
    if ((st = S.work.ensure(work_bytes)) != PQP_OK) return st;
    if ((st = mapped ? S.res.ensure(out_bytes) : S.out.ensure(out_bytes)) != PQP_OK) return st;
    if ((st = S.stage.ensure(std::max(in_bytes, out_bytes))) != PQP_OK) return st;
    char *h = static_cast<char *>(S.stage.p);
    char *d = static_cast<char *>(S.in.p);
    for (Pass &p : flight) {
      TensorArgs &a = p.a;
      const int nk = a.n;
      const size_t nn = static_cast<size_t>(nk) * nk;
      std::memcpy(h + p.o_units, p.units->data(), p.units->size() * sizeof(TensorUnit));
      for (size_t q = 0; q < p.items; ++q) {
        const int64_t k = order[p.first + q];
        reinterpret_cast<double *>(h + p.o_x)[q] = overlap[k];
        double *colp = reinterpret_cast<double *>(h + p.o_cols) + q * nn * 2;
        double *pwp = reinterpret_cast<double *>(h + p.o_cols + p.t.pw) + q * nn;
        const double y = 1.0 - overlap[k];
        for (int c = 0; c < nk; ++c)
          for (int i = 0; i < nk; ++i) {
            const double re = matrices[k][2 * (i * ld[k] + c)];
            const double im = matrices[k][2 * (i * ld[k] + c) + 1];
            colp[2 * (c * nk + i)] = re;
            colp[2 * (c * nk + i) + 1] = im;
            pwp[c * nk + i] = y * (re * re + im * im);
          }
      }
      tensor_buffers(a, p.t, static_cast<char *>(S.work.p) + p.work);
      a.cols = reinterpret_cast<double *>(d + p.o_cols);
      a.pw = reinterpret_cast<double *>(d + p.o_cols + p.t.pw);
      a.units = reinterpret_cast<const TensorUnit *>(d + p.o_units);
      a.x = reinterpret_cast<const double *>(d + p.o_x);
      a.out = static_cast<double *>(mapped ? S.res.dev : S.out.p) + 2 * p.result;
    }
    PQP_HIP(hipMemcpyAsync(d, h, in_bytes, hipMemcpyHostToDevice, S.stream));
    std::vector<TensorArgs> passes;
    for (const Pass &p : flight) passes.push_back(p.a);
    PQP_HIP(launch_tensor_signs(passes.data(), static_cast<int>(passes.size()), S.stream));
    for (const Pass &p : flight) {
      PQP_HIP(launch_tensor(p.a, S.stream));
      PQP_HIP(launch_tensor_finalize(p.a, S.stream));
    }
    if (!mapped) PQP_HIP(hipMemcpyAsync(h, S.out.p, out_bytes, hipMemcpyDeviceToHost, S.stream));
    PQP_HIP(hipStreamSynchronize(S.stream));
    const double *r = static_cast<const double *>(mapped ? S.res.host : static_cast<void *>(h));
    for (const Pass &p : flight)
      for (size_t q = 0; q < p.items; ++q) {
        out[order[p.first + q]] = r[2 * (p.result + q)];
        if (abs_sum) abs_sum[order[p.first + q]] = r[2 * (p.result + q) + 1];
      }
    flight.clear();
    in_bytes = work_bytes = items = 0;
    return PQP_OK;
  };
  for (size_t at = 0; at < order.size();) {
    const int nk = static_cast<int>(n[order[at]]);
    size_t end = at;
    while (end < order.size() && n[order[end]] == nk) ++end;
    Pass p;
    std::memset(&p.a, 0, sizeof(p.a));
    p.a.n = nk;
    if (units[nk].empty()) tensor_units(nk, &p.a.ls, &p.a.kt, units[nk]);
    p.units = &units[nk];
    p.a.n_units = static_cast<int32_t>(units[nk].size());
    for (; at < end; at += p.items) {
      p.t = tensor_pass(nk, static_cast<int64_t>(end - at), units[nk].size());
      p.first = at;
      p.items = static_cast<size_t>(p.t.items);
      p.a.n_items = static_cast<int32_t>(p.items);
      if (work_bytes + p.t.bytes > kTensorBytes && (st = run()) != PQP_OK) return st;
      p.o_units = in_bytes;
      p.o_x = align256(p.o_units + units[nk].size() * sizeof(TensorUnit));
      p.o_cols = align256(p.o_x + p.items * sizeof(double));
      in_bytes = align256(p.o_cols + p.t.signs);
      p.work = work_bytes;
      work_bytes = align256(work_bytes + p.t.bytes);
      p.result = items;
      items += p.items;
      flight.push_back(p);
    }
  }
  return run();
}

int pqp_overlap_table_c128(const double *matrix, int64_t modes, int64_t ld, const int32_t *input,
                           int64_t count, const int64_t *outputs, double overlap, double input_norm,
                           double *out) {
  CallRange range_("pqp_overlap_table_c128");
  if (modes < 1 || modes > 65535 || count < 0 || !matrix || ld < modes || !input ||
      (count > 0 && (!outputs || !out)))
    return fail(PQP_ERR_INVALID, "invalid overlap table arguments");
  int64_t n64 = 0;
  for (int64_t j = 0; j < modes; ++j) {
    if (input[j] < 0) return fail(PQP_ERR_INVALID, "occupation numbers must be non-negative");
    n64 += input[j];
  }
  if (n64 > kTensorMaxN)
    return fail(PQP_ERR_RANGE, "overlap tables support at most " + std::to_string(kTensorMaxN) + " particles");
  const int n = static_cast<int>(n64);
  // the outputs of n particles: their rows in first-quantized order, and
  // input norm x prod t!
  std::vector<uint16_t> rows;
  std::vector<double> norm;
  std::vector<int64_t> kept;
  rows.reserve(static_cast<size_t>(count * n));
  norm.reserve(static_cast<size_t>(count));
  kept.reserve(static_cast<size_t>(count));
  for (int64_t q = 0; q < count; ++q) {
    const int64_t *t = outputs + q * modes;
    int64_t sum = 0;
    for (int64_t j = 0; j < modes; ++j) {
      if (t[j] < 0) return fail(PQP_ERR_INVALID, "occupation numbers must be non-negative");
      sum += std::min<int64_t>(t[j], kTensorMaxN + 1);
    }
    out[q] = 0.0;
    if (sum != n) continue;
    double f = 1.0;
    for (int64_t j = 0; j < modes; ++j)
      for (int64_t k = 1; k <= t[j]; ++k) {
        rows.push_back(static_cast<uint16_t>(j));
        f *= static_cast<double>(k);
      }
    norm.push_back(input_norm * f);
    kept.push_back(q);
  }
  if (kept.empty()) return PQP_OK;
  if (!std::isfinite(overlap)) return fail(PQP_ERR_INVALID, "particle overlap is not finite");
  int st;
  if ((st = require_device()) != PQP_OK) return st;
  if (n == 0) {
    for (size_t q = 0; q < kept.size(); ++q) out[kept[q]] = 1.0 / norm[q];
    return PQP_OK;
  }
  TensorState &S = tensor_state();
  std::lock_guard<std::mutex> lock(S.mu);
  if ((st = ensure_stream(S.stream)) != PQP_OK) return st;
  TensorArgs a;
  std::memset(&a, 0, sizeof(a));
  a.n = n;
  std::vector<TensorUnit> units;
  tensor_units(n, &a.ls, &a.kt, units);
  a.n_units = static_cast<int32_t>(units.size());
  const TensorPass t = tensor_pass(n, static_cast<int64_t>(kept.size()), units.size());
  const size_t most = static_cast<size_t>(t.items), all = kept.size();
  const size_t o_x = align256(units.size() * sizeof(TensorUnit));
  const size_t o_u = align256(o_x + most * sizeof(double));
  const size_t o_rows = align256(o_u + static_cast<size_t>(modes) * n * 16);
  const size_t o_norm = align256(o_rows + all * n * sizeof(uint16_t));
  const size_t in_bytes = o_norm + all * sizeof(double);
  if ((st = S.in.ensure(in_bytes)) != PQP_OK) return st;
  if ((st = S.work.ensure(t.bytes)) != PQP_OK) return st;
  if ((st = S.out.ensure(all * sizeof(double))) != PQP_OK) return st;
  if ((st = S.stage.ensure(std::max(in_bytes, all * sizeof(double)))) != PQP_OK) return st;
  char *h = static_cast<char *>(S.stage.p);
  char *d = static_cast<char *>(S.in.p);
  std::memcpy(h, units.data(), units.size() * sizeof(TensorUnit));
  for (size_t q = 0; q < most; ++q) reinterpret_cast<double *>(h + o_x)[q] = overlap;
  double *hu = reinterpret_cast<double *>(h + o_u);
  for (int64_t i = 0; i < modes; ++i)
    for (int64_t j = 0; j < modes; ++j)
      for (int32_t k = 0; k < input[j]; ++k) {
        *hu++ = matrix[2 * (i * ld + j)];
        *hu++ = matrix[2 * (i * ld + j) + 1];
      }
  std::memcpy(h + o_rows, rows.data(), rows.size() * sizeof(uint16_t));
  std::memcpy(h + o_norm, norm.data(), norm.size() * sizeof(double));
  PQP_HIP(hipMemcpyAsync(d, h, in_bytes, hipMemcpyHostToDevice, S.stream));
  tensor_buffers(a, t, static_cast<char *>(S.work.p));
  a.units = reinterpret_cast<const TensorUnit *>(d);
  a.x = reinterpret_cast<const double *>(d + o_x);
  a.u = reinterpret_cast<const double *>(d + o_u);
  for (size_t p0 = 0; p0 < all; p0 += most) {
    a.n_items = static_cast<int32_t>(std::min(most, all - p0));
    a.rows = reinterpret_cast<const uint16_t *>(d + o_rows) + p0 * n;
    a.norm = reinterpret_cast<const double *>(d + o_norm) + p0;
    a.prob = static_cast<double *>(S.out.p) + p0;
    PQP_HIP(launch_tensor_gather(a, S.stream));
    PQP_HIP(launch_tensor_signs(&a, 1, S.stream));
    PQP_HIP(launch_tensor(a, S.stream));
    PQP_HIP(launch_tensor_finalize(a, S.stream));
  }
  PQP_HIP(hipMemcpyAsync(h, S.out.p, all * sizeof(double), hipMemcpyDeviceToHost, S.stream));
  PQP_HIP(hipStreamSynchronize(S.stream));
  const double *r = reinterpret_cast<const double *>(h);
  for (size_t q = 0; q < all; ++q) out[kept[q]] = r[q];
  return PQP_OK;
}

int pqp_tensor_permanent_c128(const double *matrix, int64_t n, int64_t ld, double overlap,
                              double *out, double *abs_sum) {
  const double *m[1] = {matrix};
  return pqp_tensor_permanent_batch_c128(1, m, &n, &ld, &overlap, out, abs_sum);
}

int pqp_output_table_c128(const double *matrix, int64_t modes, int64_t ld, const int32_t *input,
                          int64_t count, const int64_t *outputs, int probabilities, double *out) {
  CallRange range_("pqp_output_table_c128");
  if (modes < 1 || count < 0 || !matrix || ld < modes || !input || (count > 0 && (!outputs || !out)))
    return fail(PQP_ERR_INVALID, "invalid output table arguments");
  if (modes > kTableMaxModes)
    return fail(PQP_ERR_RANGE, "output tables support at most " + std::to_string(kTableMaxModes) + " modes");
  int64_t n = 0;
  int width = 0;
  bool ones = true;
  double in_norm = 1.0;
  for (int64_t j = 0; j < modes; ++j) {
    if (input[j] < 0) return fail(PQP_ERR_INVALID, "occupation numbers must be non-negative");
    n += input[j];
    width += input[j] > 0;
    ones = ones && input[j] <= 1;
  }
  if (n < 1 || n > kTableMaxN)
    return fail(PQP_ERR_RANGE, "output tables support 1.." + std::to_string(kTableMaxN) + " particles");
  for (int64_t j = 0; j < modes; ++j)
    for (int32_t q = 2; q <= input[j]; ++q) in_norm *= q;
  const int per = probabilities ? 1 : 2;
  const DeviceState &dev = device_state();
  if (!dev.ok) {
    // argument errors first, and a table without a matching row needs no device
    bool any = false;
    for (int64_t r = 0; r < count; ++r) {
      int64_t sum = 0;
      for (int64_t j = 0; j < modes; ++j) {
        const int64_t v = outputs[r * modes + j];
        if (v < 0) return fail(PQP_ERR_INVALID, "occupation numbers must be non-negative");
        sum += v;
      }
      any = any || sum == n;
    }
    if (any) return fail(PQP_ERR_DEVICE, dev.error);
    std::fill(out, out + per * count, 0.0);
    return PQP_OK;
  }
  TableState &S = table_state();
  std::lock_guard<std::mutex> lock(S.mu);
  int st;
  if ((st = ensure_stream(S.stream)) != PQP_OK) return st;
  // input buffer: the occupied columns, their occupations, the outputs
  const size_t o_mult = static_cast<size_t>(modes) * width * 2 * sizeof(double);
  const size_t o_outs = align256(o_mult + static_cast<size_t>(width) * sizeof(int32_t));
  const int64_t most = std::min(count, kTableSegment);
  const size_t in_bytes = o_outs + static_cast<size_t>(most) * static_cast<size_t>(modes);
  const size_t out_bytes = static_cast<size_t>(most) * per * sizeof(double);
  if ((st = S.in.ensure(in_bytes)) != PQP_OK) return st;
  if ((st = S.out.ensure(out_bytes)) != PQP_OK) return st;
  if ((st = S.stage.ensure(align256(in_bytes) + out_bytes)) != PQP_OK) return st;
  char *h = static_cast<char *>(S.stage.p);
  char *d = static_cast<char *>(S.in.p);
  double *hrows = reinterpret_cast<double *>(h);
  int32_t *hmult = reinterpret_cast<int32_t *>(h + o_mult);
  int at = 0;
  for (int64_t j = 0; j < modes; ++j) {
    if (input[j] == 0) continue;
    hmult[at] = input[j];
    for (int64_t i = 0; i < modes; ++i) {
      hrows[2 * (i * width + at)] = matrix[2 * (i * ld + j)];
      hrows[2 * (i * width + at) + 1] = matrix[2 * (i * ld + j) + 1];
    }
    ++at;
  }
  TableArgs a;
  a.rows = reinterpret_cast<const double *>(d);
  a.mult = reinterpret_cast<const int32_t *>(d + o_mult);
  a.in_norm = in_norm;
  a.modes = static_cast<int32_t>(modes);
  a.n = static_cast<int32_t>(n);
  a.prob = probabilities ? 1 : 0;
  a.states = 0;
  a.width = width;
  a.first = 0;
  a.per_given = 0.0;
  a.sums = nullptr;
  a.weights = nullptr;
  if (!ones) {
    // the sweep over the input's digits: at most 3 2^13 states
    int most_in = 0;
    for (int q = 0; q < width; ++q) {
      if (hmult[q] < hmult[a.first]) a.first = q;
      most_in = std::max(most_in, static_cast<int>(hmult[q]));
    }
    a.states = 1;
    for (int q = 0; q < width; ++q) a.states *= hmult[q] + (q == a.first ? 0 : 1);
    a.per_given = sweep_term_cost(width, most_in, static_cast<int>(n));
    const size_t sums = static_cast<size_t>(a.states) * modes * 2 * sizeof(double);
    if ((st = S.states.ensure(sums + static_cast<size_t>(a.states) * sizeof(double))) != PQP_OK) return st;
    a.sums = static_cast<double2 *>(S.states.p);
    a.weights = reinterpret_cast<double *>(static_cast<char *>(S.states.p) + sums);
  }
  double *hout = reinterpret_cast<double *>(h + align256(in_bytes));
  for (int64_t s0 = 0; s0 < count; s0 += kTableSegment) {
    const int64_t rows = std::min(count - s0, kTableSegment);
    for (int64_t c0 = 0; c0 < rows; c0 += kTableChunk) {
      const int64_t c = std::min(rows - c0, kTableChunk);
      // the first copy also brings the columns
      const size_t to = o_outs + static_cast<size_t>(c0 * modes);
      const size_t from = c0 == 0 ? 0 : to;
      if (!pack_occupations(outputs + (s0 + c0) * modes, c * modes, reinterpret_cast<uint8_t *>(h + to))) {
        PQP_HIP(hipStreamSynchronize(S.stream));  // copies out of the staging buffer
        return fail(PQP_ERR_INVALID, "occupation numbers must be non-negative");
      }
      PQP_HIP(hipMemcpyAsync(d + from, h + from, to + static_cast<size_t>(c * modes) - from,
                             hipMemcpyHostToDevice, S.stream));
      a.outs = reinterpret_cast<const uint8_t *>(d + to);
      a.out = static_cast<double *>(S.out.p) + per * c0;
      a.count = c;
      if (!ones && s0 == 0 && c0 == 0) PQP_HIP(launch_table_states(a, S.stream));
      PQP_HIP(launch_table(width, ones, a, S.stream));
    }
    PQP_HIP(hipMemcpyAsync(hout, S.out.p, static_cast<size_t>(rows) * per * sizeof(double),
                           hipMemcpyDeviceToHost, S.stream));
    PQP_HIP(hipStreamSynchronize(S.stream));
    std::memcpy(out + per * s0, hout, static_cast<size_t>(rows) * per * sizeof(double));
  }
  return PQP_OK;
}

int pqp_sample_shots_c128(const double *matrix, int64_t modes, int64_t ld, int64_t shots, int64_t photons,
                          const uint8_t *pools, const int32_t *steps, const int32_t *picks, const double *draws,
                          int32_t *out) {
  CallRange range_("pqp_sample_shots_c128");
  if (modes < 1 || shots < 0 || photons < 0 || !matrix || ld < modes ||
      (shots > 0 && (!steps || !out || (photons > 0 && (!pools || !picks || !draws)))))
    return fail(PQP_ERR_INVALID, "invalid sampling arguments");
  if (modes > kMinorsWaveMaxModes || photons > kMinorsWaveMaxCols)
    return fail(PQP_ERR_RANGE, "sampling on the device supports at most " + std::to_string(kMinorsWaveMaxModes) +
                                   " modes and " + std::to_string(kMinorsWaveMaxCols) + " photons");
  for (int64_t s = 0; s < shots; ++s) {
    if (steps[s] < 0 || steps[s] > photons) return fail(PQP_ERR_INVALID, "a shot's photons exceed its pool");
    for (int32_t p = 0; p < steps[s]; ++p)
      if (picks[p * shots + s] < 0 || picks[p * shots + s] >= photons - p)
        return fail(PQP_ERR_INVALID, "a pick is out of the pool");
    for (int64_t p = 0; p < photons; ++p)
      if (pools[s * photons + p] >= modes) return fail(PQP_ERR_INVALID, "an input mode is out of range");
  }
  if (shots == 0) return PQP_OK;
  int st;
  if ((st = require_device()) != PQP_OK) return st;
  MinorsState &S = sample_state();
  std::lock_guard<std::mutex> lock(S.mu);
  if ((st = ensure_stream(S.stream)) != PQP_OK) return st;
  const SamplePasses passes = sample_passes(shots, photons);
  const int64_t most = passes.most;
  // input: matrix, columns, photons, draws; work: the shots' columns,
  // outputs, wave counts, the failure flag, partials
  const size_t m2 = static_cast<size_t>(modes) * modes * 2 * sizeof(double);
  const size_t o_draws = align256(m2);
  const size_t o_steps = align256(o_draws + static_cast<size_t>(photons * most) * sizeof(double));
  const size_t o_cols = align256(o_steps + static_cast<size_t>(most) * sizeof(int32_t));
  const size_t in_bytes = o_cols + static_cast<size_t>(most * photons) + 1;
  const size_t w_occ = align256(static_cast<size_t>(most * modes * photons) * 2 * sizeof(double));
  const size_t w_units = align256(w_occ + static_cast<size_t>(most * modes));
  const size_t w_failed = align256(w_units + static_cast<size_t>(most) * sizeof(int32_t));
  const size_t w_part = w_failed + 256;
  if ((st = S.in.ensure(in_bytes)) != PQP_OK) return st;
  if ((st = S.work.ensure(w_part + passes.partials)) != PQP_OK) return st;
  if ((st = S.stage.ensure(std::max(in_bytes, w_failed + 256 - w_occ))) != PQP_OK) return st;
  char *h = static_cast<char *>(S.stage.p);
  char *d = static_cast<char *>(S.in.p);
  char *w = static_cast<char *>(S.work.p);
  for (int64_t s0 = 0; s0 < shots; s0 += most) {
    const int64_t n = std::min(most, shots - s0);
    for (int64_t i = 0; i < modes; ++i)
      std::memcpy(h + static_cast<size_t>(i * modes) * 16, matrix + 2 * i * ld, static_cast<size_t>(modes) * 16);
    for (int64_t p = 0; p < photons; ++p)
      std::memcpy(h + o_draws + static_cast<size_t>(p * n) * 8, draws + p * shots + s0, static_cast<size_t>(n) * 8);
    std::memcpy(h + o_steps, steps + s0, static_cast<size_t>(n) * sizeof(int32_t));
    for (int64_t s = 0; s < n; ++s) {  // the input modes in the order they join
      uint8_t pool[kMinorsWaveMaxCols];
      uint8_t *cols = reinterpret_cast<uint8_t *>(h + o_cols) + s * photons;
      if (photons) std::memcpy(pool, pools + (s0 + s) * photons, static_cast<size_t>(photons));
      for (int64_t p = 0; p < photons; ++p) {
        if (p >= steps[s0 + s]) {
          cols[p] = 0;
          continue;
        }
        const int32_t at = picks[p * shots + s0 + s];
        cols[p] = pool[at];
        std::memmove(pool + at, pool + at + 1, static_cast<size_t>(photons - p - 1 - at));
      }
    }
    PQP_HIP(hipMemcpyAsync(d, h, in_bytes, hipMemcpyHostToDevice, S.stream));
    SampleArgs a;
    a.u_t = reinterpret_cast<const double *>(d);
    a.draws = reinterpret_cast<const double *>(d + o_draws);
    a.steps = reinterpret_cast<const int32_t *>(d + o_steps);
    a.cols = reinterpret_cast<const uint8_t *>(d + o_cols);
    a.v = reinterpret_cast<double *>(w);
    a.occ = reinterpret_cast<uint8_t *>(w + w_occ);
    a.units = reinterpret_cast<int32_t *>(w + w_units);
    a.failed = reinterpret_cast<int32_t *>(w + w_failed);
    a.partials = reinterpret_cast<const double *>(w + w_part);
    a.shots = static_cast<int32_t>(n);
    a.modes = static_cast<int32_t>(modes);
    a.photons = static_cast<int32_t>(photons);
    a.waves = 1;
    PQP_HIP(launch_sample_columns(a, S.stream));
    int64_t last = 0;
    for (int64_t s = 0; s < n; ++s) last = std::max<int64_t>(last, steps[s0 + s]);
    for (int64_t step = 0; step < last; ++step) {
      if (step > 0) {
        MinorsWaveArgs m;
        m.rows = a.v;
        m.occ = a.occ;
        m.units = a.units;
        m.partials = reinterpret_cast<double *>(w + w_part);
        m.out = nullptr;
        m.item_stride = 2 * modes * photons;
        m.ld = static_cast<int32_t>(photons);
        m.modes = static_cast<int32_t>(modes);
        m.waves = passes.waves[step];
        m.k_max = passes.digits[step];
        m.last_counter = nullptr;
        m.done = nullptr;
        m.seq = 0;
        PQP_HIP(launch_minors_wave(static_cast<int>(step) + 1, m, static_cast<int>(n), S.stream));
        a.waves = m.waves;
      }
      a.step = static_cast<int32_t>(step);
      a.next_waves = passes.waves[step + 1];
      a.next_k_max = passes.digits[step + 1];
      PQP_HIP(launch_sample_step(a, S.stream));
    }
    PQP_HIP(hipMemcpyAsync(h, w + w_occ, w_failed + sizeof(int32_t) - w_occ, hipMemcpyDeviceToHost, S.stream));
    PQP_HIP(hipStreamSynchronize(S.stream));
    int32_t failed = 0;
    std::memcpy(&failed, h + (w_failed - w_occ), sizeof(failed));
    if (failed) return fail(PQP_ERR_INVALID, "probabilities contain NaN");
    const uint8_t *occ = reinterpret_cast<const uint8_t *>(h);
    for (int64_t t = 0; t < n * modes; ++t) out[s0 * modes + t] = occ[t];
  }
  return PQP_OK;
}

int pqp_sample_plan_info(int64_t shots, int64_t photons, int64_t first, int64_t *info) {
  if (!info || photons < 0 || first < 0 || first >= shots) return fail(PQP_ERR_INVALID, "invalid sampling plan arguments");
  if (photons > kMinorsWaveMaxCols)
    return fail(PQP_ERR_RANGE, "sampling on the device supports at most " + std::to_string(kMinorsWaveMaxCols) + " photons");
  const SamplePasses p = sample_passes(shots, photons);
  info[0] = std::min(p.most, shots - first / p.most * p.most);
  info[1] = static_cast<int64_t>(p.partials);
  for (int64_t step = 0; step < photons; ++step) {
    info[2 + 2 * step] = p.digits[step];
    info[3 + 2 * step] = p.waves[step];
  }
  return PQP_OK;
}

int pqp_perm_poly_plan_info(int64_t n, int64_t n_vars, int64_t n_out, const int32_t *exponents,
                            int64_t *info) {
  if (!info) return fail(PQP_ERR_INVALID, "info is null");
  PolyPlan p;
  std::string err;
  int st = poly_plan_build(n, n_vars, n_out, exponents, p, err);
  if (st != PQP_OK) return fail(st, err);
  info[0] = p.n_mono;
  info[1] = static_cast<int64_t>(p.links.size());
  info[2] = p.M;
  info[3] = p.L;
  info[4] = p.flops_per_subset;
  info[5] = static_cast<int64_t>(p.out_index.size());
  return PQP_OK;
}

int pqp_perm_poly_coefficients_c128(int64_t n, int64_t n_vars, const double *b0, const double *bm,
                                    int64_t n_out, const int32_t *exponents, double *out,
                                    int64_t *info) {
  CallRange range_("pqp_perm_poly_coefficients_c128");
  if (n_out < 0 || (n_out > 0 && !out) || (n >= 1 && !b0) || (n_vars > 0 && n >= 1 && !bm) ||
      (n_out > 0 && n_vars > 0 && !exponents))
    return fail(PQP_ERR_INVALID, "invalid matrix polynomial arguments");
  PolyState &S = poly_state();
  std::lock_guard<std::mutex> lock(S.mu);
  // The plan depends only on (n, the exponent rows): a call with the same
  // rows as the previous one reuses it and the tables already on the device.
  // Other rows of the same sizes must not cost an evaluation, so the rows are
  // compared before anything runs, of a long list on the layer path its first
  // kPolyCompareFirst bytes, and the others while the device works (7.4 MB
  // for 184756 outputs of 10 modes: 0.3 ms): lists that differ only there
  // start again with a plan of their own, which takes ten times as long.
  const size_t ex_bytes =
      (n_out > 0 && n_vars > 0) ? static_cast<size_t>(n_out) * static_cast<size_t>(n_vars) * sizeof(int32_t) : 0;
  const size_t n_ex = ex_bytes / sizeof(int32_t);
  if (S.have_plan && S.key_n == n && S.key_vars == n_vars && S.key_out == n_out) {
    const char *key = reinterpret_cast<const char *>(S.key_exps.data());
    const char *given = reinterpret_cast<const char *>(exponents);
    size_t layer_bytes = 0;
    const size_t first = S.tables_on_device && poly_layers_fit(S.plan, &layer_bytes)
                             ? std::min(ex_bytes, kPolyCompareFirst) : ex_bytes;
    bool same = first == 0 || std::memcmp(key, given, first) == 0;
    if (same) {
      auto rest = [&] { return same = first == ex_bytes || std::memcmp(key + first, given + first, ex_bytes - first) == 0; };
      bool asked = false;
      const int st = poly_run(S, b0, bm, n_out, out, info, [&] { asked = true; return rest(); });
      if (asked ? same : rest()) return st;
      g_error.clear();
    }
  }
  S.have_plan = false;
  S.tables_on_device = false;
  std::string err;
  const int st = poly_plan_build(n, n_vars, n_out, exponents, S.plan, err);
  if (st != PQP_OK) return fail(st, err);
  S.subsets.clear();
  S.subset_bits.clear();
  size_t layer_bytes = 0;
  if (poly_layers_fit(S.plan, &layer_bytes)) poly_subsets(S.plan.n, S.subsets, S.subset_bits, S.subset_first);
  S.key_n = n;
  S.key_vars = n_vars;
  S.key_out = n_out;
  S.key_exps.assign(exponents, exponents + n_ex);
  S.have_plan = true;
  return poly_run(S, b0, bm, n_out, out, info, [] { return true; });
}

int pqp_grad_batch_c128(int64_t count, const double *const *matrices, const int64_t *m_r,
                        const int64_t *m_c, const int64_t *ld, const int32_t *const *rows,
                        const int32_t *const *cols, double *perms, double *const *grads) {
  CallRange range_("pqp_grad_batch_c128");
  if (count < 0 || (count > 0 && (!matrices || !m_r || !m_c || !ld || !rows || !cols || !grads)))
    return fail(PQP_ERR_INVALID, "invalid gradient batch arguments");
  std::vector<PermInput> inputs;
  for (int64_t k = 0; k < count; ++k)
    inputs.push_back(PermInput{matrices[k], false, m_r[k], m_c[k], ld[k], rows[k], cols[k]});
  Plan plan;
  std::string err;
  PlanOptions opt;
  if (!gradients_fit_single_sweep(inputs)) return grad_batch_minors(inputs, perms, grads);
  opt.total_units = static_cast<int64_t>(std::max(device_state().cus, 1)) * kGradUnitsPerCu;
  opt.grad = true;
  int st = plan_build(inputs, opt, plan, err);
  if (st != PQP_OK) return fail(st, err);
  if (count == 0) return PQP_OK;
  if ((st = require_device()) != PQP_OK) return st;
  SingleState &S = single_state();
  std::lock_guard<std::mutex> lock(S.mu);
  Exec &x = S.x;
  if ((st = ensure_stream(x.stream)) != PQP_OK) return st;
  x.plan = std::move(plan);
  index_units(x);
  x.flags = PQP_FLAG_STATIC;
  if ((st = upload(x)) != PQP_OK) return st;
  if ((st = enqueue(x, PQP_RUN_EAGER, nullptr, nullptr)) != PQP_OK) return st;
  std::vector<double> res;
  if ((st = fetch_out(x, res)) != PQP_OK) return st;
  scatter_grad_items(x.plan, res, inputs, perms, grads);
  return PQP_OK;
}

int pqp_batch_create(int64_t count, const void *const *matrices, int is_c64, const int64_t *m_r,
                     const int64_t *m_c, const int64_t *ld, const int32_t *const *rows,
                     const int32_t *const *cols, uint32_t flags, int64_t target_inner,
                     int64_t total_units, pqp_batch **out) {
  CallRange range_("pqp_batch_create");
  if (!out) return fail(PQP_ERR_INVALID, "out is null");
  *out = nullptr;
  if (count < 0 || (count > 0 && (!matrices || !m_r || !m_c || !ld || !rows || !cols)))
    return fail(PQP_ERR_INVALID, "invalid batch arguments");
  if (count > INT32_MAX) return fail(PQP_ERR_RANGE, "too many items");
  std::vector<PermInput> inputs(static_cast<size_t>(count));
  for (int64_t k = 0; k < count; ++k)
    inputs[k] = PermInput{matrices[k], is_c64 != 0, m_r[k], m_c[k], ld[k], rows[k], cols[k]};
  // every early return (including a failed HIP call) releases what the
  // batch holds so far
  std::unique_ptr<pqp_batch, void (*)(pqp_batch *)> b(new (std::nothrow) pqp_batch(), pqp_batch_destroy);
  if (!b) return fail(PQP_ERR_NOMEM, "out of host memory");
  PlanOptions opt;
  opt.fp32_products = (flags & PQP_FLAG_FP32) != 0 || is_c64 != 0;
  opt.expand_cols = expand_mode(flags);
  opt.orient = (flags & PQP_FLAG_AS_GIVEN) == 0;
  opt.target_inner = target_inner;
  // about kBatchUnitsPerCu waves per CU over the whole batch, split by cost
  opt.total_units = total_units > 0
                        ? total_units
                        : static_cast<int64_t>(std::max(device_state().cus, 1)) * kBatchUnitsPerCu;
  std::string err;
  if (flags & PQP_FLAG_GRADIENT) {
    if (is_c64) return fail(PQP_ERR_INVALID, "gradients need complex128 input");
    b->grad = true;
    for (int64_t k = 0; k < count; ++k) {
      b->m_r.push_back(m_r[k]);
      b->m_c.push_back(m_c[k]);
      b->rows.emplace_back(rows[k], rows[k] + m_r[k]);
      b->cols.emplace_back(cols[k], cols[k] + m_c[k]);
      inputs[k].rows = b->rows.back().data();
      inputs[k].cols = b->cols.back().data();
    }
    b->grad_minors = !gradients_fit_single_sweep(inputs);
    opt.grad = !b->grad_minors;
    if (opt.grad && total_units <= 0)
      opt.total_units = static_cast<int64_t>(std::max(device_state().cus, 1)) * kGradUnitsPerCu;
  }
  int st = plan_build(inputs, opt, b->x.plan, err);
  if (st != PQP_OK) return fail(st, err);
  if (b->grad_minors) {
    std::vector<PermInput> minputs;
    minor_inputs(inputs, b->minor_rows, b->minor_item, b->minor_row, minputs);
    PlanOptions mopt;
    mopt.total_units = opt.total_units;
    MinorsPlan mp;
    st = build_minors_plan(minputs, mopt, mp, err);
    if (st != PQP_OK) return fail(st, err);
    b->xm.plan = std::move(mp.plan);
    b->minor_slot = std::move(mp.slot);
  }
  if ((st = require_device()) != PQP_OK) return st;
  index_units(b->x);
  b->x.flags = flags;
  if ((st = ensure_stream(b->x.stream)) != PQP_OK) return st;
  if ((st = upload(b->x)) != PQP_OK) return st;
  if (b->grad_minors) {
    index_units(b->xm);
    b->xm.flags = PQP_FLAG_STATIC;
    b->xm.stream = b->x.stream;  // shares the batch stream (and its graph)
    if ((st = upload(b->xm)) != PQP_OK) return st;
  }
  PQP_HIP(hipStreamSynchronize(b->x.stream));
  *out = b.release();
  return PQP_OK;
}

int pqp_permanent_batch_c128(int64_t count, const double *const *matrices, const int64_t *m_r,
                             const int64_t *m_c, const int64_t *ld, const int32_t *const *rows,
                             const int32_t *const *cols, uint32_t flags, int64_t target_inner,
                             int64_t total_units, double *out) {
  CallRange range_("pqp_permanent_batch_c128");
  if (count < 0 || (count > 0 && (!matrices || !m_r || !m_c || !ld || !rows || !cols || !out)))
    return fail(PQP_ERR_INVALID, "invalid batch arguments");
  if (count > INT32_MAX) return fail(PQP_ERR_RANGE, "too many items");
  std::vector<PermInput> inputs(static_cast<size_t>(count));
  for (int64_t k = 0; k < count; ++k)
    inputs[k] = PermInput{matrices[k], false, m_r[k], m_c[k], ld[k], rows[k], cols[k]};
  PlanOptions opt;
  opt.fp32_products = (flags & PQP_FLAG_FP32) != 0;
  opt.expand_cols = expand_mode(flags);
  opt.orient = (flags & PQP_FLAG_AS_GIVEN) == 0;
  opt.target_inner = target_inner;
  opt.total_units = total_units > 0
                        ? total_units
                        : static_cast<int64_t>(std::max(device_state().cus, 1)) * kBatchUnitsPerCu;
  Plan plan;
  std::string err;
  int st = plan_build(inputs, opt, plan, err);
  if (st != PQP_OK) return fail(st, err);
  if ((st = require_device()) != PQP_OK) return st;
  if (count == 0) return PQP_OK;
  OneShotLease lease;
  Exec &x = *lease.x;
  if ((st = ensure_stream(x.stream)) != PQP_OK) return st;
  x.plan = std::move(plan);
  index_units(x);
  x.flags = flags;
  const size_t out_bytes = static_cast<size_t>(count) * 2 * sizeof(double);
  if ((st = x.stage.ensure(std::max(x.plan.arena.size(), out_bytes))) != PQP_OK) return st;
  if ((st = upload(x)) != PQP_OK) return st;
  if ((st = enqueue(x, PQP_RUN_EAGER, nullptr, nullptr)) != PQP_OK) return st;
  // item k's value is result k; the copy follows the upload out of the
  // staging buffer on the stream
  PQP_HIP(hipMemcpyAsync(x.stage.p, x.results.p, out_bytes, hipMemcpyDeviceToHost, x.stream));
  PQP_HIP(hipStreamSynchronize(x.stream));
  std::memcpy(out, x.stage.p, out_bytes);
  lease.finished = true;
  return PQP_OK;
}

int pqp_batch_run(pqp_batch *b, int mode) {
  CallRange range_("pqp_batch_run");
  if (!b) return fail(PQP_ERR_INVALID, "batch is null");
  int st;
  if (mode == PQP_RUN_GRAPH) {
    if (!b->graph_exec) {
      PQP_HIP(hipStreamBeginCapture(b->x.stream, hipStreamCaptureModeThreadLocal));
      st = enqueue_all(b, PQP_RUN_EAGER, nullptr, nullptr);
      hipGraph_t g = nullptr;
      hipError_t e = hipStreamEndCapture(b->x.stream, &g);
      if (st != PQP_OK) {
        if (g) (void)hipGraphDestroy(g);
        return st;
      }
      if (e != hipSuccess) return fail(PQP_ERR_DEVICE, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
      b->graph = g;
      PQP_HIP(hipGraphInstantiate(&b->graph_exec, b->graph, nullptr, nullptr, 0));
    }
    PQP_HIP(hipGraphLaunch(b->graph_exec, b->x.stream));
  } else if (mode == PQP_RUN_EAGER || mode == PQP_RUN_PLAIN || mode == PQP_RUN_KERNEL) {
    if ((st = enqueue_all(b, mode, nullptr, nullptr)) != PQP_OK) return st;
  } else {
    return fail(PQP_ERR_INVALID, "unknown run mode");
  }
  b->ran = true;
  return PQP_OK;
}

int pqp_batch_sync(pqp_batch *b) {
  CallRange range_("pqp_batch_sync");
  if (!b) return fail(PQP_ERR_INVALID, "batch is null");
  PQP_HIP(hipStreamSynchronize(b->x.stream));
  return PQP_OK;
}

int pqp_batch_results(pqp_batch *b, double *out, double *out_dd) {
  CallRange range_("pqp_batch_results");
  if (!b) return fail(PQP_ERR_INVALID, "batch is null");
  if (!b->ran) return fail(PQP_ERR_INVALID, "batch has not been run");
  const size_t n = b->x.plan.items.size();
  PQP_HIP(hipStreamSynchronize(b->x.stream));
  if (b->grad && !b->grad_minors && n) {
    // gradient plans: the permanent of item k sits at its first output slot
    std::vector<double> all(2 * b->x.n_results), all_dd(4 * b->x.n_results);
    PQP_HIP(hipMemcpy(all.data(), b->x.results.p, all.size() * sizeof(double), hipMemcpyDeviceToHost));
    if (out_dd)
      PQP_HIP(hipMemcpy(all_dd.data(), static_cast<double *>(b->x.results.p) + 2 * b->x.n_results,
                        all_dd.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (size_t k = 0; k < n; ++k) {
      const int64_t o = b->x.plan.info[k].out_offset;
      if (out) std::memcpy(out + 2 * k, all.data() + 2 * o, 2 * sizeof(double));
      if (out_dd) std::memcpy(out_dd + 4 * k, all_dd.data() + 4 * o, 4 * sizeof(double));
    }
    return PQP_OK;
  }
  if (out && n) PQP_HIP(hipMemcpy(out, b->x.results.p, n * 2 * sizeof(double), hipMemcpyDeviceToHost));
  if (out_dd && n)
    PQP_HIP(hipMemcpy(out_dd, static_cast<double *>(b->x.results.p) + 2 * b->x.n_results,
                      n * 4 * sizeof(double), hipMemcpyDeviceToHost));
  return PQP_OK;
}

int pqp_batch_error_bounds(pqp_batch *b, double *bounds) {
  CallRange range_("pqp_batch_error_bounds");
  if (!b || (!bounds && !b->x.plan.items.empty())) return fail(PQP_ERR_INVALID, "invalid arguments");
  if (!b->ran) return fail(PQP_ERR_INVALID, "batch has not been run");
  const size_t n = b->x.plan.items.size();
  if (!n) return PQP_OK;
  PQP_HIP(hipStreamSynchronize(b->x.stream));
  const double nan = std::numeric_limits<double>::quiet_NaN();
  // the gradient kernels and the plain baseline keep no term magnitudes
  if (!b->x.abs_valid) {
    for (size_t k = 0; k < n; ++k) bounds[k] = nan;
    return PQP_OK;
  }
  const size_t nr = b->x.n_results;
  std::vector<double> all(7 * nr);
  PQP_HIP(hipMemcpy(all.data(), b->x.results.p, all.size() * sizeof(double), hipMemcpyDeviceToHost));
  for (size_t k = 0; k < n; ++k) {
    const int64_t o = b->x.plan.info[k].out_offset;
    bounds[k] = sweep_error_bound(b->x.plan.items[k].n, b->x.plan.fp32, all[6 * nr + o],
                                  all[2 * o], all[2 * o + 1]);
  }
  return PQP_OK;
}

int pqp_batch_time(pqp_batch *b, int mode, int reps, float *ms) {
  CallRange range_("pqp_batch_time");
  if (!b || reps < 0 || (reps > 0 && !ms)) return fail(PQP_ERR_INVALID, "invalid timing arguments");
  hipEvent_t e0, e1;
  PQP_HIP(hipEventCreate(&e0));
  PQP_HIP(hipEventCreate(&e1));
  int st = PQP_OK;
  for (int r = 0; r < reps && st == PQP_OK; ++r) {
    if (mode == PQP_RUN_GRAPH) {
      if (!b->graph_exec) st = pqp_batch_run(b, PQP_RUN_GRAPH);  // builds the graph
      if (st != PQP_OK) break;
      (void)hipStreamSynchronize(b->x.stream);
      (void)hipEventRecord(e0, b->x.stream);
      (void)hipGraphLaunch(b->graph_exec, b->x.stream);
      (void)hipEventRecord(e1, b->x.stream);
    } else {
      st = enqueue_all(b, mode, e0, e1);
      if (st != PQP_OK) break;
    }
    hipError_t e = hipEventSynchronize(e1);
    if (e != hipSuccess) {
      st = fail(PQP_ERR_DEVICE, std::string("hipEventSynchronize: ") + hipGetErrorString(e));
      break;
    }
    (void)hipEventElapsedTime(&ms[r], e0, e1);
    b->ran = true;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return st;
}

int pqp_batch_time_span(pqp_batch *b, int mode, int reps, float *ms) {
  CallRange range_("pqp_batch_time_span");
  if (!b || reps < 1 || !ms) return fail(PQP_ERR_INVALID, "invalid timing arguments");
  if (mode != PQP_RUN_GRAPH && mode != PQP_RUN_EAGER)
    return fail(PQP_ERR_INVALID, "span timing takes the graph or eager mode");
  // the graph is built outside the timed span
  if (mode == PQP_RUN_GRAPH && !b->graph_exec) {
    int st = pqp_batch_run(b, PQP_RUN_GRAPH);
    if (st != PQP_OK) return st;
  }
  PQP_HIP(hipStreamSynchronize(b->x.stream));
  hipEvent_t e0, e1;
  PQP_HIP(hipEventCreate(&e0));
  hipError_t he = hipEventCreate(&e1);
  if (he != hipSuccess) {
    (void)hipEventDestroy(e0);
    return fail(PQP_ERR_DEVICE, std::string("hipEventCreate: ") + hipGetErrorString(he));
  }
  int st = PQP_OK;
  (void)hipEventRecord(e0, b->x.stream);
  for (int r = 0; r < reps && st == PQP_OK; ++r) st = pqp_batch_run(b, mode);
  (void)hipEventRecord(e1, b->x.stream);
  he = hipEventSynchronize(e1);
  if (he != hipSuccess && st == PQP_OK)
    st = fail(PQP_ERR_DEVICE, std::string("hipEventSynchronize: ") + hipGetErrorString(he));
  if (st == PQP_OK) (void)hipEventElapsedTime(ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return st;
}

int pqp_batch_stats(const pqp_batch *b, double *flops, int64_t *terms, int64_t *units,
                    int64_t *arena_bytes, int64_t *lane_terms) {
  if (!b) return fail(PQP_ERR_INVALID, "batch is null");
  const bool m = b->grad_minors;
  if (lane_terms) {
    int64_t lt = 0;
    for (const Plan *p : {&b->x.plan, &b->xm.plan})
      for (const ItemDesc &d : p->items) lt += static_cast<int64_t>(d.units) * kWave * d.S_in;
    *lane_terms = lt;
  }
  if (flops) *flops = b->x.plan.total_flops + (m ? b->xm.plan.total_flops : 0.0);
  if (terms) *terms = b->x.plan.total_terms + (m ? b->xm.plan.total_terms : 0);
  if (units) *units = static_cast<int64_t>(b->x.plan.units.size() + (m ? b->xm.plan.units.size() : 0));
  if (arena_bytes)
    *arena_bytes = static_cast<int64_t>(b->x.plan.arena.size() + (m ? b->xm.plan.arena.size() : 0));
  return PQP_OK;
}

int pqp_batch_gradients(pqp_batch *b, double *const *grads) {
  CallRange range_("pqp_batch_gradients");
  if (!b || !grads) return fail(PQP_ERR_INVALID, "invalid arguments");
  if (!b->grad) return fail(PQP_ERR_INVALID, "batch was not created with PQP_FLAG_GRADIENT");
  if (!b->ran) return fail(PQP_ERR_INVALID, "batch has not been run");
  std::vector<double> res;
  int st;
  std::vector<PermInput> inputs;
  for (size_t k = 0; k < b->m_r.size(); ++k)
    inputs.push_back(PermInput{nullptr, false, b->m_r[k], b->m_c[k], b->m_c[k],
                               b->rows[k].data(), b->cols[k].data()});
  if (b->grad_minors) {
    if (!b->minor_item.empty() && (st = fetch_out(b->xm, res)) != PQP_OK) return st;
    scatter_gradients(b->minor_slot, res, b->minor_item, b->minor_row, inputs, grads);
    return PQP_OK;
  }
  if ((st = fetch_out(b->x, res)) != PQP_OK) return st;
  scatter_grad_items(b->x.plan, res, inputs, nullptr, grads);
  return PQP_OK;
}

int pqp_plan_image(const double *matrix, int64_t m_r, int64_t m_c, int64_t ld,
                   const int32_t *rows, const int32_t *cols, uint32_t flags,
                   int64_t target_inner, int64_t min_units, void *buf, int64_t buf_bytes,
                   int64_t *needed_bytes) {
  PermInput in{matrix, false, m_r, m_c, ld, rows, cols};
  PlanOptions opt;
  opt.fp32_products = (flags & PQP_FLAG_FP32) != 0;
  opt.expand_cols = expand_mode(flags);
  opt.orient = (flags & PQP_FLAG_AS_GIVEN) == 0;
  opt.target_inner = target_inner;
  opt.min_units = min_units;
  opt.minors = (flags & PQP_FLAG_GRADIENT) != 0;
  opt.grad = !opt.minors && (flags & PQP_PLAN_GRADIENT_SWEEP) != 0;
  Plan p;
  std::string err;
  const int st = plan_build(std::vector<PermInput>{in}, opt, p, err);
  if (st != PQP_OK) return fail(st, err);
  if (needed_bytes) *needed_bytes = static_cast<int64_t>(p.arena.size());
  if (buf && buf_bytes >= static_cast<int64_t>(p.arena.size()))
    std::memcpy(buf, p.arena.data(), p.arena.size());
  else if (buf)
    return fail(PQP_ERR_INVALID, "buffer too small for the plan image");
  return PQP_OK;
}

void pqp_batch_destroy(pqp_batch *b) {
  if (!b) return;
  if (b->x.stream) (void)hipStreamSynchronize(b->x.stream);
  if (b->graph_exec) (void)hipGraphExecDestroy(b->graph_exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  release_exec(b->xm, false);  // shares b->x's stream
  release_exec(b->x, true);
  delete b;
}

}  // extern "C"
