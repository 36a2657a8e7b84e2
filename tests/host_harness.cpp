// The host side of the handle (su2higgs_amd/csrc/su2hip_api.cpp) on the CPU:
// device memory is host memory, kernels are the records of their launches,
// and the runtime's calls can be made to fail.  Built and run by
// test_host_side.py; argv[1] names a scenario, a failed check ends with 1.
#include <hip/hip_runtime.h>
#undef __align__
#define __align__(n)
#define HIP_SYMBOL(x) ((const void *)&(x))

#include <stdlib.h>
#include <string.h>
#include <time.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <functional>
#include <set>
#include <vector>

namespace fake {
hipError_t last = hipSuccess;  // as hipGetLastError: a later success does not clear it
std::function<bool(size_t)> refuse = [](size_t) { return false; };
std::function<hipError_t()> launch_fails = [] { return hipSuccess; };
int wait_ms = 0;  // of an event
std::atomic<int> waits{0};
int singles = 0, pairs = 0;
int alt = 0;  // the fields in second buffers
std::set<void *> live;

hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
hipError_t alloc(void **p, size_t n) {
  if (refuse(n)) return ret(hipErrorOutOfMemory);
  *p = aligned_alloc(256, (n + 255) / 256 * 256);
  live.insert(*p);
  return hipSuccess;
}
hipError_t release(void *p) {
  if (!p) return hipSuccess;
  if (!live.erase(p)) abort();
  free(p);
  return hipSuccess;
}
hipError_t launch() {
  ret(launch_fails());
  return hipGetLastError();
}
}  // namespace fake

extern "C" {
hipError_t hipGetLastError(void) {
  hipError_t e = fake::last;
  fake::last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipMalloc(void **p, size_t n) { return fake::alloc(p, n); }
hipError_t hipFree(void *p) { return fake::release(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return fake::alloc(p, n); }
hipError_t hipHostFree(void *p) { return fake::release(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *s) { *p = (void *)s; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = (hipGraph_t)1; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) { *x = (hipGraphExec_t)1; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
  // the work before the first piece takes its time
  if (fake::waits++ == 0 && fake::wait_ms) usleep(1000 * fake::wait_ms);
  return hipSuccess;
}
int roctxRangePushA(const char *) { return 0; }
int roctxRangePop(void) { return 0; }
}

#include "../su2higgs_amd/csrc/su2hip_api.cpp"

namespace su2 {
hipError_t launch_pass(const LaunchCtx &, int, int, int, int, int) { fake::singles++; return fake::launch(); }
bool pair_kind(int kind, int, int) { return kind != SU2HIP_K_LINK_METROPOLIS; }
int pair_bit(int kind, int dir) {
  return kind <= SU2HIP_K_LINK_OVERRELAX ? 1 << dir
         : kind == SU2HIP_K_U1_METROPOLIS ? 1 << (ALT_U1_SHIFT + dir)
         : kind <= SU2HIP_K_DOUBLET_METROPOLIS ? ALT_F
         : kind <= SU2HIP_K_TRIPLET_METROPOLIS ? ALT_G : ALT_S;
}
hipError_t launch_pair(const LaunchCtx &, const PairTile *, int, int, int kind, int dir, int, long long *, int) {
  fake::pairs++;
  const hipError_t e = fake::launch();
  if (e == hipSuccess) fake::alt ^= pair_bit(kind, dir);
  return e;
}
hipError_t launch_pair_close(const LaunchCtx &c) {
  if (c.alt == fake::alt) fake::alt = 0;
  return fake::launch();
}
hipError_t launch_order(const LaunchCtx &, uint8_t *, const uint16_t *, int, int, int) { return fake::launch(); }
hipError_t launch_hop(const LaunchCtx &) { return fake::launch(); }
hipError_t launch_end_sweep(const LaunchCtx &c, int passes) {
  for (int i = 0; i < c.max_slots; i++) {
    LatDesc &L = c.desc[i];
    if (!L.active || L.budget == 0) continue;
    L.pass += passes;
    if (L.budget > 0) L.budget--;
  }
  return fake::launch();
}
hipError_t launch_cold(const LaunchCtx &, int, double, double, double) { return fake::launch(); }
hipError_t launch_measure(const LaunchCtx &) { return fake::launch(); }
hipError_t launch_orderparam_init(const LaunchCtx &, int) { return fake::launch(); }
hipError_t launch_flow_stage(const LaunchCtx &, int, const void *, void *, const void *, void *, void *, void *, double, double, int) { return fake::launch(); }
hipError_t launch_to_host_layout(const LaunchCtx &, int, int Vh, int f, double *h) {
  const int dofs[6] = {12, 3, 4, 3, 1, 4};
  for (size_t i = 0; i < (size_t)2 * Vh * dofs[f]; i++) h[i] = 1e8 * f + (double)i;
  return fake::launch();
}
hipError_t launch_copy(const void *s, void *d, size_t n, hipStream_t) { memcpy(d, s, n); return fake::launch(); }
}  // namespace su2

static void must(bool ok, const char *what, int line) {
  if (ok) return;
  fprintf(stderr, "line %d: %s (%s)\n", line, what, g_err.c_str());
  exit(1);
}
#define MUST(x) must(x, #x, __LINE__)

static su2hip_params params(int L0, int L1, int L2, int nhiggs = 1, int u1 = 0) {
  su2hip_params p{};
  p.L[0] = L0;
  p.L[1] = L1;
  p.L[2] = L2;
  p.precision = SU2HIP_FP32;
  p.nhiggs = nhiggs;
  p.u1 = u1;
  p.betasu2 = 9.0;
  p.betau1 = 9.0;
  p.r_u1 = 1.0;
  p.algorithm_su2link = SU2HIP_HEATBATH;
  p.algorithm_u1link = SU2HIP_METROPOLIS;
  p.algorithm_su2doublet = p.algorithm_su2triplet = p.algorithm_singlet = SU2HIP_OVERRELAX;
  p.update_links = p.update_su2doublet = p.update_su2triplet = p.update_singlet = 1;
  p.link_overrelax = 4;
  p.scalar_sweeps = 2;
  p.link_format = SU2HIP_LINKS_FULL;
  return p;
}

static su2hip_batch_t *made(const std::vector<su2hip_params> &v, int max_slots = 0, uint64_t budget = 0) {
  su2hip_batch_t *b = nullptr;
  const int rc = su2hip_create((int)v.size(), v.data(), std::max(max_slots, (int)v.size()), budget, &b);
  MUST(rc == SU2HIP_OK);
  return b;
}

// a sweep's launches: whether the links were paired
static bool sweep_pairs(su2hip_batch_t *b) {
  fake::singles = fake::pairs = 0;
  MUST(su2hip_update(b, 1) == SU2HIP_OK);
  MUST(fake::singles + fake::pairs > 0);
  return fake::pairs > 0;
}

// The optional second buffers are refused: sweeps of single passes, no error
// left behind for the next launch.
static void refused_buffers() {
  const std::vector<su2hip_params> v{params(8, 8, 8)};
  int refused = 0;
  size_t slot = slot_bytes(v[0]);
  int seen = 0;
  fake::refuse = [&](size_t n) { return n == slot && ++seen == 2 && ++refused; };
  su2hip_batch_t *b = made(v);
  MUST(refused == 1);
  MUST(!sweep_pairs(b));
  MUST(hipGetLastError() == hipSuccess);
  MUST(su2hip_destroy(b) == SU2HIP_OK);
}

// A call that is refused for want of memory leaves no error behind either.
static void refused_call() {
  su2hip_batch_t *b = made({params(8, 8, 8)});
  fake::refuse = [](size_t) { return true; };
  double rows[1 + SU2HIP_NSUMS];
  int n = 0;
  MUST(su2hip_flow(b, 0, SU2HIP_FLOW_RK3, 0.05, 0.5, 1, rows, 1, &n) == SU2HIP_ENOMEM);
  MUST(su2hip_autotune(b, 1, nullptr) == SU2HIP_ENOMEM);
  fake::refuse = [](size_t) { return false; };
  MUST(sweep_pairs(b));
  MUST(su2hip_destroy(b) == SU2HIP_OK);
}

// The tables of paired passes, allocated after the second buffers, are refused:
// single passes, and paired ones when the tables are next built.
static void refused_tables() {
  const size_t slot = slot_bytes(params(8, 8, 8));
  for (int k = 0; k < 2; k++) {
    int buffers = 0, tables = 0;
    fake::refuse = [&](size_t n) {
      if (n == slot) return ++buffers > 2;
      return buffers == 2 && tables++ == k;
    };
    su2hip_batch_t *b = made({params(8, 8, 8)}, 2);
    MUST(tables > k);
    fake::refuse = [](size_t) { return false; };
    MUST(!sweep_pairs(b));
    int i = -1;
    const su2hip_params p = params(4, 4, 4);
    MUST(su2hip_add(b, &p, &i) == SU2HIP_OK);
    MUST(sweep_pairs(b));
    MUST(su2hip_destroy(b) == SU2HIP_OK);
  }
}

// A buffer that could not grow is not taken for one of its old size.
static void refused_growth() {
  int i = -1;
  const su2hip_params p = params(64, 64, 64);
  // each of the block tables, in su2hip_add
  for (int k = 0; k < 7; k++) {
    su2hip_batch_t *b = made({params(8, 8, 8)}, 2);
    int left = k;
    fake::refuse = [&](size_t n) { return n < slot_bytes(p) / 2 && left-- == 0; };
    MUST(su2hip_add(b, &p, &i) == SU2HIP_ENOMEM);
    fake::refuse = [](size_t) { return false; };
    MUST(su2hip_remove(b, 1) == SU2HIP_OK);
    MUST(b->d_blk && b->d_cnt && b->d_partial);
    for (const auto &m : b->alt) MUST(m.d_blk && m.d_cnt);
    MUST(su2hip_update(b, 1) == SU2HIP_OK);
    MUST(su2hip_destroy(b) == SU2HIP_OK);
  }
  // the staging buffer
  su2hip_batch_t *b = made({params(8, 8, 8), p});
  std::vector<double> small(12 * 512), big((size_t)12 << 18);
  MUST(su2hip_get_fields(b, 0, small.data(), nullptr, nullptr, nullptr, nullptr) == SU2HIP_OK);
  fake::refuse = [](size_t) { return true; };
  MUST(su2hip_get_fields(b, 1, big.data(), nullptr, nullptr, nullptr, nullptr) == SU2HIP_ENOMEM);
  fake::refuse = [](size_t) { return false; };
  MUST(su2hip_get_fields(b, 0, small.data(), nullptr, nullptr, nullptr, nullptr) == SU2HIP_OK);
  MUST(b->d_stage);
  MUST(su2hip_destroy(b) == SU2HIP_OK);
}

// The second buffers give way to a request that fits without them, and only to
// such a one; where it is given back they return.
static void budget_requests() {
  const std::vector<su2hip_params> v{params(8, 8, 8), params(8, 8, 8)};
  const uint64_t slots = 2 * slot_bytes(v[0]), hop = hop_cache_bytes(v[0]);
  double rows[1 + SU2HIP_NSUMS];
  int n = 0;
  // the fields, their caches and the second buffers
  su2hip_batch_t *b = made(v, 2, 2 * slots + 2 * hop);
  MUST(sweep_pairs(b));
  // flow buffers of a lattice: more than the second buffers hold
  MUST(flow_words(v[0]) * wsize(v[0]) > slots);
  MUST(su2hip_flow(b, 0, SU2HIP_FLOW_RK3, 0.05, 0.5, 1, rows, 1, &n) == SU2HIP_ENOMEM);
  MUST(sweep_pairs(b));
  MUST(su2hip_destroy(b) == SU2HIP_OK);
  // room for the caches or for the second buffers
  b = made(v, 2, 2 * slots + hop);
  MUST(!sweep_pairs(b));
  MUST(su2hip_set_hop_cache(b, 0) == SU2HIP_OK);
  MUST(sweep_pairs(b));
  MUST(su2hip_set_hop_cache(b, 1) == SU2HIP_OK);
  MUST(!sweep_pairs(b));
  MUST(su2hip_destroy(b) == SU2HIP_OK);
}

// Installing a weight leaves every lattice at its place in its stream of draws.
static void weight_keeps_draws() {
  su2hip_batch_t *b = made({params(8, 8, 8), params(4, 4, 4)});
  su2hip_muca m{};
  m.enabled = 1;
  m.bins = 4;
  m.checks_per_sweep = 1;
  m.orderparam = SU2HIP_PHISQ;
  const double pos[6] = {0, 1, 2, 3, 4, 5}, W[6] = {};
  MUST(su2hip_set_budget(b, 1, 7) == SU2HIP_OK);
  MUST(su2hip_update(b, 5) == SU2HIP_OK);
  MUST(su2hip_muca_set(b, 0, &m, pos, W) == SU2HIP_OK);
  uint64_t seed, pass;
  for (int i = 0; i < 2; i++) {
    MUST(su2hip_rng_get(b, i, &seed, &pass) == SU2HIP_OK);
    MUST(pass == 5 * (uint64_t)b->passes);
  }
  int64_t left[2];
  MUST(su2hip_get_budgets(b, left) == SU2HIP_OK);
  MUST(left[0] == -1 && left[1] == 2);
  MUST(su2hip_destroy(b) == SU2HIP_OK);
}

// A lattice added to a handle is swept like those it was created with.
static void added_lattice_sweeps() {
  for (int n = 0; n < 2; n++) {
    su2hip_batch_t *b = nullptr;
    const su2hip_params p = params(8, 8, 8), q = params(4, 4, 4);
    MUST(su2hip_create(n, &p, 3, 0, &b) == SU2HIP_OK);
    for (int k = 0; k < 2; k++) {  // a new slot, and one used before
      int i = -1;
      MUST(su2hip_add(b, &q, &i) == SU2HIP_OK && i == n);
      MUST(su2hip_update(b, 2) == SU2HIP_OK);
      int64_t left[3];
      uint64_t seed, pass;
      MUST(su2hip_get_budgets(b, left) == SU2HIP_OK && left[i] == -1);
      MUST(su2hip_rng_get(b, i, &seed, &pass) == SU2HIP_OK && pass == 2 * (uint64_t)b->passes);
      MUST(su2hip_remove(b, i) == SU2HIP_OK);
    }
    MUST(su2hip_destroy(b) == SU2HIP_OK);
  }
}

// Fetching fields behind queued sweeps: no thread is busy while the GPU is, and
// every value arrives.
static void fetch_waits_idle() {
  const su2hip_params p = params(64, 48, 32, 1, 1);
  su2hip_batch_t *b = made({p});
  const size_t V = (size_t)vol_of(p);
  std::vector<double> u(12 * V), a(3 * V), f(4 * V);
  fake::waits = 0;
  fake::wait_ms = 400;
  timespec t0, t1;
  clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t0);
  MUST(su2hip_get_fields(b, 0, u.data(), a.data(), f.data(), nullptr, nullptr) == SU2HIP_OK);
  clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t1);
  const double cpu = (t1.tv_sec - t0.tv_sec) + 1e-9 * (t1.tv_nsec - t0.tv_nsec);
  MUST(fake::waits > DOWN_SLOTS);
  for (size_t i = 0; i < u.size(); i++) MUST(u[i] == (double)i);
  for (size_t i = 0; i < a.size(); i++) MUST(a[i] == 1e8 + (double)i);
  for (size_t i = 0; i < f.size(); i++) MUST(f[i] == 2e8 + (double)i);
  MUST(cpu < 0.3);  // four threads in a loop: 1.6 s
  MUST(su2hip_destroy(b) == SU2HIP_OK);
}

// Choosing the tiles of paired passes, on every admission of a lattice, costs by
// the shapes of lattice in the handle and not by the lattices.
static void many_alike() {
  double cpu[2];
  for (int k = 0; k < 2; k++) {
    su2hip_batch_t *b = made(std::vector<su2hip_params>(k ? 1500 : 1, params(4, 4, 4, 0)));
    cpu[k] = 1e9;
    for (int r = 0; r < 9; r++) {
      timespec t0, t1;
      clock_gettime(CLOCK_THREAD_CPUTIME_ID, &t0);
      MUST(build_pairs(b) == SU2HIP_OK && b->pair_on);
      clock_gettime(CLOCK_THREAD_CPUTIME_ID, &t1);
      cpu[k] = std::min(cpu[k], (t1.tv_sec - t0.tv_sec) + 1e-9 * (t1.tv_nsec - t0.tv_nsec));
    }
    MUST(su2hip_destroy(b) == SU2HIP_OK);
  }
  // the tables grow with the lattices; the search alone grew by 900
  MUST(cpu[1] < 300 * cpu[0]);
}

// A launch that fails in the middle of a sweep leaves no field in its second
// buffer, which nothing reads between sweeps.
static void failed_launch() {
  su2hip_batch_t *b = made({params(8, 8, 8, 1, 1)});
  int n = 0;
  fake::launch_fails = [&] { return n++, hipSuccess; };
  MUST(sweep_pairs(b));
  MUST(fake::alt == 0);
  const int launches = n;
  MUST(launches > 12);
  for (int k = 0; k < launches; k++) {
    n = 0;
    fake::launch_fails = [&] { return n++ == k ? hipErrorLaunchFailure : hipSuccess; };
    MUST(su2hip_update(b, 1) == SU2HIP_EDEVICE);
    MUST(fake::alt == 0);
  }
  MUST(su2hip_destroy(b) == SU2HIP_OK);
}

// Which passes of a sweep are paired, for the handles of test_gpu_pairs.py and
// test_gpu_pairs_mixed.py.
static su2hip_params shaped(int form, int a, int b, int c, int nhiggs, int u1, int triplet, int singlet) {
  su2hip_params p = params(a, b, c, nhiggs, u1);
  p.precision = form ? SU2HIP_FP32 : SU2HIP_FP64;
  p.link_format = form == 2 ? SU2HIP_LINKS_PACKED : form == 1 ? SU2HIP_LINKS_FULL : SU2HIP_LINKS_AUTO;
  p.triplet = triplet;
  p.singlet = singlet;
  return p;
}
static uint64_t footprints(const std::vector<su2hip_params> &v) {
  uint64_t total = 0;
  for (const auto &p : v) {
    uint64_t n = 0;
    MUST(su2hip_footprint(&p, 0, &n) == SU2HIP_OK);
    total += n;
  }
  return total;
}
static void which_sweeps_pair() {
  using Ext = std::vector<std::array<int, 3>>;
  const std::vector<Ext> small = {
      {{4, 4, 2}, {2, 4, 6}, {8, 8, 8}}, {{34, 10, 14}}, {{128, 6, 4}, {4, 26, 12}},
      {{24, 24, 24}, {16, 30, 10}, {12, 6, 50}}, {{12, 10, 14}, {8, 8, 8}, {4, 26, 12}},
      {{8, 8, 8}, {12, 10, 8}, {16, 16, 16}, {6, 8, 10}}};
  const std::vector<Ext> links = {{{40, 34, 30}}, {{24, 30, 26}, {34, 26, 22}}};
  const std::vector<Ext> none = {{{64, 48, 40}}, {{130, 4, 4}}};
  const int models[][4] = {{0, 0, 0, 0}, {1, 1, 0, 0}, {1, 1, 0, 1}, {0, 0, 1, 0}, {1, 0, 1, 0}};
  auto batch = [&](const Ext &x, int form, const int *m) {
    std::vector<su2hip_params> v;
    for (const auto &e : x) v.push_back(shaped(form, e[0], e[1], e[2], m[0], m[1], m[2], m[3]));
    return v;
  };
  for (int form = 0; form < 3; form++)
    for (const auto &m : models) {
      for (const auto &x : small) {
        su2hip_batch_t *b = made(batch(x, form, m));
        MUST(sweep_pairs(b) && b->pair_fields);
        MUST(su2hip_destroy(b) == SU2HIP_OK);
        // a budget of the footprints leaves no room
        b = made(batch(x, form, m), 0, footprints(batch(x, form, m)));
        MUST(!sweep_pairs(b));
        MUST(su2hip_destroy(b) == SU2HIP_OK);
      }
      for (const auto &x : links) {
        su2hip_batch_t *b = made(batch(x, form, m));
        MUST(sweep_pairs(b) && !b->pair_fields);
        MUST(fake::pairs == 15 && (fake::singles > 0) == (m[0] + m[2] > 0));
        MUST(su2hip_destroy(b) == SU2HIP_OK);
        b = made(batch(x, form, m), 0, footprints(batch(x, form, m)));
        MUST(!sweep_pairs(b));
        MUST(su2hip_destroy(b) == SU2HIP_OK);
      }
      for (const auto &x : none) {
        su2hip_batch_t *b = made(batch(x, form, m));
        MUST(!sweep_pairs(b));
        MUST(su2hip_destroy(b) == SU2HIP_OK);
      }
    }
  // one round of Metropolis, one of overrelaxation
  su2hip_params p = params(12, 10, 8, 1, 1);
  p.algorithm_su2link = SU2HIP_METROPOLIS;
  p.link_overrelax = 1;
  su2hip_batch_t *b = made({p});
  MUST(sweep_pairs(b) && fake::singles == 6);
  // the shuffled order
  MUST(su2hip_set_random_order(b, 1) == SU2HIP_OK);
  MUST(!sweep_pairs(b));
  MUST(su2hip_destroy(b) == SU2HIP_OK);
  // two doublets
  b = made({params(8, 8, 8, 2)});
  MUST(!sweep_pairs(b));
  MUST(su2hip_destroy(b) == SU2HIP_OK);
  // a flow's buffers in place of the second ones, until its lattice leaves
  const std::vector<su2hip_params> v(3, params(12, 10, 14));
  b = made(v, 0, footprints(v) * 29 / 20);
  std::vector<double> rows(100 * (1 + SU2HIP_NSUMS));
  int n = 0;
  MUST(sweep_pairs(b));
  MUST(su2hip_flow(b, 0, SU2HIP_FLOW_RK3, 0.05, 0.2, 2, rows.data(), 100, &n) == SU2HIP_OK);
  MUST(!sweep_pairs(b));
  MUST(su2hip_remove(b, 0) == SU2HIP_OK);
  MUST(sweep_pairs(b));
  MUST(su2hip_destroy(b) == SU2HIP_OK);
}

int main(int argc, char **argv) {
  const std::string s = argc > 1 ? argv[1] : "";
  if (s == "refused_buffers") refused_buffers();
  else if (s == "refused_call") refused_call();
  else if (s == "refused_tables") refused_tables();
  else if (s == "refused_growth") refused_growth();
  else if (s == "budget_requests") budget_requests();
  else if (s == "weight_keeps_draws") weight_keeps_draws();
  else if (s == "added_lattice_sweeps") added_lattice_sweeps();
  else if (s == "fetch_waits_idle") fetch_waits_idle();
  else if (s == "many_alike") many_alike();
  else if (s == "failed_launch") failed_launch();
  else if (s == "which_sweeps_pair") which_sweeps_pair();
  else return 2;
  MUST(fake::live.empty());
  return 0;
}
