// The GPU as the host code of the solver sees it, for tests of its error paths
// without one: memory is the host's, a stream is a queue of what was enqueued,
// run when the host waits (hipStreamQuery runs one entry), and the solver's
// launches do only what the host code reads back: the loop test of an outer
// iteration stops the loop after `stub_stop` iterations.  stub_fail(name, n): the
// n-th call of `name` from now on fails.
#include <deque>
#include <functional>
#include <map>
#include <string>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../simple-ts_amd/csrc/host_copy.h"
#include "../simple-ts_amd/csrc/sts_internal.h"
#include "../simple-ts_amd/csrc/sts_launch.h"

namespace {
std::deque<std::function<void()>> queue;
std::map<std::string, int> fails;
int stop_after = 3;
std::vector<BeginArgs> begins;

hipError_t call(const char *name, std::function<void()> f = nullptr) {
  auto it = fails.find(name);
  if (it != fails.end() && --it->second == 0) {
    fails.erase(it);
    return std::string(name) == "hipMalloc" ? hipErrorOutOfMemory : hipErrorLaunchFailure;
  }
  if (f) queue.push_back(f);
  return hipSuccess;
}
void run_one() {
  auto f = queue.front();
  queue.pop_front();
  f();
}
hipError_t run_all() {
  while (!queue.empty()) run_one();
  return hipSuccess;
}
}  // namespace

extern "C" {
void stub_fail(const char *name, int n) { fails[name] = n; }
void stub_clear() { fails.clear(), begins.clear(); }
void stub_stop(int iterations) { stop_after = iterations; }
int stub_begins() { return (int)begins.size(); }
int stub_order(int q) { return begins[q].order; }  // degree of the q-th start
int stub_whole(int q) {                            // its levels are there, the one that takes x^n and those it reads
  const BeginArgs &a = begins[q];
  for (int f = 0; f < 4; f++) {
    if (!a.to[f]) return 0;
    for (int h = 0; h < a.order; h++)
      if (!a.hist.f[h][f]) return 0;
  }
  return 1;
}

hipError_t hipMalloc(void **p, size_t n) {
  hipError_t e = call("hipMalloc");
  if (e == hipSuccess) *p = calloc(1, n ? n : 1);
  return e;
}
hipError_t hipFree(void *p) {
  (void)run_all();
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = calloc(1, n ? n : 1);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  (void)run_all();
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
  if (k != hipMemcpyHostToDevice) return call("hipMemcpyAsync", [=] { memmove(d, s, n); });
  std::vector<char> b((const char *)s, (const char *)s + n);  // (pageable: taken when called)
  return call("hipMemcpyAsync", [=] { memcpy(d, b.data(), n); });
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  return call("hipMemsetAsync", [=] { memset(d, v, n); });
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = (hipStream_t)malloc(1);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  (void)run_all();
  free((void *)s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return run_all(); }
hipError_t hipStreamQuery(hipStream_t) {
  if (!queue.empty()) run_one();
  return queue.empty() ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = (hipEvent_t)malloc(1);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  free((void *)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return run_all(); }
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) {
  *t = 0;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidValue; }
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}

// (the networks' entry points, which no test here calls)
#define NET(n)                             \
  int net_##n() asm("sts_unet_" #n);       \
  int net_##n() { return STS_ERR_UNSUPPORTED; }
NET(create) NET(destroy) NET(set_params) NET(get_params) NET(get_grads) NET(forward) NET(infer) NET(backward_mse)
NET(backward) NET(adam) NET(dataset) NET(record) NET(train_step) NET(eval) NET(record_correction) NET(param_count)
}

int sts_internal_unet_correct(sts_unet *, const StsView &, const sts_unet_corr_norm *, double *const *) { return -4; }
int sts_internal_unet_predict(sts_unet *, const StsView &, const sts_unet_norm *, double *, double *) { return -4; }
void HostCopy::reserve(size_t) {}
void HostCopy::release() {}
hipError_t HostCopy::get(void *h, const void *d, size_t n, hipStream_t) { return hipMemcpy(h, d, n, hipMemcpyDefault); }
hipError_t HostCopy::put(void *d, const void *h, size_t n, hipStream_t) { return hipMemcpy(d, h, n, hipMemcpyDefault); }

const int CELL_TILES[NVARIANT][2] = {{64, 4}, {64, 8}, {128, 2}, {32, 8}};
const int SWEEP_TILES[NVARIANT][2] = {{60, 6}, {60, 4}, {60, 8}, {60, 5}};
int aa_store_blocks(int) { return 1; }
int aa_case_tiles(int, int, int) { return 1; }
int continuity_blocks(const KGrid &) { return 1; }

template <typename R>
hipError_t launch_edges(const KGridT<R> &, const KFieldsT<R> &, int, bool, double *, hipStream_t, Gate gate,
                        LoopTest lt, const WallOp *, int) {
  const int last = std::min(stop_after, lt.N_I) - 1;
  return call("launch_edges", [=] {
    if (!lt.ctrl || (gate.ctrl && gate.k > gate.ctrl->stop_at)) return;
    const bool cont = gate.k < last;
    if (!cont) lt.ctrl->stop_at = gate.k;
    if (lt.host && (!cont || gate.k >= lt.host_from))
      *lt.host = (unsigned long long)(gate.k + 1) | (cont ? 0ull : LOOP_STOPPED);
  });
}
hipError_t launch_loop_open(LoopCtrl *c, unsigned long long *, int, unsigned long long *, hipStream_t) {
  return call("launch_loop_open", [=] { *c = LoopCtrl{0x7fffffff, 0}; });
}
hipError_t launch_begin(const BeginArgs &a, hipStream_t) {
  begins.push_back(a);
  return call("launch_begin");
}
hipError_t launch_batch_begin(int, const BeginArgs *A, const BatchTile *, int, hipStream_t) {
  const hipError_t e = call("launch_batch_begin");
  (void)run_all();
  for (int q = 0; q < 2; q++) begins.push_back(A[q]);  // (the test's batches have two cases)
  return e;
}
template <typename R>
hipError_t launch_batch(int kernel, int, const BatchCase<R> *C, int n, const BatchTile *, int, int k, int, int, int,
                        hipStream_t) {
  const int last = stop_after - 1;
  return call("launch_batch", [=] {
    for (int q = 0; q < n; q++) {
      if (kernel == BK_LOOP_OPEN) *C[q].ctrl = LoopCtrl{C[q].skip ? -1 : 0x7fffffff, 0};
      else if (kernel == BK_EDGES && k >= last && k <= C[q].ctrl->stop_at) C[q].ctrl->stop_at = k;
    }
  });
}

// What the host code reads nothing back from.
template <typename R>
hipError_t launch_assemble(const KGridT<R> &, const KFieldsT<R> &, hipStream_t, Gate, bool) { return call("launch_assemble"); }
template <typename R>
hipError_t launch_sweep(const KGridT<R> &, const KFieldsT<R> &, const R *, const R *, R *, R *, unsigned long long *,
                        unsigned long long *, hipStream_t, unsigned long long *, unsigned long long *, Gate) { return call("launch_sweep"); }
template <typename R>
hipError_t launch_sweep2(const KGridT<R> &, const KFieldsT<R> &, const R *, const R *, R *, R *, unsigned long long *,
                         unsigned long long *, unsigned long long *, unsigned long long *, hipStream_t, Gate) { return call("launch_sweep2"); }
template <typename R>
hipError_t launch_correct(const KGridT<R> &, const KFieldsT<R> &, unsigned long long *, unsigned long long *, int, bool,
                          hipStream_t, Gate) { return call("launch_correct"); }
template <typename R>
hipError_t launch_wall(const KGridT<R> &, const KFieldsT<R> &, int, hipStream_t) { return call("launch_wall"); }
template <typename R>
hipError_t launch_wall_ops(const KGridT<R> &, const KFieldsT<R> &, const WallOp *, int, bool, hipStream_t, Gate) { return call("launch_wall_ops"); }
hipError_t launch_wall_plan(const KGrid &, const unsigned *, int, WallOp *, hipStream_t) { return call("launch_wall_plan"); }
template <typename R>
hipError_t launch_flux_diff(const KGridT<R> &, const KFieldsT<R> &, hipStream_t, Gate, int) { return call("launch_flux_diff"); }
hipError_t launch_properties(const KGrid &, const KFields &, hipStream_t) { return call("launch_properties"); }
hipError_t launch_rho_mid(const KGrid &, const KFields &, hipStream_t) { return call("launch_rho_mid"); }
hipError_t launch_apply_bodies(const KGrid &, const KFields &, hipStream_t) { return call("launch_apply_bodies"); }
hipError_t launch_jump_overwrite(const KGrid &, const KFields &, hipStream_t) { return call("launch_jump_overwrite"); }
template <int N>
hipError_t launch_copies(const CopySet &, int, hipStream_t) { return call("launch_copies"); }
hipError_t launch_set_inflow(const KGrid &, const KFields &, double, hipStream_t) { return call("launch_set_inflow"); }
template <typename R>
hipError_t launch_aa_begin(const AAFieldsT<R> &, const AABuf &, int, hipStream_t) { return call("launch_aa_begin"); }
template <typename R>
hipError_t launch_aa_store(const AAFieldsT<R> &, const AABuf &, const AASel &, int, hipStream_t, Gate) { return call("launch_aa_store"); }
template <typename R>
hipError_t launch_aa_mix(const KGridT<R> &, const KFieldsT<R> &, const AAFieldsT<R> &, const AABuf &, const AASel &,
                         hipStream_t, Gate) { return call("launch_aa_mix"); }
template <typename S, typename D>
hipError_t launch_convert(const KFieldsT<S> &, const KFieldsT<D> &, unsigned long long, int, hipStream_t) { return call("launch_convert"); }
hipError_t launch_fold(unsigned long long *, int, unsigned long long *, hipStream_t) { return call("launch_fold"); }
hipError_t launch_drag(const KGrid &, const KFields &, const unsigned *, int, double *, double *, hipStream_t) { return call("launch_drag"); }
hipError_t launch_continuity(const KGrid &, const KFields &, double *, double *, double *, hipStream_t) { return call("launch_continuity"); }
hipError_t launch_tile_lists(const TileRun *, const TileLists &, hipStream_t) { return call("launch_tile_lists"); }
hipError_t launch_batch_aa(int, int, const BatchCase<double> *, int, const BatchTile *, int, int, int, const AABatchSel &,
                           hipStream_t) { return call("launch_batch_aa"); }

#define INSTANTIATE(R)                                                                                              \
  template hipError_t launch_edges<R>(const KGridT<R> &, const KFieldsT<R> &, int, bool, double *, hipStream_t, Gate, \
                                      LoopTest, const WallOp *, int);                                               \
  template hipError_t launch_batch<R>(int, int, const BatchCase<R> *, int, const BatchTile *, int, int, int, int, int, \
                                      hipStream_t);                                                                 \
  template hipError_t launch_assemble<R>(const KGridT<R> &, const KFieldsT<R> &, hipStream_t, Gate, bool);          \
  template hipError_t launch_sweep<R>(const KGridT<R> &, const KFieldsT<R> &, const R *, const R *, R *, R *,       \
                                      unsigned long long *, unsigned long long *, hipStream_t, unsigned long long *, \
                                      unsigned long long *, Gate);                                                  \
  template hipError_t launch_sweep2<R>(const KGridT<R> &, const KFieldsT<R> &, const R *, const R *, R *, R *,      \
                                       unsigned long long *, unsigned long long *, unsigned long long *,            \
                                       unsigned long long *, hipStream_t, Gate);                                    \
  template hipError_t launch_correct<R>(const KGridT<R> &, const KFieldsT<R> &, unsigned long long *,               \
                                        unsigned long long *, int, bool, hipStream_t, Gate);                        \
  template hipError_t launch_wall<R>(const KGridT<R> &, const KFieldsT<R> &, int, hipStream_t);                     \
  template hipError_t launch_wall_ops<R>(const KGridT<R> &, const KFieldsT<R> &, const WallOp *, int, bool,         \
                                         hipStream_t, Gate);                                                        \
  template hipError_t launch_flux_diff<R>(const KGridT<R> &, const KFieldsT<R> &, hipStream_t, Gate, int);          \
  template hipError_t launch_aa_begin<R>(const AAFieldsT<R> &, const AABuf &, int, hipStream_t);                    \
  template hipError_t launch_aa_store<R>(const AAFieldsT<R> &, const AABuf &, const AASel &, int, hipStream_t, Gate); \
  template hipError_t launch_aa_mix<R>(const KGridT<R> &, const KFieldsT<R> &, const AAFieldsT<R> &, const AABuf &, \
                                       const AASel &, hipStream_t, Gate);
INSTANTIATE(double)
INSTANTIATE(float)
template hipError_t launch_copies<4>(const CopySet &, int, hipStream_t);
template hipError_t launch_copies<5>(const CopySet &, int, hipStream_t);
template hipError_t launch_convert<double, float>(const KFieldsT<double> &, const KFieldsT<float> &, unsigned long long, int, hipStream_t);
template hipError_t launch_convert<float, double>(const KFieldsT<float> &, const KFieldsT<double> &, unsigned long long, int, hipStream_t);
