// A HIP runtime of plain host memory for the tests of the host code (driver,
// sessions, server, host copies): no kernel runs, and what a real GPU does
// at its own time is at the test's command.  Every stream and event carries
// the devices and the work it is ordered behind, so that a missing wait
// shows without a race.  The launchers below stand for the kernels whose
// results the host reads; all others are empty (the build adds them).
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "../../include/pmg_mi355x.h"
#include "../../multigrid_amd/csrc/pmg_internal.h"

namespace {
std::recursive_mutex mu;
struct Clock {
  std::map<const void *, long> at;  // stream -> its work that lies behind
  void merge(const Clock &o) {
    for (auto &q : o.at)
      if (at[q.first] < q.second) at[q.first] = q.second;
  }
};
struct Stream {
  int dev;
  long work = 0;
  Clock seen;
};
struct Event {
  int dev;
  Clock seen;
};
thread_local int device = 0;
std::map<char *, std::pair<size_t, Stream *>> owner;  // allocation -> stream

struct {
  int devices = 1;
  bool land = true;        // reductions reach the host
  double value = 0.0;      // what they hold
  double zero_value = 0.0; // the residual of the iterate 0
  hipError_t launch = hipSuccess, sync = hipSuccess;
  int unordered = 0;       // grouped launches not behind a member's stream
} fk;

Stream *tick(hipStream_t s) {
  auto *S = (Stream *)s;
  if (S) S->seen.at[S] = ++S->work;
  return S;
}
void put(const pmg::Red *r, double v) {
  if (!r) return;
  if (r->out) *r->out = v;
  if (r->host && fk.land) *r->host = v;
}
}  // namespace

extern "C" {
void fk_reset(int devices) {
  fk = {};
  fk.devices = devices;
}
void fk_set(int land, double value, double zero_value, int launch_error,
            int sync_error) {
  std::lock_guard<std::recursive_mutex> lk(mu);
  fk.land = land, fk.value = value, fk.zero_value = zero_value;
  fk.launch = (hipError_t)launch_error, fk.sync = (hipError_t)sync_error;
}
int fk_unordered() { return fk.unordered; }
// A copy of bytes to host memory from a stream of device `on`, asked for by
// a thread whose device is `cur`: its status, or -1 for wrong data or a
// current device that has changed.
int fk_copy(size_t bytes, int on, int cur) {
  device = on;
  hipStream_t s;
  hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
  std::vector<char> a(bytes), b(bytes, 0);
  for (size_t q = 0; q < bytes; q++) a[q] = (char)(q * 2654435761u >> 13);
  device = cur;
  pmg::host_ring_ref();
  const pmg::HostSeg g{b.data(), a.data(), bytes};
  int rc = pmg::copy_to_host(s, &g, 1);
  if (device != cur || (rc == PMG_OK && a != b)) rc = -1;
  pmg::host_ring_unref();
  hipStreamDestroy(s);
  device = 0;
  return rc;
}

hipError_t hipGetDeviceCount(int *n) {
  *n = fk.devices;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  device = d;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return fk.sync; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  *f = *t = (size_t)1 << 36;
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  *p = calloc(1, n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::recursive_mutex> lk(mu);
  owner.erase((char *)p);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = calloc(1, n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
  free(p);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) {
  return hipErrorInvalidValue;  // pageable
}
hipError_t hipGetSymbolAddress(void **p, const void *sym) {
  *p = (void *)sym;
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int, size_t n, hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lk(mu);  // fresh memory: zero already
  owner[(char *)p] = {n, tick(s)};
  return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
  memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *p, size_t n, hipMemcpyKind,
                          hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lk(mu);
  tick(s);
  memcpy(d, p, n);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = (hipStream_t) new Stream{device};
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) {
  *d = s ? ((Stream *)s)->dev : device;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return fk.sync; }
hipError_t hipStreamQuery(hipStream_t) { return fk.sync; }  // idle, or lost
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  std::lock_guard<std::recursive_mutex> lk(mu);
  ((Stream *)s)->seen.merge(((Event *)e)->seen);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = (hipEvent_t) new Event{device};
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  return hipEventCreate(e);
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (Event *)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lk(mu);
  auto *E = (Event *)e;
  auto *S = (Stream *)s;
  if (E->dev != (S ? S->dev : device)) return hipErrorInvalidHandle;
  if (tick(s)) E->seen = S->seen;
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) {
  *t = 0.f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = (hipGraph_t)malloc(1);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *,
                               char *, size_t) {
  *x = (hipGraphExec_t)malloc(1);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lk(mu);
  tick(s);
  return fk.launch;  // its iteration's scalar does not land
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  free(g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
  free(x);
  return hipSuccess;
}
}  // extern "C"

namespace pmg {
bool cg_fits(const Dim &) { return true; }
bool cg_class_fits(const Dim &, int) { return true; }
size_t max_partials(const Dim &) { return 64; }
void start_mixed(const Dim &, const double *, float *, double *,
                 const Red *red, hipStream_t s) {
  tick(s);
  put(red, 1.0);
}
template <>
void nrm1<double>(const Dim &, const double *, const Red &red, hipStream_t s) {
  tick(s);
  put(&red, 1.0);
}
template <>
void fill<double>(double *x, size_t n, double v, hipStream_t s) {
  tick(s);
  for (size_t q = 0; q < n; q++) x[q] = v;
}
template <>
void resid<double, double>(const Dim &d, int, const double *, const double *,
                           const double *, const double *x, double *r,
                           const Red *red, hipStream_t s, const double *) {
  tick(s);
  bool zero = !r;
  for (size_t q = 0; q < d.n(); q++) zero &= x[q] == 0.0;
  put(red, zero ? fk.zero_value : fk.value);
}
template <>
void resid<double, float>(const Dim &, int, const double *, const double *,
                          const double *, const double *, float *,
                          const Red *red, hipStream_t s, const double *) {
  tick(s);
  put(red, fk.value);
}
void nmresid(const Dim &, int, const double *, const double *, const double *,
             const double *, double *, const Red *red, hipStream_t s) {
  tick(s);
  put(red, fk.value);
}
void matvec7_dot(const Dim &, const double *, const double *, const double *,
                 const double *, double *, const Red &red, hipStream_t s) {
  tick(s);
  put(&red, 1.0);
}
void pcg_xr(const Dim &, double *, double *, const double *, const double *,
            const double *, const double *, const Red *red, hipStream_t s) {
  tick(s);
  put(red, fk.value);
}
// the grouped step's last kernel: by now its stream must be behind all that
// each member's own stream holds
template <class TO>
static void grouped(const GResid<double, TO> *j, int n, hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lk(mu);
  auto *S = (Stream *)s;
  for (int q = 0; q < n; q++) {
    auto it = owner.upper_bound((char *)j[q].x);
    if (it != owner.begin()) {
      --it;
      Stream *o = it->second.second;
      if (o && o != S && S->seen.at[o] < o->work) fk.unordered++;
    }
    if (j[q].out2) *j[q].out2 = fk.value;
  }
}
template <>
void g_resid<double, double>(const GResid<double, double> *j, int n,
                             hipStream_t s) {
  grouped(j, n, s);
}
template <>
void g_resid<double, float>(const GResid<double, float> *j, int n,
                            hipStream_t s) {
  grouped(j, n, s);
}
}  // namespace pmg
