// pmg_hostcopy.hip -- results to the caller's host memory (internal).
//
// A potential goes to ordinary pageable memory, often pages never touched
// before.  The runtime's own pageable copy moves it through its staging
// buffer with one thread, so the page faults and the memcpy (8 to 17 GB/s)
// bound it, not the link (52 GB/s).  Here the caller and up to seven
// helper threads drain a ring of pinned pieces: each waits for its piece,
// moves it to its place (faulting the pages in on several cores) and
// enqueues the next copy into the freed slot, so the link stays busy.
// Threads live for one call only (about 20 us each to start), which leaves
// no state behind; below kLeast bytes they cost more than they save and the
// runtime's copy is used.  A potential to a new array (MI355X, 16 cores):
// 289^3 (193 MB) 18.8 -> 4.1 ms, 161^3 (33 MB) 2.19 -> 0.88, 129^3 1.14 ->
// 0.56, 97^3 (7 MB) 0.53 -> 0.26.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "../../include/pmg_mi355x.h"
#include "pmg_internal.h"

namespace pmg {
namespace {

constexpr size_t kPiece = (size_t)2 << 20;
constexpr size_t kLeast = (size_t)4 << 20;
constexpr size_t kTwoStreams = (size_t)32 << 20;
constexpr int kThreads = 8, kSlots = 2 * kThreads;

// Pinned rings (kSlots * kPiece = 32 MB), at most kRings of them, made when
// first needed and given back with the last context; a call that finds
// none free takes the runtime's copy.
constexpr int kRings = 2;
std::mutex ring_mu;
struct Ring {
  char *p = nullptr;
  bool busy = false;
  // a second stream (of device dev) for every other piece of a large copy:
  // between two copies of one stream the link idles about 19 us (289^3 5000
  // -> 4130 us, the drop-in's 45 MB in 20 arrays 9.0 -> 6.6 ms a call).
  // From kTwoStreams on: with 17 MB the solve that follows lost more to the
  // further stream (129^3 Newton 8234 -> 8490 us) than the copy gained
  hipStream_t s2 = nullptr;
  int dev = -1;
} rings[kRings];
int ring_users = 0;

Ring *ring_take() {
  std::lock_guard<std::mutex> lk(ring_mu);
  for (Ring &r : rings)
    if (r.p && !r.busy) {
      r.busy = true;
      return &r;
    }
  for (Ring &r : rings)
    if (!r.p) {
      if (hipHostMalloc((void **)&r.p, kSlots * kPiece,
                        hipHostMallocPortable) != hipSuccess) {
        hipGetLastError();
        r.p = nullptr;
        return nullptr;
      }
      r.busy = true;
      return &r;
    }
  return nullptr;
}

void ring_give(Ring *r) {
  std::lock_guard<std::mutex> lk(ring_mu);
  r->busy = false;
}

// Runs work(0) .. work(n - 1), the first on the calling thread; a helper
// that cannot be started has its share done here.
template <class F>
void on_threads(int n, F &&work) {
  std::vector<std::thread> th;
  int started = 1;
  try {
    th.reserve(n);
    for (; started < n; started++) th.emplace_back([&work, started] { work(started); });
  } catch (const std::exception &) {
  }
  work(0);
  for (int w = started; w < n; w++) work(w);
  for (auto &t : th) t.join();
}

int threads_for(size_t pieces) {
  const int cores = std::max(1, (int)std::thread::hardware_concurrency());
  return (int)std::min<size_t>({(size_t)kThreads, (size_t)cores, pieces});
}

bool pageable(const void *p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

int copy_plain(hipStream_t s, const HostSeg *seg, int n) {
  bool ok = true;
  for (int q = 0; q < n; q++)
    ok &= hipMemcpyAsync(seg[q].dst, seg[q].src, seg[q].bytes,
                         hipMemcpyDeviceToHost, s) == hipSuccess;
  return hipStreamSynchronize(s) == hipSuccess && ok ? PMG_OK : PMG_EDEVICE;
}

int copy_pieces(hipStream_t s, const std::vector<HostSeg> &pc, Ring &r, int nt,
                bool two) {
  // events, threads and the second stream are those of the stream's device,
  // whatever the caller's current one is
  int cur = 0;
  hipDevice_t dev = 0;
  char *const ring = r.p;
  hipEvent_t ev[kSlots] = {}, start = nullptr;
  std::atomic<bool> ok{hipGetDevice(&cur) == hipSuccess &&
                       hipStreamGetDevice(s, &dev) == hipSuccess &&
                       (cur == dev || hipSetDevice(dev) == hipSuccess)};
  const int np = (int)pc.size(), ns = 2 * nt;
  // the second stream starts behind what s holds already
  hipStream_t st[2] = {s, s};
  if (ok && two && !r.s2) {
    if (hipStreamCreateWithFlags(&r.s2, hipStreamNonBlocking) == hipSuccess) {
      r.dev = dev;
    } else {
      hipGetLastError();
      r.s2 = nullptr;
    }
  }
  if (ok && two && r.s2 && r.dev == dev &&
      hipEventCreateWithFlags(&start, hipEventDisableTiming) == hipSuccess &&
      hipEventRecord(start, s) == hipSuccess &&
      hipStreamWaitEvent(r.s2, start, 0) == hipSuccess)
    st[1] = r.s2;
  // slot q % ns holds piece q; piece q is thread (q % nt)'s
  auto fetch = [&](int q) {
    const int b = q % ns;
    if (hipMemcpyAsync(ring + b * kPiece, pc[q].src, pc[q].bytes,
                       hipMemcpyDeviceToHost, st[q & 1]) != hipSuccess ||
        hipEventRecord(ev[b], st[q & 1]) != hipSuccess)
      ok = false;
  };
  for (int b = 0; b < ns; b++)
    if (hipEventCreateWithFlags(&ev[b], hipEventDisableTiming) != hipSuccess)
      ok = false;
  for (int q = 0; ok && q < std::min(ns, np); q++) fetch(q);
  on_threads(nt, [&](int w) {
    if (w && hipSetDevice(dev) != hipSuccess) ok = false;
    for (int q = w; ok && q < np; q += nt) {
      const int b = q % ns;
      if (hipEventSynchronize(ev[b]) != hipSuccess) {
        ok = false;
        return;
      }
      std::memcpy(pc[q].dst, ring + b * kPiece, pc[q].bytes);
      if (q + ns < np) fetch(q + ns);
    }
  });
  // nothing may still write the ring, also after a failure
  for (hipStream_t t : st)
    if (hipStreamSynchronize(t) != hipSuccess) ok = false;
  for (hipEvent_t e : ev)
    if (e) hipEventDestroy(e);
  if (start) hipEventDestroy(start);
  if (cur != dev && hipSetDevice(cur) != hipSuccess) ok = false;
  return ok ? PMG_OK : PMG_EDEVICE;
}

}  // namespace

void host_ring_ref() {
  std::lock_guard<std::mutex> lk(ring_mu);
  ring_users++;
}

void host_ring_unref() {
  std::lock_guard<std::mutex> lk(ring_mu);
  if (--ring_users) return;
  for (Ring &r : rings)
    if (r.p && !r.busy) {
      if (r.s2) hipStreamDestroy(r.s2);
      hipHostFree(r.p);
      r = Ring{};
    }
}

int copy_to_host(hipStream_t s, const HostSeg *seg, int n) {
  size_t total = 0;
  bool plain = false;
  for (int q = 0; q < n; q++) {
    total += seg[q].bytes;
    plain |= !pageable(seg[q].dst);
  }
  if (plain || total < kLeast) return copy_plain(s, seg, n);
  std::vector<HostSeg> pc;
  try {
    for (int q = 0; q < n; q++)
      for (size_t o = 0; o < seg[q].bytes; o += kPiece)
        pc.push_back({(char *)seg[q].dst + o, (const char *)seg[q].src + o,
                      std::min(kPiece, seg[q].bytes - o)});
  } catch (const std::exception &) {
    return copy_plain(s, seg, n);
  }
  Ring *r = ring_take();
  if (!r) return copy_plain(s, seg, n);
  const int rc = copy_pieces(s, pc, *r, threads_for(pc.size()),
                             total >= kTwoStreams);
  ring_give(r);
  return rc;
}

void copy_host(void *dst, const void *src, size_t bytes) {
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  if (bytes < kLeast) {
    std::memcpy(dst, src, bytes);
    return;
  }
  const int nt = threads_for(pieces);
  on_threads(nt, [&](int w) {
    for (size_t q = w; q < pieces; q += nt)
      std::memcpy((char *)dst + q * kPiece, (const char *)src + q * kPiece,
                  std::min(kPiece, bytes - q * kPiece));
  });
}

}  // namespace pmg
