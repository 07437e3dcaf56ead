// Copies between pageable host arrays and device memory.  The runtime's own
// pageable copies run on one core (27 GB/s in, 18 GB/s out, of the 57 GB/s
// that pinned memory reaches), and so does the first touch of a new output
// array's pages.  Here four threads move pieces through a ring of pinned
// slots, two of a thread's own: one is filled or drained while the other is
// in transfer.  M^+ on host arrays at 12^3x24 Ls12 (96 MB each way): 12.7 ->
// 5.3 ms, at 8^3x16 Ls8 (13 MB) 1.26 -> 0.90 ms.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>
#include "dwf_internal.h"
#include "dwf_rules.h"

namespace qdwf {
namespace {

// A transfer command costs some 15 us beside its bytes: at 96 MB pieces of
// 0.5, 1, 2 and 4 MB give 9.3, 6.6, 5.3 and 5.2 ms.  Eight threads are no
// faster than four.
constexpr size_t kPiece = (size_t)2 << 20;
constexpr int kCopyThreads = 4;
// below two pieces nothing overlaps: the runtime's copy
constexpr size_t kRingMin = 2 * kPiece;

// One ring per process, made when ring_pays says so, used by one transfer at
// a time and given back with the last inverter.
struct Ring {
  std::mutex mu;
  char* buf = nullptr;
  int without = 0;  // transfers that went without it
  int users = 0;
} g_ring;

// runs work(0) ... work(n - 1), as far as threads can be had at once
template <class Work>
void run_threads(int n, Work&& work)
{
  std::vector<std::thread> th;
  th.reserve(n);
  int started = 1;  // (work(0) is this thread's)
  try {
    for (; started < n; ++started) th.emplace_back(work, started);
  } catch (...) {  // (no more threads: the rest runs here)
  }
  work(0);
  for (int t = started; t < n; ++t) work(t);
  for (auto& t : th) t.join();
}

// A transfer through the ring; false: it is for the runtime's copy (small,
// not pageable, too early to make the ring, another thread's transfer in it,
// no pinned memory).
bool ring_copy(int device, hipStream_t st, char* dev, char* host, size_t bytes, bool in, size_t ring_min,
               hipError_t* err)
{
  if (bytes < std::max(kRingMin, ring_min)) return false;
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, host) != hipSuccess) (void)hipGetLastError();
  else if (at.type != hipMemoryTypeUnregistered) return false;
  std::unique_lock<std::mutex> lock(g_ring.mu, std::try_to_lock);
  if (!lock.owns_lock() || !g_ring.users) return false;
  if (!g_ring.buf) {
    if (!ring_pays(bytes, g_ring.without)) {
      ++g_ring.without;
      return false;
    }
    if (hipHostMalloc((void**)&g_ring.buf, kCopyThreads * 2 * kPiece, hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();
      g_ring.buf = nullptr;
      return false;
    }
  }
  const size_t np = (bytes + kPiece - 1) / kPiece;
  const unsigned hc = std::thread::hardware_concurrency();
  const int nt = (int)std::min<size_t>(hc ? std::min<unsigned>(hc, kCopyThreads) : 1, np);
  hipError_t e[kCopyThreads] = {};
  if (!in) {  // (the threads would spin on the work before the copy)
    *err = hipStreamSynchronize(st);
    if (*err != hipSuccess) return true;
  }
  run_threads(nt, [&](int t) {
    hipEvent_t ev[2] = {nullptr, nullptr};
    e[t] = hipSetDevice(device);
    for (auto& x : ev)
      if (e[t] == hipSuccess) e[t] = hipEventCreateWithFlags(&x, hipEventDisableTiming);
    char* slot[2] = {g_ring.buf + (size_t)2 * t * kPiece, g_ring.buf + (size_t)(2 * t + 1) * kPiece};
    bool busy[2] = {false, false};
    auto start = [&](size_t p, int k) {  // piece p to or from slot k
      const size_t n = std::min(kPiece, bytes - p * kPiece);
      e[t] = in ? hipMemcpyAsync(dev + p * kPiece, slot[k], n, hipMemcpyHostToDevice, st)
                : hipMemcpyAsync(slot[k], dev + p * kPiece, n, hipMemcpyDeviceToHost, st);
      if (e[t] == hipSuccess) e[t] = hipEventRecord(ev[k], st);
      busy[k] = true;
    };
    auto wait = [&](int k) {
      if (busy[k] && e[t] == hipSuccess) e[t] = hipEventSynchronize(ev[k]);
      if (e[t] == hipSuccess) busy[k] = false;
    };
    if (!in)
      for (int k = 0; k < 2; ++k)
        if (e[t] == hipSuccess && (size_t)(t + k * nt) < np) start(t + k * nt, k);
    int k = 0;
    for (size_t p = t; p < np && e[t] == hipSuccess; p += nt, k ^= 1) {
      wait(k);
      if (e[t] != hipSuccess) break;
      const size_t n = std::min(kPiece, bytes - p * kPiece);
      if (in) {
        std::memcpy(slot[k], host + p * kPiece, n);
        start(p, k);
      } else {
        std::memcpy(host + p * kPiece, slot[k], n);
        if (p + 2 * nt < np) start(p + 2 * nt, k);
      }
    }
    for (int j = 0; j < 2; ++j) wait(j);
    // (after an error the slots may still be in transfer)
    if ((busy[0] || busy[1])) (void)hipStreamSynchronize(st);
    for (auto& x : ev)
      if (x) (void)hipEventDestroy(x);
  });
  *err = hipSuccess;
  for (hipError_t x : e)
    if (x != hipSuccess) *err = x;
  return true;
}

}  // namespace

void copy_ring_retain()
{
  std::lock_guard<std::mutex> lock(g_ring.mu);
  ++g_ring.users;
}

void copy_ring_release()
{
  std::lock_guard<std::mutex> lock(g_ring.mu);
  if (--g_ring.users > 0) return;
  g_ring.without = 0;
  if (g_ring.buf) (void)hipHostFree(g_ring.buf);
  g_ring.buf = nullptr;
}

hipError_t copy_to_device(int device, hipStream_t st, void* dev, const void* host, size_t bytes, size_t ring_min)
{
  hipError_t err;
  if (ring_copy(device, st, (char*)dev, (char*)const_cast<void*>(host), bytes, true, ring_min, &err)) return err;
  return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
}

hipError_t copy_to_host(int device, hipStream_t st, void* host, const void* dev, size_t bytes)
{
  hipError_t err;
  if (ring_copy(device, st, (char*)const_cast<void*>(dev), (char*)host, bytes, false, 0, &err)) return err;
  err = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
  return err != hipSuccess ? err : hipStreamSynchronize(st);
}

}  // namespace qdwf
