// Host side of a CG whose scalars stay on the device: the state that its
// kernels pass on and the loop that queues them.  HIP's host API only, so that
// the loop can be tested without a GPU.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <stdexcept>
#include <string>

namespace qdwf {

struct HipError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

#define QDWF_HIP(expr)                                                                      \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess)                                                                   \
      throw qdwf::HipError(std::string(#expr) + " failed: " + hipGetErrorString(e_) + " (" + \
                     __FILE__ + ":" + std::to_string(__LINE__) + ")");                     \
  } while (0)

// Scalars of the FP64 CG on the device, one slot for the even and one for
// the odd iterations: an iteration reads slot it & 1 and writes the other.
struct CgState64 {
  double rr;      // |r|^2 before the iteration
  double target;  // stop when |r|^2 <= target
  double alpha;   // of the iteration (k_cg_residual_d)
  int64_t iter;   // iterations done before this one
  int done;       // 0 running, 1 converged, 2 non-finite
};

void launch_cg_init_d(CgState64* st, double rr, double target, hipStream_t s);

// A device-driven CG: the iteration's scalars live in two state slots on the
// device (CgState64; an iteration reads slot it & 1 and writes the other),
// and iterations are queued kCgAhead at a time, one group ahead of the group
// the host waits for; those behind the converged one find its state and do
// nothing.  No iteration waits for the host: 8^3x16 Ls8, 155 FP64 iterations
// of 65 us, the solve 18.0 -> 10.7 ms with two host round trips less each.
constexpr int kCgAhead = 2;
struct CgControl {
  CgState64* dev = nullptr;      // [2], the caller's
  CgState64* map = nullptr;      // mapped host copy of the newest state
  CgState64* map_dev = nullptr;
  bool own_map = false;
  hipEvent_t ev[2] = {nullptr, nullptr};
  // map_host null: a mapped page of its own
  CgControl(void* dev_states, void* map_host, void* map_device)
      : dev((CgState64*)dev_states), map((CgState64*)map_host), map_dev((CgState64*)map_device)
  {
    try {
      if (!map) {
        QDWF_HIP(hipHostMalloc((void**)&map, sizeof(CgState64), hipHostMallocMapped | hipHostMallocCoherent));
        own_map = true;
        QDWF_HIP(hipHostGetDevicePointer((void**)&map_dev, map, 0));
      }
      for (auto& e : ev) QDWF_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    } catch (...) {
      release();
      throw;
    }
  }
  ~CgControl() { release(); }
  CgControl(const CgControl&) = delete;
  CgControl& operator=(const CgControl&) = delete;
  void release()
  {
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    if (own_map && map) (void)hipHostFree(map);
  }
  // queue(slot) launches one iteration; returns the last state.  After an
  // error the iterations queued so far are waited for: they write the states,
  // the mapped copy and the caller's fields, which may be freed or reset next.
  template <class Queue>
  CgState64 run(double rr, double target, long max_num_iter, hipStream_t st, Queue&& queue)
  {
    *map = CgState64{};
    launch_cg_init_d(dev, rr, target, st);
    QDWF_HIP(hipGetLastError());
    long queued = 0;
    auto group = [&](hipEvent_t e) {
      for (int j = 0; j < kCgAhead && queued < max_num_iter; ++j, ++queued) queue((int)(queued & 1));
      QDWF_HIP(hipEventRecord(e, st));
    };
    try {
      group(ev[0]);
      for (long g = 1;; ++g) {
        const bool last = queued >= max_num_iter;
        if (!last) group(ev[g & 1]);
        QDWF_HIP(hipEventSynchronize(ev[(g - 1) & 1]));
        if (last || *(volatile int*)&map->done) break;
      }
    } catch (...) {
      (void)hipStreamSynchronize(st);
      throw;
    }
    QDWF_HIP(hipStreamSynchronize(st));  // the group queued behind
    return *map;
  }
};

}  // namespace qdwf
