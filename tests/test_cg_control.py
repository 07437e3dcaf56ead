"""The loop that queues a device-driven CG (dwf_cg_control.h) on a model of a
stream: work runs only when the host waits for it, and writes through the
mapped copy, so that work left behind a freed or reset copy shows."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = "/opt/rocm/include"

SOURCE = r"""
#define __HIP_PLATFORM_AMD__
#include "dwf_cg_control.h"

#include <cstdio>
#include <cstdlib>
#include <deque>
#include <functional>
#include <map>

using qdwf::CgControl;
using qdwf::CgState64;

static std::deque<std::function<void()>> work;  // the stream
static size_t done_work = 0;                    // pieces run so far
static std::map<hipEvent_t, size_t> recorded;   // pieces before an event
static bool freed_under_work = false;
static CgState64 page;

static void run_to(size_t n)
{
  for (; done_work < n; ++done_work) work[done_work]();
}
extern "C" {
hipError_t hipHostMalloc(void** p, size_t, unsigned) { *p = &page; return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** p, void* h, unsigned) { *p = h; return hipSuccess; }
hipError_t hipHostFree(void*) { freed_under_work = freed_under_work || done_work < work.size(); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { static long n; *e = (hipEvent_t)(++n); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { recorded[e] = work.size(); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { run_to(recorded[e]); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { run_to(work.size()); return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}
namespace qdwf {
void launch_cg_init_d(CgState64* st, double rr, double target, hipStream_t)
{
  work.push_back([=] { st[0] = st[1] = CgState64{rr, target, 0.0, 0, 0}; });
}
}  // namespace qdwf

// an iteration halves |r|^2; `bad`: it becomes NaN instead at that iteration
static void iteration(CgState64* st, int slot, CgState64* host, long bad)
{
  work.push_back([=] {
    const CgState64 s = st[slot];
    if (s.done) { st[1 - slot] = s; return; }
    const double rr = s.iter + 1 == bad ? 0.0 / 0.0 : s.rr / 2;
    const CgState64 n{rr, s.target, 0.0, s.iter + 1, rr != rr ? 2 : rr <= s.target ? 1 : 0};
    st[1 - slot] = n;
    *host = n;
  });
}
static int fail(const char* what, long a, long b) { std::printf("%s %ld %ld\n", what, a, b); return 1; }

int main()
{
  CgState64 st[2];
  for (long target = 1; target <= 9; ++target)
    for (long limit = 0; limit <= 12; ++limit) {
      CgControl c(st, nullptr, nullptr);
      const CgState64 e = c.run(1.0, 1.0 / (1 << target), limit, nullptr,
                                [&](int slot) { iteration(c.dev, slot, c.map_dev, -1); });
      if (done_work != work.size()) return fail("left behind", target, limit);
      if (e.iter != (limit < target ? limit : target)) return fail("iterations", target, limit);
      if (e.done != (limit >= target ? 1 : 0)) return fail("done", target, limit);
    }
  for (long bad = 1; bad <= 5; ++bad) {
    CgControl c(st, nullptr, nullptr);
    long queued = 0;
    const CgState64 e = c.run(1.0, 1e-300, 1000000, nullptr, [&](int slot) { ++queued; iteration(c.dev, slot, c.map_dev, bad); });
    if (e.done != 2 || e.iter != bad || queued > bad + 2 * qdwf::kCgAhead) return fail("breakdown", bad, queued);
  }
  // a launch that fails after some iterations are queued
  for (long at = 0; at <= 6; ++at) {
    bool thrown = false;
    try {
      CgControl c(st, nullptr, nullptr);
      long n = 0;
      c.run(1.0, 1e-300, 100, nullptr, [&](int slot) {
        if (n++ == at) throw qdwf::HipError("launch");
        iteration(c.dev, slot, c.map_dev, -1);
      });
    } catch (const qdwf::HipError&) {
      thrown = true;
    }
    if (!thrown) return fail("no error", at, 0);
    if (freed_under_work) return fail("copy freed under queued work", at, 0);
    if (done_work != work.size()) return fail("queued work outlives the call", at, 0);
  }
  std::puts("ok");
  return 0;
}
"""


def test_queued_iterations(tmp_path):
    """Stops at convergence, at odd and even limits and at a breakdown; after a
    failed launch nothing that was queued is still to run when the call
    returns, so that nothing writes a state that is freed or reset."""
    cxx = shutil.which("g++")
    if cxx is None or not os.path.exists(os.path.join(HIP, "hip", "hip_runtime_api.h")):
        pytest.skip("no host compiler or HIP headers")
    src, exe = tmp_path / "cg.cpp", str(tmp_path / "cg")
    src.write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wno-attributes", "-I", HIP, "-I",
                    os.path.join(ROOT, "qlattice_amd", "csrc"), str(src), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
