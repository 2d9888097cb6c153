"""HsaCopier (csrc/hsa_copy.cpp) on the CPU: the source compiled against a stand-in for the HSA runtime whose copy engine is
a host thread - it runs a copy once the signals it names are 0, then brings the copy's own signal from 1 to 0, or, for a
source the test marks bad, to -1, which is how the runtime reports a failed copy (hsa_ext_amd.h,
hsa_amd_memory_async_copy). A failed copy must be reported, and neither a wait for it, a copy that names it nor the
copier's end may last for good."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "tierstream_amd" / "csrc"

RUNTIME = r"""
#include <hsa/hsa.h>
#include <hsa/hsa_ext_amd.h>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <mutex>
#include <thread>
#include <vector>
namespace {
using Sig = std::atomic<int64_t>;
struct Job { void* dst; const void* src; size_t n; std::vector<Sig*> deps; Sig* done; };
std::mutex mu;
std::deque<Job> jobs;
std::atomic<bool> stop{false}, hold{false};
std::thread engine;
Sig* of(hsa_signal_t s) { return reinterpret_cast<Sig*>(s.handle); }
void run() {
  while (!stop) {
    Job j; bool got = false;
    {
      std::lock_guard<std::mutex> l(mu);
      for (auto it = jobs.begin(); !hold && it != jobs.end() && !got; ++it) {
        bool ready = true;
        for (Sig* d : it->deps) ready = ready && d->load() == 0;
        if (ready) { j = *it; jobs.erase(it); got = true; }
      }
    }
    if (!got) { std::this_thread::sleep_for(std::chrono::microseconds(50)); continue; }
    if (static_cast<const char*>(j.src)[0] == 'X') { j.done->store(-1); continue; }
    std::memcpy(j.dst, j.src, j.n);
    j.done->fetch_sub(1);
  }
}
}
extern "C" {
void fake_hold(int on) { hold = on != 0; }
hsa_status_t hsa_init() { engine = std::thread(run); return HSA_STATUS_SUCCESS; }
hsa_status_t hsa_shut_down() { stop = true; engine.join(); return HSA_STATUS_SUCCESS; }
hsa_status_t hsa_iterate_agents(hsa_status_t (*cb)(hsa_agent_t, void*), void* d) {
  cb(hsa_agent_t{1}, d);
  return cb(hsa_agent_t{2}, d);
}
hsa_status_t hsa_agent_get_info(hsa_agent_t a, hsa_agent_info_t what, void* out) {
  if (what == HSA_AGENT_INFO_DEVICE) *static_cast<hsa_device_type_t*>(out) = a.handle == 1 ? HSA_DEVICE_TYPE_CPU : HSA_DEVICE_TYPE_GPU;
  else *static_cast<uint32_t*>(out) = 0;
  return HSA_STATUS_SUCCESS;
}
hsa_status_t hsa_system_get_info(hsa_system_info_t, void* out) { *static_cast<uint64_t*>(out) = 1000000000; return HSA_STATUS_SUCCESS; }
hsa_status_t hsa_signal_create(hsa_signal_value_t v, uint32_t, const hsa_agent_t*, hsa_signal_t* s) {
  s->handle = reinterpret_cast<uint64_t>(new Sig(v));
  return HSA_STATUS_SUCCESS;
}
hsa_status_t hsa_signal_destroy(hsa_signal_t s) { delete of(s); return HSA_STATUS_SUCCESS; }
void hsa_signal_store_screlease(hsa_signal_t s, hsa_signal_value_t v) { of(s)->store(v); }
hsa_signal_value_t hsa_signal_load_scacquire(hsa_signal_t s) { return of(s)->load(); }
hsa_status_t hsa_amd_memory_async_copy(void* dst, hsa_agent_t, const void* src, hsa_agent_t, size_t n, uint32_t nd,
                                       const hsa_signal_t* deps, hsa_signal_t done) {
  if ((nd == 0) != (deps == nullptr)) return HSA_STATUS_ERROR_INVALID_ARGUMENT;
  Job j{dst, src, n, {}, of(done)};
  for (uint32_t i = 0; i < nd; ++i) j.deps.push_back(of(deps[i]));
  std::lock_guard<std::mutex> l(mu);
  jobs.push_back(j);
  return HSA_STATUS_SUCCESS;
}
hsa_status_t hsa_amd_profiling_async_copy_enable(bool) { return HSA_STATUS_SUCCESS; }
hsa_status_t hsa_amd_profiling_get_async_copy_time(hsa_signal_t, hsa_amd_profiling_async_copy_time_t* t) {
  *t = {1, 2};
  return HSA_STATUS_SUCCESS;
}
}
"""

DRIVER = r"""
#include <hip/hip_runtime_api.h>
#include <dlfcn.h>
#include <cstdio>
#include <cstring>
#include <memory>
#include <string>
#include <unistd.h>
#include "common.hpp"
#include "hsa_copy.hpp"
extern "C" hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) { std::memset(p, 0, sizeof *p); return hipSuccess; }
namespace tsa { void hip_check(hipError_t, const char*) {} }
using namespace tsa;
static char buf[8][64];
static int fails(const char* what) { std::printf("failed: %s\n", what); return 1; }
// Ends when the copy has (0), or with 1 when its failure is reported.
static int wait_for(HsaCopier& c, uint32_t sig) {
  try {
    while (!c.done(sig)) usleep(50);
  } catch (const Error& e) {
    return e.status() == SS_E_BACKEND ? 1 : 2;
  }
  return 0;
}
int main(int argc, char** argv) {
  alarm(20);  // (a wait that lasts for good ends the program)
  const std::string what = argv[1];
  auto hold = reinterpret_cast<void (*)(int)>(dlsym(dlopen("libhsa-runtime64.so.1", RTLD_NOW), "fake_hold"));
  auto c = std::make_unique<HsaCopier>(0);
  std::strcpy(buf[0], what == "chain" ? "good" : "X");
  hold(1);
  uint32_t s[4] = {c->copy(buf[1], buf[0], 64, false, nullptr, 0)};
  for (int i = 1; i < 4; ++i) s[i] = c->copy(buf[i + 1], buf[i], 64, i & 1, &s[i - 1], 1);  // each behind the last
  if (c->done(s[3])) return fails("a held copy has ended");
  hold(0);
  if (what == "chain") {
    for (uint32_t x : s) if (wait_for(*c, x)) return fails("a copy of the chain");
    if (std::strcmp(buf[4], "good")) return fails("the bytes");
    uint64_t ns = 0;
    if (!c->copy_ns(s[0], &ns)) return fails("its time");
    for (uint32_t x : s) c->unref(x);
    for (int i = 0; i < 100; ++i) {  // signals are used again
      const uint32_t x = c->copy(buf[5], buf[0], 64, false, &s[3], 0);
      if (wait_for(*c, x)) return fails("a copy on a used signal");
      c->unref(x);
    }
  } else if (what == "wait") {
    if (wait_for(*c, s[0]) != 1) return fails("the failure is not reported to a wait for the copy");
    if (wait_for(*c, s[3]) != 1) return fails("the failure is not reported to a wait for a later copy");
    try {
      c->copy(buf[5], buf[6], 64, false, &s[3], 1);
      return fails("a copy is taken after a failure");
    } catch (const Error&) {
    }
  }  // "end": the copier ends with the failure and the copies behind it pending
  c.reset();
  std::printf("ok\n");
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("hsa")
    (d / "runtime.cpp").write_text(RUNTIME)
    (d / "driver.cpp").write_text(DRIVER)
    flags = ["g++", "-std=c++17", "-O1", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT / 'include'}", f"-I{CSRC}"]
    for cmd in ([*flags, "-shared", "-fPIC", str(d / "runtime.cpp"), "-Wl,-soname,libhsa-runtime64.so.1", "-lpthread",
                 "-o", str(d / "libhsa-runtime64.so.1")],
                [*flags, str(d / "driver.cpp"), str(CSRC / "hsa_copy.cpp"), "-ldl", "-lpthread", "-o", str(d / "driver")]):
        p = subprocess.run(cmd, capture_output=True, text=True)
        assert p.returncode == 0, p.stderr[-3000:]
    return d


@pytest.mark.parametrize("what", ["chain", "wait", "end"])
def test_copier(program, what):
    r = subprocess.run([str(program / "driver"), what], capture_output=True, text=True, timeout=60,
                       env={"LD_LIBRARY_PATH": str(program)})
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
