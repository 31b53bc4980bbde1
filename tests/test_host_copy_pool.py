"""csrc/host_copy.h compiled for the host over stand-ins for the HIP calls: the
pool of pinned slots is held by copies that use it only, and never while a copy
waits on the runtime's path for what is queued on its stream."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "entropicthreadsafe_amd", "csrc")
PROGRAM = r"""
#include <sched.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <atomic>
#include <mutex>
#include <thread>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
typedef int hipStream_t;
typedef void *hipEvent_t;
enum { hipMemcpyDeviceToHost, hipMemcpyHostToDevice, hipEventDisableTiming, hipHostMallocDefault };
namespace {
constexpr int kMaxDevices = 1;
bool no_memory = false;
int copies = 0, waits_free = 0, waits_held = 0;
bool pool_free();
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, int) { return *e = (void *)e, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, int) {
  *p = no_memory ? nullptr : malloc(n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) {
  static std::mutex m;
  memcpy(d, s, n);
  std::lock_guard<std::mutex> lk(m);
  copies++;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return (pool_free() ? waits_free : waits_held)++, hipSuccess; }
#include "host_copy.h"
bool pool_free() {
  bool ok = false;
  std::thread([&] {
    if ((ok = g_stage[0].mu.try_lock())) g_stage[0].mu.unlock();
  }).join();
  return ok;
}
template <bool OUT>
void run(const char *what, size_t bytes) {
  std::vector<char> host(bytes), dev(bytes);
  for (size_t i = 0; i < bytes; i++) (OUT ? dev : host)[i] = (char)(i * 7 + i / 251);
  copies = waits_free = waits_held = 0;
  const hipError_t e = host_copy<OUT>(0, 0, host.data(), dev.data(), bytes);
  printf("%s %d %d %d %d %d %d\n", what, (int)e, (int)(host == dev), copies, waits_free, waits_held, (int)pool_free());
}
}
int main() {
  run<true>("small", 4096);
  run<true>("below", kStageMinOut - 1);
  run<true>("staged", kStageMinOut + 12345);
  run<false>("upload", kStageMinIn - 1);
  run<false>("staged-in", kStageMinIn + 4097);
  stage_retain(0);
  stage_release(0);
  no_memory = true;
  run<true>("no-memory", kStageMinOut + 1);
  g_stage[0].mu.lock();
  std::thread([] { run<true>("taken", kStageMinOut + 1); }).join();
  g_stage[0].mu.unlock();
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_pool_is_held_by_staged_copies_only(tmp_path):
    src, exe = tmp_path / "p.cpp", tmp_path / "p"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I" + CSRC, "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=120).stdout
    rows = {r.split()[0]: list(map(int, r.split()[1:])) for r in out.splitlines()}
    for what, (err, equal, copies, waits_free, waits_held, free_after) in rows.items():
        assert err == 0 and equal == 1, what
        if what != "taken":  # held by another thread throughout
            assert waits_held == 0 and free_after, what  # no wait on the stream with the pool held
        assert (copies == 1) == (what not in ("staged", "staged-in")), what
    assert all(rows[w][3] == 1 for w in ("small", "below", "no-memory"))
