// host_copy.h -- copies between callers' arrays and the device, included by
// tslb.hip inside its anonymous namespace.
//
// Callers' arrays are pageable.  The runtime copies to one through a pinned
// buffer on one thread, which for a fresh array also takes the page faults:
// 10 GB/s, and the frame of a 512^3 run took as long as 100 of its steps.  So a
// large copy is cut in chunks that several threads move through pinned slots:
// each thread takes the next chunk, queues its transfer on the context's
// stream and meanwhile copies its previous one.  Five fields of 512^3 to the
// host: 265 -> 65 ms (41 GB/s), of 256^3 31 -> 10 ms, four of 301x130x187 12 ->
// 4.4 ms.  Making the pool costs a run's first frame of five 10 MB fields 0.7 ms
// (3.3 -> 4.0) and saves 0.5 ms in each of the next; a frame of four 7.6 MB fields
// is as fast either way.  From the host the runtime pins the array in place, which moves
// 20-28 GB/s; the slots are ahead of that only on the largest arrays (537 MB:
// 19 -> 12 ms; 134 MB: 4.0 ms either way; 67 MB: 2.5 ms against 2.9).
//
// The slots are as large as the copies so far needed, 64 MiB in all at most (a
// pool of that size made the first frame of a 10 MB field, and the uploads after
// it, slower than the runtime's path).  They belong to the device, are shared by its
// contexts and freed with the last of them.  A copy that finds them taken by
// another thread's takes the runtime's path.
#pragma once

constexpr size_t kStageMinOut = 8u << 20, kStageMinIn = 256u << 20;  // bytes from which a copy is cut
constexpr size_t kStageSlotMax = 4u << 20;
constexpr int kStageThreads = 8;

struct StagePool {
  std::mutex mu;      // held for the length of a staged copy
  std::mutex ref_mu;  // guards users
  int users = 0;
  char *mem = nullptr;
  size_t slot = 0;    // bytes of each of its 2 * kStageThreads slots
  hipEvent_t ev[2 * kStageThreads] = {};
};
StagePool g_stage[kMaxDevices];

void stage_retain(int dev) {
  std::lock_guard<std::mutex> lk(g_stage[dev].ref_mu);
  g_stage[dev].users++;
}
// with `dev` current
void stage_release(int dev) {
  StagePool &s = g_stage[dev];
  std::lock_guard<std::mutex> lk(s.ref_mu);
  if (--s.users > 0) return;
  std::lock_guard<std::mutex> lk2(s.mu);
  for (auto &e : s.ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (s.mem) (void)hipHostFree(s.mem);
  s.mem = nullptr;
  s.slot = 0;
}
bool stage_ready(StagePool &s, size_t slot) {
  if (s.slot >= slot) return true;
  if (s.mem) (void)hipHostFree(s.mem);
  s.mem = nullptr;
  s.slot = 0;
  for (auto &e : s.ev)
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return (void)hipGetLastError(), false;
  if (hipHostMalloc((void **)&s.mem, 2 * kStageThreads * slot, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    s.mem = nullptr;
    return false;
  }
  s.slot = slot;
  return true;
}
int stage_threads() {
  cpu_set_t set;
  const int n = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
  return n < 1 ? 1 : (n < kStageThreads ? n : kStageThreads);
}

// host <- dev (TO_HOST) or dev <- host, after the work queued on the stream; the
// host array is written by the time it returns, read by the next wait on the
// stream
template <bool TO_HOST>
hipError_t host_copy(int device, hipStream_t st, void *host, void *dev, size_t bytes) {
  auto runtime = [&] {
    const hipError_t e = TO_HOST ? hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st)
                                 : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
    return TO_HOST && e == hipSuccess ? hipStreamSynchronize(st) : e;
  };
  // the runtime's path may wait for long work on the stream: never with the pool
  if (bytes < (TO_HOST ? kStageMinOut : kStageMinIn)) return runtime();
  StagePool &s = g_stage[device];
  std::unique_lock<std::mutex> lk(s.mu, std::try_to_lock);
  if (!lk.owns_lock()) return runtime();
  const int nthr = stage_threads();
  // two chunks per thread at least, of whole 64 KiB, at most 2 MiB, or 4 MiB
  // where a large array is worth the larger pool (512^3: 65 ms a frame, 90 with
  // 1 MiB)
  size_t chunk = (bytes / (2 * (size_t)nthr) + 0xffff) & ~(size_t)0xffff;
  const size_t most = bytes < kStageMinIn ? kStageSlotMax / 2 : kStageSlotMax;
  if (chunk > most) chunk = most;
  if (!stage_ready(s, chunk)) {
    lk.unlock();
    return runtime();
  }
  const size_t nchunk = (bytes + chunk - 1) / chunk;
  std::atomic<size_t> next{0};
  std::atomic<int> err{(int)hipSuccess};
  auto work = [&](int w) {
    auto ck = [&](hipError_t e) {
      int none = (int)hipSuccess;
      if (e != hipSuccess) err.compare_exchange_strong(none, (int)e);
      return e == hipSuccess;
    };
    if (!ck(hipSetDevice(device))) return;
    size_t held[2] = {SIZE_MAX, SIZE_MAX};  // chunk in flight in each slot
    auto slot = [&](int k) { return s.mem + (size_t)(2 * w + k) * s.slot; };
    auto len = [&](size_t i) { return i + 1 < nchunk ? chunk : bytes - i * chunk; };
    // waits for a slot's transfer and, to the host, copies it out
    auto finish = [&](int k) {
      if (held[k] == SIZE_MAX) return;
      if (ck(hipEventSynchronize(s.ev[2 * w + k])) && TO_HOST)
        memcpy((char *)host + held[k] * chunk, slot(k), len(held[k]));
      held[k] = SIZE_MAX;
    };
    int k = 0;
    for (size_t i; err == (int)hipSuccess && (i = next.fetch_add(1)) < nchunk; k ^= 1) {
      finish(k);
      char *h = slot(k), *d = (char *)dev + i * chunk;
      if (!TO_HOST) memcpy(h, (char *)host + i * chunk, len(i));
      const hipError_t e = TO_HOST ? hipMemcpyAsync(h, d, len(i), hipMemcpyDeviceToHost, st)
                                   : hipMemcpyAsync(d, h, len(i), hipMemcpyHostToDevice, st);
      if (!ck(e) || !ck(hipEventRecord(s.ev[2 * w + k], st))) break;
      held[k] = i;
    }
    finish(k);
    finish(k ^ 1);
  };
  std::thread th[kStageThreads];
  for (int w = 1; w < nthr && (size_t)w < nchunk; w++) {
    try {
      th[w] = std::thread(work, w);
    } catch (...) {
      break;  // the others take its chunks
    }
  }
  work(0);
  for (auto &t : th)
    if (t.joinable()) t.join();
  if (err != (int)hipSuccess) (void)hipStreamSynchronize(st);
  return (hipError_t)err.load();
}
