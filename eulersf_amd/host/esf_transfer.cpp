// esf_transfer.cpp -- large copies from device memory into the caller's
// (pageable) host arrays.
//
// hipMemcpyAsync into pageable memory runs through the runtime's own staging
// on one thread: 9 GB/s into a fresh 51 MB array, where most of the time goes
// to that thread's page faults and memcpy while the link could carry 56 GB/s.
// Here a few threads each move chunks through pinned slots of their own, two
// per thread so that one is on the link while the other is copied out: 51 MB
// in 2.1 ms against 5.5, 6.6 MB in 0.36 against 0.50.  (The other way the
// runtime's 25 GB/s from warm pages is as fast as this measured.)
//
// Memory that the caller pinned is written by the link itself: 51 MB in 0.91
// ms (1.81 through the slots), 3.2 MB in 0.07 (0.21).
//
// The pinned slots belong to the process: at most kStages sets of 16 MB,
// taken for one copy at a time, made once the copies repay it (kRepays) and
// freed when the last context goes.  A copy that finds none free or a small one
// uses hipMemcpyAsync; one whose threads cannot be started moves their shares
// on the calling thread.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "../csrc/esf_internal.h"

namespace esf {

namespace {

constexpr size_t kChunk = size_t(1) << 20;
constexpr int kThreads = 8;
constexpr int kStages = 4;
// below this a copy is over before the threads are up
constexpr size_t kLeast = size_t(3) << 20;
// Bytes of such copies, since there was no context, that go the plain way
// before a set is pinned for them.  Pinning and freeing one costs 1 to 2 ms and
// it saves 20 to 55 us a MB: a program with one context at a time and one 22 MB
// copy of each waited 2.1 ms for it where the plain copy takes 1.25.
constexpr size_t kRepays = size_t(48) << 20;

struct Stages {
  std::mutex lock;
  int contexts = 0;
  size_t asked = 0;  // bytes, up to kRepays
  char* mem[kStages] = {};
  bool taken[kStages] = {};

  // a set of 2 kThreads slots for a copy of `bytes`, or -1
  int take(size_t bytes) {
    std::lock_guard<std::mutex> g(lock);
    asked = std::min(kRepays, asked + std::min(kRepays, bytes));
    if (asked < kRepays) return -1;
    for (int i = 0; i < kStages; i++) {
      if (taken[i]) continue;
      if (!mem[i] && hipHostMalloc((void**)&mem[i], 2 * kThreads * kChunk) != hipSuccess) {
        mem[i] = nullptr;
        (void)hipGetLastError();
        return -1;
      }
      taken[i] = true;
      return i;
    }
    return -1;
  }
  void give(int i) {
    std::lock_guard<std::mutex> g(lock);
    taken[i] = false;
  }
};
Stages gStages;

// thread w of `threads`: chunks w, w + threads, ..
void moveChunks(esf_ctx* ctx, char* host, const char* dev, size_t bytes, char* slots, int w,
                int threads, std::atomic<int>* failed) {
  hipEvent_t ev[2] = {nullptr, nullptr};
  auto check = [&](hipError_t e) {
    if (e != hipSuccess) failed->store((int)e);
  };
  // (worker 0 is the calling thread, whose current device is the caller's)
  int was = ctx->device;
  check(hipGetDevice(&was));
  if (was != ctx->device) check(hipSetDevice(ctx->device));
  for (hipEvent_t& e : ev) check(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  size_t at[2] = {0, 0}, len[2] = {0, 0};
  int k = 0;
  auto settle = [&](int s) {
    if (!len[s]) return;
    check(hipEventSynchronize(ev[s]));
    if (!failed->load()) std::memcpy(host + at[s], slots + s * kChunk, len[s]);
    len[s] = 0;
  };
  for (size_t off = w * kChunk; off < bytes && !failed->load(); off += threads * kChunk, k ^= 1) {
    settle(k);
    const size_t n = std::min(kChunk, bytes - off);
    check(hipMemcpyAsync(slots + k * kChunk, dev + off, n, hipMemcpyDeviceToHost, ctx->stream));
    check(hipEventRecord(ev[k], ctx->stream));
    at[k] = off;
    len[k] = n;
  }
  settle(k);
  settle(k ^ 1);
  for (hipEvent_t e : ev)
    if (e) (void)hipEventDestroy(e);
  if (was != ctx->device) (void)hipSetDevice(was);
}

}  // namespace

// memory the runtime has not pinned (or does not know)
static bool pageable(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

esf_status copyToHost(esf_ctx* ctx, void* dst, const void* src, size_t bytes) {
  const int cpus = (int)std::thread::hardware_concurrency();
  const int threads = std::min<int>(std::min(kThreads, std::max(cpus / 2, 1)),
                                    (int)((bytes + kChunk - 1) / kChunk));
  const int stage = bytes >= kLeast && threads > 1 && pageable(dst) ? gStages.take(bytes) : -1;
  if (stage < 0) {
    ESF_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    ESF_HIP(streamSync(ctx));
    return ESF_OK;
  }
  char* slots = gStages.mem[stage];
  std::atomic<int> failed{0};
  std::vector<std::thread> team;
  int started = 1;  // this thread is worker 0
  try {
    team.reserve(threads);
    for (; started < threads; started++)
      team.emplace_back(moveChunks, ctx, (char*)dst, (const char*)src, bytes,
                        slots + 2 * started * kChunk, started, threads, &failed);
  } catch (...) {
    // the shares of the threads that did not start fall to this one, below
  }
  moveChunks(ctx, (char*)dst, (const char*)src, bytes, slots, 0, threads, &failed);
  for (int w = started; w < threads; w++)
    moveChunks(ctx, (char*)dst, (const char*)src, bytes, slots, w, threads, &failed);
  for (std::thread& t : team) t.join();
  // (after a failure copies may still be queued: none outlives the slots' lease)
  const hipError_t e = streamSync(ctx);
  gStages.give(stage);
  if (failed.load() || e != hipSuccess) {
    ctx->err = std::string("host copy: ") +
               hipGetErrorString(failed.load() ? (hipError_t)failed.load() : e);
    return ESF_ERR_DEVICE;
  }
  return ESF_OK;
}

void transferContext(int change) {
  std::lock_guard<std::mutex> g(gStages.lock);
  gStages.contexts += change;
  if (gStages.contexts > 0) return;
  gStages.asked = 0;
  for (char*& m : gStages.mem) {
    if (m) (void)hipHostFree(m);
    m = nullptr;
  }
}

}  // namespace esf
