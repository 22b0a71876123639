// Host copies (eulersf_amd/host/esf_transfer.cpp) against a stand-in for the
// HIP runtime: device memory is host memory, copies are made at once, an
// event belongs to the device that was current when it was made and may only
// be recorded on that device's streams.  transfer_check SCENARIO prints what
// the caller could see.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "../../eulersf_amd/csrc/esf_internal.h"

namespace {
std::mutex lk;
thread_local int current = 0;
int streamDevice = 0;
std::map<char*, size_t> pinned;
long mallocs = 0, frees = 0, chunks = 0, direct = 0, events = 0;

bool inPinned(const void* p) {
  std::lock_guard<std::mutex> g(lk);
  for (auto& m : pinned)
    if ((const char*)p >= m.first && (const char*)p < m.first + m.second) return true;
  return false;
}
}  // namespace

extern "C" {
hipError_t hipSetDevice(int d) {
  current = d;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = current;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  std::lock_guard<std::mutex> g(lk);
  events++;
  *e = (hipEvent_t) new int(current);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> g(lk);
  events--;
  delete (int*)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  return *(int*)e == streamDevice ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  std::lock_guard<std::mutex> g(lk);
  pinned[(char*)*p] = n;
  mallocs++;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> g(lk);
  pinned.erase((char*)p);
  std::free(p);
  frees++;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::memset(a, 0, sizeof(*a));
  a->type = inPinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(dst, src, n);
  std::lock_guard<std::mutex> g(lk);
  (n <= (size_t(1) << 20) ? chunks : direct)++;
  return hipSuccess;
}
}

namespace esf {
hipEvent_t fiberMark(esf_ctx*) { return nullptr; }
hipError_t fiberWait(esf_ctx*, hipEvent_t) { return hipErrorUnknown; }
}  // namespace esf

static std::vector<char> numbers(size_t n) {
  std::vector<char> v(n);
  unsigned s = 12345;
  for (char& c : v) c = (char)((s = s * 1664525u + 1013904223u) >> 24);
  return v;
}

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  const size_t MB = size_t(1) << 20;
  esf_ctx ctx;
  const std::vector<char> dev = numbers(52 * MB + 1234);
  std::vector<char> host(dev.size());
  auto copy = [&](char* dst, size_t n) {
    std::memset(dst, 0, n);
    if (esf::copyToHost(&ctx, dst, dev.data(), n) != ESF_OK) {
      std::printf("failed %s\n", ctx.err.c_str());
      std::exit(1);
    }
    if (std::memcmp(dst, dev.data(), n)) {
      std::printf("wrong bytes\n");
      std::exit(1);
    }
  };
  auto report = [&](const char* name) {
    std::printf("%s chunks %ld direct %ld mallocs %ld frees %ld events %ld device %d\n", name,
                chunks, direct, mallocs, frees, events, current);
    chunks = direct = 0;
  };
  if (!std::strcmp(what, "device")) {
    // a context of GPU 1 and a caller whose current device is 0
    ctx.device = streamDevice = 1;
    esf::transferContext(1);
    copy(host.data(), dev.size());
    report("large");
    copy(host.data(), MB / 2);
    report("small");
    esf::transferContext(-1);
    report("end");
  }
  if (!std::strcmp(what, "pinned")) {
    // a destination the caller pinned, whole and from its middle
    esf::transferContext(1);
    copy(host.data(), dev.size());
    report("pageable");
    char* p = nullptr;
    (void)hipHostMalloc((void**)&p, dev.size(), 0);
    copy(p, dev.size());
    report("pinned");
    copy(p + 5 * MB, 4 * MB);
    report("inside");
    (void)hipHostFree(p);
    esf::transferContext(-1);
  }
  if (!std::strcmp(what, "pool")) {
    // one context at a time, one copy each: 20 MB, and 52 at once
    for (int k = 0; k < 3; k++) {
      esf::transferContext(1);
      copy(host.data(), 20 * MB);
      esf::transferContext(-1);
    }
    report("single");
    esf::transferContext(1);
    copy(host.data(), dev.size());
    esf::transferContext(-1);
    report("big");
    // a context that goes on: 20 MB four times
    esf::transferContext(1);
    for (int k = 0; k < 4; k++) {
      copy(host.data(), 20 * MB);
      report(("copy" + std::to_string(k)).c_str());
    }
    esf::transferContext(-1);
    report("end");
  }
  return 0;
}
