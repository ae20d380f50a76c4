// A HIP runtime of queues on the CPU for csrc/fr_host_copy.cpp: work is put into a queue per stream
// (hipStreamPerThread: per thread) and runs only when somebody waits for that queue.  Device memory is
// host memory.  Prints one line per check and returns the number of failed ones.
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "fr_common.h"

namespace {
struct Queue {
  std::mutex mu;
  std::vector<std::function<void()>> work;
  void push(std::function<void()> f) {
    std::lock_guard<std::mutex> l(mu);
    work.push_back(std::move(f));
  }
  void drain() {
    std::lock_guard<std::mutex> l(mu);
    for (auto &f : work) f();
    work.clear();
  }
};
std::mutex mu;  // of the maps
std::map<std::pair<hipStream_t, std::thread::id>, Queue> queues;
std::map<hipEvent_t, Queue *> events;

const void *pinned = nullptr;  // the one array that the runtime knows
int copies = 0;

Queue &queue(hipStream_t s) {
  std::lock_guard<std::mutex> l(mu);
  return queues[{s, s == hipStreamPerThread ? std::this_thread::get_id() : std::thread::id()}];
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = std::malloc(n), hipSuccess; }
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t) new char, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (char *)e, hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  if (p != pinned) return hipErrorInvalidValue;
  return a->type = hipMemoryTypeHost, hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  Queue &q = queue(s);
  std::lock_guard<std::mutex> l(mu);
  events[e] = &q;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  Queue *q;
  {
    std::lock_guard<std::mutex> l(mu);
    q = events[e];
  }
  return q->drain(), hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { return queue(s).drain(), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  queue(st).push([=] {
    ++copies;
    std::memcpy(d, s, n);
  });
  return hipSuccess;
}
}

namespace fr {
int fail(int code, const std::string &) { return code; }
int hip_fail(hipError_t, const char *, const char *, int) { return FR_E_HIP; }
}  // namespace fr

static int failed = 0;
static void check(const char *what, bool ok) {
  std::printf("%s %s\n", ok ? "ok  " : "FAIL", what);
  failed += !ok;
}

// a copy each way behind queued work on the same stream: the work adds one to every device value
static void ordered(const char *what, hipStream_t st) {
  const size_t n = fr::HostStaging::kFromIn / 8 + 3 * fr::HostStaging::kChunk / 8 + 1;
  std::vector<double> dev(n, 1.0), host(n, 0.0);
  auto step = [&] {
    queue(st).push([&] {
      std::this_thread::sleep_for(std::chrono::milliseconds(50));
      for (double &v : dev) v += 1.0;
    });
  };
  fr::HostStaging s;
  step();
  int rc = fr::copy_to_host(s, host.data(), dev.data(), n, st);
  check((std::string(what) + ": the host state holds the queued step").c_str(), rc == 0 && host == std::vector<double>(n, 2.0));
  step();
  const std::vector<double> next(n, 7.0);
  rc = fr::copy_to_device(s, dev.data(), next.data(), n, st);
  (void)hipStreamSynchronize(st);
  check((std::string(what) + ": the new state comes after the queued step").c_str(), rc == 0 && dev == next);
  s.release();
}

// arrays that the runtime knows are copied as they are, by one copy each way
static void straight(hipStream_t st) {
  const size_t n = fr::HostStaging::kFromIn / 8 + 1;
  std::vector<double> dev(n, 1.0), host(n, 2.0);
  pinned = host.data();
  copies = 0;
  fr::HostStaging s;
  int rc = fr::copy_to_device(s, dev.data(), host.data(), n, st);
  check("pinned array: one copy in", rc == 0 && copies == 1 && !s.buf && dev == host);
  dev.assign(n, 3.0);
  rc = fr::copy_to_host(s, host.data(), dev.data(), n, st);
  check("pinned array: one copy out", rc == 0 && copies == 2 && !s.buf && dev == host);
  s.release();
  pinned = nullptr;
}

// 28 MiB: one copy in, which the chunks would make slower, and chunks out
static void lines(hipStream_t st) {
  const size_t n = (28u << 20) / 8;
  std::vector<double> dev(n, 1.0), host(n, 2.0);
  copies = 0;
  fr::HostStaging s;
  int rc = fr::copy_to_device(s, dev.data(), host.data(), n, st);
  check("28 MiB: one copy in", rc == 0 && copies == 1 && dev == host);
  dev.assign(n, 3.0);
  rc = fr::copy_to_host(s, host.data(), dev.data(), n, st);
  check("28 MiB: chunks out", rc == 0 && copies == 1 + 14 && dev == host);
  s.release();
}

int main() {
  int own = 0;
  ordered("own stream", (hipStream_t)&own);
  ordered("null stream", nullptr);
  ordered("per-thread stream", hipStreamPerThread);
  straight((hipStream_t)&own);
  lines((hipStream_t)&own);
  return failed;
}
