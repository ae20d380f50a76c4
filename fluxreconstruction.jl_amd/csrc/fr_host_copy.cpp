// fr_host_copy.cpp -- copies between pageable host arrays and the device.
//
// One hipMemcpyAsync on a pageable array pins and copies piece by piece in the calling thread, and a
// fresh result array takes its page faults there too.  Large copies go through pinned chunks instead:
// a few worker threads, each with two chunks, move the caller's pages while the other chunk is on the
// bus.  Plain and staged, into a fresh array: 8 MB 474 / 328 us, 16 MB 916 / 512, 24 MB 1742 / 1080, 32 MB
// 2234 / 1273, 53 MB 5.27 / 1.74 ms; from one: 24 MB 668 / 714 us, 28 MB 798 / 815, 30 MB 864 / 864, 32 MB
// 931 / 907, 40 MB 1350 / 1131, 53 MB 1849 / 1514.  The chunks (16 MB) take about 0.7 ms to pin, once per
// context, hence HostStaging::kFromOut and kFromIn.  Chunks of 1 MB took 2.0 and 1.87 ms at 53 MB, of 4 MB
// 1.74 and 1.34.
#include <algorithm>
#include <cstring>
#include <exception>
#include <thread>

#include "fr_common.h"

namespace fr {

// the chunks and events belong to the stream's device, whichever is current
int HostStaging::ensure(hipStream_t st) {
  if (buf) return FR_OK;
  int now = 0;
  hipError_t e = hipGetDevice(&now);
  device = now;
  if (e == hipSuccess && st) e = hipStreamGetDevice(st, &device);
  if (e == hipSuccess && device != now) e = hipSetDevice(device);
  if (e == hipSuccess) e = hipHostMalloc((void **)&buf, 2 * kWorkers * kChunk, hipHostMallocDefault);
  for (hipEvent_t &v : ev)
    if (e == hipSuccess) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
  if (device != now) (void)hipSetDevice(now);
  if (e == hipSuccess) return FR_OK;
  release();
  (void)hipGetLastError();  // the copy goes without staging
  return FR_E_NOMEM;
}

void HostStaging::release() {
  for (hipEvent_t &e : ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (buf) (void)hipHostFree(buf);
  buf = nullptr;
}

// chunks w, w + kWorkers, ... of the array, by way of the worker's two pinned chunks; an event per
// pinned chunk tells when its copy over the bus is done
static hipError_t work(const HostStaging &s, int w, char *dev, char *host, size_t bytes, bool up, hipStream_t st) {
  constexpr size_t C = HostStaging::kChunk;
  hipError_t e = hipSetDevice(s.device);
  const size_t n = (bytes + C - 1) / C;
  auto size = [&](size_t c) { return std::min(C, bytes - c * C); };
  auto pinned = [&](int b) { return s.buf + (2 * w + b) * C; };
  size_t at[2] = {n, n};  // chunk on its way in each pinned chunk
  int b = 0;
  for (size_t c = w; e == hipSuccess; c += HostStaging::kWorkers, b ^= 1) {
    if (at[b] < n) {  // this pinned chunk's last copy
      e = hipEventSynchronize(s.ev[2 * w + b]);
      if (e == hipSuccess && !up) std::memcpy(host + at[b] * C, pinned(b), size(at[b]));
      at[b] = n;
    }
    if (c >= n) {
      if (at[b ^ 1] == n) break;
      continue;
    }
    if (e != hipSuccess) break;
    if (up) std::memcpy(pinned(b), host + c * C, size(c));
    e = hipMemcpyAsync(up ? dev + c * C : pinned(b), up ? pinned(b) : dev + c * C, size(c),
                       up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipEventRecord(s.ev[2 * w + b], st);
    if (e == hipSuccess) at[b] = c;
  }
  return e;
}

static int staged(HostStaging &s, char *dev, char *host, size_t bytes, bool up, hipStream_t st) {
  int now = 0;
  FR_HIP(hipGetDevice(&now));
  hipError_t err[HostStaging::kWorkers];
  std::thread th[HostStaging::kWorkers];
  for (int w = 1; w < HostStaging::kWorkers; ++w) {
    try {
      th[w] = std::thread([&, w] { err[w] = work(s, w, dev, host, bytes, up, st); });
    } catch (const std::exception &) {  // no thread to be had: this one does its part below
    }
  }
  err[0] = work(s, 0, dev, host, bytes, up, st);
  for (int w = 1; w < HostStaging::kWorkers; ++w) {
    if (th[w].joinable())
      th[w].join();
    else
      err[w] = work(s, w, dev, host, bytes, up, st);
  }
  // after an error a chunk may still be on its way: none outlives the call
  hipError_t e = hipStreamSynchronize(st);
  if (s.device != now) (void)hipSetDevice(now);
  for (hipError_t q : err)
    if (e == hipSuccess) e = q;
  FR_HIP(e);
  return FR_OK;
}

// Whether the runtime knows the array: pinned, managed or on a device.
static bool registered(const void *host) {
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, host) == hipSuccess) return at.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return false;
}

// Whether the chunks serve a copy.  The workers all name the caller's stream, so its handle has to mean one
// stream in every thread: hipStreamPerThread is another stream in each of them, whose copies would not
// wait for the work that the caller has queued.  An array that the runtime knows goes over the bus as it
// is: 40 MB pinned 739 us in and 745 us out, by way of the chunks 1128 and 1140.
static bool staging_serves(const void *host, size_t bytes, size_t from, hipStream_t st) {
  return bytes >= from && st != hipStreamPerThread && !registered(host);
}

int copy_to_device(HostStaging &s, double *dev, const double *host, size_t n, hipStream_t st) {
  const size_t bytes = n * sizeof(double);
  if (staging_serves(host, bytes, HostStaging::kFromIn, st) && s.ensure(st) == FR_OK)
    return staged(s, (char *)dev, (char *)const_cast<double *>(host), bytes, true, st);
  FR_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st));
  FR_HIP(hipStreamSynchronize(st));
  return FR_OK;
}

int copy_to_host(HostStaging &s, double *host, const double *dev, size_t n, hipStream_t st) {
  const size_t bytes = n * sizeof(double);
  if (staging_serves(host, bytes, HostStaging::kFromOut, st) && s.ensure(st) == FR_OK)
    return staged(s, (char *)const_cast<double *>(dev), (char *)host, bytes, false, st);
  FR_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st));
  FR_HIP(hipStreamSynchronize(st));
  return FR_OK;
}

}  // namespace fr
