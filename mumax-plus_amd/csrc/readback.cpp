// A copy into pageable memory runs at 9 GB/s: the driver bounces it through a
// pinned buffer with one thread, and that thread also takes every page fault
// of a freshly allocated destination.  Here several host threads share the
// bytes out in chunks; each moves its chunks through two pinned buffers of its
// own, so the device's copies, the memory copies and the page faults of
// different chunks overlap.
#include "readback.hpp"

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "common.hpp"

namespace mpa {

namespace {

constexpr size_t CHUNK = (size_t)1 << 20;
constexpr int THREADS = 8;
constexpr size_t MIN_BYTES = (size_t)3 << 20;  // below, one thread's copy is as fast
// Allocating the buffers takes as long as their copies save on this many bytes
// (1.5 ms; 0.15 ms saved on 3 MiB, 3.5 on 50): a program that reads less in all
// never has them.
constexpr size_t SETUP_BYTES = (size_t)32 << 20;

struct Lane {
  char* pin[2] = {nullptr, nullptr};
  hipEvent_t ev[2] = {nullptr, nullptr};
};

// One set of buffers (16 MiB pinned) per process and one device; a second
// reader at the same time, or one on another device, takes the plain copy.
// The last world to go leaves them if any world read through them since there
// was none before it, so a program with one world and one read a point keeps
// them (with an allocation and a release a point, reading and dropping a 512 x
// 512 magnet's world took 6.7 ms instead of 2.2); otherwise it gives them back.
std::mutex mu;       // held for the length of a read
std::mutex count_mu;
int worlds = 0;
int device = -1;
bool used = false;   // since there was no world
size_t plain_bytes = 0;  // read without buffers
char* pinned = nullptr;
Lane lanes[THREADS];

void drop() {
  for (Lane& l : lanes)
    for (int b = 0; b < 2; ++b) {
      if (l.ev[b]) (void)hipEventDestroy(l.ev[b]);
      l.ev[b] = nullptr;
    }
  if (pinned) (void)hipHostFree(pinned);
  pinned = nullptr;
  plain_bytes = 0;
  device = -1;
}

void plain(void* host, const void* dev, size_t bytes, hipStream_t s) {
  HIP_CHECK(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
}

// Whether a read of this many bytes on stream s has the buffers.  Their events
// belong to one device: a thread that reads with another one current (a host
// thread starts on device 0, wherever the stream lives) takes the plain copy.
bool ready(size_t bytes, hipStream_t s) {
  int dev = 0;
  hipDevice_t sdev = -1;
  if (hipGetDevice(&dev) != hipSuccess || hipStreamGetDevice(s, &sdev) != hipSuccess || (int)sdev != dev) return false;
  if (device == dev) return true;
  if (device >= 0) return false;
  plain_bytes += bytes;
  if (plain_bytes < SETUP_BYTES) return false;
  bool ok = hipHostMalloc(reinterpret_cast<void**>(&pinned), 2 * THREADS * CHUNK, hipHostMallocDefault) == hipSuccess;
  if (!ok) pinned = nullptr;
  for (int i = 0; ok && i < 2 * THREADS; ++i) {
    Lane& l = lanes[i / 2];
    l.pin[i & 1] = pinned + i * CHUNK;
    ok = hipEventCreateWithFlags(&l.ev[i & 1], hipEventDisableTiming) == hipSuccess;
  }
  if (!ok) {
    (void)hipGetLastError();
    drop();
    return false;
  }
  device = dev;
  return true;
}

}  // namespace

void readback_retain() {
  std::lock_guard<std::mutex> lk(count_mu);
  ++worlds;
}

void readback_release() {
  std::lock_guard<std::mutex> lk(count_mu);
  if (--worlds > 0) return;
  std::lock_guard<std::mutex> lk2(mu);
  if (!used) drop();
  used = false;
}

void read_back(void* host, const void* dev, size_t bytes, hipStream_t s) {
  std::unique_lock<std::mutex> lk(mu, std::defer_lock);
  if (bytes < MIN_BYTES || !lk.try_lock() || !ready(bytes, s)) {
    plain(host, dev, bytes, s);
    return;
  }
  used = true;
  const size_t n = (bytes + CHUNK - 1) / CHUNK;
  const int T = (int)std::min<size_t>(THREADS, n);
  std::exception_ptr failed[THREADS];
  auto work = [&](int t) {
    try {
      HIP_CHECK(hipSetDevice(device));
      Lane& l = lanes[t];
      auto issue = [&](size_t c, int b) {
        const size_t off = c * CHUNK, len = std::min(CHUNK, bytes - off);
        HIP_CHECK(hipMemcpyAsync(l.pin[b], static_cast<const char*>(dev) + off, len, hipMemcpyDeviceToHost, s));
        HIP_CHECK(hipEventRecord(l.ev[b], s));
      };
      int b = 0;
      if ((size_t)t < n) issue(t, 0);
      for (size_t c = t; c < n; c += T, b ^= 1) {
        if (c + T < n) issue(c + T, b ^ 1);
        HIP_CHECK(hipEventSynchronize(l.ev[b]));
        const size_t off = c * CHUNK;
        std::memcpy(static_cast<char*>(host) + off, l.pin[b], std::min(CHUNK, bytes - off));
      }
    } catch (...) {
      failed[t] = std::current_exception();
    }
  };
  std::vector<std::thread> pool;
  pool.reserve(T);
  int started = 1;
  try {
    for (; started < T; ++started) pool.emplace_back(work, started);
  } catch (...) {
    // no more threads: the started ones end, and their shares are copied again below
  }
  work(0);
  for (std::thread& th : pool) th.join();
  // every queued copy ends before the buffers are used again
  HIP_CHECK(hipStreamSynchronize(s));
  for (int t = 0; t < started; ++t)
    if (failed[t]) std::rethrow_exception(failed[t]);
  if (started < T) plain(host, dev, bytes, s);
}

}  // namespace mpa
