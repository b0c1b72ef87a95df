// Device-to-host read-out of large arrays into the caller's memory.
//
// A copy into pageable memory goes through the runtime's own staging on one
// thread, and the caller's array is usually fresh, so that thread also takes
// its page faults: 275 MB of moments of the 256^3 cavity came at 10 GB/s, a
// quarter of the time of 300 steps and a read-out. Here the array crosses in
// chunks into a ring of pinned buffers while worker threads empty the ring
// into the caller's memory (converting where the caller wants FP64 of an FP32
// array).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "flb_host.hpp"

namespace flbh {

namespace {

constexpr size_t kChunk = size_t(2) << 20;
constexpr int kRing = 16;     // 32 MiB of pinned memory while the ring lives
constexpr int kWorkers = 8;
constexpr int kCopiesFirst = 4;  // DirectOut

// The ring serves one read-out at a time (busy); it is made at the first large
// read-out and given back when the last block or box of the process goes.
// Small moments have a buffer of their own (DirectOut): in the ring, the first
// of them pinned 32 MiB, and a large read-out beside it found the ring taken.
// Never destroyed itself: blocks may outlive static objects.
struct Ring {
  std::mutex busy;
  std::mutex users_mu;
  int users = 0;
  char* buf = nullptr;
  hipEvent_t ev[kRing] = {};
  int device = -1;  // of the events
  std::mutex direct_busy;
  char* direct = nullptr;
  int small = 0;  // small moments read by a copy since the buffer was given back
  std::atomic<int64_t> paths[FLB_READ_PATHS] = {};  // flb_readout_paths
};
Ring& ring() {
  static Ring* r = new Ring();
  return *r;
}

bool pin(Ring& r, char** p, size_t bytes) {
  if (hipHostMalloc(reinterpret_cast<void**>(p), bytes, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    *p = nullptr;
    return false;
  }
  r.paths[FLB_READ_PINNED] += int64_t(bytes);
  return true;
}
void unpin(Ring& r, char** p, size_t bytes) {
  if (!*p) return;
  (void)hipHostFree(*p);
  *p = nullptr;
  r.paths[FLB_READ_PINNED] -= int64_t(bytes);
}

void drop(Ring& r) {
  for (hipEvent_t& e : r.ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  unpin(r, &r.buf, kChunk * kRing);
  r.device = -1;
}

// The ring with events of the current device; false where it cannot be had.
bool ready(Ring& r) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  if (r.buf && r.device == dev) return true;
  drop(r);
  if (!pin(r, &r.buf, kChunk * kRing)) return false;
  for (hipEvent_t& e : r.ev)
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      e = nullptr;
      drop(r);
      return false;
    }
  r.device = dev;
  return true;
}

void put(void* host, const char* src, size_t bytes, bool widen) {
  if (!widen) {
    std::memcpy(host, src, bytes);
    return;
  }
  const float* f = reinterpret_cast<const float*>(src);
  double* d = static_cast<double*>(host);
  for (size_t i = 0; i < bytes / sizeof(float); ++i) d[i] = double(f[i]);
}

// One read-out through the ring, chunk c (at most kChunk bytes of one part) in
// buffer c % kRing. The calling thread enqueues the copies; worker w empties
// chunks w, w + n, ...
struct Job {
  Ring& r;
  bool widen;
  hipStream_t stream;
  int device;
  std::vector<ReadPart> list;        // chunks
  std::vector<char> emptied;         // per chunk
  std::mutex mu;
  std::condition_variable cv;
  size_t issued = 0;                 // chunks enqueued
  hipError_t err = hipSuccess;

  Job(Ring& ring, const ReadPart* parts, size_t n, bool wide, hipStream_t s)
      : r(ring), widen(wide), stream(s), device(ring.device) {
    for (size_t k = 0; k < n; ++k)
      for (size_t at = 0; at < parts[k].bytes; at += kChunk)
        list.push_back({static_cast<char*>(parts[k].host) + at * (wide ? 2 : 1),
                        static_cast<const char*>(parts[k].dev) + at, std::min(kChunk, parts[k].bytes - at)});
    emptied.assign(list.size(), 0);
  }
  size_t chunks() const { return list.size(); }

  hipError_t enqueue(size_t c) {
    const hipError_t e = hipMemcpyAsync(r.buf + (c % kRing) * kChunk, list[c].dev, list[c].bytes,
                                        hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipEventRecord(r.ev[c % kRing], stream);
  }
  hipError_t empty(size_t c) {
    const hipError_t e = hipEventSynchronize(r.ev[c % kRing]);
    if (e == hipSuccess) put(list[c].host, r.buf + (c % kRing) * kChunk, list[c].bytes, widen);
    return e;
  }
  void fail_all(hipError_t e) {
    std::lock_guard<std::mutex> l(mu);
    if (err == hipSuccess) err = e;
    cv.notify_all();
  }
  void worker(size_t w, size_t n) {
    (void)hipSetDevice(device);
    for (size_t c = w; c < chunks(); c += n) {
      {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return issued > c || err != hipSuccess; });
        if (err != hipSuccess) return;
      }
      const hipError_t e = empty(c);
      if (e != hipSuccess) return fail_all(e);
      std::lock_guard<std::mutex> l(mu);
      emptied[c] = 1;
      cv.notify_all();
    }
  }
  void issue() {
    for (size_t c = 0; c < chunks(); ++c) {
      if (c >= kRing) {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return emptied[c - kRing] || err != hipSuccess; });
        if (err != hipSuccess) return;
      }
      const hipError_t e = enqueue(c);
      if (e != hipSuccess) return fail_all(e);
      std::lock_guard<std::mutex> l(mu);
      issued = c + 1;
      cv.notify_all();
    }
  }
};

// Pageable copies of all parts, one wait.
hipError_t plain(const ReadPart* parts, size_t n, size_t bytes, bool widen, hipStream_t s) {
  const std::unique_ptr<char[]> t(widen ? new (std::nothrow) char[bytes] : nullptr);
  if (widen && !t) return hipErrorOutOfMemory;
  hipError_t e = hipSuccess;
  char* to = t.get();
  for (size_t k = 0; e == hipSuccess && k < n; ++k) {
    e = hipMemcpyAsync(widen ? to : parts[k].host, parts[k].dev, parts[k].bytes, hipMemcpyDeviceToHost, s);
    to += widen ? parts[k].bytes : 0;
  }
  const hipError_t w = hipStreamSynchronize(s);
  if (e == hipSuccess) e = w;
  if (e != hipSuccess || !widen) return e;
  to = t.get();
  for (size_t k = 0; k < n; to += parts[k].bytes, ++k) put(parts[k].host, to, parts[k].bytes, true);
  return hipSuccess;
}

}  // namespace

void readout_retain() {
  Ring& r = ring();
  std::lock_guard<std::mutex> l(r.users_mu);
  ++r.users;
}

void readout_release() {
  Ring& r = ring();
  std::lock_guard<std::mutex> l(r.users_mu);
  if (--r.users > 0) return;
  std::lock_guard<std::mutex> b(r.busy);
  drop(r);
  std::lock_guard<std::mutex> d(r.direct_busy);
  unpin(r, &r.direct, kDirect);
  r.small = 0;
}

// A kernel's output of at most kDirect bytes may go straight into pinned
// memory instead of a device buffer that is copied afterwards: one operation
// less on the stream (a step of 16^3 cells and its moments 39 -> 28 us). Holds the
// buffer while it lives; ptr is null where another thread holds it, and for
// the first four such read-outs: pinning and giving back cost 47 us, as much
// as four read-outs save. A program that makes a 16^3 block, steps and reads
// it k times and closes it, copies only -> buffer from the second read-out on
// -> now: k = 1 174 -> 169 -> 172 us, k = 2 206 -> 244 -> 203, k = 4 285 -> 300
// -> 278, k = 8 440 -> 410 -> 446, k = 32 1380 -> 1078 -> 1107.
DirectOut::DirectOut(size_t bytes) {
  Ring& r = ring();
  if (bytes > kDirect || !r.direct_busy.try_lock()) return;
  if (r.direct || (r.small >= kCopiesFirst && pin(r, &r.direct, kDirect))) {
    ptr = r.direct;
    r.paths[FLB_READ_DIRECT] += 1;
    return;
  }
  r.small += r.small < kCopiesFirst;
  r.direct_busy.unlock();
}
DirectOut::~DirectOut() {
  if (ptr) ring().direct_busy.unlock();
}

// Workers pay from two chunks on; a second read-out at the same time takes the
// plain copy. Several arrays are one read-out: one by one, the 10 gradients of
// a batch of 2.45 M cells were 10 waits and 10 cleared buffers (iteration less
// its kernels 1.8 -> 1.3 ms).
hipError_t readout(const ReadPart* parts, size_t n, bool widen, hipStream_t s) {
  size_t bytes = 0;
  for (size_t k = 0; k < n; ++k) bytes += parts[k].bytes;
  Ring& r = ring();
  std::unique_lock<std::mutex> busy(r.busy, std::defer_lock);
  if (bytes < 2 * kChunk || !busy.try_lock() || !ready(r)) {
    r.paths[FLB_READ_PLAIN] += 1;
    return plain(parts, n, bytes, widen, s);
  }
  r.paths[FLB_READ_RING] += 1;
  Job job(r, parts, n, widen, s);
  const size_t workers = std::min<size_t>(kWorkers, job.chunks());
  std::vector<std::thread> pool;
  pool.reserve(workers);
  try {
    for (size_t w = 0; w < workers; ++w) pool.emplace_back([&job, w, workers] { job.worker(w, workers); });
  } catch (const std::system_error&) {
    job.fail_all(hipErrorOutOfMemory);
  }
  if (pool.size() == workers) job.issue();
  for (std::thread& t : pool) t.join();
  if (pool.size() < workers) return plain(parts, n, bytes, widen, s);
  // copies of an abandoned read-out must not land in the ring later
  if (job.err != hipSuccess) (void)hipStreamSynchronize(s);
  return job.err;
}

hipError_t readout(void* host, const void* dev, size_t bytes, bool widen, hipStream_t s) {
  const ReadPart p{host, dev, bytes};
  return readout(&p, 1, widen, s);
}

}  // namespace flbh

int flb_readout_paths(int64_t* counts, int n) {
  int64_t now[FLB_READ_PATHS];
  for (int k = 0; k < FLB_READ_PATHS; ++k) now[k] = flbh::ring().paths[k];
  return flbh::copy_paths(now, FLB_READ_PATHS, counts, n);
}
