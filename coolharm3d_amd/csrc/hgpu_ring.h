// hgpu_ring.h -- the host side of the copies between device and (pageable) host
// memory: a ring of pinned chunks that the GPU fills or empties (kernels in
// hgpu_xfer.h) while host threads move them, and the plain copies that take its
// place where no memory can be pinned.  Host API of the runtime only.
#pragma once
#include <hip/hip_runtime_api.h>
#include <sched.h>
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace hgpu {

// The calling thread's current device while in scope
struct DeviceScope {
  int before = 0;
  bool moved = false;
  explicit DeviceScope(int device) {
    if (hipGetDevice(&before) == hipSuccess && before != device) moved = hipSetDevice(device) == hipSuccess;
  }
  ~DeviceScope() { if (moved) (void)hipSetDevice(before); }
};

// Ring of pinned chunks of one context, on its device; sized by the largest
// copy so far (at most cap chunks), released with the context.  One copy at a time
// (busy): threads that read from one context wait for each other.
struct XferRing {
  static constexpr size_t SLOT = 2u << 20;     // a multiple of 64 B (a zone) and 16 B
  static constexpr int SLOTS = 8;
  char* host = nullptr;
  char* dev = nullptr;                         // the device's address of host
  hipEvent_t ev[SLOTS] = {};
  int slots = 0;
  int device = 0;                              // the context's, whatever the calling thread's is
  std::mutex busy;
  int cap = SLOTS;                             // most chunks to ask for; lowered where pinned memory ran short

  void release() {
    for (int s = 0; s < slots; s++) (void)hipEventDestroy(ev[s]);
    if (host) (void)hipHostFree(host);
    host = dev = nullptr;
    slots = 0;
  }
  // A ring of n > slots chunks in place of the present one, which stays where
  // the larger one cannot be had; nothing may be in flight
  bool grow(int n) {
    void *p = nullptr, *d = nullptr;
    int have = slots;
    hipError_t e = hipHostMalloc(&p, n * SLOT, hipHostMallocDefault);
    if (e == hipSuccess) e = hipHostGetDevicePointer(&d, p, 0);
    for (; e == hipSuccess && have < n; have++) {
      e = hipEventCreateWithFlags(&ev[have], hipEventDisableTiming);
      if (e != hipSuccess) break;
    }
    if (e != hipSuccess) {
      while (have > slots) (void)hipEventDestroy(ev[--have]);
      if (p) (void)hipHostFree(p);
      (void)hipGetLastError();
      return false;
    }
    if (host) (void)hipHostFree(host);
    host = static_cast<char*>(p);
    dev = static_cast<char*>(d);
    slots = n;
    return true;
  }
  // Chunks for a copy of `bytes`: as many as it can use, or fewer where pinned
  // memory is short (which is remembered: asking costs more than it gives).
  // False: not one, the copy goes without.
  bool reserve(size_t bytes) {
    const size_t want = (bytes + SLOT - 1) / SLOT;
    int n = (int)std::min<size_t>((size_t)cap, std::max<size_t>(1, want));
    const int asked = n;
    while (n > slots && !grow(n)) n /= 2;
    if (n < asked && slots < asked) cap = slots;
    return slots > 0;
  }
};

// Host threads beside the caller for a copy of `bytes`: none below 4 MB (a few
// chunks: starting threads would cost what they save), else enough to keep up
// with the link (a core copies about 29 GB/s, less into fresh pages), and at most
// half the CPUs that the process may run on (the ranks of a node share its CPUs).
inline int xfer_threads(size_t bytes) {
  if (bytes < (4u << 20)) return 0;
  cpu_set_t cpus;
  const unsigned hw = sched_getaffinity(0, sizeof(cpus), &cpus) == 0 ? (unsigned)CPU_COUNT(&cpus)
                                                                     : std::thread::hardware_concurrency();
  return (int)std::min<unsigned>(hw > 2 ? hw / 2 : 0, bytes < (32u << 20) ? 3 : 6);
}

// Device to host: fill(offset, bytes, chunk) enqueues on st the kernel that
// fills a chunk (a device address) with bytes [offset, offset + bytes) of the
// result; plain() is the copy where no memory can be pinned.  Returns when host
// holds all of it.
template <class Fill, class Plain>
hipError_t xfer_to_host(XferRing& R, hipStream_t st, void* host, size_t bytes, Fill&& fill, Plain&& plain) {
  std::lock_guard<std::mutex> one(R.busy);
  const DeviceScope on(R.device);
  if (!R.reserve(bytes)) return plain();
  hipError_t e = hipSuccess;
  const long long n = (long long)((bytes + XferRing::SLOT - 1) / XferRing::SLOT);
  const int S = R.slots;
  const auto len = [&](long long c) { return std::min(XferRing::SLOT, bytes - (size_t)c * XferRing::SLOT); };
  const auto enqueue = [&](long long c) {
    const size_t off = (size_t)c * XferRing::SLOT;
    fill(off, len(c), R.dev + (size_t)(c % S) * XferRing::SLOT);
    hipError_t r = hipGetLastError();
    return r == hipSuccess ? hipEventRecord(R.ev[c % S], st) : r;
  };
  const auto take = [&](long long c) {
    const hipError_t r = hipEventSynchronize(R.ev[c % S]);
    if (r == hipSuccess)
      std::memcpy(static_cast<char*>(host) + (size_t)c * XferRing::SLOT, R.host + (size_t)(c % S) * XferRing::SLOT, len(c));
    return r;
  };
  std::atomic<long long> enqueued{0}, next{0};
  std::atomic<long long> copied[XferRing::SLOTS];   // chunks taken out of each slot
  for (auto& x : copied) x.store(0);
  std::atomic<int> err{(int)hipSuccess};
  // The workers sleep until the first chunk is there: work queued on the stream
  // before the copy may take long, and the caller alone waits for that.  (The caller
  // only keeps the chunks filled: taking some itself made 93 MB 0.9 ms slower.)
  std::mutex gate;
  std::condition_variable opened;
  bool open = false;
  const auto worker = [&]() {
    if (hipSetDevice(R.device) != hipSuccess) err = (int)hipErrorInvalidDevice;
    {
      std::unique_lock<std::mutex> l(gate);
      opened.wait(l, [&]() { return open; });
    }
    for (;;) {
      const long long c = next.fetch_add(1);
      if (c >= n) return;
      while (enqueued.load(std::memory_order_acquire) <= c) {
        if (err.load() != (int)hipSuccess) return;
        std::this_thread::yield();
      }
      const hipError_t r = take(c);
      if (r != hipSuccess) { err = (int)r; return; }
      copied[c % S].fetch_add(1, std::memory_order_release);
    }
  };
  std::vector<std::thread> pool;
  try {
    const int w = n > 1 ? xfer_threads(bytes) : 0;
    pool.reserve(w);
    for (int k = 0; k < w; k++) pool.emplace_back(worker);
  } catch (...) {
    // fewer threads than wanted (or none): the copy below works with any number
  }
  if (pool.empty()) {   // the caller alone: fill ahead, take in order
    long long filled = 0;
    for (long long c = 0; c < n && e == hipSuccess; c++) {
      for (; filled < n && filled < c + S && e == hipSuccess; filled++) e = enqueue(filled);
      if (e == hipSuccess) e = take(c);
    }
  } else {
    const auto put = [&](long long c) {
      const hipError_t r = enqueue(c);
      if (r != hipSuccess) err = (int)r;
      else enqueued.store(c + 1, std::memory_order_release);
    };
    long long c = 0;
    for (; c < n && c < S && err.load() == (int)hipSuccess; c++) put(c);
    if (err.load() == (int)hipSuccess && (e = hipEventSynchronize(R.ev[0])) != hipSuccess) err = (int)e;
    {
      std::lock_guard<std::mutex> l(gate);
      open = true;
    }
    opened.notify_all();
    for (; c < n && err.load() == (int)hipSuccess; c++) {
      while (copied[c % S].load(std::memory_order_acquire) < c / S && err.load() == (int)hipSuccess) std::this_thread::yield();
      put(c);
    }
    for (auto& t : pool) t.join();
    e = (hipError_t)err.load();
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(st);   // no kernel may still write a chunk
  return e;
}

// Host to device: empty(offset, bytes, chunk) enqueues on st the kernel that
// reads bytes [offset, offset + bytes) of the source from a chunk; plain() as
// above.  Returns when the device holds all of it.
template <class Empty, class Plain>
hipError_t xfer_to_device(XferRing& R, hipStream_t st, const void* host, size_t bytes, Empty&& empty, Plain&& plain) {
  std::lock_guard<std::mutex> one(R.busy);
  const DeviceScope on(R.device);
  if (!R.reserve(bytes)) return plain();
  hipError_t e = hipSuccess;
  const long long n = (long long)((bytes + XferRing::SLOT - 1) / XferRing::SLOT);
  const int S = R.slots;
  for (long long c = 0; c < n && e == hipSuccess; c++) {
    const size_t off = (size_t)c * XferRing::SLOT, len = std::min(XferRing::SLOT, bytes - off);
    const size_t at = (size_t)(c % S) * XferRing::SLOT;
    if (c >= S) e = hipEventSynchronize(R.ev[c % S]);
    if (e != hipSuccess) break;
    std::memcpy(R.host + at, static_cast<const char*>(host) + off, len);
    empty(off, len, R.dev + at);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipEventRecord(R.ev[c % S], st);
  }
  const hipError_t s = hipStreamSynchronize(st);
  return e == hipSuccess ? s : e;
}

// Without pinned memory: the runtime's own copies of pageable memory; a state
// ([nv][nt] on the device, [nt][nv] on the host) goes through a buffer of a chunk's
// size and is transposed on the host.
inline hipError_t plain_to_host(hipStream_t st, void* host, const void* dev, size_t bytes) {
  const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
  const hipError_t s = hipStreamSynchronize(st);
  return e == hipSuccess ? s : e;
}
template <class Move>   // move(buffer, first zone, zones): one buffer's worth, waited for
hipError_t plain_state(long long nt, int nv, Move&& move) {
  const long long nz = std::min<long long>(nt, (long long)(XferRing::SLOT / (sizeof(double) * nv)));
  std::unique_ptr<double[]> buf(new (std::nothrow) double[(size_t)nz * nv]);
  if (!buf) return hipErrorOutOfMemory;
  hipError_t e = hipSuccess;
  for (long long z0 = 0; z0 < nt && e == hipSuccess; z0 += nz) e = move(buf.get(), z0, std::min(nz, nt - z0));
  return e;
}
inline hipError_t plain_state_to_host(hipStream_t st, double* host, const double* S, long long nt, int nv) {
  return plain_state(nt, nv, [&](double* buf, long long z0, long long n) {
    hipError_t e = hipSuccess;
    for (int v = 0; v < nv && e == hipSuccess; v++)
      e = hipMemcpyAsync(buf + v*n, S + v*nt + z0, sizeof(double) * n, hipMemcpyDeviceToHost, st);
    const hipError_t s = hipStreamSynchronize(st);
    if (e == hipSuccess) e = s;
    if (e == hipSuccess)
      for (long long z = 0; z < n; z++) for (int v = 0; v < nv; v++) host[(z0 + z)*nv + v] = buf[v*n + z];
    return e;
  });
}
inline hipError_t plain_state_to_device(hipStream_t st, double* S, const double* host, long long nt, int nv) {
  return plain_state(nt, nv, [&](double* buf, long long z0, long long n) {
    for (long long z = 0; z < n; z++) for (int v = 0; v < nv; v++) buf[v*n + z] = host[(z0 + z)*nv + v];
    hipError_t e = hipSuccess;
    for (int v = 0; v < nv && e == hipSuccess; v++)
      e = hipMemcpyAsync(S + v*nt + z0, buf + v*n, sizeof(double) * n, hipMemcpyHostToDevice, st);
    const hipError_t s = hipStreamSynchronize(st);
    return e == hipSuccess ? s : e;
  });
}

}  // namespace hgpu
