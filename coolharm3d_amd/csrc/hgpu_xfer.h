// hgpu_xfer.h -- copies of large arrays between device and (pageable) host
// memory, through a ring of pinned chunks.
//
// The reference's arrays hold a zone's variables together ([zone][8]), the
// device's hold a variable's zones together ([8][zone]).  The GPU turns one into
// the other as it fills or empties a pinned chunk, and a few host threads move
// the chunks to or from the caller's memory meanwhile, so a copy runs at the
// link's rate (57 GB/s pinned) instead of one host core's (transposing 336 MB
// on the host took 50 ms beside the copy).  Measured, 192x192x128 with ghosts
// (336 MB) to fresh numpy memory: 57 -> 8.1 ms down, 12 ms up.
#pragma once
#include "hgpu_launch.h"
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace hgpu {

constexpr int XFER_B = 256;

// nz zones from zone z0 of S ([8][nt]) to out ([nz][8]); a workgroup turns 256
// zones around in LDS so that both sides are read and written in whole lines.
// The LDS rows are 264 words of 8 B apart: a wavefront's 8 variables x 8 zones
// then meet on at most two lanes per bank.
__global__ __launch_bounds__(XFER_B) void k_soa_to_aos(const double* __restrict__ S, long long nt, long long z0,
                                                       long long nz, double* __restrict__ out) {
  __shared__ double buf[NP][XFER_B + 8];
  const long long zb = (long long)blockIdx.x * XFER_B;
  const long long z = zb + threadIdx.x;
  if (z < nz) {
#pragma unroll
    for (int v = 0; v < NP; v++) buf[v][threadIdx.x] = S[v*nt + z0 + z];
  }
  __syncthreads();
  const long long n = (nz - zb < XFER_B ? nz - zb : XFER_B) * NP;
#pragma unroll
  for (int r = 0; r < NP; r++) {
    const int e = r*XFER_B + threadIdx.x;
    if (e < n) out[zb*NP + e] = buf[e % NP][e / NP];
  }
}

__global__ __launch_bounds__(XFER_B) void k_aos_to_soa(const double* __restrict__ in, long long nt, long long z0,
                                                       long long nz, double* __restrict__ S) {
  __shared__ double buf[NP][XFER_B + 8];
  const long long zb = (long long)blockIdx.x * XFER_B;
  const long long n = (nz - zb < XFER_B ? nz - zb : XFER_B) * NP;
#pragma unroll
  for (int r = 0; r < NP; r++) {
    const int e = r*XFER_B + threadIdx.x;
    if (e < n) buf[e % NP][e / NP] = in[zb*NP + e];
  }
  __syncthreads();
  const long long z = zb + threadIdx.x;
  if (z < nz) {
#pragma unroll
    for (int v = 0; v < NP; v++) S[v*nt + z0 + z] = buf[v][threadIdx.x];
  }
}

// n32 words of 4 B from src to dst, 16 B at a time; both 16 B aligned
__global__ __launch_bounds__(XFER_B) void k_copy_words(const unsigned* __restrict__ src, long long n32,
                                                       unsigned* __restrict__ dst) {
  const long long n16 = n32 / 4, stride = (long long)gridDim.x * XFER_B;
  const long long t0 = (long long)blockIdx.x * XFER_B + threadIdx.x;
  for (long long t = t0; t < n16; t += stride)
    reinterpret_cast<uint4*>(dst)[t] = reinterpret_cast<const uint4*>(src)[t];
  if (t0 < n32 - 4*n16) dst[4*n16 + t0] = src[4*n16 + t0];
}

// Ring of pinned chunks of one context, on its device; sized by the largest
// copy so far (at most SLOTS chunks), released with the context.
struct XferRing {
  static constexpr size_t SLOT = 2u << 20;     // a multiple of 64 B (a zone) and 16 B
  static constexpr int SLOTS = 8;
  char* host = nullptr;
  char* dev = nullptr;                         // the device's address of host
  hipEvent_t ev[SLOTS] = {};
  int slots = 0, device = 0;

  void release() {
    for (int s = 0; s < slots; s++) (void)hipEventDestroy(ev[s]);
    if (host) (void)hipHostFree(host);
    host = dev = nullptr;
    slots = 0;
  }
  // at least the chunks that `bytes` can use; nothing may be in flight
  hipError_t reserve(size_t bytes) {
    const size_t want = (bytes + SLOT - 1) / SLOT;
    int n = (int)std::min<size_t>(SLOTS, std::max<size_t>(1, want));
    if (n <= slots) return hipSuccess;
    release();
    void *p = nullptr, *d = nullptr;
    hipError_t e = hipGetDevice(&device);
    if (e == hipSuccess) e = hipHostMalloc(&p, n * SLOT, hipHostMallocDefault);
    while (e == hipErrorOutOfMemory && n > 1) {   // pinned memory is short: a smaller ring, down to one chunk
      (void)hipGetLastError();
      n /= 2;
      e = hipHostMalloc(&p, n * SLOT, hipHostMallocDefault);
    }
    if (e != hipSuccess) return e;
    host = static_cast<char*>(p);
    e = hipHostGetDevicePointer(&d, p, 0);
    for (; e == hipSuccess && slots < n; slots++) {
      e = hipEventCreateWithFlags(&ev[slots], hipEventDisableTiming);
      if (e != hipSuccess) break;
    }
    if (e != hipSuccess) { release(); return e; }
    dev = static_cast<char*>(d);
    return hipSuccess;
  }
};

// Host threads beside the caller for a copy of `bytes`: none below 4 MB (a few
// chunks: starting threads would cost what they save), else enough to keep up
// with the link (a core copies about 29 GB/s, less into fresh pages).
inline int xfer_threads(size_t bytes) {
  if (bytes < (4u << 20)) return 0;
  const unsigned hw = std::thread::hardware_concurrency();
  return (int)std::min<unsigned>(hw > 2 ? hw / 2 : 0, bytes < (32u << 20) ? 3 : 6);
}

// Device to host: fill(offset, bytes, chunk) enqueues on st the kernel that
// fills a chunk (a device address) with bytes [offset, offset + bytes) of the
// result.  Returns when host holds all of it.
template <class Fill>
hipError_t xfer_to_host(XferRing& R, hipStream_t st, void* host, size_t bytes, Fill&& fill) {
  hipError_t e = R.reserve(bytes);
  if (e != hipSuccess) return e;
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
  const auto worker = [&]() {
    if (hipSetDevice(R.device) != hipSuccess) err = (int)hipErrorInvalidDevice;
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
    for (long long c = 0; c < n && err.load() == (int)hipSuccess; c++) {
      while (copied[c % S].load(std::memory_order_acquire) < c / S && err.load() == (int)hipSuccess) std::this_thread::yield();
      const hipError_t r = enqueue(c);
      if (r != hipSuccess) { err = (int)r; break; }
      enqueued.store(c + 1, std::memory_order_release);
    }
    for (auto& t : pool) t.join();
    e = (hipError_t)err.load();
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(st);   // no kernel may still write a chunk
  return e;
}

// Host to device: empty(offset, bytes, chunk) enqueues on st the kernel that
// reads bytes [offset, offset + bytes) of the source from a chunk.  Returns
// when the device holds all of it.
template <class Empty>
hipError_t xfer_to_device(XferRing& R, hipStream_t st, const void* host, size_t bytes, Empty&& empty) {
  hipError_t e = R.reserve(bytes);
  if (e != hipSuccess) return e;
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

}  // namespace hgpu
