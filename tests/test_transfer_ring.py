"""The host side of the copies to and from the device (hgpu_ring.h) against a small
stand-in for the runtime: host and device memory are one, a launch runs at once,
and pinned memory, events and copies can be made to fail."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "coolharm3d_amd", "csrc")

STUB = r"""
#pragma once
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <sched.h>
#include <mutex>
#include <thread>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
typedef int* hipStream_t;
struct Ev { int device; };
typedef Ev* hipEvent_t;
struct Rt {
  std::mutex m;
  std::map<void*, size_t> pinned;
  size_t budget = ~(size_t)0, used = 0, most = 0;
  int mallocs = 0, events = 0, event_limit = 1 << 20, copies = 0;
  int busy_ms = 0, waiters_then = 0;
  std::thread::id first_waiter;
  hipError_t malloc_error = hipErrorOutOfMemory;
} rt;
static thread_local int t_device = 0;
static thread_local hipError_t t_last = hipSuccess;
inline hipError_t fails(hipError_t e) { if (e) t_last = e; return e; }
inline hipError_t hipGetLastError() { hipError_t e = t_last; t_last = hipSuccess; return e; }
inline hipError_t hipGetDevice(int* d) { *d = t_device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  std::lock_guard<std::mutex> l(rt.m);
  rt.mallocs++;
  if (rt.used + n > rt.budget) return fails(rt.malloc_error);
  *p = malloc(n);
  rt.pinned[*p] = n;
  rt.used += n;
  if (rt.used > rt.most) rt.most = rt.used;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> l(rt.m);
  rt.used -= rt.pinned.at(p);
  rt.pinned.erase(p);
  free(p);
  return hipSuccess;
}
inline hipError_t hipHostGetDevicePointer(void** d, void* p, unsigned) { *d = p; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  std::lock_guard<std::mutex> l(rt.m);
  if (rt.events >= rt.event_limit) return fails(hipErrorOutOfMemory);
  rt.events++;
  *e = new Ev{t_device};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { std::lock_guard<std::mutex> l(rt.m); rt.events--; delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) { return e->device == *st ? hipSuccess : fails(hipErrorInvalidHandle); }
inline hipError_t hipEventSynchronize(hipEvent_t) {
  std::unique_lock<std::mutex> l(rt.m);
  if (rt.first_waiter == std::thread::id()) {
    rt.first_waiter = std::this_thread::get_id();
    l.unlock();
    std::this_thread::sleep_for(std::chrono::milliseconds(rt.busy_ms));
    l.lock();
    rt.busy_ms = 0;
  } else if (rt.busy_ms) {
    rt.waiters_then++;
  }
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::lock_guard<std::mutex> l(rt.m);
  rt.copies++;
  memcpy(d, s, n);
  return hipSuccess;
}
"""

COMMON = r"""
#include "hgpu_ring.h"
#include <cstdio>
#include <random>
using namespace hgpu;
#define CHECK(x) do { if (!(x)) { printf("%d: %s\n", __LINE__, #x); return 1; } } while (0)
constexpr int NV = 8;
constexpr size_t CH = XferRing::SLOT;
static int stream_device = 0;
static hipStream_t ST = &stream_device;
static std::vector<double> values(long long nt, unsigned seed) {
  std::mt19937_64 g(seed);
  std::vector<double> a((size_t)nt * NV);
  for (double& x : a) x = (double)(long long)g();
  return a;
}
// the state S ([NV][nt]) to h ([nt][NV]) and back, as the library's callers do it
static hipError_t down(XferRing& R, double* h, const double* S, long long nt) {
  return xfer_to_host(R, ST, h, sizeof(double) * NV * nt, [&](size_t off, size_t len, char* chunk) {
    const long long z0 = (long long)(off / (8 * NV)), nz = (long long)(len / (8 * NV));
    double* out = reinterpret_cast<double*>(chunk);
    for (long long z = 0; z < nz; z++) for (int v = 0; v < NV; v++) out[z*NV + v] = S[v*nt + z0 + z];
  }, [&]() { return plain_state_to_host(ST, h, S, nt, NV); });
}
static hipError_t up(XferRing& R, double* S, const double* h, long long nt) {
  return xfer_to_device(R, ST, h, sizeof(double) * NV * nt, [&](size_t off, size_t len, const char* chunk) {
    const long long z0 = (long long)(off / (8 * NV)), nz = (long long)(len / (8 * NV));
    const double* in = reinterpret_cast<const double*>(chunk);
    for (long long z = 0; z < nz; z++) for (int v = 0; v < NV; v++) S[v*nt + z0 + z] = in[z*NV + v];
  }, [&]() { return plain_state_to_device(ST, S, h, nt, NV); });
}
static bool round_trip(XferRing& R, long long nt, unsigned seed) {
  const std::vector<double> a = values(nt, seed);
  std::vector<double> S(a.size()), b(a.size());
  if (up(R, S.data(), a.data(), nt) != hipSuccess || down(R, b.data(), S.data(), nt) != hipSuccess) return false;
  for (long long z = 0; z < nt; z++) for (int v = 0; v < NV; v++) if (S[v*nt + z] != a[z*NV + v]) return false;
  return a == b;
}
constexpr long long ZC = CH / (8 * NV);   // zones of a chunk
"""

CASES = {
    "sizes": r"""
  XferRing R;
  for (long long nt : {1ll, ZC - 1, ZC, ZC + 1, 3*ZC + 5, 7*ZC, 23*ZC + 1}) CHECK(round_trip(R, nt, (unsigned)nt));
  CHECK(R.slots == XferRing::SLOTS && rt.used == XferRing::SLOTS * CH && rt.copies == 0);
  R.release();
  CHECK(rt.used == 0 && rt.events == 0);
""",
    # a ring of fewer chunks than wanted, asked for once
    "short": r"""
  for (int have : {1, 2, 4, 5}) {
    rt.budget = have * CH;
    XferRing R;
    CHECK(round_trip(R, 23*ZC + 7, 3));
    const int slots = R.slots, asked = rt.mallocs;
    CHECK(slots >= 1 && slots <= have && rt.copies == 0);
    CHECK(round_trip(R, 23*ZC + 7, 4) && round_trip(R, 40*ZC + 1, 5) && round_trip(R, 3, 6));
    CHECK(rt.mallocs == asked && R.slots == slots);
    R.release();
    CHECK(rt.used == 0 && rt.events == 0);
  }
""",
    # a larger ring cannot be had: the present one stays
    "kept": r"""
  XferRing R;
  CHECK(round_trip(R, 2*ZC, 1));
  CHECK(R.slots == 2);
  char* const held = R.host;
  rt.budget = rt.used;
  CHECK(round_trip(R, 23*ZC + 7, 2));
  CHECK(R.slots == 2 && R.host == held && rt.copies == 0);
  rt.budget = ~(size_t)0;
  rt.event_limit = 2;
  R.cap = XferRing::SLOTS;
  CHECK(round_trip(R, 23*ZC + 7, 3));                    // no events for more chunks
  CHECK(R.slots == 2 && R.host == held && rt.events == 2 && rt.used == 2 * CH);
  CHECK(hipGetLastError() == hipSuccess);
""",
    # no pinned memory at all, whatever the runtime calls it: the plain copies
    "none": r"""
  for (hipError_t e : {hipErrorOutOfMemory, hipErrorInvalidValue}) {
    rt.budget = 0;
    rt.malloc_error = e;
    XferRing R;
    for (long long nt : {1ll, ZC + 1, 23*ZC + 7}) CHECK(round_trip(R, nt, (unsigned)nt));
    std::vector<char> a(100, 'x'), b(100);
    CHECK(xfer_to_host(R, ST, b.data(), 100, [](size_t, size_t, char*) {}, [&]() { return plain_to_host(ST, b.data(), a.data(), 100); }) == hipSuccess);
    CHECK(a == b && rt.used == 0 && rt.events == 0 && hipGetLastError() == hipSuccess);
    R.cap = 0;                                           // none wanted
    const int asked = rt.mallocs;
    CHECK(round_trip(R, 2*ZC, 9) && rt.mallocs == asked);
  }
""",
    # several threads with a ring between them
    "threads": r"""
  XferRing R;
  std::atomic<int> bad{0};
  std::vector<std::thread> t;
  for (int k = 0; k < 4; k++)
    t.emplace_back([&, k]() { for (int q = 0; q < 12; q++) if (!round_trip(R, (q % 3) * ZC + 900*k + 7, 100*k + q)) bad++; });
  for (auto& x : t) x.join();
  CHECK(bad == 0);
""",
    # a thread whose current device is another than the context's
    "device": r"""
  stream_device = 1;
  XferRing R;
  R.device = 1;
  CHECK(round_trip(R, 3*ZC + 5, 1) && rt.copies == 0 && R.slots == 4);
  int now = -1;
  CHECK(hipGetDevice(&now) == hipSuccess && now == 0);
""",
    # work queued before the copy is waited for by the caller alone; no more host threads
    # than the process's CPUs allow
    "crew": r"""
  XferRing R;
  const long long nt = 23*ZC + 7;
  const std::vector<double> S = values(nt, 1);
  std::vector<double> h(S.size());
  rt.busy_ms = 50;                                       // the first wait takes this long
  CHECK(down(R, h.data(), S.data(), nt) == hipSuccess);
  for (long long z = 0; z < nt; z++) for (int v = 0; v < NV; v++) CHECK(h[z*NV + v] == S[v*nt + z]);
  CHECK(rt.first_waiter == std::this_thread::get_id() && rt.waiters_then == 0);
  cpu_set_t all, some;
  CHECK(sched_getaffinity(0, sizeof(all), &all) == 0);
  for (int want : {1, 2, 4}) {
    CPU_ZERO(&some);
    for (int c = 0, k = 0; c < CPU_SETSIZE && k < want; c++) if (CPU_ISSET(c, &all)) { CPU_SET(c, &some); k++; }
    if (CPU_COUNT(&some) < want) break;
    CHECK(sched_setaffinity(0, sizeof(some), &some) == 0);
    CHECK(xfer_threads(64u << 20) == (want > 2 ? want / 2 : 0));
  }
""",
}


@pytest.mark.parametrize("name", list(CASES))
def test_ring(tmp_path, name):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime_api.h").write_text(STUB)
    src, exe = tmp_path / "ring.cpp", tmp_path / "ring"
    src.write_text(COMMON + "int main() {\n" + CASES[name] + "  return 0;\n}\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I" + str(tmp_path), "-I" + CSRC, "-o", str(exe), str(src)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
