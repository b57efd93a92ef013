"""The pinned ring's protocol on the CPU: host_copy.hip compiled by g++ against a
small stand-in of the HIP runtime (streams as threads, events as marks on them,
the copy kernel run as written), so that what it asks of the runtime and the order
of its transfers can be checked without a GPU."""
import os
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "mdwtracker_amd" / "csrc"

RUNTIME = r"""
#pragma once
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>
#define __global__
#define __launch_bounds__(...)
#define __restrict__
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101 };
enum { hipHostMallocDefault = 0, hipHostMallocPortable = 1, hipHostMallocCoherent = 0x40000000 };
enum { hipEventDefault = 0, hipEventDisableTiming = 2, hipEventReleaseToSystem = (int)0x80000000 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
struct uint4 { uint32_t x, y, z, w; };
struct dim3 { unsigned x, y = 1, z = 1; dim3(unsigned n) : x(n) {} };
struct Idx { unsigned x; };
inline thread_local Idx blockIdx, threadIdx, gridDim;
namespace fake {
inline thread_local hipError_t last = hipSuccess;
inline thread_local int device = 0;
inline std::mutex mu;
inline unsigned host_flags = 0, event_flags = 0;
inline std::map<int, int> rings, launches, copies;  // by device
inline hipError_t set(hipError_t e) { if (e) last = e; return e; }
struct Stream {
  std::mutex m;
  std::condition_variable cv, idle;
  std::deque<std::function<void()>> q;
  uint64_t pushed = 0, done = 0;
  bool stop = false;
  std::thread t{[this] {
    while (true) {
      std::function<void()> f;
      {
        std::unique_lock<std::mutex> l(m);
        cv.wait(l, [&] { return stop || !q.empty(); });
        if (q.empty()) return;
        f = std::move(q.front());
        q.pop_front();
      }
      f();
      std::lock_guard<std::mutex> l(m);
      ++done;
      idle.notify_all();
    }
  }};
  uint64_t push(std::function<void()> f) {
    std::lock_guard<std::mutex> l(m);
    q.push_back(std::move(f));
    cv.notify_one();
    return ++pushed;
  }
  void wait(uint64_t n) {
    std::unique_lock<std::mutex> l(m);
    idle.wait(l, [&] { return done >= n; });
  }
  ~Stream() {
    { std::lock_guard<std::mutex> l(m); stop = true; }
    cv.notify_one();
    t.join();
  }
};
struct Event { std::mutex m; Stream* s = nullptr; uint64_t n = 0; };
}  // namespace fake
typedef fake::Stream* hipStream_t;
typedef fake::Event* hipEvent_t;
inline hipError_t hipGetLastError() { hipError_t e = fake::last; fake::last = hipSuccess; return e; }
inline hipError_t hipSetDevice(int d) { fake::device = d; return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = fake::device; return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
  std::lock_guard<std::mutex> l(fake::mu);
  fake::host_flags = flags;
  ++fake::rings[fake::device];
  *p = std::aligned_alloc(4096, n);
  std::memset(*p, 0xA5, n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> l(fake::mu);
  --fake::rings[fake::device];
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
  std::lock_guard<std::mutex> l(fake::mu);
  fake::event_flags = flags;
  *e = new fake::Event();
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> l(e->m);
  e->s = s;
  e->n = s->push([] {});
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  fake::Stream* s;
  uint64_t n;
  { std::lock_guard<std::mutex> l(e->m); s = e->s; n = e->n; }
  if (s) s->wait(n);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t q) {
  { std::lock_guard<std::mutex> l(fake::mu); ++fake::copies[fake::device]; }
  q->wait(q->push([=] { std::memcpy(d, s, n); }));
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) { s->wait(s->push([] {})); return hipSuccess; }
template <class F>
inline void fake_launch(F&& kernel, dim3 grid, dim3 block, hipStream_t s) {
  { std::lock_guard<std::mutex> l(fake::mu); ++fake::launches[fake::device]; }
  s->push([=] {
    gridDim.x = grid.x;
    for (blockIdx.x = 0; blockIdx.x < grid.x; ++blockIdx.x)
      for (threadIdx.x = 0; threadIdx.x < block.x; ++threadIdx.x) kernel();
  });
}
#define hipLaunchKernelGGL(f, grid, block, lds, stream, ...)                                  \
  do { auto args_ = std::make_tuple(__VA_ARGS__);                                             \
       fake_launch([args_] { std::apply(f, args_); }, grid, block, stream); } while (0)
inline hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** a, size_t, hipStream_t s) {
  auto k = reinterpret_cast<void (*)(const uint8_t*, uint8_t*, uint32_t)>(const_cast<void*>(f));
  auto* src = *static_cast<const uint8_t**>(a[0]);
  auto* dst = *static_cast<uint8_t**>(a[1]);
  const uint32_t n = *static_cast<uint32_t*>(a[2]);
  fake_launch([=] { k(src, dst, n); }, grid, block, s);
  return hipSuccess;
}
"""

PROLOGUE = r"""
#include <tuple>
#include <dirent.h>
#include <sched.h>
#include <cstdio>
#include "host_copy.hip"
using namespace mdwt;
static int bad = 0;
#define EXPECT(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); ++bad; } } while (0)
static const size_t kRing = kChunk * kSlots;
static std::vector<uint8_t> pattern(size_t n, uint32_t seed) {
  std::vector<uint8_t> v(n);
  uint64_t x = seed * 0x9E3779B97F4A7C15ull + 1;
  for (size_t i = 0; i < n; i += 8) {
    x = x * 6364136223846793005ull + 1442695040888963407ull;
    const uint64_t y = x >> 8;
    std::memcpy(&v[i], &y, std::min<size_t>(8, n - i));
  }
  return v;
}
// n bytes to the "device" and back; the device copy is compared with the source
static void round_trip(size_t n, uint32_t seed, int device, hipStream_t s) {
  const std::vector<uint8_t> src = pattern(n, seed);
  void* dev = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  std::vector<uint8_t> back(n, 0xEE);
  EXPECT(copy_to_device(dev, src.data(), n, device, s) == hipSuccess);
  EXPECT(hipStreamSynchronize(s) == hipSuccess);
  EXPECT(std::memcmp(dev, src.data(), n) == 0);
  EXPECT(copy_to_host(back.data(), dev, n, device, s) == hipSuccess);
  EXPECT(back == src);
  std::free(dev);
}
[[maybe_unused]] static int threads_now() {
  int n = 0;
  DIR* d = opendir("/proc/self/task");
  while (readdir(d)) ++n;
  closedir(d);
  return n - 2;
}
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("ring")
    (tmp / "hip").mkdir()
    (tmp / "hip" / "hip_runtime.h").write_text(RUNTIME)

    def go(body):
        src, exe = tmp / "t.cpp", tmp / "t"
        src.write_text(PROLOGUE + "int main() {\n" + body + '\n  if (!bad) std::printf("ok\\n");\n  return bad;\n}\n')
        r = subprocess.run(["g++", "-O2", "-std=c++17", f"-I{tmp}", f"-I{CSRC}", str(src), "-o", str(exe), "-pthread"],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
        assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
    return go


def test_sizes_around_the_ring(run):
    """Up to several times the ring's slots, with ragged tails, both ways."""
    run(r"""
  host_copy_acquire();
  fake::Stream stream;
  hipStream_t s = &stream;
  uint32_t seed = 0;
  for (size_t n : {size_t(1), kMinBytes - 1, kMinBytes, kMinBytes + 3, kChunk - 1, kChunk, kChunk + 17,
                   kRing - 5, kRing, kRing + 1, kRing + kChunk, 2 * kRing + 12345, 3 * kRing - 7})
    round_trip(n, ++seed, 0, s);
  EXPECT(fake::rings[0] == 1);
  host_copy_release();
  EXPECT(fake::rings[0] == 0);""")


def test_threads_and_streams_side_by_side(run):
    run(r"""
  host_copy_acquire();
  fake::Stream streams[6];
  std::vector<std::thread> t;
  for (uint32_t k = 0; k < 6; ++k)
    t.emplace_back([k, s = &streams[k]] {
      for (uint32_t i = 0; i < 4; ++i) round_trip(kRing + 1000 * k + i, 10 * k + i, 0, s);
    });
  for (auto& x : t) x.join();
  EXPECT(fake::rings[0] >= 1 && fake::rings[0] <= 4);
  host_copy_release();
  EXPECT(fake::rings[0] == 0);""")


def test_what_kernels_write_is_visible_to_the_host(run):
    """The copy kernel writes and reads the ring while host threads do: coherent
    memory, and events that release to the system."""
    run(r"""
  host_copy_acquire();
  fake::Stream s;
  round_trip(kRing + 1, 1, 0, &s);
  EXPECT(fake::host_flags & hipHostMallocCoherent);
  EXPECT(fake::event_flags & hipEventReleaseToSystem);
  EXPECT(fake::event_flags & hipEventDisableTiming);
  host_copy_release();""")


def test_an_earlier_error_of_the_thread_is_not_the_copys(run):
    """An error that an earlier call of the calling thread left behind (the
    runtime keeps it until it is asked for)."""
    run(r"""
  host_copy_acquire();
  fake::Stream s;
  fake::last = hipErrorOutOfMemory;
  round_trip(kRing + 1, 1, 0, &s);
  EXPECT(hipGetLastError() == hipErrorOutOfMemory);
  host_copy_release();""")


def test_every_device_gets_rings(run):
    """One thread that goes over several devices, twice: each keeps a ring of its
    own, however many others there are, and the current device stays."""
    run(r"""
  host_copy_acquire();
  fake::Stream s;
  for (int round = 0; round < 2; ++round)
    for (int d = 0; d < 7; ++d) {
      hipSetDevice(d);
      const int before = fake::launches[d];
      round_trip(kRing, 1, d, &s);
      EXPECT(fake::launches[d] == before + 2 * kSlots && fake::copies[d] == 0);
      EXPECT(fake::rings[d] == 1);
      EXPECT(fake::device == d);
    }
  hipSetDevice(3);
  host_copy_release();
  EXPECT(fake::device == 3);
  for (const auto& r : fake::rings) EXPECT(r.second == 0);""")


@pytest.mark.parametrize("cores", [1, 2, 3, 4, 6])
def test_no_more_threads_than_cores(run, cores):
    """The calling thread and its helpers, on a process of few cores."""
    if len(os.sched_getaffinity(0)) < cores:
        pytest.skip("fewer cores here")
    run(r"""
  cpu_set_t all, some;
  sched_getaffinity(0, sizeof(all), &all);
  CPU_ZERO(&some);
  for (int i = 0, n = 0; i < CPU_SETSIZE && n < %d; ++i)
    if (CPU_ISSET(i, &all)) CPU_SET(i, &some), ++n;
  sched_setaffinity(0, sizeof(some), &some);
  host_copy_acquire();
  fake::Stream s;
  round_trip(kRing + 100, 1, 0, &s);
  EXPECT(threads_now() == 1 + 1 + std::min(3, %d - 1));  // main, the stream, the helpers
  host_copy_release();
  EXPECT(threads_now() == 2);""" % (cores, cores))
