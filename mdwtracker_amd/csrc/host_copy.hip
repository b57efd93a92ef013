// See host_copy.hpp. A lane is a pinned ring of kSlots chunks, an event per slot
// and up to kWorkers threads; a call takes a free lane of its device (or makes one, up
// to kMaxLanes per device; past that, or where pinned memory is not to be had, it copies
// as the runtime does), so calls of several threads, handles and streams run
// side by side and share nothing but the list of free lanes.
#include "host_copy.hpp"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace mdwt {
namespace {

// Bytes of a ring slot. A chunk costs about 5 us beside its transfer, so small
// ones are slow (a 1024^2 denoiser inference: 2.58 / 2.30 / 2.00 ms at 512 KiB / 1 /
// 2 MiB), and large ones overlap less (a 4 MiB frame buffer: 308 against 312 us
// at 1 / 2 MiB).
constexpr size_t kChunk = size_t(2) << 20;
constexpr int kSlots = 8;                     // 16 MiB per lane
constexpr size_t kPiece = size_t(256) << 10;  // bytes a thread copies at a time
constexpr int kWorkers = 3;                   // beside the calling thread, at most
constexpr size_t kMaxLanes = 4;               // per device
// below this, waking the workers costs more than they save
constexpr size_t kMinBytes = size_t(512) << 10;

// 16-byte words of a chunk, then its last bytes. One side is pinned host memory,
// read or written over the link: a copy engine's transfer costs about 25 us
// beside the bytes, a launch about 5 (the inference above: 2.17 against 2.00 ms).
__global__ __launch_bounds__(256) void move_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                   uint32_t bytes) {
  const uint32_t n = bytes / 16u, step = gridDim.x * 256u;
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += step)
    reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
  const uint32_t t = n * 16u + threadIdx.x;
  if (blockIdx.x == 0 && t < bytes) dst[t] = src[t];
}

class Lane {
 public:
  static std::unique_ptr<Lane> make(int device) {
    std::unique_ptr<Lane> l(new (std::nothrow) Lane(device));
    if (!l) return nullptr;
    // Kernels and host threads take turns on a slot: coherent memory, so that
    // each sees the other's writes whatever the runtime's default, and events that
    // release to the system, since a host thread reads what lies before one.
    if (hipHostMalloc(reinterpret_cast<void**>(&l->ring_), kChunk * kSlots,
                      hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
      l->ring_ = nullptr;
      (void)hipGetLastError();
      return nullptr;
    }
    for (auto& e : l->ev_)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventReleaseToSystem) != hipSuccess) {
        e = nullptr;
        (void)hipGetLastError();
        return nullptr;
      }
    // a thread per core that this process may use: with fewer cores than threads
    // the copies would take them from each other while they wait for transfers
    cpu_set_t cores;
    const int n = sched_getaffinity(0, sizeof(cores), &cores) == 0 ? CPU_COUNT(&cores) : kWorkers + 1;
    const int workers = std::min(kWorkers, n - 1);
    try {
      for (int i = 0; i < workers; ++i) l->threads_.emplace_back([p = l.get()] { p->worker(); });
    } catch (const std::system_error&) {
      // fewer workers: the calling thread does the rest
    } catch (const std::bad_alloc&) {
    }
    return l;
  }
  ~Lane() {
    {
      std::lock_guard<std::mutex> lock(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (auto& t : threads_) t.join();
    int current = device_;
    (void)hipGetDevice(&current);
    (void)hipSetDevice(device_);
    for (auto& e : ev_)
      if (e) {
        (void)hipEventSynchronize(e);  // a slot may still be on its way to the device
        (void)hipEventDestroy(e);
      }
    if (ring_) (void)hipHostFree(ring_);
    (void)hipSetDevice(current);
  }
  int device() const { return device_; }

  // One copy; the caller owns the lane meanwhile.
  hipError_t run(bool to_host, uint8_t* host, uint8_t* dev, size_t bytes, hipStream_t s) {
    to_host_ = to_host;
    host_ = host;
    dev_ = dev;
    bytes_ = bytes;
    stream_ = s;
    chunks_ = (bytes + kChunk - 1) / kChunk;
    pieces_ = (bytes + kPiece - 1) / kPiece;
    next_.store(0);
    error_.store(hipSuccess);
    for (int i = 0; i < kSlots; ++i) {
      // a slot of the previous copy may still be read by its transfer
      if (used_[i]) {
        const hipError_t e = hipEventSynchronize(ev_[i]);
        if (e != hipSuccess) return e;
      }
      used_[i] = false;
      issued_[i].store(0);
      left_[i].store(pieces_of(size_t(i)));
    }
    if (to_host)
      for (size_t c = 0; c < chunks_ && c < size_t(kSlots); ++c) issue(c);
    if (error_.load() == hipSuccess) {
      {
        std::lock_guard<std::mutex> lock(mu_);
        busy_ = int(threads_.size());
        ++job_;
      }
      cv_.notify_all();
      chunk_loop();
      std::unique_lock<std::mutex> lock(mu_);
      done_.wait(lock, [&] { return busy_ == 0; });
    }
    return hipError_t(error_.load());
  }

 private:
  explicit Lane(int device) : device_(device) {}

  size_t size(size_t c) const { return c + 1 < chunks_ ? kChunk : bytes_ - c * kChunk; }
  int pieces_of(size_t c) const { return c < chunks_ ? int((size(c) + kPiece - 1) / kPiece) : 0; }
  void fail(hipError_t e) {
    int none = hipSuccess;
    error_.compare_exchange_strong(none, int(e));
  }
  // the transfer of chunk c and the event behind it; marks the slot as chunk c's
  void issue(size_t c) {
    const size_t k = c % kSlots;
    uint8_t *slot = ring_ + k * kChunk, *dev = dev_ + c * kChunk;
    const uint8_t* src = to_host_ ? dev : slot;
    uint8_t* dst = to_host_ ? slot : dev;
    uint32_t n = uint32_t(size(c));
    void* args[] = {&src, &dst, &n};
    // the launch's own status: hipGetLastError would give the error of any
    // earlier call of this thread, and the copy would fail with it
    hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(move_kernel), dim3(256), dim3(256), args, 0,
                                   stream_);
    if (e == hipSuccess) e = hipEventRecord(ev_[k], stream_);
    if (e != hipSuccess) fail(e);
    used_[k] = true;
    issued_[k].store(c + 1, std::memory_order_release);
  }
  // waits until chunk c's transfer was issued (by the thread that took chunk c -
  // kSlots, or by run) and is done
  void await(size_t c) {
    const size_t k = c % kSlots;
    while (issued_[k].load(std::memory_order_acquire) != c + 1) {
      if (error_.load() != hipSuccess) return;
      std::this_thread::yield();
    }
    const hipError_t e = hipEventSynchronize(ev_[k]);
    if (e != hipSuccess) fail(e);
  }
  // Pieces are taken in order, so the chunk that a thread waits for is always
  // another thread's own or done; after an error nobody waits. The thread that
  // finishes a chunk's last piece passes it on.
  void chunk_loop() {
    while (error_.load() == hipSuccess) {
      const size_t p = next_.fetch_add(1);
      if (p >= pieces_) return;
      const size_t c = p * kPiece / kChunk, k = c % kSlots, at = p * kPiece;
      const size_t n = std::min(kPiece, bytes_ - at);
      uint8_t* slot = ring_ + k * kChunk + (at - c * kChunk);
      if (to_host_)
        await(c);
      else if (c >= size_t(kSlots))
        await(c - kSlots);
      if (error_.load() != hipSuccess) return;
      if (to_host_)
        std::memcpy(host_ + at, slot, n);
      else
        std::memcpy(slot, host_ + at, n);
      if (left_[k].fetch_sub(1) == 1) {
        left_[k].store(pieces_of(c + kSlots));
        if (!to_host_)
          issue(c);
        else if (c + kSlots < chunks_)
          issue(c + kSlots);
      }
    }
  }
  void worker() {
    uint64_t seen = 0;
    while (true) {
      {
        std::unique_lock<std::mutex> lock(mu_);
        cv_.wait(lock, [&] { return stop_ || job_ != seen; });
        if (stop_) return;
        seen = job_;
      }
      const hipError_t e = hipSetDevice(device_);
      if (e != hipSuccess) fail(e);
      chunk_loop();
      std::lock_guard<std::mutex> lock(mu_);
      if (--busy_ == 0) done_.notify_one();
    }
  }

  const int device_;
  uint8_t* ring_ = nullptr;
  hipEvent_t ev_[kSlots] = {};
  bool used_[kSlots] = {};
  std::atomic<size_t> issued_[kSlots] = {};
  std::atomic<int> left_[kSlots] = {};  // pieces of the slot's chunk still to be copied
  std::vector<std::thread> threads_;
  std::mutex mu_;
  std::condition_variable cv_, done_;
  uint64_t job_ = 0;
  int busy_ = 0;
  bool stop_ = false;
  // the copy being done
  bool to_host_ = false;
  uint8_t *host_ = nullptr, *dev_ = nullptr;
  size_t bytes_ = 0, chunks_ = 0, pieces_ = 0;
  hipStream_t stream_ = nullptr;
  std::atomic<size_t> next_{0};
  std::atomic<int> error_{hipSuccess};
};

// Never destroyed: threads must not be joined while the process is going down.
struct Pool {
  std::mutex mu;
  int handles = 0;
  std::vector<size_t> lanes;  // by device: made, free or in use
  std::vector<std::unique_ptr<Lane>> free;
};
Pool& pool() {
  static Pool* p = new Pool();
  return *p;
}

std::unique_ptr<Lane> take(int device) {
  Pool& p = pool();
  {
    std::lock_guard<std::mutex> lock(p.mu);
    for (auto& l : p.free)
      if (l->device() == device) {
        std::unique_ptr<Lane> got = std::move(l);
        l = std::move(p.free.back());
        p.free.pop_back();
        return got;
      }
    try {
      if (p.lanes.size() <= size_t(device)) p.lanes.resize(size_t(device) + 1, 0);
    } catch (const std::bad_alloc&) {
      return nullptr;
    }
    if (p.lanes[size_t(device)] >= kMaxLanes) return nullptr;
    ++p.lanes[size_t(device)];
  }
  std::unique_ptr<Lane> l = Lane::make(device);
  if (!l) {
    std::lock_guard<std::mutex> lock(p.mu);
    --p.lanes[size_t(device)];
  }
  return l;
}
void give(std::unique_ptr<Lane> l) {
  Pool& p = pool();
  std::lock_guard<std::mutex> lock(p.mu);
  const size_t device = size_t(l->device());
  try {
    p.free.push_back(std::move(l));
  } catch (const std::bad_alloc&) {
    --p.lanes[device];
  }
}

hipError_t copy(bool to_host, void* host, void* dev, size_t bytes, int device, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  if (bytes >= kMinBytes) {
    if (std::unique_ptr<Lane> l = take(device)) {
      const hipError_t e = l->run(to_host, static_cast<uint8_t*>(host), static_cast<uint8_t*>(dev), bytes, s);
      give(std::move(l));
      return e;
    }
  }
  if (!to_host) return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
  const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

}  // namespace

void host_copy_acquire() {
  Pool& p = pool();
  std::lock_guard<std::mutex> lock(p.mu);
  ++p.handles;
}

void host_copy_release() {
  Pool& p = pool();
  std::vector<std::unique_ptr<Lane>> gone;
  {
    std::lock_guard<std::mutex> lock(p.mu);
    if (--p.handles > 0) return;
    gone.swap(p.free);
    for (const auto& l : gone) --p.lanes[size_t(l->device())];
  }
}

hipError_t copy_to_host(void* dst, const void* src, size_t bytes, int device, hipStream_t s) {
  return copy(true, dst, const_cast<void*>(src), bytes, device, s);
}
hipError_t copy_to_device(void* dst, const void* src, size_t bytes, int device, hipStream_t s) {
  return copy(false, const_cast<void*>(src), dst, bytes, device, s);
}

}  // namespace mdwt
