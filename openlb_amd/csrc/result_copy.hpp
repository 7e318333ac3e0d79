// Results on their way to the host (host code).
//
// An export evaluates a field into device memory and copies it to the caller's
// pageable buffer.  Handed that buffer, hipMemcpy moved 10 GB/s (275 MB of
// density and velocity of a 256^3 block: 27.6 ms): one thread copies out of the
// runtime's staging memory and takes the page faults of a fresh array, 8-13 GB/s
// where the link gives 52 GB/s.  Here helper threads copy chunks through a
// pinned buffer, so that transfers, host copies and page faults overlap: 8.3 ms
// into memory the program has used before with the HIP runtime that torch
// brings, 14.9 ms with ROCm 7.2's own (hipMemcpy alone 17.6 and 22.5).  Smaller
// results take one transfer, during which the helpers touch the caller's pages,
// and a workspace that stays allocated.
//
// A reading of a few words (lbmh_statistics) has pinned memory of its own, which
// a running kernel writes and the host polls.
//
// One pinned buffer (12 MB), one device workspace (up to 64 MB) and five idle
// helper threads per process serve whoever holds the lease; a second thread
// exporting at the same time allocates and copies for itself.  The workspace
// goes with the last lattice or ensemble; it grows by doubling, as an
// allocation of a few hundred KB takes 1 us and one of 4 MB 13.  The pinned
// buffer and the threads outlive it: a program that makes one lattice after
// another and reads FP64 moments of each paid for them every time (48^3 cells
// 1040 us and 135 us at the destruction, now 167 and 35; 24^3 159 and 89, now
// 66 and 4).  lbmh_release_buffers gives them back.
#pragma once

#include <hip/hip_runtime.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "lbmh_common.hpp"

namespace lbmh {

constexpr size_t kCopyChunk = size_t(2) << 20;     // bytes of one transfer
constexpr int kCopyThreads = 6;                    // slots; the caller and its helpers
constexpr size_t kCopyDirect = size_t(64) << 10;   // up to here hipMemcpy's own path is as fast
// From here on the helpers pay for their wake-up: 432 KB into memory in use take
// 42 us without and 54 with them, 549 KB 49 and 53, 1 MB 79 and 68; the velocities
// of a split cavity's eight pieces, 890 KB each, 980 and 870 us.
constexpr size_t kCopyHelped = size_t(448) << 10;
constexpr size_t kWorkspaceLimit = size_t(64) << 20;
constexpr size_t kReadingBytes = 128;  // the values, and from byte 64 on the reading's number

// Threads that run one job together with the caller.  Used under the lease.
class CopyHelpers {
 public:
  // job(slot) for slot 0 on this thread and the others on the helpers that
  // could be started; returns when all are done.
  void run(const std::function<void(int)>& job)
  {
    if (threads_.empty()) pid_ = getpid();
    try {
      while (int(threads_.size()) < kCopyThreads - 1) {
        const int slot = int(threads_.size()) + 1;
        threads_.emplace_back([this, slot, round = round_] { serve(slot, round); });
      }
    } catch (const std::exception&) {
      // fewer helpers
    }
    {
      std::lock_guard<std::mutex> l(mutex_);
      job_ = &job;
      pending_ = int(threads_.size());
      ++round_;
    }
    wake_.notify_all();
    job(0);
    std::unique_lock<std::mutex> l(mutex_);
    done_.wait(l, [this] { return pending_ == 0; });
    job_ = nullptr;
  }

  void stop()
  {
    {
      std::lock_guard<std::mutex> l(mutex_);
      quit_ = true;
    }
    wake_.notify_all();
    // in a forked child the helpers do not exist
    for (std::thread& t : threads_) {
      if (pid_ == getpid()) t.join();
      else t.detach();
    }
    threads_.clear();
    quit_ = false;
  }

 private:
  void serve(int slot, uint64_t seen)
  {
    std::unique_lock<std::mutex> l(mutex_);
    for (;;) {
      wake_.wait(l, [&] { return quit_ || round_ != seen; });
      if (quit_) return;
      seen = round_;
      const std::function<void(int)>* job = job_;
      l.unlock();
      (*job)(slot);
      l.lock();
      if (--pending_ == 0) done_.notify_one();
    }
  }

  std::mutex mutex_;
  std::condition_variable wake_, done_;
  std::vector<std::thread> threads_;
  const std::function<void(int)>* job_ = nullptr;
  uint64_t round_ = 0;
  int pending_ = 0;
  bool quit_ = false;
  pid_t pid_ = 0;
};

// What the helpers wait for while the steps queued before a result run: they
// spin for a few ms and then sleep.  Waking them takes 25 to 200 us of the
// caller's time, so only waits it does not show in are slept through (48^3 D3Q27,
// 300 steps and FP64 moments: 2357 us, with a spin of 200 us 2385).  An event
// before the result's kernel, to wake them in time, took 5 to 10 us itself.
class Gate {
 public:
  void set(bool good)
  {
    {
      std::lock_guard<std::mutex> l(mutex_);
      state_ = good ? 1 : -1;
    }
    changed_.notify_all();
  }

  bool decided() const { return state_ != 0; }

  bool wait()
  {
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(5);
    while (!decided() && std::chrono::steady_clock::now() < until) std::this_thread::yield();
    if (!decided()) {
      std::unique_lock<std::mutex> l(mutex_);
      changed_.wait(l, [this] { return decided(); });
    }
    return state_ > 0;
  }

 private:
  std::mutex mutex_;
  std::condition_variable changed_;
  std::atomic<int> state_{0};
};

// The pages of n bytes of the caller's memory, which the result overwrites.
inline void touch(char* at, size_t n)
{
  constexpr size_t kPage = 4096;
  for (size_t k = 0; k < n; k += kPage) const_cast<volatile char*>(at)[k] = 0;
}

struct ResultPool {
  std::mutex lease;        // held while an export uses the buffers
  std::mutex count_mutex;
  int users = 0;           // lattices and ensembles alive
  void* pinned = nullptr;
  void* device = nullptr;
  size_t device_bytes = 0;
  int ordinal = -1;        // device the workspace lies on
  void* reading = nullptr; // pinned and coherent, kReadingBytes
  uint64_t number = 0;     // under the lease: readings so far
  CopyHelpers helpers;

  static ResultPool& get()
  {
    // never destroyed: helpers that wait when the process exits are left to it
    static ResultPool& pool = *new ResultPool;
    return pool;
  }

  void retain()
  {
    std::lock_guard<std::mutex> c(count_mutex);
    ++users;
  }

  void release()
  {
    std::lock_guard<std::mutex> c(count_mutex);
    if (--users > 0) return;
    std::lock_guard<std::mutex> l(lease);
    drop_workspace();
  }

  // Everything the pool holds; the next export sets up again what it needs.
  void give_back()
  {
    std::lock_guard<std::mutex> l(lease);
    helpers.stop();
    if (pinned) (void)hipHostFree(pinned);
    pinned = nullptr;
    if (reading) (void)hipHostFree(reading);
    reading = nullptr;
    drop_workspace();
  }

  void drop_workspace()
  {
    if (!device) return;
    DeviceGuard guard(ordinal);
    (void)hipFree(device);
    device = nullptr;
    device_bytes = 0;
    ordinal = -1;
  }
};

// hipMalloc that gives the idle workspace back where the card has no room
// otherwise: what an export leaves allocated refuses no later call.
inline hipError_t device_alloc(void** p, size_t bytes)
{
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  ResultPool& pool = ResultPool::get();
  std::unique_lock<std::mutex> l(pool.lease, std::try_to_lock);
  if (!l.owns_lock() || !pool.device) return e;
  (void)hipGetLastError();
  pool.drop_workspace();
  return hipMalloc(p, bytes);
}

// Device memory for one export, and its way to the host.
class ResultBuffer {
 public:
  ResultBuffer() : lock_(ResultPool::get().lease, std::try_to_lock) {}
  ~ResultBuffer()
  {
    if (own_) (void)hipFree(own_);
  }
  ResultBuffer(const ResultBuffer&) = delete;
  ResultBuffer& operator=(const ResultBuffer&) = delete;

  // `bytes` on the current device `ordinal`
  int allocate(int ordinal, size_t bytes)
  {
    ordinal_ = ordinal;
    ResultPool& pool = ResultPool::get();
    if (lock_.owns_lock() && bytes <= kWorkspaceLimit) {
      if (pool.ordinal != ordinal || pool.device_bytes < bytes) {
        pool.drop_workspace();
        size_t size = kCopyDirect;  // doubled up to what is needed
        while (size < bytes) size *= 2;
        void* fresh = nullptr;
        hipError_t e = hipMalloc(&fresh, size);
        if (e == hipErrorOutOfMemory && size > bytes) {  // a full card: no more than needed
          (void)hipGetLastError();
          size = bytes;
          e = hipMalloc(&fresh, size);
        }
        if (e != hipSuccess) return hip_fail(e, "hipMalloc");
        pool.device = fresh;
        pool.device_bytes = size;
        pool.ordinal = ordinal;
      }
      p = pool.device;
      return LBMH_OK;
    }
    hipError_t e = hipMalloc(&own_, bytes);
    if (e == hipErrorOutOfMemory && lock_.owns_lock() && pool.device) {
      (void)hipGetLastError();
      pool.drop_workspace();
      e = hipMalloc(&own_, bytes);
    }
    if (e != hipSuccess) return hip_fail(e, "hipMalloc");
    p = own_;
    return LBMH_OK;
  }

  // Memory for a reading that the host takes while the kernel runs, or null
  // without the lease.  Such a poll needs coherent memory: without the flag an
  // allocation follows the environment (HIP_HOST_COHERENT).
  void* reading()
  {
    ResultPool& pool = ResultPool::get();
    if (!lock_.owns_lock()) return nullptr;
    if (!pool.reading) {
      if (hipHostMalloc(&pool.reading, kReadingBytes, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
        pool.reading = nullptr;
        (void)hipGetLastError();
        return nullptr;
      }
      std::memset(pool.reading, 0, kReadingBytes);
    }
    return pool.reading;
  }

  // The pinned buffer, or null without the lease.
  void* pinned()
  {
    ResultPool& pool = ResultPool::get();
    if (!lock_.owns_lock()) return nullptr;
    if (!pool.pinned && hipHostMalloc(&pool.pinned, kCopyChunk * kCopyThreads, hipHostMallocPortable) != hipSuccess) {
      pool.pinned = nullptr;
      (void)hipGetLastError();
    }
    return pool.pinned;
  }

  // A number no earlier holder of the lease was given.
  uint64_t next_number() { return lock_.owns_lock() ? ++ResultPool::get().number : 0; }

  // The first `bytes` to host memory, after the null stream's work.  Memory that
  // the runtime has pinned or allocated takes them straight from the link (45 MB
  // in 0.87 ms; through the pinned buffer 1.06 ms).
  int to_host(void* host, size_t bytes)
  {
    ResultPool& pool = ResultPool::get();
    if (bytes <= kCopyDirect || known_to_runtime(host) || !pinned()) {
      LBMH_HIP(hipMemcpy(host, p, bytes, hipMemcpyDeviceToHost));
      return LBMH_OK;
    }
    char* const to = static_cast<char*>(host);
    std::atomic<int> error{hipSuccess};
    if (bytes <= kCopyChunk * kCopyThreads) {
      // one transfer; meanwhile the helpers touch their part of the caller's
      // pages, and copy it when the transfer is done
      char* const stage = static_cast<char*>(pool.pinned);
      if (bytes < kCopyHelped) {
        // (hipMemcpyAsync, the pages touched meanwhile and a wait for the stream:
        // 15 us more for 166 KB with the runtime that torch brings)
        LBMH_HIP(hipMemcpy(stage, p, bytes, hipMemcpyDeviceToHost));
        std::memcpy(to, stage, bytes);
        return LBMH_OK;
      }
      Gate arrived;  // the transfer's data
      constexpr size_t kPage = 4096;
      const size_t part = (bytes / kCopyThreads + kPage) / kPage * kPage;
      std::atomic<size_t> next{0};
      pool.helpers.run([&](int slot) {
        if (slot == 0) {
          const hipError_t e = hipMemcpy(stage, p, bytes, hipMemcpyDeviceToHost);
          if (e != hipSuccess) error = e;
          arrived.set(e == hipSuccess);
        }
        for (;;) {
          const size_t at = next.fetch_add(part);
          if (at >= bytes) return;
          const size_t n = std::min(part, bytes - at);
          if (!arrived.decided()) touch(to + at, n);
          if (!arrived.wait()) return;
          std::memcpy(to + at, stage + at, n);
        }
      });
    } else {
      // a transfer waits in a busy loop for the work queued before it: one thread
      // does, while the others touch the pages of their first chunk
      Gate drained;
      std::atomic<size_t> next{0};
      pool.helpers.run([&](int slot) {
        if (slot == 0) {
          const hipError_t e = hipStreamSynchronize(nullptr);
          if (e != hipSuccess) error = e;
          drained.set(e == hipSuccess);
        }
        const hipError_t d = hipSetDevice(ordinal_);
        if (d != hipSuccess) error = d;
        char* const stage = static_cast<char*>(pool.pinned) + size_t(slot) * kCopyChunk;
        while (error == hipSuccess) {
          const size_t at = next.fetch_add(kCopyChunk);
          if (at >= bytes) return;
          const size_t n = std::min(kCopyChunk, bytes - at);
          if (!drained.decided()) touch(to + at, n);
          if (!drained.wait()) return;
          const hipError_t e = hipMemcpy(stage, static_cast<const char*>(p) + at, n, hipMemcpyDeviceToHost);
          if (e != hipSuccess) error = e;
          else std::memcpy(to + at, stage, n);
        }
      });
    }
    if (error != hipSuccess) return hip_fail(static_cast<hipError_t>(error.load()), "hipMemcpy(device to host)");
    return LBMH_OK;
  }

  void* p = nullptr;

 private:
  static bool known_to_runtime(const void* host)
  {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();  // pageable memory, to some versions
    return false;
  }

  std::unique_lock<std::mutex> lock_;
  void* own_ = nullptr;
  int ordinal_ = 0;
};

}  // namespace lbmh
