// Results on their way to the host (host code).
//
// An export evaluates a field into device memory and copies it to the caller's
// pageable buffer.  Handed that buffer, hipMemcpy moved 10 GB/s (275 MB of
// density and velocity of a 256^3 block: 27.6 ms): one thread copies out of the
// runtime's staging memory and takes the page faults of a fresh array, 13 GB/s
// where the link gives 52 GB/s.  Here several threads each copy one chunk to
// their slot of a pinned buffer and on to the caller's, so that transfers and
// host copies overlap.  Small exports (the 96 members of a study, 1 MB each)
// cost a hipMalloc and a hipFree more than the copy: 230 us each.
//
// One pinned buffer (12 MB) and one device workspace (up to 64 MB) per process
// serve whoever holds the lease; a second thread exporting at the same time
// allocates for itself.  They are freed with the last lattice or ensemble.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "lbmh_common.hpp"

namespace lbmh {

constexpr size_t kCopyChunk = size_t(2) << 20;     // bytes of one transfer
constexpr int kCopyThreads = 6;                    // slots, and threads of a large copy
constexpr size_t kCopyDirect = size_t(64) << 10;   // up to here hipMemcpy's own path is as fast
constexpr size_t kWorkspaceLimit = size_t(64) << 20;

struct ResultPool {
  std::mutex lease;        // held while an export uses the buffers
  std::mutex count_mutex;
  int users = 0;           // lattices and ensembles alive
  void* pinned = nullptr;
  void* device = nullptr;
  size_t device_bytes = 0;
  int ordinal = -1;        // device the workspace lies on

  static ResultPool& get()
  {
    static ResultPool pool;
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
    if (pinned) (void)hipHostFree(pinned);
    drop_workspace();
    pinned = nullptr;
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
        const size_t size = std::min(kWorkspaceLimit, std::max(bytes, size_t(4) << 20));
        void* fresh = nullptr;
        LBMH_HIP(hipMalloc(&fresh, size));
        pool.device = fresh;
        pool.device_bytes = size;
        pool.ordinal = ordinal;
      }
      p = pool.device;
      return LBMH_OK;
    }
    LBMH_HIP(hipMalloc(&own_, bytes));
    p = own_;
    return LBMH_OK;
  }

  // The first `bytes` to pageable host memory, after the null stream's work.
  int to_host(void* host, size_t bytes)
  {
    ResultPool& pool = ResultPool::get();
    if (bytes > kCopyDirect && lock_.owns_lock() && !pool.pinned) {
      if (hipHostMalloc(&pool.pinned, kCopyChunk * kCopyThreads, hipHostMallocPortable) != hipSuccess) {
        pool.pinned = nullptr;
        (void)hipGetLastError();
      }
    }
    if (bytes <= kCopyDirect || !lock_.owns_lock() || !pool.pinned) {
      LBMH_HIP(hipMemcpy(host, p, bytes, hipMemcpyDeviceToHost));
      return LBMH_OK;
    }
    std::atomic<size_t> next{0};
    std::atomic<int> error{hipSuccess};
    auto work = [&](int slot, bool set_device) {
      if (set_device) {
        const hipError_t e = hipSetDevice(ordinal_);
        if (e != hipSuccess) {
          error = e;
          return;
        }
      }
      char* stage = static_cast<char*>(pool.pinned) + size_t(slot) * kCopyChunk;
      while (error == hipSuccess) {
        const size_t at = next.fetch_add(kCopyChunk);
        if (at >= bytes) return;
        const size_t n = std::min(kCopyChunk, bytes - at);
        const hipError_t e = hipMemcpy(stage, static_cast<const char*>(p) + at, n, hipMemcpyDeviceToHost);
        if (e != hipSuccess) {
          error = e;
          return;
        }
        std::memcpy(static_cast<char*>(host) + at, stage, n);
      }
    };
    // a thread pays from two chunks each on
    const int threads = int(std::min<size_t>(kCopyThreads, bytes / (2 * kCopyChunk)));
    std::vector<std::thread> helpers;
    try {
      for (int t = 1; t < threads; ++t) helpers.emplace_back(work, t, true);
    } catch (const std::exception&) {
      // fewer helpers: the others, or this thread alone, take all chunks
    }
    work(0, false);
    for (std::thread& t : helpers) t.join();
    if (error != hipSuccess) return hip_fail(static_cast<hipError_t>(error.load()), "hipMemcpy(device to host)");
    return LBMH_OK;
  }

  void* p = nullptr;

 private:
  std::unique_lock<std::mutex> lock_;
  void* own_ = nullptr;
  int ordinal_ = 0;
};

}  // namespace lbmh
