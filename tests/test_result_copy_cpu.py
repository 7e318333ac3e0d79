"""The buffers and helper threads that bring results to the host
(openlb_amd/csrc/result_copy.hpp), compiled with g++ against stand-ins for the
HIP calls they make: device memory is host memory of a set size, and a call that
waits for the null stream waits out its backlog, busily, as the runtime does."""
import os
import subprocess


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEAD = r"""
#include <sys/resource.h>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <thread>
#include <vector>
#include "result_copy.hpp"

namespace lbmh { thread_local std::string g_error; }
using namespace lbmh;

static int bad = 0;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); ++bad; } } while (0)

// the stand-in device
static std::mutex fake;
static std::map<void*, size_t> device_blocks, host_blocks;
static size_t device_limit = size_t(1) << 40, device_used = 0;
static std::vector<unsigned> host_flags;             // of every hipHostMalloc
static std::vector<std::pair<void*, size_t>> copies;  // destination and size of every transfer
static std::atomic<int64_t> drained_at{0};            // ns of the steady clock
static std::map<void*, size_t> registered;            // host memory the runtime knows

static int64_t now() { return std::chrono::steady_clock::now().time_since_epoch().count(); }

static void drain()
{
  while (now() < drained_at) {
  }
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
  std::lock_guard<std::mutex> l(fake);
  if (device_used + n > device_limit) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  device_blocks[*p] = n;
  device_used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p)
{
  std::lock_guard<std::mutex> l(fake);
  device_used -= device_blocks.at(p);
  device_blocks.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags)
{
  std::lock_guard<std::mutex> l(fake);
  *p = std::malloc(n);
  host_blocks[*p] = n;
  host_flags.push_back(flags);
  return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
  std::lock_guard<std::mutex> l(fake);
  host_blocks.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind)
{
  drain();
  std::memcpy(to, from, n);
  std::lock_guard<std::mutex> l(fake);
  copies.push_back({to, n});
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
  drain();
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
  std::memset(a, 0, sizeof(*a));
  a->type = hipMemoryTypeUnregistered;
  for (auto& r : registered)
    if (p >= r.first && p < static_cast<char*>(r.first) + r.second) a->type = hipMemoryTypeHost;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
}

// One result of `n` bytes into `host`, as an export brings it there.
static int bring(std::vector<unsigned char>& host, size_t n)
{
  host.assign(n, 0xee);
  ResultBuffer out;
  const int rc = out.allocate(0, n);
  if (rc != LBMH_OK) return rc;
  for (size_t k = 0; k < n; k += 1009) static_cast<unsigned char*>(out.p)[k] = static_cast<unsigned char>(k >> 8);
  const int rt = out.to_host(host.data(), n);
  for (size_t k = 0; k < n; k += 1009) CHECK(host[k] == static_cast<unsigned char>(k >> 8));
  return rt;
}

static size_t threads()
{
  FILE* f = std::fopen("/proc/self/status", "r");
  char line[256];
  size_t n = 0;
  while (std::fgets(line, sizeof line, f)) std::sscanf(line, "Threads: %zu", &n);
  std::fclose(f);
  return n;
}
"""

# one lattice after another, each read a few times: nothing is set up again
LIFETIME = r"""
int main() {
  ResultPool& pool = ResultPool::get();
  std::vector<unsigned char> host;
  size_t made = 0, alive = 0;
  for (int k = 0; k < 8; ++k) {
    pool.retain();
    for (size_t n : {size_t(100) << 10, size_t(3) << 20, size_t(30) << 20}) {
      CHECK(bring(host, n) == LBMH_OK);
      CHECK(device_used >= n && device_used < 2 * n);  // a small result keeps a small workspace
    }
    pool.release();
    CHECK(device_used == 0);  // the workspace goes with the last lattice
    if (k == 0) { made = host_flags.size(); alive = threads(); }
    CHECK(host_flags.size() == made && threads() == alive);
  }
  size_t held = 0;
  for (auto& b : host_blocks) held += b.second;
  CHECK(held <= (size_t(12) << 20) + 4096 && alive <= 6);  // bounded
  pool.give_back();
  CHECK(host_blocks.empty() && device_used == 0 && threads() == 1);
  pool.retain();
  CHECK(bring(host, size_t(3) << 20) == LBMH_OK);  // and set up again when needed
  pool.give_back();  // a lattice is still alive
  CHECK(host_blocks.empty() && device_used == 0);
  CHECK(bring(host, size_t(3) << 20) == LBMH_OK);
  pool.release();
"""

# what a kernel writes while the host polls lies in coherent memory of its own
READING = r"""
int main() {
  ResultPool& pool = ResultPool::get();
  pool.retain();
  uint64_t last = 0;
  void* at = nullptr;
  {
    ResultBuffer b;
    at = b.reading();
    CHECK(at && host_flags.size() == 1 && (host_flags[0] & hipHostMallocCoherent) && host_blocks[at] <= 4096);
    for (size_t k = 0; k < kReadingBytes; ++k) CHECK(static_cast<char*>(at)[k] == 0);
    last = b.next_number();
    CHECK(last > 0);
    ResultBuffer other;  // no lease: no memory and no number to wait for
    CHECK(!other.reading() && other.next_number() == 0);
  }
  std::vector<unsigned char> host;
  CHECK(bring(host, size_t(20) << 20) == LBMH_OK);
  ResultBuffer b;
  CHECK(b.reading() == at && b.next_number() > last);
  for (size_t k = 0; k < kReadingBytes; ++k) CHECK(static_cast<char*>(at)[k] == 0);  // untouched by exports
"""

# one thread waits for the work queued before a result, whatever the size
BACKLOG = r"""
static double cpu_ms()
{
  rusage u;
  getrusage(RUSAGE_SELF, &u);
  return (u.ru_utime.tv_sec + u.ru_stime.tv_sec) * 1e3 + (u.ru_utime.tv_usec + u.ru_stime.tv_usec) * 1e-3;
}
int main() {
  ResultPool::get().retain();
  for (size_t n : {size_t(100) << 10, size_t(3) << 20, size_t(12) << 20, size_t(30) << 20}) {
    std::vector<unsigned char> host;
    CHECK(bring(host, n) == LBMH_OK);  // sets up
    const double idle = cpu_ms();
    CHECK(bring(host, n) == LBMH_OK);
    const double alone = cpu_ms() - idle;
    constexpr int kWait = 400;
    drained_at = now() + int64_t(kWait) * 1000000;
    const double before = cpu_ms();
    CHECK(bring(host, n) == LBMH_OK);
    const double used = cpu_ms() - before;
    std::printf("%zu bytes: %.0f ms of CPU time behind %d ms, %.0f ms alone\n", n, used, kWait, alone);
    // the caller's wait, the copy itself, and half a wait to spare
    CHECK(used < 1.5 * kWait + alone);
  }
"""

# below kCopyHelped no helper is started or woken
SMALL = r"""
int main() {
  ResultPool::get().retain();
  std::vector<unsigned char> host;
  for (size_t n : {size_t(2000), kCopyDirect, kCopyDirect + 1, size_t(300) << 10, kCopyHelped - 1}) CHECK(bring(host, n) == LBMH_OK);
  CHECK(threads() == 1);
  CHECK(bring(host, kCopyHelped) == LBMH_OK && threads() == 6);
"""

# a destination the runtime knows takes one transfer, straight into it
PINNED = r"""
int main() {
  ResultPool::get().retain();
  for (size_t n : {size_t(100) << 10, size_t(3) << 20, size_t(30) << 20}) {
    std::vector<unsigned char> host(n);
    registered[host.data()] = n;
    copies.clear();
    CHECK(bring(host, n) == LBMH_OK);  // assign() keeps the allocation
    CHECK(copies.size() == 1 && copies[0].first == host.data() && copies[0].second == n);
    registered.clear();
  }
  CHECK(host_flags.empty() && threads() == 1);
"""

# a card with little room left refuses nothing for what earlier results left allocated
FULL = r"""
int main() {
  constexpr size_t MB = size_t(1) << 20;
  ResultPool::get().retain();
  std::vector<unsigned char> host;
  void* a = nullptr;
  void* b = nullptr;
  device_limit = 100 * MB;
  CHECK(device_alloc(&a, 97 * MB) == hipSuccess);
  CHECK(bring(host, 5 * MB / 2) == LBMH_OK);  // 4 MB would not fit
  CHECK(hipFree(a) == hipSuccess);
  CHECK(bring(host, 60 * MB) == LBMH_OK);
  CHECK(device_used == 64 * MB);
  CHECK(bring(host, 80 * MB) == LBMH_OK);     // needs the workspace's room
  CHECK(bring(host, 60 * MB) == LBMH_OK);
  CHECK(device_alloc(&a, 90 * MB) == hipSuccess && device_used == 90 * MB);
  CHECK(bring(host, 30 * MB) != LBMH_OK && device_alloc(&b, 30 * MB) == hipErrorOutOfMemory);
  CHECK(bring(host, 10 * MB) == LBMH_OK);
  {
    // another thread's export holds the lease: its workspace stays
    ResultBuffer out;
    CHECK(out.allocate(0, 8 * MB) == LBMH_OK);
    std::thread other([&] { CHECK(device_alloc(&b, 30 * MB) == hipErrorOutOfMemory); });
    other.join();
    CHECK(device_blocks.count(out.p));
  }
"""

TAIL = r"""
  std::printf("bad %d\n", bad);
  std::fflush(stdout);
  std::_Exit(bad != 0);
}
"""


def run(body, tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(HEAD + body + TAIL)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                    f"-I{os.path.join(ROOT, 'include')}", f"-I{os.path.join(ROOT, 'openlb_amd', 'csrc')}",
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr


def test_buffers_outlive_the_last_lattice(tmp_path):
    """A program with one lattice at a time sets the pinned buffer and the
    helper threads up once; the device workspace goes with the last lattice, and
    lbmh_release_buffers gives everything back."""
    run(LIFETIME, tmp_path)


def test_readings_are_polled_in_coherent_memory(tmp_path):
    """lbmh_statistics' result and number: a small coherent allocation, no part of the export buffer."""
    run(READING, tmp_path)


def test_one_thread_waits_for_the_queued_steps(tmp_path):
    """A result behind a long backlog takes one thread's CPU time, not every helper's."""
    run(BACKLOG, tmp_path)


def test_small_results_wake_no_helpers(tmp_path):
    run(SMALL, tmp_path)


def test_pinned_destinations_take_one_transfer(tmp_path):
    run(PINNED, tmp_path)


def test_kept_workspace_refuses_no_later_call(tmp_path):
    run(FULL, tmp_path)
