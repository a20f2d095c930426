// device.cpp -- device set-up, stream, timers, errors and the device-memory
// helpers of the additive ABI.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <unordered_map>

#include "lsamd_internal.hpp"

namespace lsamd {
namespace {

std::mutex g_mutex;
bool g_device_ready = false;
bool g_device_failed = false;
hipStream_t g_stream = nullptr;
thread_local std::string g_last_error;

hipEvent_t g_ev_begin[kTimerCount] = {};
hipEvent_t g_ev_end[kTimerCount] = {};
bool g_ev_used[kTimerCount] = {};

} // namespace

void set_last_error(std::string const &msg) { g_last_error = msg; }

bool fail(std::string const &msg) {
  g_last_error = msg;
  return false;
}

bool ensure_device() {
  std::lock_guard<std::mutex> lock(g_mutex);
  if (g_device_ready) return true;
  if (g_device_failed) {
    g_last_error = "no usable gfx950 device";
    return false;
  }
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count == 0) {
    g_device_failed = true;
    g_last_error = "no HIP device visible";
    return false;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, 0) != hipSuccess) {
    g_device_failed = true;
    g_last_error = "hipGetDeviceProperties failed";
    return false;
  }
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    g_device_failed = true;
    g_last_error = std::string("device is ") + prop.gcnArchName + ", engine is built for gfx950";
    return false;
  }
  if (hipSetDevice(0) != hipSuccess || hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking) != hipSuccess) {
    g_device_failed = true;
    g_last_error = "stream creation failed";
    return false;
  }
  for (int i = 0; i < kTimerCount; ++i) {
    (void)hipEventCreate(&g_ev_begin[i]);
    (void)hipEventCreate(&g_ev_end[i]);
  }
  g_device_ready = true;
  return true;
}

hipStream_t stream() { return g_stream; }

void timer_begin(int family) {
  if (family < 0 || family >= kTimerCount || !g_device_ready) return;
  (void)hipEventRecord(g_ev_begin[family], g_stream);
}

void timer_end(int family) {
  if (family < 0 || family >= kTimerCount || !g_device_ready) return;
  (void)hipEventRecord(g_ev_end[family], g_stream);
  g_ev_used[family] = true;
}

// ---------------------------------------------------------------------------
// Block pool.  The driver clears the pages of freed device memory before it
// hands them out again, at about 35 GB/s: a program that builds one operator
// after another (38 GB of temporaries and results on the 6x6 lattice) waited
// 0.8 s per build for that, and a call on a small host batch spent most of
// its time in hipMalloc / hipFree.  A block is released only after the whole
// device has finished (as hipFree does), so whatever stream still used it is
// done when it is handed out again.
// ---------------------------------------------------------------------------
namespace {

struct BlockPool {
  std::mutex mutex;
  std::unordered_map<void *, size_t> live;
  struct Free {
    void *ptr;
    uint64_t stamp;
  };
  std::multimap<size_t, Free> free; // by size
  size_t cached = 0, capacity = 0;
  uint64_t clock = 0;

  // Called with the mutex held: down to `limit` cached bytes.
  void shrink(size_t limit) {
    while (cached > limit && !free.empty()) {
      auto oldest = free.begin();
      for (auto it = free.begin(); it != free.end(); ++it)
        if (it->second.stamp < oldest->second.stamp) oldest = it;
      (void)hipFree(oldest->second.ptr);
      cached -= oldest->first;
      free.erase(oldest);
    }
  }
};

// Never destroyed: arrays of static duration are released at process exit.
BlockPool &pool() {
  static BlockPool *const p = new BlockPool;
  return *p;
}

size_t block_size(size_t bytes) {
  size_t const unit = bytes < (size_t{1} << 20) ? 256 : (bytes < (size_t{64} << 20) ? size_t{64} << 10 : size_t{2} << 20);
  return (bytes + unit - 1) / unit * unit;
}

// LSAMD_POOL_BYTES, or a twelfth of the device's memory.
size_t pool_capacity() {
  if (char const *e = std::getenv("LSAMD_POOL_BYTES")) return static_cast<size_t>(std::strtoull(e, nullptr, 10));
  size_t free_b = 0, total_b = 0;
  (void)hipMemGetInfo(&free_b, &total_b);
  return total_b / 12;
}

} // namespace

void *pool_allocate(size_t bytes) {
  size_t const want = block_size(bytes);
  BlockPool &p = pool();
  std::lock_guard<std::mutex> lock(p.mutex);
  void *ptr = nullptr;
  auto const it = p.free.lower_bound(want);
  size_t size = want;
  if (it != p.free.end() && it->first - want <= want / 8) {
    ptr = it->second.ptr;
    size = it->first;
    p.cached -= size;
    p.free.erase(it);
  } else if (hipMalloc(&ptr, want) != hipSuccess) {
    (void)hipGetLastError();
    p.shrink(0);
    if (hipMalloc(&ptr, want) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
  }
  p.live[ptr] = size;
  return ptr;
}

void pool_release(void *ptr) {
  bool const idle = hipDeviceSynchronize() == hipSuccess;
  BlockPool &p = pool();
  std::lock_guard<std::mutex> lock(p.mutex);
  auto const it = p.live.find(ptr);
  size_t const size = it->second;
  p.live.erase(it);
  if (p.capacity == 0) p.capacity = std::max<size_t>(1, pool_capacity());
  if (!idle || size > p.capacity) {
    (void)hipFree(ptr);
    return;
  }
  p.free.emplace(size, BlockPool::Free{ptr, ++p.clock});
  p.cached += size;
  p.shrink(p.capacity);
}

size_t pool_trim() {
  std::lock_guard<std::mutex> lock(pool().mutex);
  size_t const before = pool().cached;
  pool().shrink(0);
  return before - pool().cached;
}

size_t pool_cached_bytes() {
  std::lock_guard<std::mutex> lock(pool().mutex);
  return pool().cached;
}

} // namespace lsamd

using namespace lsamd;

extern "C" int ls_amd_device_available(void) { return ensure_device() ? 0 : 1; }

extern "C" char const *ls_amd_last_error(void) { return g_last_error.c_str(); }

extern "C" void ls_amd_clear_error(void) { g_last_error.clear(); }

extern "C" void *ls_amd_device_malloc(size_t bytes) {
  if (!ensure_device()) return nullptr;
  void *p = nullptr;
  if (hipMalloc(&p, bytes == 0 ? 1 : bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  pool_trim(); // the blocks kept for reuse may be what is missing
  if (hipMalloc(&p, bytes == 0 ? 1 : bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  set_last_error("hipMalloc failed");
  return nullptr;
}

extern "C" int64_t ls_amd_device_trim(void) { return static_cast<int64_t>(pool_trim()); }

extern "C" void ls_amd_device_free(void *ptr) {
  if (ptr != nullptr) (void)hipFree(ptr);
}

extern "C" int ls_amd_memcpy_h2d(void *dst, void const *src, size_t bytes) {
  if (!ensure_device()) return -1;
  if (hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream()) != hipSuccess) return -1;
  return hipStreamSynchronize(stream()) == hipSuccess ? 0 : -1;
}

extern "C" int ls_amd_memcpy_d2h(void *dst, void const *src, size_t bytes) {
  if (!ensure_device()) return -1;
  if (hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream()) != hipSuccess) return -1;
  return hipStreamSynchronize(stream()) == hipSuccess ? 0 : -1;
}

extern "C" int ls_amd_synchronize(void) {
  if (!ensure_device()) return -1;
  return hipStreamSynchronize(stream()) == hipSuccess ? 0 : -1;
}

extern "C" double ls_amd_last_kernel_ms(int family) {
  if (family < 0 || family >= kTimerCount || !g_ev_used[family]) return -1.0;
  if (hipEventSynchronize(g_ev_end[family]) != hipSuccess) return -1.0;
  float ms = 0;
  if (hipEventElapsedTime(&ms, g_ev_begin[family], g_ev_end[family]) != hipSuccess) return -1.0;
  return static_cast<double>(ms);
}
