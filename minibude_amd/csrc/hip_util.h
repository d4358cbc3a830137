// hip_util.h -- small HIP helpers shared by the C-ABI translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdlib>
#include <string>

#include "bude_internal.h"

namespace bude {

inline int hip_fail(hipError_t e, const char *what) {
  return fail(e == hipErrorOutOfMemory ? BUDE_ERR_OUT_OF_MEMORY : BUDE_ERR_RUNTIME,
              std::string(what) + ": " + hipGetErrorName(e) + ": " + hipGetErrorString(e));
}

inline int hip_check(hipError_t e, const char *what) { return e == hipSuccess ? BUDE_OK : hip_fail(e, what); }

// Bytes all DeviceBuffers hold, and whether BUDE_MI355X_MAX_MEMORY_MB (not set:
// no bound) lets them be n more; an allocation beyond it is out of memory.
inline std::atomic<size_t> device_bytes{0};
inline bool take_device_bytes(size_t n) {
  const size_t held = device_bytes.fetch_add(n) + n;
  const char *mb = std::getenv("BUDE_MI355X_MAX_MEMORY_MB");
  if (!mb || held <= size_t(std::strtoull(mb, nullptr, 10)) << 20) return true;
  device_bytes.fetch_sub(n);
  return false;
}

// Owning device allocation (hipMalloc / hipFree).
struct DeviceBuffer {
  void *ptr = nullptr;
  size_t bytes = 0;

  DeviceBuffer() = default;
  DeviceBuffer(const DeviceBuffer &) = delete;
  DeviceBuffer &operator=(const DeviceBuffer &) = delete;
  ~DeviceBuffer() { reset(); }

  void reset() {
    if (ptr) (void)hipFree(ptr);
    device_bytes.fetch_sub(bytes);
    ptr = nullptr;
    bytes = 0;
  }
  int alloc(size_t n) {
    reset();
    if (n == 0) n = 4;
    const bool room = take_device_bytes(n);
    if (int st = hip_check(room ? hipMalloc(&ptr, n) : hipErrorOutOfMemory, "hipMalloc")) {
      if (room) device_bytes.fetch_sub(n);
      (void)hipGetLastError();  // (reported here: a caller that goes on without the memory is not to find it after its next launch)
      ptr = nullptr;
      return st;
    }
    bytes = n;
    return BUDE_OK;
  }
  // Keeps the current allocation when it already holds n bytes; a growing
  // buffer gets a quarter of headroom where there is memory for it, so sizes
  // that vary a little from call to call settle on one allocation.  The old
  // allocation goes before the new one is made.
  int reserve(size_t n) {
    if (ptr && bytes >= n) return BUDE_OK;
    const int st = alloc(ptr ? n + n / 4 : n);
    return st == BUDE_ERR_OUT_OF_MEMORY ? alloc(n) : st;
  }
  // Copies n bytes in, reusing the allocation when it is large enough.
  int assign(const void *src, size_t n) {
    if (int st = reserve(n)) return st;
    return n ? hip_check(hipMemcpy(ptr, src, n, hipMemcpyHostToDevice), "hipMemcpy H2D") : BUDE_OK;
  }
  int upload(const void *src, size_t n) {
    if (int st = alloc(n)) return st;
    return n ? hip_check(hipMemcpy(ptr, src, n, hipMemcpyHostToDevice), "hipMemcpy H2D") : BUDE_OK;
  }
};

// Owning pinned host allocation (hipHostMalloc / hipHostFree): the source of
// copies that run asynchronously to the host.
struct PinnedBuffer {
  void *ptr = nullptr;
  PinnedBuffer() = default;
  PinnedBuffer(const PinnedBuffer &) = delete;
  PinnedBuffer &operator=(const PinnedBuffer &) = delete;
  ~PinnedBuffer() {
    if (ptr) (void)hipHostFree(ptr);
  }
  int alloc(size_t n) {
    if (ptr) (void)hipHostFree(ptr);
    ptr = nullptr;
    if (int st = hip_check(hipHostMalloc(&ptr, n ? n : 4, hipHostMallocDefault), "hipHostMalloc")) {
      (void)hipGetLastError();  // (as above)
      ptr = nullptr;
      return st;
    }
    return BUDE_OK;
  }
};

}  // namespace bude
