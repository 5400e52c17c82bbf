// common.hpp -- error handling, logging and the per-device HIP context of
// libspined.  Everything here is host code shared by the C-ABI objects and
// the kernel launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <mutex>
#include <stdexcept>
#include <string>

#include "../../include/lattice_symmetries.h"

namespace spined {

// An error that maps onto an ls_error_code at the C boundary.
struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string &what) : std::runtime_error(what), code(c) {}
};

[[noreturn]] void throw_hip(hipError_t e, const char *expr, const char *file, int line);

#define SPINED_HIP(expr)                                                       \
  do {                                                                         \
    hipError_t _e = (expr);                                                    \
    if (_e != hipSuccess) ::spined::throw_hip(_e, #expr, __FILE__, __LINE__);   \
  } while (0)

#define SPINED_CHECK_LAUNCH() SPINED_HIP(hipGetLastError())

bool logging_enabled();
void log_line(const char *fmt, ...) __attribute__((format(printf, 1, 2)));

// Library-owned stream of the current device (created on first use, default
// priority, non-blocking w.r.t. the null stream).
hipStream_t stream();
int current_device();

// Pools of device blocks.  Every library kernel and copy runs on the device's
// library stream, so a block that is handed on is only touched after the work
// that used it before; host copies into a block go through that stream too
// (copy_in).  Large blocks (allocate_pooled, at least kPoolMinBytes): the
// eigensolver's vectors (6.9 GB each at D = 8.6e8, dozens per solve) and the
// entry blocks of dropped gather caches, of exactly the size asked for,
// instead of hipFree, which unmaps them page by page.  Small blocks
// (everything else below kPoolMinBytes): rounded up to a quarter of a power
// of two, at most kSmallPoolBytes of them kept per device; a hipMalloc and
// hipFree pair costs 20 to 200 us.  An allocation that the driver refuses
// drops the gather caches not in use (into the pool), returns the pooled
// blocks of the device and retries once.
constexpr size_t kPoolMinBytes = size_t(256) << 20;
constexpr size_t kSmallPoolBytes = size_t(1) << 30;
enum class Pool { none, large, small };
size_t small_class(size_t bytes);              // size of the small block for `bytes`
void *device_alloc(size_t bytes, Pool pool);   // throws Error(LS_OUT_OF_MEMORY)
void device_free(void *p, size_t bytes, Pool pool, int device);
void pool_release_device();                    // hipFree the current device's pooled blocks
size_t pool_bytes(size_t bytes);               // pooled bytes in large blocks of this size (current device)
// Host -> device copy of `bytes`, complete on return, in stream order.
void copy_in(void *dst, const void *src, size_t bytes);

// Device buffer with RAII release (any thread).  allocate_pooled(count,
// bytes) takes a block of max(count * sizeof(T), bytes) bytes from the pool.
template <class T> struct DeviceBuffer {
  T *ptr = nullptr;
  size_t n = 0;
  size_t cap = 0;      // bytes of the block
  Pool pooled = Pool::none;
  int dev = 0;         // device of a pooled block
  DeviceBuffer() = default;
  explicit DeviceBuffer(size_t count) { allocate(count); }
  DeviceBuffer(const DeviceBuffer &) = delete;
  DeviceBuffer &operator=(const DeviceBuffer &) = delete;
  DeviceBuffer(DeviceBuffer &&o) noexcept
      : ptr(o.ptr), n(o.n), cap(o.cap), pooled(o.pooled), dev(o.dev) {
    o.ptr = nullptr;
    o.n = 0;
    o.cap = 0;
  }
  DeviceBuffer &operator=(DeviceBuffer &&o) noexcept {
    if (this != &o) {
      release();
      ptr = o.ptr;
      n = o.n;
      cap = o.cap;
      pooled = o.pooled;
      dev = o.dev;
      o.ptr = nullptr;
      o.n = 0;
      o.cap = 0;
    }
    return *this;
  }
  ~DeviceBuffer() { release(); }
  void allocate(size_t count) { take(count, 0, false); }
  void allocate_pooled(size_t count, size_t bytes = 0) { take(count, bytes, true); }
  void release() {
    if (ptr) device_free(ptr, cap, pooled, dev);
    ptr = nullptr;
    n = 0;
    cap = 0;
  }
  size_t bytes() const { return n * sizeof(T); }

private:
  void take(size_t count, size_t bytes, bool pool) {
    release();
    size_t b = std::max(count * sizeof(T), bytes);
    if (b) {
      pooled = b < kPoolMinBytes ? Pool::small : pool ? Pool::large : Pool::none;
      if (pooled == Pool::small) b = small_class(b);
      if (pooled != Pool::none) dev = current_device();
      ptr = static_cast<T *>(device_alloc(b, pooled));
      cap = b;
    }
    n = count;
  }
};

// Converts exceptions into status codes at the C boundary.
template <class F> int guarded(F &&f) {
  try {
    f();
    return LS_SUCCESS;
  } catch (const Error &e) {
    if (logging_enabled()) log_line("error %d: %s", e.code, e.what());
    return e.code;
  } catch (const std::bad_alloc &) {
    return LS_OUT_OF_MEMORY;
  } catch (const std::exception &e) {
    if (logging_enabled()) log_line("internal error: %s", e.what());
    return LS_INTERNAL_ERROR;
  }
}

} // namespace spined
