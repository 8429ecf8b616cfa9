// Copies between pageable host arrays and device memory, and device scratch of calls that own no operator.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "cmx_internal.h"

namespace cmx {

// dev[0..bytes) = host[0..bytes), ordered on stream s; host stays valid until the stream has passed the copy
void host_to_device(void* dev, const void* host, size_t bytes, hipStream_t s);
// host[0..bytes) = dev[0..bytes) after the work queued on s; host holds the data when this returns
void device_to_host(void* host, const void* dev, size_t bytes, hipStream_t s);
// Gives back the pinned staging buffers, the copy threads and the cached scratch that no call is using
void xfer_release();
// device bytes of the current device that the cache holds: free memory to a caller that counts it, since an
// allocation that fails releases them
size_t scratch_cached();

// Device memory from the bounded cache of earlier calls' buffers (cap: its size, dev: its device), and back
// to it; work on a buffer that is given back must have completed
void* scratch_take(size_t bytes, size_t& cap, int& dev);
void scratch_give(void* p, size_t cap, int dev);
// Buffers above this are not worth caching where many live at once: a sixteenth of what the cache holds
constexpr size_t SCRATCH_LARGE = (size_t)256 << 20;
// Small pinned host blocks (PINNED_BLOCK bytes), cached likewise
constexpr size_t PINNED_BLOCK = 8192;
void* pinned_take();
void pinned_give(void* p);

// Device memory of one call, from a bounded cache of earlier calls' buffers.  The caller's work on it must
// have completed (stream synchronised) when the object goes out of scope.
class DevScratch {
 public:
  explicit DevScratch(size_t bytes);
  ~DevScratch();
  DevScratch(const DevScratch&) = delete;
  DevScratch& operator=(const DevScratch&) = delete;
  template <typename T> T* as() const { return static_cast<T*>(p_); }
  void* get() const { return p_; }
  size_t bytes() const { return bytes_; }

 private:
  void* p_ = nullptr;
  size_t bytes_ = 0, cap_ = 0;
  int dev_ = 0, throwing_;
};

}  // namespace cmx
