// Copies between device memory and a caller's host arrays: pageable ones through
// pinned memory that the object owning the stream keeps (host_copy.cpp), others
// as they are.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <mutex>

class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy &) = delete;
  HostCopy &operator=(const HostCopy &) = delete;
  ~HostCopy() { release(); }

  // Pinned memory for copies of up to `bytes` (at most MOST; larger ones go in
  // pieces).  Without it -- none could be had, or never called -- get and put
  // leave the copy to the runtime.
  void reserve(size_t bytes);
  void release();

  // Ordered after the work enqueued on s; complete when they return.
  hipError_t get(void *host, const void *dev, size_t bytes, hipStream_t s);
  hipError_t put(void *dev, const void *host, size_t bytes, hipStream_t s);

  static constexpr size_t MOST = (size_t)32 << 20;    // pinned memory of one object
  static constexpr size_t CHUNK = (size_t)4 << 20;    // one transfer
  static constexpr size_t PIECE = (size_t)256 << 10;   // one memcpy
  static constexpr size_t HELP = (size_t)2 << 20;     // bytes per helper thread
  static constexpr size_t POPULATE = (size_t)4 << 20;  // results below this: pages are had at once
  static constexpr int MOST_CHUNKS = (int)(MOST / CHUNK), HELPERS = 4;

 private:
  std::mutex lock_;  // one copy at a time
  char *pinned_ = nullptr;
  size_t size_ = 0;
  hipEvent_t ev_[MOST_CHUNKS] = {};
};
