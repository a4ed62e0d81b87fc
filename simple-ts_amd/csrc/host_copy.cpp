// A pageable copy runs at 17 GB/s here and, into an array that its caller has
// just allocated, at 10 (its pages are had one by one, at their first touch, by
// one thread); a transfer into pinned memory at 50.  So a result is transferred
// into pinned memory in chunks, and the chunks that have arrived are copied out
// by the caller and a few helper threads, which share the page faults; an input
// is copied in by them and each chunk transferred as soon as it is filled.  5.9
// MB into a new array: 633 -> 380 us, into an old one 330 -> 180; 23.6 MB: 1,750
// -> 780; 0.66 MB: 99 -> 70 (its pages are had during the transfer).
#include "host_copy.h"

#include <stdint.h>
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <thread>

namespace {

// The pieces of [0, bytes) of a copy from src to dst, taken in order by several
// threads; a piece may be copied once `ready` bytes reach its end.
struct Pieces {
  char *dst;
  const char *src;
  size_t bytes, piece, chunk;                      // chunk: a multiple of piece
  std::atomic<size_t> next{0}, ready{0};           // pieces taken, bytes available
  std::atomic<size_t> done[HostCopy::MOST_CHUNKS] = {};  // bytes copied of each chunk

  // Copies the next piece; false when none is left.
  bool one() {
    const size_t at = next.fetch_add(1, std::memory_order_relaxed) * piece;
    if (at >= bytes) return false;
    const size_t n = std::min(piece, bytes - at);
    while (ready.load(std::memory_order_acquire) < at + n) std::this_thread::yield();
    memcpy(dst + at, src + at, n);
    done[at / chunk].fetch_add(n, std::memory_order_release);
    return true;
  }
  void work() {
    while (one()) {
    }
  }
  bool copied(int k) const {
    return done[k].load(std::memory_order_acquire) == std::min(chunk, bytes - chunk * (size_t)k);
  }
};

// Has the system put pages behind [p, p + bytes), whole ones, at once rather than
// at each one's first touch; what it cannot do it leaves to those.
void populate(void *p, size_t bytes) {
#ifdef MADV_POPULATE_WRITE
  const uintptr_t page = 4096, from = ((uintptr_t)p + page - 1) & ~(page - 1), to = ((uintptr_t)p + bytes) & ~(page - 1);
  if (to > from) (void)madvise((void *)from, to - from, MADV_POPULATE_WRITE);
#else
  (void)p, (void)bytes;
#endif
}

// Whether the runtime knows the array (pinned, managed or device memory): its own
// copy is then one transfer, at the rate of one into pinned_.
bool known(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return false;
}

// Helper threads on the pieces, joined when it goes out of scope (their pieces
// are then copied); fewer when the system gives fewer.
struct Helpers {
  std::thread t[HostCopy::HELPERS];
  int n = 0;
  void start(Pieces &p, size_t bytes) {
    const int want = (int)std::min<size_t>(HostCopy::HELPERS, bytes / HostCopy::HELP);
    try {
      for (; n < want; n++) t[n] = std::thread([&p] { p.work(); });
    } catch (...) {
    }
  }
  ~Helpers() {
    for (int k = 0; k < n; k++) t[k].join();
  }
};

}  // namespace

void HostCopy::reserve(size_t bytes) {
  std::lock_guard<std::mutex> hold(lock_);
  const size_t want = std::min(std::max(bytes, (size_t)4096), MOST);
  if (pinned_ || want == 0) return;
  for (hipEvent_t &e : ev_)
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      return;
    }
  if (hipHostMalloc((void **)&pinned_, want, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    pinned_ = nullptr;
    return;
  }
  size_ = want;
}

void HostCopy::release() {
  if (pinned_) (void)hipHostFree(pinned_);
  pinned_ = nullptr;
  for (hipEvent_t &e : ev_) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

hipError_t HostCopy::get(void *host, const void *dev, size_t bytes, hipStream_t s) {
  std::lock_guard<std::mutex> hold(lock_);
  hipError_t e = hipSuccess;
  if (!pinned_ || known(host)) {
    e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
  }
  for (size_t off = 0; off < bytes; off += size_) {
    const size_t len = std::min(size_, bytes - off);
    const int chunks = (int)((len + CHUNK - 1) / CHUNK);
    for (int k = 0; k < chunks; k++) {
      const size_t at = CHUNK * k;
      e = hipMemcpyAsync(pinned_ + at, (const char *)dev + off + at, std::min(CHUNK, len - at), hipMemcpyDeviceToHost, s);
      if (e == hipSuccess && k + 1 < chunks) e = hipEventRecord(ev_[k], s);
      if (e != hipSuccess) {
        (void)hipStreamSynchronize(s);
        return e;
      }
    }
    if (len < POPULATE) populate((char *)host + off, len);  // while the transfer runs
    Pieces p;
    p.dst = (char *)host + off, p.src = pinned_, p.bytes = len, p.piece = PIECE, p.chunk = CHUNK;
    Helpers h;
    for (int k = 0; k < chunks && e == hipSuccess; k++) {
      e = k + 1 < chunks ? hipEventSynchronize(ev_[k]) : hipStreamSynchronize(s);
      p.ready.store(std::min(CHUNK * (k + 1), len), std::memory_order_release);
      if (k == 0) h.start(p, len);  // the earlier work on s is done: helpers do not wait for that
    }
    p.ready.store(len, std::memory_order_release);  // (also after an error: the helpers come to their end)
    p.work();
    if (e != hipSuccess) return e;
  }
  return e;
}

hipError_t HostCopy::put(void *dev, const void *host, size_t bytes, hipStream_t s) {
  std::lock_guard<std::mutex> hold(lock_);
  hipError_t e = hipSuccess;
  if (!pinned_ || known(host)) {
    e = hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
  }
  for (size_t off = 0; off < bytes; off += size_) {
    const size_t len = std::min(size_, bytes - off);
    const int chunks = (int)((len + CHUNK - 1) / CHUNK);
    Pieces p;
    p.dst = pinned_, p.src = (const char *)host + off, p.bytes = len, p.piece = PIECE, p.chunk = CHUNK;
    p.ready.store(len, std::memory_order_relaxed);
    {
      Helpers h;
      h.start(p, len);
      bool more = true;
      for (int k = 0; k < chunks && e == hipSuccess;) {
        if (p.copied(k)) {
          const size_t at = CHUNK * (size_t)k;
          e = hipMemcpyAsync((char *)dev + off + at, pinned_ + at, std::min(CHUNK, len - at), hipMemcpyHostToDevice, s);
          k++;
        } else if (more) more = p.one();
        else std::this_thread::yield();
      }
      p.work();  // (after an error)
    }
    const hipError_t w = hipStreamSynchronize(s);  // the pinned memory is free again
    if (e != hipSuccess || w != hipSuccess) return e != hipSuccess ? e : w;
  }
  return e;
}
