// sphdem_hostcopy.h -- copies from device memory into a caller's pageable
// memory.
//
// What bounds them: the host.  The runtime stages such a copy through pinned
// memory and moves it on by one thread, which also takes the page faults of
// memory that was just allocated.  Here the caller's thread and helpers that
// live for the copy (kWays together) each take every kWays-th piece, with a
// piece of their own on its way from the device while they copy the one before.
// One field,
// the runtime's copy and this one: 4.5 MB 288 and 215 us, 9.5 MB 575 and 378,
// 28 MB 1615 and 960 (29 GB/s; eight threads the same, pieces of 0.5 MB 1330).
// Threads kept for the context's life save some 20 us a copy.
// Below kShared the runtime's copy is as fast (0.1 MB 29 and 35 us).
#pragma once

#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <exception>
#include <thread>

namespace sphdem {

class HostCopy {
 public:
  static constexpr int kWays = 4;
  static constexpr size_t kPiece = 1u << 20;   // bytes
  static constexpr size_t kShared = 4u << 20;  // bytes; smaller copies are left to the runtime

  HostCopy() = default;
  HostCopy(const HostCopy&) = delete;
  HostCopy& operator=(const HostCopy&) = delete;
  ~HostCopy() { release(); }

  // The pinned pieces, for copies of up to `most` bytes.  Without them copy()
  // leaves all to the runtime.
  void prepare(size_t most) {
    if (pinned_ || most < kShared) return;
    void* p = nullptr;
    if (hipHostMalloc(&p, 2 * kWays * kPiece, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      return;
    }
    pinned_ = (char*)p;
    for (int i = 0; i < 2 * kWays; i++)
      if (hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        ev_[i] = nullptr;
        release();
        return;
      }
  }

  // dst[0..bytes) = src, ordered after what stream holds; returns when done.
  hipError_t copy(int device, hipStream_t stream, void* dst, const void* src, size_t bytes) {
    bool own = bytes >= kShared && pinned_;
    if (own) {  // the caller's memory pageable?
      hipPointerAttribute_t at;
      own = hipPointerGetAttributes(&at, dst) != hipSuccess || at.type == hipMemoryTypeUnregistered;
      (void)hipGetLastError();  // an unknown pointer may be reported as an error
    }
    if (!own) {
      const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
      return e != hipSuccess ? e : hipStreamSynchronize(stream);
    }
    const Job job{device, stream, (char*)dst, (const char*)src, bytes};
    std::thread helper[kWays];
    hipError_t err[kWays] = {};
    for (int w = 1; w < kWays; w++) {
      try {
        helper[w] = std::thread([&, w] {
          err[w] = hipSetDevice(job.device);
          if (err[w] == hipSuccess) err[w] = part(job, w);
        });
      } catch (const std::exception&) {  // its pieces are left to this thread
      }
    }
    err[0] = part(job, 0);
    for (int w = 1; w < kWays; w++)
      if (!helper[w].joinable()) err[w] = part(job, w);
    hipError_t e = err[0];
    for (int w = 1; w < kWays; w++) {
      if (helper[w].joinable()) helper[w].join();
      if (e == hipSuccess) e = err[w];
    }
    return e;
  }

  // gives the pinned memory back
  void release() {
    for (int i = 0; i < 2 * kWays; i++)
      if (ev_[i]) {
        (void)hipEventDestroy(ev_[i]);
        ev_[i] = nullptr;
      }
    if (pinned_) (void)hipHostFree(pinned_);
    pinned_ = nullptr;
  }

 private:
  struct Job {
    int device;
    hipStream_t stream;
    char* dst;
    const char* src;
    size_t bytes;
  };

  // pieces w, w + kWays, ... by the two buffers of thread w
  hipError_t part(const Job& J, int w) {
    const size_t n = (J.bytes + kPiece - 1) / kPiece;
    hipError_t e = hipSuccess;
    auto fetch = [&](size_t k, int b) {
      const size_t at = k * kPiece, len = std::min(kPiece, J.bytes - at);
      e = hipMemcpyAsync(pinned_ + (size_t)(2 * w + b) * kPiece, J.src + at, len,
                         hipMemcpyDeviceToHost, J.stream);
      if (e == hipSuccess) e = hipEventRecord(ev_[2 * w + b], J.stream);
    };
    int b = 0;
    if ((size_t)w < n) fetch(w, 0);
    for (size_t k = w; k < n && e == hipSuccess; k += kWays, b ^= 1) {
      hipError_t wait = hipEventSynchronize(ev_[2 * w + b]);
      if (wait != hipSuccess) return wait;
      if (k + kWays < n) fetch(k + kWays, b ^ 1);
      const size_t at = k * kPiece;
      memcpy(J.dst + at, pinned_ + (size_t)(2 * w + b) * kPiece, std::min(kPiece, J.bytes - at));
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(J.stream);  // nothing left on its way
    return e;
  }

  char* pinned_ = nullptr;
  hipEvent_t ev_[2 * kWays] = {};
};

}  // namespace sphdem
