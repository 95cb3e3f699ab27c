// sphdem_hostcopy.h -- copies from device memory into a caller's pageable
// memory.
//
// What bounds them: the host.  The runtime stages such a copy through pinned
// memory and moves it on by one thread, which also takes the page faults of
// memory that was just allocated.  Here the caller's thread and the context's
// helpers (kWays together) each take every kWays-th piece, with a piece of their
// own on its way from the device while they copy the one before.  One field,
// the runtime's copy and this one: 4.5 MB 288 and 200 us, 9.5 MB 575 and 360,
// 28 MB 1615 and 930 (30 GB/s; eight threads the same, pieces of 0.5 MB 1330).
// Below kShared the runtime's copy is as fast (0.1 MB 29 and 35 us).
#pragma once

#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <condition_variable>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

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

  // The pinned pieces and the helpers, for copies of up to `most` bytes.  Without
  // them (no memory, no threads) copy() leaves all to the runtime, or more to the
  // caller's thread.
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
    const int cpus = (int)std::max(1u, std::thread::hardware_concurrency());
    try {
      helpers_.reserve(kWays);
      for (int w = 1; w < std::min((int)kWays, cpus); w++) helpers_.emplace_back([this, w] { help(w); });
    } catch (const std::exception&) {  // as many as can be had
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
    job_ = Job{device, stream, (char*)dst, (const char*)src, bytes, 1 + (int)helpers_.size()};
    if (job_.ways > 1) {
      std::lock_guard<std::mutex> lock(mu_);
      pending_ = job_.ways - 1;
      turn_++;
      wake_.notify_all();
    }
    hipError_t e = part(0);
    if (job_.ways > 1) {
      std::unique_lock<std::mutex> lock(mu_);
      done_.wait(lock, [&] { return pending_ == 0; });
      for (int w = 1; w < job_.ways; w++)
        if (e == hipSuccess) e = err_[w];
    }
    return e;
  }

  // ends the helpers and gives the pinned memory back
  void release() {
    if (!helpers_.empty()) {
      {
        std::lock_guard<std::mutex> lock(mu_);
        stop_ = true;
        wake_.notify_all();
      }
      for (std::thread& t : helpers_) t.join();
      helpers_.clear();
      stop_ = false;
    }
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
    int ways;
  };

  void help(int w) {
    unsigned seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> lock(mu_);
        wake_.wait(lock, [&] { return stop_ || turn_ != seen; });
        if (stop_) return;
        seen = turn_;
      }
      err_[w] = hipSetDevice(job_.device);
      if (err_[w] == hipSuccess) err_[w] = part(w);
      std::lock_guard<std::mutex> lock(mu_);
      if (--pending_ == 0) done_.notify_one();
    }
  }
  // pieces w, w + ways, ... by the two buffers of thread w
  hipError_t part(int w) {
    const Job& J = job_;
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
    for (size_t k = w; k < n && e == hipSuccess; k += J.ways, b ^= 1) {
      hipError_t wait = hipEventSynchronize(ev_[2 * w + b]);
      if (wait != hipSuccess) return wait;
      if (k + J.ways < n) fetch(k + J.ways, b ^ 1);
      const size_t at = k * kPiece;
      memcpy(J.dst + at, pinned_ + (size_t)(2 * w + b) * kPiece, std::min(kPiece, J.bytes - at));
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(J.stream);  // nothing left on its way
    return e;
  }

  char* pinned_ = nullptr;
  hipEvent_t ev_[2 * kWays] = {};
  std::vector<std::thread> helpers_;
  std::mutex mu_;
  std::condition_variable wake_, done_;
  Job job_{};
  unsigned turn_ = 0;
  int pending_ = 0;
  bool stop_ = false;
  hipError_t err_[kWays] = {};
};

}  // namespace sphdem
