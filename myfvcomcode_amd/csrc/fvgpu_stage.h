// fvgpu_stage.h -- copies between device memory and the caller's ordinary
// (pageable) host memory through pinned staging.
//
// A copy straight to pageable memory runs at about 10 GB/s here and costs
// tens of microseconds at any size: the runtime pins or stages the pages one
// after another, and the first touch of a fresh result array happens inside
// it.  Here small copies go through one pinned buffer, and large ones by
// chunks over a few threads, each with two pinned chunks: one is moved over
// the bus while the other is copied to or from the caller's memory, so that
// the page faults and the memory copies of several chunks run side by side.
// Measured to fresh memory, direct / staged: 14 KB 25 / 12 us, 280 KB 118 /
// 19, 1 MB 410 / 49, 8 MB 1025 / 535, 41 MB 4065 / 1316, 328 MB 31.2 / 8.2 ms
// (4 threads of 2 MB chunks; 2 threads 12.4 ms, 8 threads 8.2 ms).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

class HostStage {
 public:
  static constexpr size_t SMALL = 2u << 20;   // copies up to this size go through one buffer
  static constexpr size_t CHUNK = 2u << 20;
  static constexpr int THREADS = 4;

  // Allocates the buffer of the small copies now, so that they allocate
  // nothing later.
  void reserve() { (void)pinned(small_, SMALL); }
  // Frees the staging; no copy may be under way.
  void release() {
    if (small_) (void)hipHostFree(small_);
    if (large_) (void)hipHostFree(large_);
    small_ = large_ = nullptr;
  }

  // Synchronous copies in the order of `stream` (of `device`).
  hipError_t to_host(void* dst, const void* src, size_t n, hipStream_t stream, int device) {
    return copy(static_cast<char*>(dst), static_cast<char*>(const_cast<void*>(src)), n, false, stream, device);
  }
  hipError_t to_device(void* dst, const void* src, size_t n, hipStream_t stream, int device) {
    return copy(static_cast<char*>(const_cast<void*>(src)), static_cast<char*>(dst), n, true, stream, device);
  }

 private:
  char *small_ = nullptr, *large_ = nullptr;
  std::mutex mu_;   // the staging serves one copy at a time

  // Clears the error of a call whose failure is an answer here -- unless an
  // error was pending before it, as that of a launch, which the caller has yet
  // to report.
  static void answered(hipError_t pending) {
    if (pending == hipSuccess) (void)hipGetLastError();
  }

  static bool pinned(char*& p, size_t n) {
    if (p) return true;
    const hipError_t pending = hipPeekAtLastError();
    if (hipHostMalloc((void**)&p, n, hipHostMallocDefault) != hipSuccess) {
      answered(pending);   // no staging: the caller copies directly
      p = nullptr;
    }
    return p != nullptr;
  }

  // n bytes between host memory `host` and device memory `dev`, upwards to
  // the device or down to the host
  hipError_t copy(char* host, char* dev, size_t n, bool up, hipStream_t stream, int device) {
    if (n == 0) return hipStreamSynchronize(stream);
    if (!host || !dev) return hipErrorInvalidValue;
    // memory the runtime knows (pinned, or the device's) needs no staging
    hipPointerAttribute_t at_{};
    const hipError_t pending = hipPeekAtLastError();
    const hipError_t asked = hipPointerGetAttributes(&at_, host);
    if (asked != hipSuccess) answered(pending);
    const bool known = asked == hipSuccess && at_.type != hipMemoryTypeUnregistered;
    std::unique_lock<std::mutex> lock(mu_, std::defer_lock);
    if (!known) lock.lock();
    if (!known && n <= SMALL && pinned(small_, SMALL)) {
      if (up) std::memcpy(small_, host, n);
      hipError_t e = up ? hipMemcpyAsync(dev, small_, n, hipMemcpyHostToDevice, stream)
                        : hipMemcpyAsync(small_, dev, n, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
      if (e == hipSuccess && !up) std::memcpy(host, small_, n);
      return e;
    }
    if (!known && n > SMALL && pinned(large_, 2 * CHUNK * THREADS)) {
      // chunks small enough that every thread has some
      const size_t chunk = std::min(CHUNK, std::max<size_t>(CHUNK / 4, n / (2 * THREADS) / 4096 * 4096));
      hipError_t err[THREADS] = {};
      std::thread helpers[THREADS];
      int started = 1;
      // lane j of `lanes` takes the chunks j, j + lanes, ...: fixed before
      // the first helper starts, so a helper that cannot be started leaves
      // its chunks to the caller
      auto lane = [&](int j) { err[j] = run_lane(host, dev, n, chunk, j, THREADS, up, stream, device); };
      try {
        for (; started < THREADS; ++started) helpers[started] = std::thread(lane, started);
      } catch (const std::exception&) {   // no thread, or no memory for one
      }
      int here = device;
      (void)hipGetDevice(&here);
      lane(0);
      for (int j = started; j < THREADS; ++j) lane(j);
      if (here != device) (void)hipSetDevice(here);
      for (int j = 1; j < started; ++j) helpers[j].join();
      for (hipError_t e : err)
        if (e != hipSuccess) return e;
      return hipStreamSynchronize(stream);
    }
    hipError_t e = up ? hipMemcpyAsync(dev, host, n, hipMemcpyHostToDevice, stream)
                      : hipMemcpyAsync(host, dev, n, hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  }

  hipError_t run_lane(char* host, char* dev, size_t n, size_t chunk, int j, int lanes, bool up, hipStream_t stream,
                      int device) {
    hipError_t e = hipSetDevice(device);
    hipEvent_t ev[2] = {};
    char* buf[2] = {large_ + (size_t)(2 * j) * CHUNK, large_ + (size_t)(2 * j + 1) * CHUNK};
    for (int s = 0; s < 2 && e == hipSuccess; ++s) e = hipEventCreateWithFlags(&ev[s], hipEventDisableTiming);
    const size_t nch = (n + chunk - 1) / chunk;
    auto len = [&](size_t c) { return std::min(chunk, n - c * chunk); };
    auto issue = [&](size_t c, int s) {
      hipError_t r = up ? hipMemcpyAsync(dev + c * chunk, buf[s], len(c), hipMemcpyHostToDevice, stream)
                        : hipMemcpyAsync(buf[s], dev + c * chunk, len(c), hipMemcpyDeviceToHost, stream);
      return r == hipSuccess ? hipEventRecord(ev[s], stream) : r;
    };
    if (up) {
      int s = 0;
      size_t i = 0;
      for (size_t c = j; c < nch && e == hipSuccess; c += lanes, s ^= 1, ++i) {
        if (i >= 2) e = hipEventSynchronize(ev[s]);   // the buffer's last chunk has left it
        if (e != hipSuccess) break;
        std::memcpy(buf[s], host + c * chunk, len(c));
        e = issue(c, s);
      }
    } else {
      int s = 0;
      if ((size_t)j < nch && e == hipSuccess) e = issue(j, 0);
      for (size_t c = j; c < nch && e == hipSuccess; c += lanes, s ^= 1) {
        if (c + lanes < nch) e = issue(c + lanes, s ^ 1);
        if (e == hipSuccess) e = hipEventSynchronize(ev[s]);
        if (e == hipSuccess) std::memcpy(host + c * chunk, buf[s], len(c));
      }
    }
    // nothing may still be moving through the buffers when the lane ends
    for (int s = 0; s < 2; ++s)
      if (ev[s]) {
        (void)hipEventSynchronize(ev[s]);
        (void)hipEventDestroy(ev[s]);
      }
    return e;
  }
};
