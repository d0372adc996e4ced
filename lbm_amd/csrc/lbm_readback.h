// Copies of device results into the caller's (pageable) memory.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace lbm {

// A device-to-host copy into pageable memory goes through the runtime's
// staging at about 9 GB/s: one host thread copies out of it and, where the
// destination is fresh, takes its page faults.  Here a large transfer lands
// in pinned chunks while several threads empty them, the faults included (537
// MB 51 -> 14 ms, 50 MB 4.0 -> 1.8 ms, once 2 ms more for the chunks; 8 MB 0.5
// ms either way, so smaller copies stay with the runtime).  The chunks stay
// with the owner; threads live as long as the call.
// A read-back holds the staging (hold()) from the kernel that fills it to the
// end of its copy: reads of one owner from several threads go in turn.
class Readback {
 public:
  static constexpr size_t CHUNK = 2u << 20;
  static constexpr int THREADS = 8, CHUNKS = 2 * THREADS;

  std::unique_lock<std::mutex> hold() { return std::unique_lock<std::mutex>(mu_); }

  // two arrays that lie one behind the other at src
  hipError_t copy(void *dst, size_t bytes, void *dst2, size_t bytes2, const void *src, hipStream_t s) {
    const char *src2 = static_cast<const char *>(src) + bytes;
    if (bytes + bytes2 < LEAST) {
      const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
      return e != hipSuccess ? e : plain(dst2, src2, bytes2, s);
    }
    const hipError_t e = copy(dst, src, bytes, s);
    return e != hipSuccess ? e : copy(dst2, src2, bytes2, s);
  }

  // CHUNK bytes of pinned memory that a kernel of stream s may write and the
  // host reads once the stream is synchronised; null where there are none
  void *pinned(hipStream_t s) {
    const OnDevice of(s);
    return of.ok && reserve(1) ? chunk_[0] : nullptr;
  }

  // bytes from src on the device to dst, after what is queued on the stream;
  // done on return
  hipError_t copy(void *dst, const void *src, size_t bytes, hipStream_t s) {
    if (bytes < LEAST) return plain(dst, src, bytes, s);
    const OnDevice of(s);
    const size_t n = (bytes + CHUNK - 1) / CHUNK;
    if (!of.ok || !reserve(CHUNKS)) return plain(dst, src, bytes, s);
    char *to = static_cast<char *>(dst);
    const char *from = static_cast<const char *>(src);
    std::mutex mu;
    std::condition_variable moved, emptied;
    size_t issued = 0;        // chunks whose transfer is queued
    std::vector<char> empty;  // by chunk: emptied
    hipError_t error = hipSuccess;
    auto work = [&](size_t first, size_t step) {
      (void)hipSetDevice(of.device);
      for (size_t k = first; k < n; k += step) {
        {
          std::unique_lock<std::mutex> lock(mu);
          moved.wait(lock, [&] { return issued > k || error != hipSuccess; });
          if (issued <= k) return;  // an error ended the transfers
        }
        const hipError_t e = hipEventSynchronize(event_[k % CHUNKS]);
        if (e == hipSuccess) memcpy(to + k * CHUNK, chunk_[k % CHUNKS], std::min(CHUNK, bytes - k * CHUNK));
        std::lock_guard<std::mutex> lock(mu);
        if (e != hipSuccess) error = e;
        empty[k] = 1;
        emptied.notify_one();
        if (e != hipSuccess) {
          moved.notify_all();
          return;
        }
      }
    };
    std::vector<std::thread> threads;
    try {
      empty.assign(n, 0);
      threads.reserve(THREADS);
      for (size_t t = 0; t < std::min<size_t>(THREADS, n); ++t) threads.emplace_back(work, t, std::min<size_t>(THREADS, n));
    } catch (...) {  // no memory or no threads: let those that started go
      {
        std::lock_guard<std::mutex> lock(mu);
        error = hipErrorOutOfMemory;
        moved.notify_all();
      }
      for (auto &t : threads) t.join();
      return plain(dst, src, bytes, s);
    }
    for (size_t k = 0; k < n; ++k) {
      if (k >= CHUNKS) {
        std::unique_lock<std::mutex> lock(mu);
        emptied.wait(lock, [&] { return empty[k - CHUNKS] || error != hipSuccess; });
        if (error != hipSuccess) break;
      }
      hipError_t e = hipMemcpyAsync(chunk_[k % CHUNKS], from + k * CHUNK, std::min(CHUNK, bytes - k * CHUNK),
                                    hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipEventRecord(event_[k % CHUNKS], s);
      std::lock_guard<std::mutex> lock(mu);
      if (e != hipSuccess) error = e;
      else issued = k + 1;
      moved.notify_all();
      if (e != hipSuccess) break;
    }
    for (auto &t : threads) t.join();
    const hipError_t e = hipStreamSynchronize(s);
    return error != hipSuccess ? error : e;
  }

  void release() {
    for (int k = 0; k < have_; ++k) {
      (void)hipHostFree(chunk_[k]);
      (void)hipEventDestroy(event_[k]);
    }
    have_ = 0;
  }
  Readback() = default;
  Readback(const Readback &) = delete;
  Readback &operator=(const Readback &) = delete;
  ~Readback() { release(); }

 private:
  // The stream's device is current for the scope's length: events belong to
  // the device they are made on, and the caller may have another one current.
  struct OnDevice {
    int device = 0, before = 0;
    bool ok;
    explicit OnDevice(hipStream_t s)
        : ok(hipStreamGetDevice(s, &device) == hipSuccess && hipGetDevice(&before) == hipSuccess &&
             (device == before || hipSetDevice(device) == hipSuccess)) {}
    ~OnDevice() {
      if (ok && device != before) (void)hipSetDevice(before);
    }
  };
  static constexpr size_t LEAST = 16u << 20;  // below, the runtime's copy is as fast

  static hipError_t plain(void *dst, const void *src, size_t bytes, hipStream_t s) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    return e != hipSuccess ? e : hipStreamSynchronize(s);
  }
  bool reserve(int n) {
    for (; have_ < n; ++have_) {
      if (hipHostMalloc(&chunk_[have_], CHUNK, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      if (hipEventCreateWithFlags(&event_[have_], hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipHostFree(chunk_[have_]);
        return false;
      }
    }
    return true;
  }
  std::mutex mu_;
  void *chunk_[CHUNKS] = {};
  hipEvent_t event_[CHUNKS] = {};
  int have_ = 0;
};

}  // namespace lbm
