// Device complex values to a caller's array of doubles, the form every state leaves the engine
// in: pieces of kPiece bytes go through a pinned ring, each worker keeping one piece in flight
// while it widens another into the caller's pages. A pageable copy of the whole array into a
// fresh host vector and one loop over it took 1.9 ms for a 1136² complex64 object and four 256²
// modes (the vector's and the caller's page faults, the staged copy and the loop one after the
// other); this takes 0.7 once the ring is there.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <thread>
#include <vector>

#include "cplx.hpp"

namespace ptyrs {

// One engine's ring. A download is one call at a time (the engine's callers hold it exclusively);
// its workers live for the call.
class DownloadRing {
 public:
  static constexpr int kWorkers = 4;
  static constexpr size_t kPiece = 512 * 1024;
  // A worker per 2 MB from kMin on: the threads cost more than a small download has to gain (2.4 MB
  // with four of them: 0.6 ms a pass slower than the plain copy). Below kMin it is used, on the
  // calling thread, once it exists.
  static constexpr size_t kMin = 4 << 20, kPerWorker = 2 << 20;
  // Large downloads that go without: the ring's pinned memory takes 0.35 ms and its first use as
  // much again in page faults and new threads, more than one download gains (the first pass of an
  // engine in complex128: 512² with one mode 3.7 ms without, 6.7 with; 256² × 2 modes 2.7 and
  // 3.4). A program that takes one result, object and probe, does not pay for it.
  static constexpr int kPlain = 2;

  // Whether a download of `bytes` goes through the ring, which this makes if it is wanted and
  // missing. Pinned memory or events that are refused leave the caller its plain copy.
  bool ready(size_t bytes) {
    if (host_) return bytes >= 2 * kPiece;
    if (bytes < kMin || large_++ < kPlain) return false;
    if (prepare() == hipSuccess) return true;
    (void)hipGetLastError();  // the next launch's check must not report it
    return false;
  }

  DownloadRing() = default;
  DownloadRing(const DownloadRing&) = delete;
  DownloadRing& operator=(const DownloadRing&) = delete;
  ~DownloadRing() {
    for (auto& e : done_)
      if (e) (void)hipEventDestroy(e);
    if (host_) (void)hipHostFree(host_);
  }

  // `count` complex values at `src`, after what `stream` holds, into out[2·count], once the ring
  // is ready.
  template <typename T>
  hipError_t run(int device, hipStream_t stream, const cplx<T>* src, size_t count, double* out) {
    const size_t per = kPiece / sizeof(cplx<T>);
    const size_t pieces = (count + per - 1) / per;
    const size_t bytes = sizeof(cplx<T>) * count;
    const int nw =
        bytes < kMin ? 1 : int(std::min({size_t(kWorkers), bytes / kPerWorker, pieces}));
    hipError_t err[kWorkers] = {};
    auto work = [&](int w) noexcept {
      auto check = [&](hipError_t r) {
        if (r != hipSuccess && err[w] == hipSuccess) err[w] = r;
        return r == hipSuccess;
      };
      auto slot_of = [&](size_t k) { return 2 * w + int(k / size_t(nw) & 1); };
      auto issue = [&](size_t k) {
        const size_t off = k * per, len = std::min(per, count - off);
        const int s = slot_of(k);
        return check(hipMemcpyAsync(at(s), src + off, sizeof(cplx<T>) * len,
                                    hipMemcpyDeviceToHost, stream)) &&
               check(hipEventRecord(done_[s], stream));
      };
      if (!check(hipSetDevice(device))) return;
      size_t next = size_t(w);  // the next piece to issue: two of the worker's are in flight
      for (int i = 0; i < 2 && next < pieces; ++i, next += size_t(nw))
        if (!issue(next)) return;
      for (size_t k = size_t(w); k < pieces; k += size_t(nw)) {
        const int s = slot_of(k);
        if (!check(hipEventSynchronize(done_[s]))) return;
        const size_t off = k * per, len = std::min(per, count - off);
        const T* from = static_cast<const T*>(at(s));
        double* to = out + 2 * off;
        if constexpr (sizeof(T) == sizeof(double)) {
          std::memcpy(to, from, sizeof(double) * 2 * len);
        } else {
          for (size_t i = 0; i < 2 * len; ++i) to[i] = double(from[i]);
        }
        if (next < pieces) {
          if (!issue(next)) return;
          next += size_t(nw);
        }
      }
    };
    std::vector<std::thread> helpers;
    int started = 1;
    try {
      for (; started < nw; ++started) helpers.emplace_back(work, started);
    } catch (...) {
      // No further thread to be had: this one takes the remaining workers' pieces below.
    }
    work(0);
    for (int w = started; w < nw; ++w) work(w);
    for (auto& t : helpers) t.join();
    // Whatever a failed worker left in flight must not write the ring during a later call.
    for (const hipError_t e : err)
      if (e != hipSuccess) {
        (void)hipStreamSynchronize(stream);
        return e;
      }
    return hipSuccess;
  }

 private:
  static constexpr int kSlots = 2 * kWorkers;
  hipError_t prepare() {
    for (auto& e : done_) {
      if (e) continue;
      const hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
      if (r != hipSuccess) {
        e = nullptr;
        return r;
      }
    }
    const hipError_t r =
        hipHostMalloc(&host_, size_t(kSlots) * kPiece, hipHostMallocDefault);
    if (r != hipSuccess) host_ = nullptr;
    return r;
  }
  void* at(int slot) const { return static_cast<char*>(host_) + size_t(slot) * kPiece; }
  void* host_ = nullptr;
  size_t large_ = 0;  // downloads from kMin on before there was a ring
  hipEvent_t done_[kSlots] = {};
};

}  // namespace ptyrs
