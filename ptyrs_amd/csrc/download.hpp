// Device complex values to a caller's array of doubles, the form every state leaves the engine
// in: pieces of kPiece bytes go through a pinned ring and are widened into the caller's pages
// while the next ones are copied. A pageable copy of the whole array into a fresh host vector and
// one loop over it took 1.9 ms for a 1136² complex64 object and four 256² modes (the vector's and
// the caller's page faults, the staged copy and the loop one after the other); this takes 0.7.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <memory>
#include <mutex>
#include <thread>

#include "cplx.hpp"

namespace ptyrs {

// One download's pieces. The calling thread makes every runtime call and publishes the pieces as
// they land; whoever claims a published piece widens it. Helpers that come late, because the host's
// cores are taken, find every piece claimed and hold nobody up: with each thread bound to its
// share of the pieces, a first pass beside a program's other busy threads waited up to 7 ms for
// them to start.
struct DownloadJob {
  const char* ring = nullptr;
  size_t piece = 0, slots = 0;  // bytes of a slot, slots
  double* out = nullptr;
  size_t count = 0, per = 0, pieces = 0;  // values, values a piece, pieces
  void (*widen)(const void*, double*, size_t) = nullptr;
  std::atomic<size_t> landed{0}, claimed{0}, widened{0};
  std::unique_ptr<std::atomic<bool>[]> free;  // piece k has left its slot

  // Widens the next published piece; false if there is none unclaimed.
  bool step() {
    size_t k = claimed.load(std::memory_order_relaxed);
    do {
      if (k >= pieces || k >= landed.load(std::memory_order_acquire)) return false;
    } while (!claimed.compare_exchange_weak(k, k + 1, std::memory_order_acq_rel));
    const size_t off = k * per;
    widen(ring + (k % slots) * piece, out + 2 * off, std::min(per, count - off));
    free[k].store(true, std::memory_order_release);
    widened.fetch_add(1, std::memory_order_acq_rel);
    return true;
  }
  // A helper's part: until every piece is claimed.
  void help() {
    while (claimed.load(std::memory_order_acquire) < pieces)
      if (!step()) std::this_thread::yield();
  }
  // No piece is claimed from here on; returns once the claimed ones are done.
  void stop() {
    const size_t k = claimed.exchange(pieces, std::memory_order_acq_rel);
    while (widened.load(std::memory_order_acquire) < std::min(k, pieces))
      std::this_thread::yield();
  }
};

// The process's helper threads, at most kThreads, started when a download first asks for them,
// asleep between downloads and gone after kIdle without one. Never destroyed: a helper asleep at
// the process's end must find its mutex.
class DownloadHelpers {
 public:
  static constexpr int kThreads = 3;
  static constexpr std::chrono::seconds kIdle{10};
  static DownloadHelpers& get() {
    static DownloadHelpers* h = new DownloadHelpers;
    return *h;
  }
  // Up to `n` helpers join `job`. Threads that cannot be had are done without.
  void post(const std::shared_ptr<DownloadJob>& job, int n) noexcept {
    try {
      {
        std::lock_guard<std::mutex> lock(m_);
        for (int i = 0; i < n; ++i) jobs_.push_back(job);
        for (; threads_ < std::min<int>(kThreads, int(jobs_.size())); ++threads_)
          std::thread([this] { loop(); }).detach();
      }
      cv_.notify_all();
    } catch (...) {
    }
  }
  // Forgets what no helper has taken up of `job`.
  void drop(const std::shared_ptr<DownloadJob>& job) {
    std::lock_guard<std::mutex> lock(m_);
    jobs_.erase(std::remove(jobs_.begin(), jobs_.end(), job), jobs_.end());
  }

 private:
  void loop() {
    std::unique_lock<std::mutex> lock(m_);
    while (cv_.wait_for(lock, kIdle, [this] { return !jobs_.empty(); })) {
      const std::shared_ptr<DownloadJob> job = jobs_.front();
      jobs_.pop_front();
      lock.unlock();
      job->help();
      lock.lock();
    }
    --threads_;
  }
  std::mutex m_;
  std::condition_variable cv_;
  std::deque<std::shared_ptr<DownloadJob>> jobs_;
  int threads_ = 0;
};

// One engine's ring. A download is one call at a time (the engine's callers hold it exclusively).
class DownloadRing {
 public:
  static constexpr size_t kPiece = 512 * 1024, kSlots = 8;
  // A helper per 2 MB past the first from kMin on: below it the plain copy is as fast. Once the
  // ring exists smaller downloads take it too, on the calling thread.
  static constexpr size_t kMin = 4 << 20, kPerThread = 2 << 20;

  // Whether a download of `bytes` goes through the ring, which this makes if it is wanted and
  // missing. Pinned memory or events that are refused leave the caller its plain copy.
  bool ready(size_t bytes) {
    if (host_) return bytes >= 2 * kPiece;
    if (bytes < kMin) return false;
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
  hipError_t run(hipStream_t stream, const cplx<T>* src, size_t count, double* out) {
    const size_t bytes = sizeof(cplx<T>) * count;
    auto job = std::make_shared<DownloadJob>();
    DownloadJob& j = *job;
    j.ring = static_cast<const char*>(host_);
    j.piece = kPiece;
    j.slots = kSlots;
    j.out = out;
    j.count = count;
    j.per = kPiece / sizeof(cplx<T>);
    j.pieces = (count + j.per - 1) / j.per;
    j.widen = widen<T>;
    j.free.reset(new std::atomic<bool>[j.pieces]());
    size_t issued = 0, landed = 0;
    hipError_t err = hipSuccess;
    auto issue = [&] {  // every piece whose slot is free
      while (err == hipSuccess && issued < j.pieces &&
             (issued < kSlots || j.free[issued - kSlots].load(std::memory_order_acquire))) {
        const size_t off = issued * j.per, s = issued % kSlots;
        err = hipMemcpyAsync(static_cast<char*>(host_) + s * kPiece, src + off,
                             sizeof(cplx<T>) * std::min(j.per, count - off),
                             hipMemcpyDeviceToHost, stream);
        if (err == hipSuccess) err = hipEventRecord(done_[s], stream);
        if (err == hipSuccess) ++issued;
      }
    };
    auto land = [&] {  // publishes the next issued piece
      err = hipEventSynchronize(done_[landed % kSlots]);
      if (err == hipSuccess) j.landed.store(++landed, std::memory_order_release);
    };
    issue();
    // The first piece waits for the stream's work; helpers are woken only then.
    if (err == hipSuccess) land();
    const size_t helpers =
        bytes < kMin ? 0 : std::min<size_t>(DownloadHelpers::kThreads, bytes / kPerThread - 1);
    if (helpers > 0 && err == hipSuccess) DownloadHelpers::get().post(job, int(helpers));
    while (err == hipSuccess && j.widened.load(std::memory_order_acquire) < j.pieces) {
      issue();
      // A piece for every helper and this thread (a copy takes a tenth of a widening).
      while (err == hipSuccess && landed < issued &&
             landed <= j.claimed.load(std::memory_order_acquire) + helpers)
        land();
      if (err == hipSuccess && !j.step())
        std::this_thread::yield();  // helpers hold the last pieces, or the slots
    }
    j.stop();
    if (helpers > 0) DownloadHelpers::get().drop(job);
    // Whatever a failure left in flight must not write the ring during a later call.
    if (err != hipSuccess) (void)hipStreamSynchronize(stream);
    return err;
  }

 private:
  template <typename T>
  static void widen(const void* src, double* to, size_t len) {
    const T* from = static_cast<const T*>(src);
    if constexpr (sizeof(T) == sizeof(double)) {
      std::memcpy(to, from, sizeof(double) * 2 * len);
    } else {
      for (size_t i = 0; i < 2 * len; ++i) to[i] = double(from[i]);
    }
  }
  hipError_t prepare() {
    for (auto& e : done_) {
      if (e) continue;
      const hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
      if (r != hipSuccess) {
        e = nullptr;
        return r;
      }
    }
    const hipError_t r = hipHostMalloc(&host_, kSlots * kPiece, hipHostMallocDefault);
    if (r != hipSuccess) host_ = nullptr;
    return r;
  }
  void* host_ = nullptr;
  hipEvent_t done_[kSlots] = {};
};

}  // namespace ptyrs
