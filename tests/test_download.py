"""The state downloads' ring (csrc/download.hpp) on the host: compiled here against a stand-in of
the few runtime calls it makes, whose allocations can be refused and whose copies can fail; alone,
and several rings at once on the shared helpers."""

import shutil
import subprocess

from conftest import ROOT

RUNTIME = r"""
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>
using hipError_t = int;
using hipStream_t = void*;
using hipEvent_t = void*;
constexpr int hipSuccess = 0, hipErrorOutOfMemory = 2;
constexpr int hipEventDisableTiming = 2, hipHostMallocDefault = 0, hipMemcpyDeviceToHost = 2;
inline int refuse_host = 0, refuse_event = -1, last = 0, events = 0, pinned = 0;
inline int copies_left = -1;  // copies until one fails
inline std::thread::id caller;
inline std::atomic<bool> others{false};  // a runtime call from another thread than the caller's
inline hipError_t hipGetLastError() { int e = last; last = 0; return e; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  if (refuse_event >= 0 && events >= refuse_event) return last = hipErrorOutOfMemory;
  ++events;
  *e = std::malloc(1);
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { --events; std::free(e); return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (refuse_host) return last = hipErrorOutOfMemory;
  ++pinned;
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { --pinned; std::free(p); return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) {
  if (std::this_thread::get_id() != caller) others = true;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  if (std::this_thread::get_id() != caller) others = true;
  if (copies_left == 0) return hipErrorOutOfMemory;
  if (copies_left > 0) --copies_left;
  std::memcpy(d, s, n);
  return hipSuccess;
}
"""

CPLX = """
#pragma once
namespace ptyrs {
template <typename T> struct cplx { T x, y; };
}
"""

PROGRAM = r"""
#include <cstdio>
#include "download.hpp"
using namespace ptyrs;

#define CHECK(x) if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }

// Whether a download of `count` values comes back whole through a ring made by a large one.
template <typename T>
bool whole(DownloadRing& ring, size_t count) {
  std::vector<cplx<T>> src(count);
  for (size_t i = 0; i < count; ++i) src[i] = {T(i), T(-0.5 * double(i))};
  std::vector<double> out(2 * count, 1e300);
  if (ring.run(nullptr, src.data(), count, out.data()) != hipSuccess) return false;
  for (size_t i = 0; i < count; ++i)
    if (out[2 * i] != double(src[i].x) || out[2 * i + 1] != double(src[i].y)) return false;
  return true;
}

template <typename T>
int run() {
  const size_t large = 32 << 20, mid = 2 << 20, small = 100000;
  {
    DownloadRing ring;  // nothing to be had: no ring, no error left, and no second try fails
    refuse_host = 1;
    CHECK(!ring.ready(large) && last == 0);
    CHECK(!ring.ready(large) && last == 0);
    CHECK(!ring.ready(mid) && pinned == 0);
    refuse_host = 0;  // memory again: the ring is made
    CHECK(ring.ready(large) && pinned == 1);
  }
  CHECK(pinned == 0 && events == 0);
  {
    DownloadRing ring;
    CHECK(!ring.ready(mid) && events == 0);
    refuse_event = 3;
    CHECK(!ring.ready(large) && last == 0 && pinned == 0);
    refuse_event = -1;
    CHECK(ring.ready(large) && ring.ready(mid) && !ring.ready(small));
    const size_t piece = DownloadRing::kPiece / sizeof(cplx<T>);
    for (size_t count : {size_t(1), piece, piece + 1, 2 * piece, 8 * piece - 1, 17 * piece + 3,
                         40 * piece})
      for (int i = 0; i < 5; ++i) CHECK(whole<T>(ring, count));
    // A copy that fails ends the download with its error, and the ring serves the next one.
    std::vector<cplx<T>> src(40 * piece);
    std::vector<double> out(2 * src.size());
    for (int k : {0, 1, 7, 8, 13, 39}) {
      copies_left = k;
      CHECK(ring.run(nullptr, src.data(), src.size(), out.data()) == hipErrorOutOfMemory);
      copies_left = -1;
      CHECK(whole<T>(ring, src.size()));
    }
  }
  CHECK(pinned == 0 && events == 0);
  CHECK(!others);  // the helpers only widen
  {  // several engines' rings at once, sharing the helpers
    std::atomic<int> bad{0};
    std::vector<std::thread> threads;
    std::vector<DownloadRing> rings(6);
    for (auto& r : rings) CHECK(r.ready(large));
    for (auto& r : rings)
      threads.emplace_back([&] {
        for (int i = 0; i < 10; ++i) bad += !whole<T>(r, 700000);
      });
    for (auto& t : threads) t.join();
    CHECK(bad == 0);
  }
  return 0;
}

int main() {
  caller = std::this_thread::get_id();
  if (run<float>()) return 1;
  others = false;
  return run<double>();
}
"""


def test_ring_on_the_host(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "cplx.hpp").write_text(CPLX)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    shutil.copy(ROOT / "ptyrs_amd" / "csrc" / "download.hpp", tmp_path)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(tmp_path),
                    str(tmp_path / "main.cpp"), "-o", str(tmp_path / "main")], check=True)
    run = subprocess.run([str(tmp_path / "main")], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
