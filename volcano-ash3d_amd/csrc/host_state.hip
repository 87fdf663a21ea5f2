// Reading the state back when the ts1 slot follows from ts0 (zero, or ts0's
// interior with zero ghosts).
//
// Both levels over the link take twice the time of one (57 GB/s measured on
// PCIe Gen5 x16; the largest states' forecasts spent a quarter of their time
// there), so only ts0 is sure to cross it: host threads write the ts1 level
// from the rows of ts0 that have arrived, with stores that bypass the caches,
// while the copies go on.  How fast they are depends on the machine, so once
// ts0 is enqueued the link takes rows of ts1 too, from the end of the level,
// until it meets the threads: with no thread at all everything is copied, as
// before.  37 MB per level (120x80x40x10) 1.35 -> 0.90 ms, 576 MB
// (360x240x50x15) 20.4 -> 10.8, 2.8 GB (1440x720x80x4) 99.5 -> 52.0; while the
// pages of the caller's array are not mapped to the process yet (pinned
// memory that only the device has written), which the threads pay 4 us a
// page for: 1.55, 19.1 and 92.2.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "common.hpp"

namespace ash3d {

namespace {

constexpr int kDepth = 4;    // copies in flight
// Threads besides the caller's: four write as fast as the link delivers, and
// more as the level grows, for memory whose pages are not mapped yet.
constexpr int kThreadsMin = 4, kThreadsMax = 12;
constexpr long long kPerThread = 32ll << 20;
// Below this size of a level both levels are copied: the threads' start
// costs what they save (10 MB: 400 us copied, 340 with threads; 3 MB: 151
// and 167).
constexpr long long kMinLevel = 16ll << 20;
constexpr long long kCopyMin = 4ll << 20, kCopyMax = 32ll << 20;  // of one copy (70 us, 0.6 ms)
constexpr long long kTakeMin = 16ll << 10, kTakeMax = 256ll << 10;  // of what a thread takes at a time

typedef double Pair __attribute__((ext_vector_type(2)));

// dst[0..n) = src[0..n), or zeros (src null), past the caches
void stream_out(double *dst, const double *src, long long n) {
  long long q = 0;
  if (n > 0 && ((uintptr_t)dst & 15)) {
    __builtin_nontemporal_store(src ? src[0] : 0.0, dst);
    q = 1;
  }
  for (; q + 1 < n; q += 2) {
    const Pair v = src ? Pair{src[q], src[q + 1]} : Pair{0.0, 0.0};
    __builtin_nontemporal_store(v, (Pair *)(dst + q));
  }
  if (q < n) __builtin_nontemporal_store(src ? src[q] : 0.0, dst + q);
}

// Rows are x rows of the level (nx + 4 cells), the slowest index last.
struct Readback {
  Dims d;
  bool zero;            // ts1 is zero throughout
  double *h0, *h1;      // the host levels
  std::mutex m;
  std::condition_variable cv;
  long long ready = 0;  // rows of ts0 that have arrived
  long long front = 0, back = 0;  // rows of ts1 not taken yet
  bool stop = false;

  void write_rows(long long r0, long long r1) {
    const int ny4 = d.ny + 4, nz4 = d.nz + 4;
    for (long long r = r0; r < r1; ++r) {
      const int j = (int)(r % ny4) - 1, k = (int)((r / ny4) % nz4) - 1;
      double *dst = h1 + r * d.sy;
      if (zero || j < 1 || j > d.ny || k < 1 || k > d.nz) {
        stream_out(dst, nullptr, d.sy);
      } else {
        stream_out(dst, nullptr, 2);
        stream_out(dst + 2, h0 + r * d.sy + 2, d.nx);
        stream_out(dst + 2 + d.nx, nullptr, 2);
      }
    }
  }

  void work() {
    using clock = std::chrono::steady_clock;
    const long long row_b = d.sy * 8;
    long long take = kTakeMin;
    for (;;) {
      long long r0, r1;
      {
        std::unique_lock<std::mutex> lk(m);
        r0 = front;
        r1 = std::min(back, r0 + std::max(1ll, take / row_b));
        if (stop || r0 >= r1) break;
        front = r1;
        if (!zero) cv.wait(lk, [&] { return stop || ready >= r1; });
        if (stop) break;
      }
      const auto t0 = clock::now();
      write_rows(r0, r1);
      // memory that this process touches for the first time takes 20 times
      // as long (a page fault every 4 KB): small pieces there, so that the
      // link is not kept waiting for the last of them
      if (clock::now() - t0 > std::chrono::microseconds(50)) take = std::max(kTakeMin, take / 4);
      else take = std::min(kTakeMax, take * 2);
    }
    // the stores above become visible before the caller sees the thread end
    std::atomic_thread_fence(std::memory_order_seq_cst);
  }

  void arrived(long long r) {
    {
      std::lock_guard<std::mutex> lk(m);
      ready = r;
    }
    cv.notify_all();
  }
};

struct Threads {
  Readback *w;
  std::vector<std::thread> t;
  ~Threads() {
    for (auto &x : t) x.join();
  }
};

}  // namespace

hipError_t download_levels(hipStream_t s, const Dims &d, bool zero, const double *c0, double *c1, double *host,
                           hipEvent_t *ev) {
  static_assert(kDepth == kReadbackEvents, "one event per copy in flight");
  const long long n = d.ncell * d.ns, rows = n / d.sy;
  if (n * 8 < kMinLevel) {
    hipError_t e = zero ? launch_fill(s, c1, n, 0.0) : launch_mirror_interior(s, d, c0, c1, 0, rows);
    return e != hipSuccess ? e : hipMemcpyAsync(host, c0, 2 * sizeof(double) * (size_t)n, hipMemcpyDeviceToHost, s);
  }
  Readback w;
  w.d = d;
  w.zero = zero;
  w.h0 = host;
  w.h1 = host + n;
  const long long row_b = d.sy * 8;
  const long long chunk = std::max((kCopyMin + row_b - 1) / row_b, std::min(rows / 16, kCopyMax / row_b));
  w.back = rows;
  Threads pool{&w, {}};
  hipError_t e = hipSuccess;
  long long end[kDepth] = {};  // rows of ts0 complete with each event (0: a copy of ts1)
  long long issued = 0, waited = 0, r0 = 0;
  auto wait_one = [&]() {
    const int q = (int)(waited++ % kDepth);
    e = hipEventSynchronize(ev[q]);
    if (e == hipSuccess && end[q]) w.arrived(end[q]);
  };
  bool started = false;
  auto start = [&]() {
    started = true;
    cpu_set_t set;
    const int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
    const int nt = std::min(cpus - 1, (int)std::clamp<long long>(8 * n / kPerThread, kThreadsMin, kThreadsMax));
    try {
      for (int q = 0; q < nt; ++q) pool.t.emplace_back([&w] { w.work(); });
    } catch (const std::exception &) {
      // (the threads that did start; the link takes the rest)
    }
  };
  while (e == hipSuccess) {
    if (issued - waited == kDepth) {
      if (!started) start();  // (the first copies under way)
      wait_one();
      continue;
    }
    const double *src = c0;
    long long a = r0, b = std::min(rows, r0 + chunk);
    if (a < b) {
      r0 = b;
    } else {
      if (!started) start();
      // rows of ts1 from the end, where the threads are behind
      std::unique_lock<std::mutex> lk(w.m);
      if (!zero && waited < issued && w.front + 2 * chunk >= w.ready) {
        lk.unlock();
        wait_one();
        continue;
      }
      if (waited == issued && !pool.t.empty() && w.back - w.front <= 2 * chunk) break;  // (theirs)
      a = std::max(w.front, w.back - std::max(chunk, (w.back - w.front) / 4));
      b = w.back;
      w.back = a;
      src = c1;
    }
    if (a >= b) break;
    const int q = (int)(issued % kDepth);
    if (src == c1)
      e = zero ? launch_fill(s, c1 + a * d.sy, (b - a) * d.sy, 0.0) : launch_mirror_interior(s, d, c0, c1, a, b);
    if (e == hipSuccess)
      e = hipMemcpyAsync((src == c0 ? w.h0 : w.h1) + a * d.sy, src + a * d.sy, sizeof(double) * (size_t)((b - a) * d.sy),
                         hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipEventRecord(ev[q], s);
    if (e == hipSuccess) {
      end[q] = src == c0 ? b : 0;
      ++issued;
    }
  }
  while (e == hipSuccess && waited < issued) wait_one();
  if (e != hipSuccess) {
    {
      std::lock_guard<std::mutex> lk(w.m);
      w.stop = true;
    }
    // (no copy may write the caller's array after the call)
    (void)hipStreamSynchronize(s);
  }
  w.cv.notify_all();
  return e;
}

}  // namespace ash3d
