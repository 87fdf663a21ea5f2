// download_levels (csrc/host_state.hip) against a runtime that defers every
// copy until it is waited for, and fails at a chosen call: whatever fails, no
// copy is left to write the caller's array after the return, and without a
// failure both levels arrive.
//   readback_errors CALL COUNT   CALL: copy, record, wait, none; the
//   COUNT-th call of that kind (from 0) fails
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <string>
#include <vector>

#include "common.hpp"

namespace {

std::string fail_call;
int fail_count = 0;
struct Copy { double *to; const double *from; size_t bytes; };
std::deque<Copy> queue;        // enqueued, not carried out
long long enqueued = 0, done = 0;
std::map<hipEvent_t, long long> marks;

bool fails(const char *call) { return fail_call == call && fail_count-- == 0; }
void run_until(long long n) {
  for (; done < n; ++done) {
    std::memcpy(queue.front().to, queue.front().from, queue.front().bytes);
    queue.pop_front();
  }
}

}  // namespace

extern "C" {
hipError_t hipMemcpyAsync(void *to, const void *from, size_t bytes, hipMemcpyKind, hipStream_t) {
  if (fails("copy")) return hipErrorInvalidValue;
  queue.push_back({(double *)to, (const double *)from, bytes});
  ++enqueued;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  if (fails("record")) return hipErrorInvalidValue;
  marks[e] = enqueued;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (fails("wait")) return hipErrorInvalidValue;
  run_until(marks[e]);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  run_until(enqueued);
  return hipSuccess;
}
}

namespace ash3d {
// (the stream's kernels run at once: the device level they write is copied later)
hipError_t launch_fill(hipStream_t, double *p, long long n, double v) {
  for (long long q = 0; q < n; ++q) p[q] = v;
  return hipSuccess;
}
hipError_t launch_mirror_interior(hipStream_t, const Dims &d, const double *c0, double *c1, long long r0, long long r1) {
  for (long long q = r0 * d.sy; q < r1 * d.sy; ++q) {
    const long long cell = q % d.ncell;
    const int i = (int)(cell % d.sy) - 1, j = (int)(cell / d.sy % (d.ny + 4)) - 1, k = (int)(cell / d.sz) - 1;
    c1[q] = i >= 1 && i <= d.nx && j >= 1 && j <= d.ny && k >= 1 && k <= d.nz ? c0[q] : 0.0;
  }
  return hipSuccess;
}
}  // namespace ash3d

int main(int argc, char **argv) {
  if (argc != 3) return 2;
  fail_call = argv[1];
  fail_count = std::atoi(argv[2]);
  const bool expect = fail_call != "none";
  const ash3d::Dims d = ash3d::make_dims(95, 60, 44, 16);  // 39 MB a level
  const size_t n = (size_t)(d.ncell * d.ns);
  std::vector<double> c0(n), c1(n, -2.0), want(n), host(2 * n, -1.0);
  for (size_t q = 0; q < n; ++q) c0[q] = 1.0 + (double)q;
  ash3d::launch_mirror_interior(nullptr, d, c0.data(), want.data(), 0, (long long)n / d.sy);
  long long dummy[ash3d::kReadbackEvents];
  hipEvent_t ev[ash3d::kReadbackEvents];
  for (int q = 0; q < ash3d::kReadbackEvents; ++q) ev[q] = (hipEvent_t)&dummy[q];
  const hipError_t e = ash3d::download_levels(nullptr, d, false, c0.data(), c1.data(), host.data(), ev);
  if ((e != hipSuccess) != expect) return std::printf("returned %d\n", (int)e), 1;
  if (!queue.empty()) return std::printf("%zu copies left to write the array\n", queue.size()), 1;
  if (!expect && (std::memcmp(host.data(), c0.data(), n * 8) || std::memcmp(host.data() + n, want.data(), n * 8)))
    return std::printf("levels differ\n"), 1;
  std::printf("ok\n");
  return 0;
}
