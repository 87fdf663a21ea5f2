// Explicit diffusion sweeps diff_x, diff_y, diff_z (src/Diffusion.F90:
// 266-650) in place on ts0.
//
// The factors of a cell's two interfaces (three divisions each) do not
// depend on the bin: a wave forms them once and keeps them in registers for
// every bin of its group, with the next bin's cells in flight.  x rows: a
// workgroup per row, the neighbours through LDS.  y and z lines: 64
// neighbouring lines x M cells per wave, the waves of a workgroup stacked
// along the line.  A workgroup's waves load a bin before any of them stores
// it (one barrier per bin); where a line takes several workgroups, the rows
// at their borders are copied to the ts1 slot beforehand and read from there.
// The ghost cells along the lines are not read: they hold the edge cells
// (periodic x: the wrapped ones, :317-327).  Bound by HBM latency and
// bandwidth; 181x133x41x7 (6.9 M bin-cells): x, y, z 25, 40 (borders included), 27 us against
// 254 (with the transposes of the state that the x lines went through), 147
// and 58 us for one thread per line.
// The arithmetic is the reference's, expression by expression.
#include <algorithm>

#include "common.hpp"

namespace ash3d {

namespace {

struct ExpArgs {
  DiffArgs A;
  int periodic;      // x lines only
  int groups, bins;  // bin groups, bins per group
};

// lets a barrier order the LDS accesses (and, since every load that precedes
// it has been waited for, a workgroup's global loads before its later stores)
// without draining the loads in flight
__device__ __forceinline__ void wg_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// the value is in its register (its load has returned)
__device__ __forceinline__ void arrived(double &v) { asm volatile("" : "+v"(v)); }

// kds of interface I times dt (:357-359)
__device__ __forceinline__ double exp_factor(double dt, double sig, double kapm, double kap0, double Km, double K0) {
  const double ds = 2.0 * sig / (kapm + kap0);
  const double kds = 0.5 * (Km + K0) * ds;
  return dt * kds;
}

// One workgroup per x row (j, k): CPT cells per thread, cell c = tid +
// blockDim.x * m + 1.
template <int CPT>
__global__ __launch_bounds__(1024) void k_diff_explicit_x(ExpArgs T) {
  extern __shared__ double s_row[];  // two rows, by bin parity
  const DiffArgs &A = T.A;
  const Dims d = A.d;
  const int nx = d.nx, tid = threadIdx.x, BT = blockDim.x;
  const TileGroup tg = xcd_tile_group(blockIdx.x, T.groups);
  if (tg.tile >= (long long)d.ny * d.nz) return;  // padding workgroup (uniform)
  const int j = (int)(tg.tile % d.ny) + 1, k = (int)(tg.tile / d.ny) + 1;
  const bool line_on = j >= A.g.a0 && j <= A.g.a1 && k >= A.g.b0 && k <= A.g.b1;
  const long long o = d.p3(0, j, k), ok = kline_base(d, 0, j, k);  // cell 0
  const int nlo = tg.group * T.bins, nhi = min(nlo + T.bins, d.ns);
  int cell[CPT];
  bool in[CPT], keep[CPT];
  double A0[CPT], A1[CPT], sL[CPT], sR[CPT], qs[CPT];
#pragma unroll
  for (int m = 0; m < CPT; ++m) {
    const int c = tid + BT * m + 1;
    in[m] = c <= nx;
    cell[m] = min(c, nx);
    keep[m] = line_on && c >= A.g.rmin && c <= A.g.rmax;
    const int q = cell[m];
    const double kl = A.kap[o + q - 1], kc = A.kap[o + q], kr = A.kap[o + q + 1];
    const double s0 = A.sig[o + q], s1 = A.sig[o + q + 1];
    const double K0 = A.kk[ok + q];
    A0[m] = exp_factor(A.dt, s0, kl, kc, A.kk[ok + q - 1], K0);
    A1[m] = exp_factor(A.dt, s1, kc, kr, K0, A.kk[ok + q + 1]);
    sL[m] = s0 / kc;
    sR[m] = s1 / kc;
    qs[m] = A.c0[o + q + d.ncell * (long long)nlo];
  }
  for (int n = nlo; n < nhi; ++n) {
    double *s = s_row + (long long)(n & 1) * BT * CPT;
    double q[CPT];
#pragma unroll
    for (int m = 0; m < CPT; ++m) {
      q[m] = qs[m];
      if (in[m]) s[cell[m] - 1] = q[m];
    }
    const long long bn = d.ncell * (long long)min(n + 1, nhi - 1);
#pragma unroll
    for (int m = 0; m < CPT; ++m) qs[m] = A.c0[o + cell[m] + bn];
    wg_barrier();
    const bool on = A.aloft.on(n);
    double *c = A.c0 + d.ncell * (long long)n;
#pragma unroll
    for (int m = 0; m < CPT; ++m) {
      const int p = cell[m];
      const int l = p > 1 ? p - 1 : (T.periodic ? nx : 1), r = p < nx ? p + 1 : (T.periodic ? 1 : nx);
      const double dm = q[m] - s[l - 1], dp = s[r - 1] - q[m];
      const double LF = A1[m] * dp * sR[m];    // (:367-372)
      const double RF = -(A0[m] * dm * sL[m]);
      const double res = q[m] + (LF + RF);
      if (in[m]) c[o + p] = (on && keep[m]) ? res : 0.0;
    }
  }
}

// the rows on both sides of every border between the workgroups of a line
// (lines of DIR, rows per workgroup R) from c to halo, every line and bin
template <int DIR>
__global__ __launch_bounds__(256) void k_border_rows(Dims d, LineGeom g, int R, const double *c, double *halo) {
  const unsigned na = (unsigned)(g.Na + 255) / 256, nr = 2 * (unsigned)((g.N - 1) / R);  // rows R, R+1, 2R, 2R+1, ...
  const int a = (int)(blockIdx.x % na) * 256 + (int)threadIdx.x + 1;
  if (a > g.Na) return;
  const int q = (int)(blockIdx.x / na % nr), b = (int)(blockIdx.x / na / nr) + 1;
  const int r = R * (q / 2 + 1) + (q & 1);
  const long long o = line_base(d, DIR, a, b) + line_stride(d, DIR) * (long long)(r + 1);
  for (int n = blockIdx.y; n < d.ns; n += gridDim.y) halo[o + d.ncell * (long long)n] = c[o + d.ncell * (long long)n];
}

template <int DIR, int M>
__global__ __launch_bounds__(512) void k_diff_explicit_tile(ExpArgs T) {
  const DiffArgs &A = T.A;
  const Dims d = A.d;
  const LineGeom g = A.g;
  const int N = g.N, rmin = g.rmin, rmax = g.rmax;
  const int ntile = (g.Na + 63) / 64;
  const int S = (int)blockDim.y, LB = (N + M * S - 1) / (M * S);
  const TileGroup tg = xcd_tile_group(blockIdx.x, T.groups);
  if (tg.tile >= (long long)ntile * LB * g.Nb) return;  // padding workgroup (uniform)
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  const int a0 = (int)(tg.tile % ntile) * 64 + 1;
  const long long rest = tg.tile / ntile;
  const int b = (int)(rest / LB) + 1;
  const int r0 = 1 + ((int)(rest % LB) * S + w) * M;  // first cell of the tile (past the line: barriers only)
  // lanes past the last line repeat it: the same loads, values and stores
  const int al = min((int)threadIdx.x, g.Na - a0), a = a0 + al;
  const bool line_on = a >= g.a0 && a <= g.a1 && b >= g.b0 && b <= g.b1;
  const long long sL = line_stride(d, DIR), base = line_base(d, DIR, a, b);
  const long long kS = kline_stride(d, DIR), kB = kline_base(d, DIR, a, b);
  const int nlo = tg.group * T.bins, nhi = min(nlo + T.bins, d.ns);
  auto row = [&](int r) { return base + sL * (long long)(r + 1); };
  // A tile with no line or cell of the box, and a bin that is not aloft, are
  // stored as zeros and not read (uniform): y and z of a 5x5x4 box at
  // 360x240x50x15 193 us each against 284 and 290 with every tile read.  Bit
  // n - nlo of run: bin n is swept here
  const unsigned group = (1u << (nhi - nlo)) - 1, on = A.aloft.bits(nlo, nhi);
  const bool in_box = a0 <= g.a1 && a0 + 63 >= g.a0 && b >= g.b0 && b <= g.b1 && r0 <= rmax && r0 + M > rmin;
  const unsigned run = in_box ? on : 0u;
  for (unsigned z = group & ~run; z; z &= z - 1) {
    const int u = __builtin_ctz(z);
    if (on >> u & 1) wg_barrier();  // (other waves read this tile's edge cells)
    double *c = A.c0 + d.ncell * (long long)(nlo + u);
#pragma unroll
    for (int i = 0; i < M; ++i)
      if (r0 + i <= N) c[row(r0 + i)] = 0.0;
  }
  if (!run) return;
  // the neighbouring workgroups' rows come from the copies
  const double *below = w == 0 && r0 > 1 ? A.scratch_b : A.c0;
  const double *above = w == S - 1 && r0 + M <= N ? A.scratch_b : A.c0;
  double f[M + 1], fl[M], fr[M];
  {
    double kp[M + 2], K[M + 2], sg[M + 1];
#pragma unroll
    for (int i = 0; i < M + 2; ++i) {
      const int r = min(r0 - 1 + i, N + 1);
      kp[i] = A.kap[row(r)];
      K[i] = A.kk[kB + kS * (long long)r];
    }
#pragma unroll
    for (int i = 0; i <= M; ++i) sg[i] = A.sig[row(min(r0 + i, N + 1))];
#pragma unroll
    for (int i = 0; i <= M; ++i) f[i] = exp_factor(A.dt, sg[i], kp[i], kp[i + 1], K[i], K[i + 1]);
#pragma unroll
    for (int i = 0; i < M; ++i) {
      fl[i] = sg[i] / kp[i + 1];
      fr[i] = sg[i + 1] / kp[i + 1];
    }
  }
  double qs[M + 2];
  auto fetch = [&](int n) {
    const long long bo = d.ncell * (long long)n;
    qs[0] = below[row(min(max(r0 - 1, 1), N)) + bo];
#pragma unroll
    for (int i = 1; i <= M; ++i) qs[i] = A.c0[row(min(r0 - 1 + i, N)) + bo];
    qs[M + 1] = above[row(min(r0 + M, N)) + bo];
  };
  fetch(nlo + __builtin_ctz(run));
  for (unsigned left = run; left; left &= left - 1) {
    const int n = nlo + __builtin_ctz(left);
    double q[M + 2];
#pragma unroll
    for (int i = 0; i < M + 2; ++i) {
      q[i] = qs[i];
      arrived(q[i]);
    }
    const unsigned next = left & (left - 1);
    fetch(nlo + __builtin_ctz(next ? next : left));
    wg_barrier();  // every load of the bin before its first store
    double *c = A.c0 + d.ncell * (long long)n;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const int r = r0 + i;
      const double LF = f[i + 1] * (q[i + 2] - q[i + 1]) * fr[i];
      const double RF = -(f[i] * (q[i + 1] - q[i]) * fl[i]);
      const double res = q[i + 1] + (LF + RF);
      if (r <= N) c[row(r)] = (line_on && r >= rmin && r <= rmax) ? res : 0.0;
    }
  }
}

template <int DIR, int M>
hipError_t launch_tile(hipStream_t s, ExpArgs t) {
  const DiffArgs &a = t.A;
  const int S = std::min(8, (a.g.N + M - 1) / M), LB = (a.g.N + M * S - 1) / (M * S);
  if (LB > 1) {
    const long long items = 2LL * (LB - 1) * a.g.Nb * ((a.g.Na + 255) / 256);
    hipLaunchKernelGGL((k_border_rows<DIR>), dim3((unsigned)items, std::min(a.d.ns, 64)), dim3(256), 0, s, a.d, a.g,
                       M * S, a.c0, a.scratch_b);
  }
  const long long tiles = (long long)((a.g.Na + 63) / 64) * LB * a.g.Nb;
  // bin groups: two waves per SIMD, at most 8 bins
  const long long want = std::max<long long>((2048 + tiles * S - 1) / (tiles * S), (a.d.ns + 7) / 8);
  t.groups = (int)std::min<long long>(a.d.ns, want);
  t.bins = (a.d.ns + t.groups - 1) / t.groups;
  t.groups = (a.d.ns + t.bins - 1) / t.bins;
  const long long blocks = padded_tiles(tiles) * t.groups;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_diff_explicit_tile<DIR, M>), dim3((unsigned)blocks), dim3(64, S), 0, s, t);
  return hipGetLastError();
}

template <int CPT>
hipError_t launch_x(hipStream_t s, ExpArgs t, int bt) {
  const long long rows = (long long)t.A.d.ny * t.A.d.nz;
  const long long want = (2048 + rows * (bt / 64) - 1) / (rows * (bt / 64));
  t.groups = (int)std::max<long long>(1, std::min<long long>(t.A.d.ns, want));
  t.bins = (t.A.d.ns + t.groups - 1) / t.groups;
  t.groups = (t.A.d.ns + t.bins - 1) / t.bins;
  const long long blocks = padded_tiles(rows) * t.groups;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  const size_t lds = sizeof(double) * 2 * (size_t)bt * CPT;
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute((const void *)k_diff_explicit_x<CPT>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_diff_explicit_x<CPT>), dim3((unsigned)blocks), dim3(bt), lds, s, t);
  return hipGetLastError();
}

// x rows longer than one workgroup holds: from a copy of the state in the
// ts1 slot, a thread per cell
__global__ __launch_bounds__(256) void k_copy_rows(Dims d, const double *c, double *to) {
  const long long o = d.p3(1, (int)(blockIdx.x % (unsigned)d.ny) + 1, (int)(blockIdx.x / (unsigned)d.ny) + 1) +
                      d.ncell * (long long)blockIdx.y;
  for (int i = threadIdx.x; i < d.nx; i += 256) to[o + i] = c[o + i];
}
__global__ __launch_bounds__(256) void k_diff_explicit_cells(ExpArgs T) {
  const DiffArgs &A = T.A;
  const Dims d = A.d;
  const int nx = d.nx, n = blockIdx.y;
  const int j = (int)(blockIdx.x % (unsigned)d.ny) + 1, k = (int)(blockIdx.x / (unsigned)d.ny) + 1;
  const bool on = A.aloft.on(n) && j >= A.g.a0 && j <= A.g.a1 && k >= A.g.b0 && k <= A.g.b1;
  const long long o = d.p3(0, j, k), ok = kline_base(d, 0, j, k), bn = d.ncell * (long long)n;
  for (int p = threadIdx.x + 1; p <= nx; p += 256) {
    const int l = p > 1 ? p - 1 : (T.periodic ? nx : 1), r = p < nx ? p + 1 : (T.periodic ? 1 : nx);
    const double q = A.scratch_b[o + bn + p], dm = q - A.scratch_b[o + bn + l], dp = A.scratch_b[o + bn + r] - q;
    const double kc = A.kap[o + p], s0 = A.sig[o + p], s1 = A.sig[o + p + 1], K0 = A.kk[ok + p];
    const double f0 = exp_factor(A.dt, s0, A.kap[o + p - 1], kc, A.kk[ok + p - 1], K0);
    const double f1 = exp_factor(A.dt, s1, kc, A.kap[o + p + 1], K0, A.kk[ok + p + 1]);
    const double LF = f1 * dp * (s1 / kc);
    const double RF = -(f0 * dm * (s0 / kc));
    const double res = q + (LF + RF);
    A.c0[o + bn + p] = (on && p >= A.g.rmin && p <= A.g.rmax) ? res : 0.0;
  }
}

}  // namespace

hipError_t launch_diff_explicit(hipStream_t s, const DiffArgs &a, int periodic) {
  ExpArgs t{a, a.g.dir == 0 ? periodic : 0, 1, a.d.ns};
  if (a.g.dir == 1) return launch_tile<1, 8>(s, t);
  if (a.g.dir == 2) return launch_tile<2, 8>(s, t);
  // x rows: 256 threads or fewer where four cells each hold the row
  const int nx = a.d.nx;
  const int cpt = nx <= 256 ? 1 : nx <= 512 ? 2 : nx <= 1024 ? 4 : 8;
  const int bt = ((nx + cpt - 1) / cpt + 63) / 64 * 64;
  if (bt > 1024) {
    const long long rows = (long long)a.d.ny * a.d.nz;
    if (rows > 0x7fffffffLL || a.d.ns > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_copy_rows, dim3((unsigned)rows, a.d.ns), dim3(256), 0, s, a.d, a.c0, a.scratch_b);
    hipLaunchKernelGGL(k_diff_explicit_cells, dim3((unsigned)rows, a.d.ns), dim3(256), 0, s, t);
    return hipGetLastError();
  }
  switch (cpt) {
    case 1: return launch_x<1>(s, t, bt);
    case 2: return launch_x<2>(s, t, bt);
    case 4: return launch_x<4>(s, t, bt);
    default: return launch_x<8>(s, t, bt);
  }
}

}  // namespace ash3d
