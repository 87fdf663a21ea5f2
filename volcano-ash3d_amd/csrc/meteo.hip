// Per-step driver work that the reference does on the host between the
// hot-path calls, kept on the device so that the state never leaves HBM:
//   * wind time interpolation between two met steps
//     (src/MesoInterpolater.f90:203-230),
//   * the CFL and diffusion maxima of Adjust_DT (src/Adjust_dt.f90:96-285),
//   * the slab maxima of get_minmax_index (src/Calc_Mesh.f90:459-511).
// Maxima and minima are exact in any order, so the reductions (per-block
// partials, then a fixed-order host pass) reproduce the reference's loops
// bit for bit.
#include "common.hpp"

namespace ash3d {

namespace {

constexpr double MPS_2_KMPHR = 3.6;  // src/Ash3d_VariableModules.f90:286

// v_pd(1:nx,1:ny,1:nz) = (real(last) + real(next - last) * frac) * 3.6,
// the difference in FP32 as the _sp arrays give it.  A wave takes SEG cells of
// an x row of the unpadded FP32 arrays: blockIdx.y 0 the three winds, n bin
// n - 1's fall speed.  Bound by HBM bandwidth.  With fall speeds 256 cells,
// four loads of a bin in flight: 1.0 GB of 360x240x50x15 in 238 us, 250 with
// a whole row per wave and 298 with the indices of every cell divided out.
// The winds alone 64 cells: 720x360x70 173 us, 201 with a whole row.
constexpr int kRow = 256;  // threads per workgroup

template <int SEG>
__global__ __launch_bounds__(kRow) void k_met_interp(Dims d, const float *__restrict__ lx, const float *__restrict__ ly,
                                                    const float *__restrict__ lz, const float *__restrict__ lf,
                                                    const float *__restrict__ nx_, const float *__restrict__ ny_,
                                                    const float *__restrict__ nz_, const float *__restrict__ nf,
                                                    double frac, double *vx, double *vy, double *vz, double *vf) {
  const unsigned segs = (unsigned)(d.nx + SEG - 1) / SEG;
  const unsigned item = blockIdx.x * (kRow / 64) + threadIdx.x / 64, r = segs == 1 ? item : item / segs;
  if (r >= (unsigned)d.ny * (unsigned)d.nz) return;
  const int i0 = (int)(item - r * segs) * SEG + (int)(threadIdx.x & 63), end = min(i0 + SEG, d.nx);
  const long long o = d.p3(1, (int)(r % (unsigned)d.ny) + 1, (int)(r / (unsigned)d.ny) + 1);
  const long long m = (long long)d.nx * r;
  if (blockIdx.y == 0) {
#pragma unroll 2
    for (int i = i0; i < end; i += 64) {
      const float ax = lx[m + i], ay = ly[m + i], az = lz[m + i];
      const float dx = nx_[m + i] - ax, dy = ny_[m + i] - ay, dz = nz_[m + i] - az;
      vx[o + i] = ((double)ax + (double)dx * frac) * MPS_2_KMPHR;
      vy[o + i] = ((double)ay + (double)dy * frac) * MPS_2_KMPHR;
      vz[o + i] = ((double)az + (double)dz * frac) * MPS_2_KMPHR;
    }
  } else {
    const int n = (int)blockIdx.y - 1;
    const long long mf = m + (long long)d.nx * d.ny * d.nz * n;
    double *w = vf + o + d.ncell * (long long)n;
#pragma unroll 4
    for (int i = i0; i < end; i += 64) {
      const float a = lf[mf + i], dv = nf[mf + i] - a;
      w[i] = ((double)a + (double)dv * frac) * MPS_2_KMPHR;
    }
  }
}

constexpr int kRed = 256;

__device__ inline double block_max(double v, double *sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = kRed / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + s]);
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

// The largest of the bins' |at(n)|, up to eight loads in flight; the last
// group is the smallest power of two that holds the bins left (its loads past
// the last bin repeat that one's): adjust_dt at 720x360x70x1 392 us, 426 with
// eight loads throughout.
template <int U, typename T, typename F>
__device__ __forceinline__ T raise_by_bins(T m, int n0, int ns, F &&at) {
  T v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) v[u] = at(min(n0 + u, ns - 1));
#pragma unroll
  for (int u = 0; u < U; ++u) m = fmax(m, fabs(v[u]));
  return m;
}
template <typename T, typename F>
__device__ __forceinline__ T max_over_bins(int ns, F &&at) {
  T m = 0;
  int n = 0;
  for (; ns - n > 4; n += 8) m = raise_by_bins<8>(m, n, ns, at);
  if (ns - n > 2) return raise_by_bins<4>(m, n, ns, at);
  if (ns - n == 2) return raise_by_bins<2>(m, n, ns, at);
  return ns > n ? raise_by_bins<1>(m, n, ns, at) : m;
}

// Per-block partials of Adjust_DT over the interior cells:
// [0] vxmax_dx (lon-lat) or max|vx| (projected), [1] the same for y,
// [2] vzmax_dz, [3] min of the diffusion times (negated, so that all four
// reduce with max).  met != 0 reads the FP32 next met step (in m/s).
struct DtArgs {
  Dims d;
  int latlon, met, diffusion;
  const double *vx, *vy, *vz, *vf, *kap, *sx, *sy, *sz, *kx, *ky, *kz, *dz;
  const float *mx, *my, *mz, *mf;
  double *partial;  // [blocks][4]
};

template <bool PACKED>
__global__ __launch_bounds__(kRed) void k_dt_partials(DtArgs A) {
  __shared__ double sh[kRed];
  const Dims d = A.d;
  const long long n3 = (long long)d.nx * d.ny * d.nz;
  const long long kxs = d.nx + 2, kxys = (long long)(d.nx + 2) * (d.ny + 2);
  double r0 = 0.0, r1 = 0.0, r2 = 0.0, r3 = -INFINITY;
  // a wave takes 64 cells of an x row at a time (PACKED: 64 cells in the order
  // of the unpadded arrays, over the ends of the rows)
  const unsigned nx = (unsigned)d.nx, ny = (unsigned)d.ny, chunks = (nx + 63) / 64;
  const long long items = PACKED ? (n3 + 63) / 64 : (long long)chunks * ny * d.nz;
  for (long long it = (long long)blockIdx.x * (kRed / 64) + threadIdx.x / 64; it < items; it += gridDim.x * (kRed / 64)) {
    const unsigned lane = threadIdx.x & 63;
    unsigned row, qi;
    if constexpr (PACKED) {
      const long long c = 64 * it + lane;
      row = n3 <= 0xffffffffLL - 64 ? (unsigned)c / nx : (unsigned)(c / nx);
      qi = (unsigned)(c - (long long)row * nx);
      if (row >= ny * (unsigned)d.nz) continue;
    } else {
      row = (unsigned)it / chunks;
      qi = ((unsigned)it - row * chunks) * 64 + lane;
      if (qi >= nx) continue;
    }
    const int i = (int)qi + 1, j = (int)(row % ny) + 1, k = (int)(row / ny) + 1;
    const long long m = (long long)d.nx * row + (i - 1);
    const long long o = d.p3(i, j, k);
    const double kap = A.kap[o];
    if (A.met) {
      if (A.latlon) {
        double ms = fmin(A.sx[o], A.sx[o + 1]);
        r0 = fmax(r0, (double)fabsf(A.mx[m]) * MPS_2_KMPHR * ms / kap);
        ms = fmin(A.sy[o], A.sy[o + d.sy]);
        r1 = fmax(r1, (double)fabsf(A.my[m]) * MPS_2_KMPHR * ms / kap);
      } else {
        r0 = fmax(r0, (double)fabsf(A.mx[m]));
        r1 = fmax(r1, (double)fabsf(A.my[m]));
      }
      const float vfm = max_over_bins<float>(d.ns, [&](int n) { return A.mf[m + n3 * n]; });
      r2 = fmax(r2, (double)(fabsf(A.mz[m]) + vfm) * MPS_2_KMPHR / A.dz[k - 1]);
    } else {
      if (A.latlon) {
        double ms = fmin(A.sx[o], A.sx[o + 1]);
        r0 = fmax(r0, fabs(A.vx[o]) * ms / kap);
        ms = fmin(A.sy[o], A.sy[o + d.sy]);
        r1 = fmax(r1, fabs(A.vy[o]) * ms / kap);
      } else {
        r0 = fmax(r0, fabs(A.vx[o]));
        r1 = fmax(r1, fabs(A.vy[o]));
      }
      const double vfm = max_over_bins<double>(d.ns, [&](int n) { return A.vf[o + d.ncell * n]; });
      r2 = fmax(r2, (fabs(A.vz[o]) + vfm) / A.dz[k - 1]);
    }
    if (A.diffusion) {
      const long long ok = (long long)i + kxs * j + kxys * k;
      double rr = kap / fmin(A.sx[o], A.sx[o + 1]);
      const double t1 = (rr * rr) / A.kx[ok];
      rr = kap / fmin(A.sy[o], A.sy[o + d.sy]);
      const double t2 = (rr * rr) / A.ky[ok];
      rr = kap / fmin(A.sz[o], A.sz[o + d.sz]);
      const double t3 = (rr * rr) / A.kz[ok];
      r3 = fmax(r3, -(t1 + t2 + t3));
    }
  }
  r0 = block_max(r0, sh);
  r1 = block_max(r1, sh);
  r2 = block_max(r2, sh);
  r3 = block_max(r3, sh);
  if (threadIdx.x == 0) {
    double *p = A.partial + 4 * (long long)blockIdx.x;
    p[0] = r0; p[1] = r1; p[2] = r2; p[3] = r3;
  }
}

// Slab maxima of get_minmax_index: px[i] = max over (j,k,n), py[j] over
// (i,k,n), pz[k] over (i,j,n) of concen(1:nx,1:ny,1:nz,1:ns,ts0), clamped
// at zero (the reference compares them with a positive threshold) and kept
// as the bit patterns of non-negative doubles, whose unsigned order is their
// numeric order.  A workgroup takes kSlabRows rows of a (k, bin) plane, a
// wave a row at a time in blocks of kSlabCols columns, all loads of a row
// in flight: the column maxima stay in registers, a row costs one wave
// reduction, and an atomic is issued only for a value above the stored one
// (140 MB of 241x161x45x10 in 50 us against 113 us with a reduction per 64
// cells and an atomic per column and plane).
constexpr int kSlabChunks = 6, kSlabCols = 64 * kSlabChunks, kSlabRows = 64;

__device__ inline void raise(unsigned long long *p, double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  if (b > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(p, b);
}

__global__ __launch_bounds__(kRed) void k_slab_max(Dims d, const double *__restrict__ c0,
                                                   unsigned long long *px, unsigned long long *py,
                                                   unsigned long long *pz) {
  __shared__ double s_col[kRed / 64][kSlabCols], s_row[kSlabRows];
  const int k = (int)(blockIdx.x % (unsigned)d.nz) + 1;
  const int n = (int)(blockIdx.x / (unsigned)d.nz);
  const int j0 = (int)blockIdx.y * kSlabRows, j1 = min(j0 + kSlabRows, d.ny);
  const double *c = c0 + d.ncell * (long long)n;
  const int lane = threadIdx.x & 63, w = threadIdx.x / 64;
  double top = 0.0;
  for (int i0 = 0; i0 < d.nx; i0 += kSlabCols) {
    double mi[kSlabChunks];
#pragma unroll
    for (int u = 0; u < kSlabChunks; ++u) mi[u] = 0.0;
    for (int j = j0 + 1 + w; j <= j1; j += kRed / 64) {
      const double *p = c + d.p3(1, j, k);
      double v[kSlabChunks], row = 0.0;
#pragma unroll
      for (int u = 0; u < kSlabChunks; ++u) v[u] = p[min(i0 + 64 * u + lane, d.nx - 1)];
#pragma unroll
      for (int u = 0; u < kSlabChunks; ++u) {
        v[u] = (i0 + 64 * u + lane < d.nx) ? fmax(v[u], 0.0) : 0.0;
        mi[u] = fmax(mi[u], v[u]);
        row = fmax(row, v[u]);
      }
      for (int s = 32; s > 0; s >>= 1) row = fmax(row, __shfl_xor(row, s, 64));
      if (lane == 0) s_row[j - 1 - j0] = i0 ? fmax(s_row[j - 1 - j0], row) : row;
      top = fmax(top, row);
    }
    // the waves' column maxima, then one atomic per column
#pragma unroll
    for (int u = 0; u < kSlabChunks; ++u) s_col[w][64 * u + lane] = mi[u];
    __syncthreads();
    for (int q = threadIdx.x; q < kSlabCols && i0 + q < d.nx; q += kRed) {
      double m = s_col[0][q];
#pragma unroll
      for (int v = 1; v < kRed / 64; ++v) m = fmax(m, s_col[v][q]);
      raise(&px[i0 + q], m);
    }
    __syncthreads();
  }
  if (lane == 0) raise(&pz[k - 1], top);
  if ((int)threadIdx.x < j1 - j0) raise(&py[j0 + threadIdx.x], s_row[threadIdx.x]);
}

__global__ void k_zero_u64(unsigned long long *p, int n) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0ull;
}

}  // namespace

hipError_t launch_met_interp(hipStream_t s, const Dims &d, const float *const last[4], const float *const next[4],
                             double frac, bool with_vf, double *vx, double *vy, double *vz, double *vf) {
  const int seg = with_vf ? 256 : 64;
  const long long items = (long long)d.ny * d.nz * ((d.nx + seg - 1) / seg);
  const long long blocks = (items + kRow / 64 - 1) / (kRow / 64);
  if (blocks > 0x3fffffffLL) return hipErrorInvalidValue;  // (item numbers of 32 bits)
  const dim3 grid((unsigned)blocks, with_vf ? 1 + d.ns : 1);
  auto *k = with_vf ? k_met_interp<256> : k_met_interp<64>;
  hipLaunchKernelGGL(k, grid, dim3(kRow), 0, s, d, last[0], last[1], last[2], last[3], next[0], next[1], next[2],
                     next[3], frac, vx, vy, vz, vf);
  return hipGetLastError();
}

int dt_partial_blocks(const Dims &d) {
  const long long n3 = (long long)d.nx * d.ny * d.nz;
  const long long b = (n3 + kRed - 1) / kRed;
  return (int)(b < 2048 ? b : 2048);
}

hipError_t launch_dt_partials(hipStream_t s, const Dims &d, int latlon, int met, int diffusion, const double *vx,
                              const double *vy, const double *vz, const double *vf, const double *kap,
                              const double *sx, const double *sy, const double *sz, const double *kx,
                              const double *ky, const double *kz, const double *dz, const float *const met_next[4],
                              double *partial) {
  DtArgs A{d, latlon, met, diffusion, vx, vy, vz, vf, kap, sx, sy, sz, kx, ky, kz, dz,
           met_next[0], met_next[1], met_next[2], met_next[3], partial};
  // Rows that leave a fifth of the lanes or more idle are packed: adjust_dt at
  // 30x1000x20x3 50.6 us, 57.0 by rows, 65x65x33x3 42.5 and 45.5; by rows
  // 360x240x50x15 195 us, 213 packed (the divisions of every lane)
  const bool packed = 5 * (long long)d.nx <= 4 * 64 * (((long long)d.nx + 63) / 64);
  if (packed) hipLaunchKernelGGL((k_dt_partials<true>), dim3(dt_partial_blocks(d)), dim3(kRed), 0, s, A);
  else hipLaunchKernelGGL((k_dt_partials<false>), dim3(dt_partial_blocks(d)), dim3(kRed), 0, s, A);
  return hipGetLastError();
}

hipError_t launch_slab_max(hipStream_t s, const Dims &d, const double *c0, unsigned long long *prof) {
  const int np = d.nx + d.ny + d.nz;
  hipLaunchKernelGGL(k_zero_u64, dim3((np + 255) / 256), dim3(256), 0, s, prof, np);
  hipLaunchKernelGGL(k_slab_max, dim3((unsigned)(d.nz * d.ns), (unsigned)((d.ny + kSlabRows - 1) / kSlabRows)),
                     dim3(kRed), 0, s, d, c0, prof, prof + d.nx, prof + d.nx + d.ny);
  return hipGetLastError();
}

}  // namespace ash3d
