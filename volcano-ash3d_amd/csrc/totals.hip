// Per-bin mass budget on the device: the sums of Calc_AshVol_Aloft,
// Calc_AshVol_Deposit and Calc_AshVol_Outflow (src/Output_Vars.f90:1255-1293,
// :1375-1404, :1419-1459) before their conversion to volume, which
// TimeStepTotals (src/TimeStepTotals.f90:17-88) evaluates every step:
//   aloft(n)   = sum concen(1:nx,1:ny,1:nz,n,ts0) * kappa(1:nx,1:ny,1:nz)
//   deposit(n) = sum DepositGranularity(1:nx,1:ny,n) * kappa(1:nx,1:ny,0)
//   outflow(n) = sum over the yz1, yz2, xz1, xz2 and xy2 faces of the
//                outflow times the kappa of the ghost cell it belongs to.
// The reduction is deterministic: a fixed number of partial sums per bin,
// each over a fixed set of cells in a fixed order, then a fixed-order sum
// of the partials.  The aloft sum reads the state once, a wave per x row
// (lanes along x, so that a row needs one division for its indices instead
// of several per cell): 518 MB of a 360x240x50x15 state in 108 us against
// 210 us with one thread per strided cell.
#include "common.hpp"

namespace ash3d {

namespace {

constexpr int kThreads = 512;
constexpr int kParts = 128;
constexpr int kBins = 8;  // bins of a workgroup, which share the rows' kappa

__device__ inline double block_sum(double v, double *sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = kThreads / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + s];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

struct TotArgs {
  Dims d;
  const double *c0, *kap, *dep;
  const double *yz1, *yz2, *xz1, *xz2, *xy2;
  double *partial;  // [ns][kParts][3]
};

__global__ __launch_bounds__(kThreads) void k_mass_partials(TotArgs A) {
  __shared__ double sh[kThreads];
  const Dims d = A.d;
  // blockIdx.y < groups: the aloft sums of a group of bins; beyond: the
  // deposit and outflow sums of one bin
  const int groups = (d.ns + kBins - 1) / kBins, p = blockIdx.x;
  if ((int)blockIdx.y < groups) {
    const int n0 = blockIdx.y * kBins;
    double a[kBins];
    long long ofs[kBins];
#pragma unroll
    for (int u = 0; u < kBins; ++u) {
      a[u] = 0.0;
      ofs[u] = d.ncell * (long long)min(n0 + u, d.ns - 1);
    }
    // x rows (j,k), one wave each
    const int lane = threadIdx.x & 63;
    const unsigned rows = (unsigned)d.ny * (unsigned)d.nz, waves = kParts * (kThreads / 64);
    for (unsigned r = (unsigned)p * (kThreads / 64) + threadIdx.x / 64; r < rows; r += waves) {
      const long long o = d.p3(1, (int)(r % (unsigned)d.ny) + 1, (int)(r / (unsigned)d.ny) + 1);
      for (int i = lane; i < d.nx; i += 64) {
        const double kp = A.kap[o + i];
#pragma unroll
        for (int u = 0; u < kBins; ++u) a[u] += A.c0[o + i + ofs[u]] * kp;
      }
    }
#pragma unroll
    for (int u = 0; u < kBins; ++u) {
      const double s = block_sum(a[u], sh);
      if (threadIdx.x == 0 && n0 + u < d.ns) A.partial[((long long)(n0 + u) * kParts + p) * 3] = s;
    }
    return;
  }
  const int n = (int)blockIdx.y - groups;
  const long long stride = (long long)kParts * kThreads;
  const long long t0 = (long long)p * kThreads + threadIdx.x;
  // deposit
  double b = 0.0;
  const long long nxy = (long long)d.nx * d.ny;
  for (long long t = t0; t < nxy; t += stride) {
    const int i = (int)(t % d.nx) + 1, j = (int)(t / d.nx) + 1;
    b += A.dep[t + nxy * n] * A.kap[d.p3(i, j, 0)];
  }
  // outflow through five faces
  double o = 0.0;
  const long long nyz = (long long)d.ny * d.nz, nxz = (long long)d.nx * d.nz;
  const long long byz = (long long)(d.ny + 4) * (d.nz + 4) * n;
  const long long bxz = (long long)(d.nx + 4) * (d.nz + 4) * n;
  const long long bxy = (long long)(d.nx + 4) * (d.ny + 4) * n;
  for (long long t = t0; t < nyz; t += stride) {
    const int j = (int)(t % d.ny) + 1, k = (int)(t / d.ny) + 1;
    const long long f = (long long)(j + 1) + (long long)(d.ny + 4) * (k + 1) + byz;
    o += A.yz1[f] * A.kap[d.p3(0, j, k)];
    o += A.yz2[f] * A.kap[d.p3(d.nx + 1, j, k)];
  }
  for (long long t = t0; t < nxz; t += stride) {
    const int i = (int)(t % d.nx) + 1, k = (int)(t / d.nx) + 1;
    const long long f = (long long)(i + 1) + (long long)(d.nx + 4) * (k + 1) + bxz;
    o += A.xz1[f] * A.kap[d.p3(i, 0, k)];
    o += A.xz2[f] * A.kap[d.p3(i, d.ny + 1, k)];
  }
  for (long long t = t0; t < nxy; t += stride) {
    const int i = (int)(t % d.nx) + 1, j = (int)(t / d.nx) + 1;
    const long long f = (long long)(i + 1) + (long long)(d.nx + 4) * (j + 1) + bxy;
    o += A.xy2[f] * A.kap[d.p3(i, j, d.nz + 1)];
  }
  b = block_sum(b, sh);
  o = block_sum(o, sh);
  if (threadIdx.x == 0) {
    double *w = A.partial + ((long long)n * kParts + p) * 3;
    w[1] = b;
    w[2] = o;
  }
}

// one wave per (bin, sum): lane l adds partials l and l + 64, then the wave
__global__ __launch_bounds__(64) void k_mass_final(const double *partial, int ns, double *out) {
  const int n = blockIdx.x / 3, q = blockIdx.x % 3;
  double s = 0.0;
  for (int p = threadIdx.x; p < kParts; p += 64) s += partial[((long long)n * kParts + p) * 3 + q];
  for (int h = 32; h > 0; h >>= 1) s += __shfl_down(s, h, 64);
  if (threadIdx.x == 0) out[(long long)q * ns + n] = s;
}

}  // namespace

long long mass_partials_size(const Dims &d) { return (long long)d.ns * kParts * 3; }

hipError_t launch_mass_totals(hipStream_t s, const Dims &d, const double *c0, const double *kap,
                              const double *dep, const double *yz1, const double *yz2, const double *xz1,
                              const double *xz2, const double *xy2, double *partial, double *out) {
  TotArgs A{d, c0, kap, dep, yz1, yz2, xz1, xz2, xy2, partial};
  hipLaunchKernelGGL(k_mass_partials, dim3(kParts, (d.ns + kBins - 1) / kBins + d.ns), dim3(kThreads), 0, s, A);
  hipLaunchKernelGGL(k_mass_final, dim3(3 * d.ns), dim3(64), 0, s, partial, d.ns, out);
  return hipGetLastError();
}

}  // namespace ash3d
