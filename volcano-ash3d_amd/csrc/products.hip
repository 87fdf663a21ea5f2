// Output products of the transport state and their ESRI ASCII files:
//   ConcentrationCalculator  src/Output_Vars.f90:1026-1137 (cloud load,
//                            peak concentration, cloud top and bottom,
//                            cloud mask and area)
//   AshThicknessCalculator   src/Output_Vars.f90:855-893 (deposit thickness,
//                            deposit mask and area)
//   write_2D_ASCII           src/write_ASCII.f90:264-382 (header, 10f18.6
//                            rows from the northern row down, real(4) values)
// The products are one pass over the state on the device (lanes along x, so
// every load of a wavefront is one coalesced segment), in the reference's
// summation order.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <string>

#include "common.hpp"

namespace ash3d {

namespace {

constexpr double KG_2_MG = 1.0e6;    // src/Ash3d_VariableModules.f90:285
constexpr double KM3_2_M3 = 1.0e9;   // :284
constexpr double KM2_2_M2 = 1.0e6;   // :283
constexpr double M_2_MM = 1.0e3;     // :281

// Columns in workgroups of kCol columns (lanes along x) x kWaves waves: the
// waves take the levels of a chunk of kChunk between them, each level's sum
// over the bins in the reference's order with kAhead bins' loads in flight,
// into LDS; then the first wave folds the chunk's levels upward.  One pass
// over the state, bound by HBM bandwidth: 518 MB of a 360x240x50x15 state in
// 125 us (products) and 120 us (column load), against 349 and 338 us with
// one thread per column, which kept a load or two in flight per lane.
constexpr int kCol = 64, kWaves = 8, kChunk = 16, kAhead = 8;

// The sums over the bins of levels k0 .. k0+kChunk-1 (those <= nz) of the
// workgroup's columns into sum[level - k0][lane]; o: the column's offset at
// level 0 (c null: zeros).  Ends with a barrier.
__device__ inline void level_sums(const Dims &d, const double *c, long long o, int k0, double (*sum)[kCol]) {
  const int l = threadIdx.x, w = threadIdx.y;
  for (int q = w; q < kChunk && k0 + q <= d.nz; q += kWaves) {
    double s = 0.0;
    if (c != nullptr) {
      const double *p = c + o + d.sz * (long long)(k0 + q);
      for (int n0 = 0; n0 < d.ns; n0 += kAhead) {
        double v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = p[d.ncell * (long long)min(n0 + u, d.ns - 1)];
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
          if (n0 + u < d.ns) s += v[u];
      }
    }
    sum[q][l] = s;
  }
  __syncthreads();
}

// out: 5 planes of nx*ny doubles (cloud load, max concentration, max
// height, min height, deposit thickness) then 2 planes of int32 masks.
__global__ __launch_bounds__(kCol *kWaves) void k_products(ProdArgs P) {
  __shared__ double sum[2][kChunk][kCol];
  const Dims d = P.d;
  const unsigned nxy = (unsigned)d.nx * (unsigned)d.ny;
  const unsigned t = blockIdx.x * kCol + threadIdx.x, tt = min(t, nxy - 1);
  const int i = (int)(tt % (unsigned)d.nx) + 1, j = (int)(tt / (unsigned)d.nx) + 1;
  const long long o = d.p3(i, j, 0);
  double *load = P.out, *maxc = P.out + nxy, *maxh = maxc + nxy, *minh = maxh + nxy, *thick = minh + nxy;
  int *mcloud = (int *)(P.out + 5 * (long long)nxy), *mdep = mcloud + nxy;
  // ConcentrationCalculator, columns of the box imin..imax x jmin..jmax
  double L = 0.0, H = 0.0, B = 100.0, C = 0.0, tcmax = 0.0;
  bool first_le = false;
  for (int k0 = 1, par = 0; k0 <= d.nz; k0 += kChunk, par ^= 1) {
    level_sums(d, P.c, o, k0, sum[par]);
    if (threadIdx.y != 0) continue;
    for (int k = k0; k < k0 + kChunk && k <= d.nz; ++k) {
      const double tc = sum[par][k - k0][threadIdx.x];  // sum(concen_pd(i,j,k,1:n_gs_max,ts1)), bins in order
      L = L + tc * P.dz[k - 1] / 1.0e3;
      if (tc >= P.cloudcon) H = P.zcc[k - 1] + 0.5 * P.dz[k - 1];
      // the top-down scan keeps the lowest level at or below the threshold
      if (tc <= P.cloudcon && !first_le) {
        B = P.zcc[k - 1] - 0.5 * P.dz[k - 1];
        first_le = true;
      }
      tcmax = (k == 1) ? tc : fmax(tcmax, tc);  // maxval(TotalConcentration(:))
    }
  }
  if (t >= nxy) return;
  if (threadIdx.y == 0) {
    int mask = 0;
    if (i >= P.i0 && i <= P.i1 && j >= P.j0 && j <= P.j1) {
      mask = (L >= P.cloudload) ? 1 : 0;
      if (mask) {
        if (B < 0.0 && H > 0.0) B = 0.0;
        B = fmin(H, B);
        C = tcmax * KG_2_MG / KM3_2_M3;
      } else {
        L = 0.0;
        H = 0.0;
        B = 0.0;
      }
    } else {
      L = 0.0;
      H = 0.0;
      B = 100.0;
    }
    load[t] = L;
    maxc[t] = C;
    maxh[t] = H;
    minh[t] = B;
    mcloud[t] = mask;
  } else if (threadIdx.y == 1) {
    // AshThicknessCalculator, every column
    double s = 0.0;  // sum(DepositGranularity(i,j,1:n_gs_max))
    for (int n = 0; n < d.ns; ++n) s += P.dep[t + (long long)nxy * n];
    const double th = s * P.dz[0] / KM2_2_M2 / P.density * M_2_MM;
    thick[t] = th;
    mdep[t] = (th > P.depo) ? 1 : 0;
  }
}

// CloudLoad of every column (no threshold): out(nx, ny)
__global__ __launch_bounds__(kCol *kWaves) void k_column_load(Dims d, const double *c0, const double *dz,
                                                             double *out) {
  __shared__ double sum[2][kChunk][kCol];
  const unsigned nxy = (unsigned)d.nx * (unsigned)d.ny;
  const unsigned t = blockIdx.x * kCol + threadIdx.x, tt = min(t, nxy - 1);
  const int i = (int)(tt % (unsigned)d.nx) + 1, j = (int)(tt / (unsigned)d.nx) + 1;
  double L = 0.0;
  for (int k0 = 1, par = 0; k0 <= d.nz; k0 += kChunk, par ^= 1) {
    level_sums(d, c0, d.p3(i, j, 0), k0, sum[par]);
    if (threadIdx.y != 0) continue;
    for (int k = k0; k < k0 + kChunk && k <= d.nz; ++k) L = L + sum[par][k - k0][threadIdx.x] * dz[k - 1] / 1.0e3;
  }
  if (threadIdx.y == 0 && t < nxy) out[t] = L;
}

// Fortran Fw.d of a real(4) value: the exact decimal expansion rounded to d
// places, right-justified in w columns, asterisks when it does not fit.
void put_f(std::string &o, double v, int w, int dd) {
  char buf[64];
  int len = snprintf(buf, sizeof buf, "%*.*f", w, dd, v);
  if (len < 0 || len > w) o.append((size_t)w, '*');
  else o.append(buf, (size_t)len);
}

void put_i(std::string &o, int v, int w) {
  char buf[32];
  int len = snprintf(buf, sizeof buf, "%*d", w, v);
  if (len < 0 || len > w) o.append((size_t)w, '*');
  else o.append(buf, (size_t)len);
}

}  // namespace

hipError_t launch_products(hipStream_t s, const ProdArgs &p) {
  const long long nxy = (long long)p.d.nx * p.d.ny;
  hipLaunchKernelGGL(k_products, dim3((unsigned)((nxy + kCol - 1) / kCol)), dim3(kCol, kWaves), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_column_load(hipStream_t s, const Dims &d, const double *c0, const double *dz, double *out) {
  const long long nxy = (long long)d.nx * d.ny;
  hipLaunchKernelGGL(k_column_load, dim3((unsigned)((nxy + kCol - 1) / kCol)), dim3(kCol, kWaves), 0, s, d, c0, dz,
                     out);
  return hipGetLastError();
}

// write_2D_ASCII (src/write_ASCII.f90:334-373) into a string
std::string esri_ascii_text(int nx, int ny, const double *field, const int32_t *mask, const char *fill,
                            int latlon, double xll, double yll, double dx, double dy) {
  std::string o;
  o.reserve((size_t)nx * ny * 18 + (size_t)ny * (nx / 10 + 4) + 256);
  const double KM_2_M = 1.0e3;  // src/Ash3d_VariableModules.f90:280
  o += "NCOLS ";
  put_i(o, nx, 5);
  o += "\nNROWS ";
  put_i(o, ny, 5);
  o += "\nXLLCORNER ";
  // lon-lat: GIS prefers -180..180 (:343-346); projected: km to m (:350-352)
  put_f(o, latlon ? (xll > 180.0 ? xll - 360.0 : xll) : xll * KM_2_M, 15, 3);
  o += "\nYLLCORNER ";
  put_f(o, latlon ? yll : yll * KM_2_M, 15, 3);
  o += "\nCELLSIZE ";
  put_f(o, latlon ? dx : dx * KM_2_M, 15, 3);
  put_f(o, latlon ? dy : dy * KM_2_M, 15, 3);
  char fv[7] = "      ";  // Fill_Value, character(len=6), a6
  for (int c = 0; c < 6 && fill[c]; ++c) fv[c] = fill[c];
  o += "\nNODATA_VALUE ";
  o += fv;
  o += "\n";
  const float fvalue = (float)strtod(fill, nullptr);  // read(Fill_Value,*) FValue, real(op=4)
  for (int j = ny; j >= 1; --j) {
    for (int i0 = 1; i0 <= nx; i0 += 10) {  // format 10f18.6: records of ten
      for (int i = i0; i <= nx && i < i0 + 10; ++i) {
        const long long t = (long long)(i - 1) + (long long)nx * (j - 1);
        const float v = (mask == nullptr || mask[t]) ? (float)field[t] : fvalue;  // real(..., kind=op)
        put_f(o, (double)v, 18, 6);
      }
      o += "\n";
    }
    o += "  \n";  // write(fid,*)" ": list-directed blank, then the string
  }
  return o;
}

// the output file name of write_2D_ASCII (:316-331)
std::string esri_ascii_name(const char *root, double time_h, int is_final) {
  std::string r(root);
  const size_t a = r.find_first_not_of(' ');
  r = (a == std::string::npos) ? std::string() : r.substr(a);
  const size_t b = r.find_last_not_of(' ');
  r = (b == std::string::npos) ? std::string() : r.substr(0, b + 1);
  if (r.find("outvar") != std::string::npos || r.find("ArrivalTime") != std::string::npos) return r + ".dat";
  std::string cio;
  if (is_final) {
    cio = "____final";
  } else {
    std::string tbuf;
    if (time_h < 10.0) {
      cio = "00";
      put_f(tbuf, time_h, 4, 2);
    } else if (time_h < 100.0) {
      cio = "0";
      put_f(tbuf, time_h, 5, 2);
    } else {
      put_f(tbuf, time_h, 6, 2);
    }
    cio += tbuf + "hrs";
  }
  return r + cio + ".dat";
}

}  // namespace ash3d
