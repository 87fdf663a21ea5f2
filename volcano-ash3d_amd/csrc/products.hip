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
// over the bins in the reference's order with eight bins' loads in flight,
// into LDS; then the first wave folds the chunk's levels upward.  One pass
// over the state, bound by HBM bandwidth: 518 MB of a 360x240x50x15 state in
// 112 us (products) and 100 us (column load), against 347 and 338 us with
// one thread per column, which kept a load or two in flight per lane.
constexpr int kCol = 64, kWaves = 8, kChunk = 16;

// s + the U bins of p from n0 on, in order, their loads in flight together
// (those past the last bin repeat that one's and are not added)
template <int U>
__device__ __forceinline__ double add_bins(double s, const double *p, const Dims &d, int n0) {
  double v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) v[u] = p[d.ncell * (long long)min(n0 + u, d.ns - 1)];
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (n0 + u < d.ns) s += v[u];
  return s;
}

// The sums over the bins of levels k0 .. k0+kChunk-1 (those <= nz) of the
// workgroup's columns into sum[level - k0][lane], and what they add to the load
// into term (formed here: one wave folds all levels, and its divisions would
// hold up the others); o: the column's offset at level 0 (c null: zeros; sum
// null: not stored).  The last group of bins is the smallest power of two
// that holds the bins left (column load at 100x200x60x2 44 us, 50 with eight
// loads throughout).  Ends with a barrier.
__device__ inline void level_sums(const Dims &d, const double *c, long long o, const double *dz, int k0, double (*sum)[kCol],
                                  double (*term)[kCol]) {
  const int l = threadIdx.x, w = threadIdx.y;
#pragma unroll
  for (int q = w; q < kChunk; q += kWaves) {
    if (k0 + q > d.nz) break;
    double s = 0.0;
    if (c != nullptr) {
      const double *p = c + o + d.sz * (long long)(k0 + q);
      int n = 0;
      for (; d.ns - n > 4; n += 8) s = add_bins<8>(s, p, d, n);
      if (d.ns - n > 2) s = add_bins<4>(s, p, d, n);
      else if (d.ns - n == 2) s = add_bins<2>(s, p, d, n);
      else if (d.ns > n) s = add_bins<1>(s, p, d, n);
    }
    if (sum) sum[q][l] = s;
    term[q][l] = s * dz[k0 + q - 1] / 1.0e3;
  }
  __syncthreads();
}

// The same for one column by its own thread, folded upward eight levels at a
// time: fold(k, sum over the bins, its term of the load).
constexpr int kWhole = 256;  // columns (threads) of a workgroup
template <typename F>
__device__ __forceinline__ void whole_column(const Dims &d, const double *c, long long o, const double *dz, F &&fold) {
  for (int k0 = 1; k0 <= d.nz; k0 += 8) {
    double s[8] = {};
    if (c != nullptr)
      for (int n = 0; n < d.ns; ++n) {
        const double *p = c + o + d.ncell * (long long)n;
#pragma unroll
        for (int q = 0; q < 8; ++q) s[q] += p[d.sz * (long long)min(k0 + q, d.nz)];
      }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (k0 + q <= d.nz) fold(k0 + q, s[q], s[q] * dz[k0 + q - 1] / 1.0e3);
  }
}
// Few bins of many columns: a workgroup's waves would meet at a barrier for
// every two loads a lane.  Products and column load of 720x360x70x1 42 and 26
// us (the waves of a workgroup 82 and 51), 720x360x30x2 32 and 22 (45 and
// 30), 1440x300x30x4 89 and 77 (111 and 85).
inline bool whole_columns(const Dims &d) { return d.ns <= 4 && (long long)d.nx * d.ny >= 1 << 17; }

// out: 5 planes of nx*ny doubles (cloud load, max concentration, max
// height, min height, deposit thickness) then 2 planes of int32 masks.
template <bool WHOLE>
__global__ __launch_bounds__(WHOLE ? kWhole : kCol *kWaves) void k_products(ProdArgs P) {
  const Dims d = P.d;
  const unsigned nxy = (unsigned)d.nx * (unsigned)d.ny;
  const unsigned t = blockIdx.x * (WHOLE ? kWhole : kCol) + threadIdx.x, tt = min(t, nxy - 1);
  const int i = (int)(tt % (unsigned)d.nx) + 1, j = (int)(tt / (unsigned)d.nx) + 1;
  const long long o = d.p3(i, j, 0);
  double *load = P.out, *maxc = P.out + nxy, *maxh = maxc + nxy, *minh = maxh + nxy, *thick = minh + nxy;
  int *mcloud = (int *)(P.out + 5 * (long long)nxy), *mdep = mcloud + nxy;
  // ConcentrationCalculator, columns of the box imin..imax x jmin..jmax
  double L = 0.0, H = 0.0, B = 100.0, C = 0.0, tcmax = 0.0;
  bool first_le = false;
  auto fold = [&](int k, double tc, double term) {  // tc: sum(concen_pd(i,j,k,1:n_gs_max,ts1)), bins in order
    // (heights of every level, not only of the columns that take them: loads
    // under a lane's condition would wait one after the other)
    const double zc = P.zcc[k - 1], hdz = 0.5 * P.dz[k - 1], top = zc + hdz, base = zc - hdz;
    L = L + term;
    if (tc >= P.cloudcon) H = top;
    // the top-down scan keeps the lowest level at or below the threshold
    if (tc <= P.cloudcon && !first_le) {
      B = base;
      first_le = true;
    }
    tcmax = (k == 1) ? tc : fmax(tcmax, tc);  // maxval(TotalConcentration(:))
  };
  if constexpr (WHOLE) {
    whole_column(d, P.c, o, P.dz, fold);
  } else {
    __shared__ double sum[2][kChunk][kCol], term[2][kChunk][kCol];
    for (int k0 = 1, par = 0; k0 <= d.nz; k0 += kChunk, par ^= 1) {
      level_sums(d, P.c, o, P.dz, k0, sum[par], term[par]);
      if (threadIdx.y != 0) continue;
#pragma unroll 4
      for (int k = k0; k < min(k0 + kChunk, d.nz + 1); ++k)
        fold(k, sum[par][k - k0][threadIdx.x], term[par][k - k0][threadIdx.x]);
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
  }
  if (WHOLE || threadIdx.y == 1) {
    // AshThicknessCalculator, every column
    double s = 0.0;  // sum(DepositGranularity(i,j,1:n_gs_max))
    for (int n = 0; n < d.ns; ++n) s += P.dep[t + (long long)nxy * n];
    const double th = s * P.dz[0] / KM2_2_M2 / P.density * M_2_MM;
    thick[t] = th;
    mdep[t] = (th > P.depo) ? 1 : 0;
  }
}

// CloudLoad of every column (no threshold): out(nx, ny)
template <bool WHOLE>
__global__ __launch_bounds__(WHOLE ? kWhole : kCol *kWaves) void k_column_load(Dims d, const double *c0,
                                                                              const double *dz, double *out) {
  const unsigned nxy = (unsigned)d.nx * (unsigned)d.ny;
  const unsigned t = blockIdx.x * (WHOLE ? kWhole : kCol) + threadIdx.x, tt = min(t, nxy - 1);
  const int i = (int)(tt % (unsigned)d.nx) + 1, j = (int)(tt / (unsigned)d.nx) + 1;
  double L = 0.0;
  if constexpr (WHOLE) {
    whole_column(d, c0, d.p3(i, j, 0), dz, [&](int, double, double term) { L = L + term; });
  } else {
    __shared__ double term[2][kChunk][kCol];
    for (int k0 = 1, par = 0; k0 <= d.nz; k0 += kChunk, par ^= 1) {
      level_sums(d, c0, d.p3(i, j, 0), dz, k0, nullptr, term[par]);
      if (threadIdx.y != 0) continue;
      for (int k = k0; k < k0 + kChunk && k <= d.nz; ++k) L = L + term[par][k - k0][threadIdx.x];
    }
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
  if (whole_columns(p.d))
    hipLaunchKernelGGL((k_products<true>), dim3((unsigned)((nxy + kWhole - 1) / kWhole)), dim3(kWhole), 0, s, p);
  else
    hipLaunchKernelGGL((k_products<false>), dim3((unsigned)((nxy + kCol - 1) / kCol)), dim3(kCol, kWaves), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_column_load(hipStream_t s, const Dims &d, const double *c0, const double *dz, double *out) {
  const long long nxy = (long long)d.nx * d.ny;
  if (whole_columns(d))
    hipLaunchKernelGGL((k_column_load<true>), dim3((unsigned)((nxy + kWhole - 1) / kWhole)), dim3(kWhole), 0, s, d, c0,
                       dz, out);
  else
    hipLaunchKernelGGL((k_column_load<false>), dim3((unsigned)((nxy + kCol - 1) / kCol)), dim3(kCol, kWaves), 0, s, d,
                       c0, dz, out);
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
