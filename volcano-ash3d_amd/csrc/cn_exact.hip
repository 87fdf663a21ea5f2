// theta-scheme line solves in dgtsv's order (diffCN_{x,y,z}, src/
// Diffusion.F90:671-1428, with LAPACK dgtsv's elimination) for sweeps in
// which dgtsv interchanges no rows (counted when the lines are factored).
// The elimination and back substitution of a line are two serial chains,
// so a sweep is bound by their latency and by how many run side by side: a
// wave takes one bin of 64 lines (lanes are lines), and the NW waves of a
// workgroup take NW bins of the same lines.  The bin-independent row
// coefficients go through LDS a chunk of RC rows ahead, loaded once for all
// the waves, and a chunk of the state (back: of the eliminated right-hand
// sides) is in flight in registers while the one before is worked on.  x
// lines are contiguous in memory: a wave turns their chunks into its lanes'
// lines through LDS on the way in and out.  The eliminated right-hand sides
// wait in registers on lines of up to 80 cells (two registers a row), on
// longer ones in the ts1 slot, whose traffic is then half of the sweep's and,
// on larger states, what bounds it (y at 240x160x50x8: 569 MB in 148 us, 3.9
// TB/s).  Against one thread per line and 2 or 8 bins (k_diff_cn,
// k_diff_cn_xrows, which keep the sweeps with row interchanges): 240x160x50x8
// x, y, z 380, 347, 145 us -> 172, 146, 77 (z with the ts1 slot 118).
// Quotients from inverses (fewer dependent operations) and two chunks in
// flight gained nothing.  The arithmetic is dgtsv's, so the results are the
// same bits.
#include <algorithm>

#include "common.hpp"

namespace ash3d {

namespace {

// the state of x lines, in its own layout (the description A of x lines is
// the x<->y transposed grid's)
struct ExactArgs {
  DiffArgs A;
  Dims o;
  double *c;
};

// orders a wave's own LDS writes before its other lanes' reads
__device__ __forceinline__ void wave_lds() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ void wg_lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// KC > 0: the eliminated right-hand sides of up to KC chunks stay in
// registers instead of the scratch.
template <bool XR, int NW, int RC, int KC>
__global__ __launch_bounds__(64 * NW, (KC == 8 && NW == 4) ? 3 : 1) void k_cn_exact(ExactArgs E) {
  static_assert(!XR || KC == 0, "");
  constexpr int RPW = RC / NW;  // rows of a chunk that each wave loads
  static_assert(RC % NW == 0, "");
  const DiffArgs &A = E.A;
  if (A.sel == 4 && A.ndom[1] != 0) return;  // rows to interchange: the other kernels' sweep (uniform)
  __shared__ double s_f[2][4][RC][64];
  __shared__ double s_q[XR ? NW : 1][XR ? 64 * (RC + 1) : 1];
  __shared__ long long s_row[XR ? 64 : 1];
  const Dims d = A.d;
  const LineGeom g = A.g;
  const long long lines = (long long)g.Na * g.Nb;
  const TileGroup tg = xcd_tile_group(blockIdx.x, (d.ns + NW - 1) / NW);
  if (tg.tile * 64 >= lines) return;  // padding workgroup (uniform)
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.y), l64 = (int)threadIdx.x;
  const bool repeat = tg.tile * 64 + l64 >= lines;  // lanes past the last line repeat it
  const long long gid = repeat ? lines - 1 : tg.tile * 64 + l64;
  const int a = (int)(gid % g.Na) + 1, b = (int)(gid / g.Na) + 1;
  const int bin = tg.group * NW + w;
  const bool exists = bin < d.ns, on = exists && A.aloft.on(bin);  // uniform in the wave
  const int N = g.N, rmin = g.rmin, n = g.rmax - g.rmin + 1;
  const bool line_on = a >= g.a0 && a <= g.a1 && b >= g.b0 && b <= g.b1;
  const long long sL = line_stride(d, g.dir), base = line_base(d, g.dir, a, b);
  auto row = [&](int l) { return base + sL * (long long)(rmin + l); };  // row l: cell rmin-1+l
  const long long bofs = d.ncell * (long long)min(bin, d.ns - 1);
  double *sb = A.scratch_b + bofs;
  const double *Lf = A.lr, *Rf = A.lr + d.ncell, *fF = A.lu, *fD = A.lu + d.ncell, *fDU = fD + d.ncell;
  double *c = (XR ? E.c : A.c0) + (XR ? E.o.ncell : d.ncell) * (long long)min(bin, d.ns - 1);
  const long long ob = XR ? E.o.p3(-1, a, b) : base, os = XR ? 1 : sL;  // the state: cell r at ob + os*(r+1)
  if (XR && w == 0) s_row[l64] = ob;
  if (on && line_on) {
    const int singular = A.sing[gid];
    if (singular) atomicCAS(A.flag, 0, singular);
  }
  const double th = A.theta, omt = 1.0 - th;
  if (XR) wg_lds_barrier();
  // cells 1..N of the lines and one bin (its state z) to zero, split over
  // parts waves (x lines: along the lines)
  auto clear = [&](double *z, int part, int parts) {
    if constexpr (XR) {
      for (int ln = part; ln < 64 && tg.tile * 64 + ln < lines; ln += parts)
        for (int r = l64; r < N; r += 64) z[s_row[ln] + 2 + r] = 0.0;
    } else {
      if (repeat) return;
      for (int r = 1 + part; r <= N; r += parts) z[ob + os * (long long)(r + 1)] = 0.0;
    }
  };
  // lines outside the box, or bins that are not aloft, throughout the
  // workgroup (every wave has the same lines; uniform): nothing is read
  const int b0 = tg.group * NW, b1 = min(b0 + NW, d.ns);
  bool any_bin = false;
  for (int q = b0; q < b1; ++q) any_bin = any_bin || A.aloft.on(q);
  if (!any_bin || __ballot(line_on) == 0) {
    for (int q = b0; q < b1; ++q) clear((XR ? E.c : A.c0) + (XR ? E.o.ncell : d.ncell) * (long long)q, w, NW);
    return;
  }

  // ---- elimination: chunk k holds rows k*RC+1 .. k*RC+RC, with the q of
  // each row's right neighbour (cell rmin+l)
  double ff[RPW][3], qn[RC];
  auto load_f = [&](int k) {
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      const int l = min(k * RC + w * RPW + r + 1, n);
      ff[r][0] = Lf[row(l)];
      ff[r][1] = Rf[row(l)];
      ff[r][2] = fF[row(max(l - 1, 1))];  // fact of elimination step l-1 is at row l-1's cell
    }
  };
  auto put_f = [&](int k) {
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      const double L = ff[r][0], R = ff[r][1], C = L + R;
      double(*s)[RC][64] = s_f[k & 1];
      s[0][w * RPW + r][l64] = omt * L;
      s[1][w * RPW + r][l64] = 1.0 - omt * C;
      s[2][w * RPW + r][l64] = omt * R;
      s[3][w * RPW + r][l64] = ff[r][2];
    }
  };
  double *tile = s_q[XR ? w : 0];
  auto load_q = [&](int k) {  // cells rmin+l of the chunk's rows (past the line: the last cell)
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      if constexpr (XR) {
        const int f = r * 64 + l64, ln = f / RC, col = f % RC;
        qn[r] = c[s_row[ln] + min(rmin + k * RC + 1 + col, g.rmax) + 1];
      } else {
        qn[r] = c[ob + os * (long long)(min(rmin + k * RC + 1 + r, g.rmax) + 1)];
      }
    }
  };
  auto take_q = [&](double (&q)[RC]) {
    if constexpr (XR) {
      wave_lds();
#pragma unroll
      for (int r = 0; r < RC; ++r) {
        const int f = r * 64 + l64;
        tile[(f / RC) * (RC + 1) + f % RC] = qn[r];
      }
      wave_lds();
#pragma unroll
      for (int r = 0; r < RC; ++r) q[r] = tile[l64 * (RC + 1) + r];
    } else {
#pragma unroll
      for (int r = 0; r < RC; ++r) q[r] = qn[r];
    }
  };
  const int nch = (n + RC - 1) / RC;
  double ql = c[ob + os * (long long)(rmin + 1)], qc = ql;  // BC_left_t0 = q(rmin) (:822)
  double Bc = 0.0;
  load_f(0);
  load_q(0);
  put_f(0);
  wg_lds_barrier();
  double Y[KC > 0 ? KC * RC : 1];
  constexpr int kUnroll = KC > 0 ? KC : 1;  // (kept chunks: registers by constant indexes)
#pragma unroll kUnroll
  for (int k = 0; k < (KC > 0 ? KC : nch); ++k) {
    if (KC == 0 || k < nch) {
      double q[RC];
      take_q(q);
      if (k + 1 < nch) {
        load_f(k + 1);
        load_q(k + 1);
      }
      const double(*s)[RC][64] = s_f[k & 1];
      if (on) {
#pragma unroll
        for (int r = 0; r < RC; ++r) {
          const int l = k * RC + r + 1;
          if (l <= n) {
            const double qr = l < n ? q[r] : qc;  // BC_right_t0 (:845)
            const double Bn = s[0][r][l64] * ql + s[1][r][l64] * qc + s[2][r][l64] * qr;
            if (l > 1) {
              if constexpr (KC > 0) Y[k * RC + r - 1] = Bc;
              else sb[row(l - 1)] = Bc;
              Bc = Bn - s[3][r][l64] * Bc;
            } else {
              Bc = Bn;
            }
            ql = qc;
            qc = qr;
          }
        }
      }
      if (k + 1 < nch) put_f(k + 1);
      wg_lds_barrier();
    }
  }

  // ---- back substitution: chunk k holds rows top - k*RC .. top - k*RC - RC + 1
  // (row n's right-hand side is Bc; kept ones go by the elimination's chunks)
  const int top = KC > 0 ? nch * RC : n;
  double fb[RPW][2], yn[KC > 0 ? 1 : RC];
  auto load_b = [&](int k) {
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      const int i = max(top - k * RC - (w * RPW + r), 1);
      const long long o = row(KC > 0 ? min(i, n) : i);
      fb[r][0] = fD[o];
      fb[r][1] = fDU[o];
    }
  };
  auto put_b = [&](int k) {
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      s_f[k & 1][0][w * RPW + r][l64] = fb[r][0];
      s_f[k & 1][1][w * RPW + r][l64] = fb[r][1];
    }
  };
  auto load_y = [&](int k) {
    if constexpr (KC == 0) {
#pragma unroll
      for (int r = 0; r < RC; ++r) yn[r] = sb[row(min(max(n - k * RC - r, 1), max(n - 1, 1)))];
    }
  };
  double x1 = 0.0, x2 = 0.0;
  load_b(0);
  load_y(0);
  put_b(0);
  wg_lds_barrier();
#pragma unroll kUnroll
  for (int j = 0; j < (KC > 0 ? KC : nch); ++j) {
    const int kk = KC - 1 - j;  // the kept chunk
    const int k = KC > 0 ? nch - 1 - kk : j;
    if (KC == 0 || kk < nch) {
      double y[RC], x[RC];
#pragma unroll
      for (int r = 0; r < RC; ++r) {
        if constexpr (KC > 0) y[r] = Y[kk * RC + RC - 1 - r];
        else y[r] = yn[r];
      }
      if (k + 1 < nch) {
        load_b(k + 1);
        load_y(k + 1);
      }
      const double(*s)[RC][64] = s_f[k & 1];
      if (on) {
#pragma unroll
        for (int r = 0; r < RC; ++r) {
          const int i = top - k * RC - r;
          x[r] = 0.0;
          if (i >= 1 && (KC == 0 || i <= n)) {
            const double D = s[0][r][l64], DU = s[1][r][l64];
            double xi;
            if (i == n) xi = Bc / D;
            else if (i == n - 1) xi = (y[r] - DU * x1) / D;
            else xi = (y[r] - DU * x1 - 0.0 * x2) / D;  // (the second super-diagonal is zero)
            x2 = x1;
            x1 = xi;
            x[r] = line_on ? xi : 0.0;
            if constexpr (!XR) c[ob + os * (long long)(rmin + i)] = x[r];
          }
        }
        if constexpr (XR) {
          wave_lds();
#pragma unroll
          for (int r = 0; r < RC; ++r) tile[l64 * (RC + 1) + (RC - 1 - r)] = x[r];
          wave_lds();
          const int lo = n - k * RC - RC;  // row of column 0, less one
#pragma unroll
          for (int r = 0; r < RC; ++r) {
            const int f = r * 64 + l64, ln = f / RC, col = f % RC, i = lo + 1 + col;
            if (tg.tile * 64 + ln < lines && i >= 1) c[s_row[ln] + rmin + i] = tile[ln * (RC + 1) + col];
          }
        }
      }
      if (k + 1 < nch) put_b(k + 1);
      wg_lds_barrier();
    }
  }
  // cells the reference leaves at zero: bins that are not aloft, and cells
  // outside [rmin, rmax] (off lines above)
  if (!exists) return;
  if (!on) return clear(c, 0, 1);
  if (repeat) return;
  for (int r = 1; r <= N; ++r)
    if (r < rmin || r > g.rmax) c[ob + os * (long long)(r + 1)] = 0.0;
}

template <bool XR, int NW, int RC, int KC = 0>
hipError_t launch(hipStream_t s, const ExactArgs &e) {
  const long long lines = (long long)e.A.g.Na * e.A.g.Nb;
  const long long blocks = padded_tiles((lines + 63) / 64) * ((e.A.d.ns + NW - 1) / NW);
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_cn_exact<XR, NW, RC, KC>), dim3((unsigned)blocks), dim3(64, NW), 0, s, e);
  return hipGetLastError();
}

}  // namespace

// Four waves per workgroup share the row coefficients (two or one for fewer
// bins), eight rows per chunk.  Measured when every line's right-hand sides
// still went through the ts1 slot, 240x160x50x8 x, y, z: 161, 138, 110 us; two
// waves 178, 133, 134; eight 240, 143, 121 (too few workgroups for the
// serial chains of one to fill the others' waits); 16 rows 152, 136, 117 but
// 254 against 238 on 241-cell rows, at 250 more registers.
hipError_t launch_cn_exact(hipStream_t s, const DiffArgs &a, const Dims *orig, double *c_orig) {
  const ExactArgs e{a, orig ? *orig : a.d, c_orig};
  if (orig) {
    if (a.d.ns >= 4) return launch<true, 4, 8>(s, e);
    return a.d.ns >= 2 ? launch<true, 2, 8>(s, e) : launch<true, 1, 8>(s, e);
  }
  // Right-hand sides kept in registers: z 118 -> 78 us at 240x160x50x8, 504 ->
  // 315 at 360x240x50x15, 142 -> 97 at 300x120x64x8; 10 chunks (two waves per
  // SIMD) 3.07 -> 1.92 ms at 1440x720x80x4, 35 us either way for the 80-cell y
  // lines of 120x80x40x10
  const int n = a.g.rmax - a.g.rmin + 1;
  if (n <= 64) {
    if (a.d.ns >= 4) return launch<false, 4, 8, 8>(s, e);
    return a.d.ns >= 2 ? launch<false, 2, 8, 8>(s, e) : launch<false, 1, 8, 8>(s, e);
  }
  if (n <= 80) {
    if (a.d.ns >= 4) return launch<false, 4, 8, 10>(s, e);
    return a.d.ns >= 2 ? launch<false, 2, 8, 10>(s, e) : launch<false, 1, 8, 10>(s, e);
  }
  if (a.d.ns >= 4) return launch<false, 4, 8>(s, e);
  return a.d.ns >= 2 ? launch<false, 2, 8>(s, e) : launch<false, 1, 8>(s, e);
}

}  // namespace ash3d
