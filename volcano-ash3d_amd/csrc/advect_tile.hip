// y and z sweeps of the limited donor-cell-upwind update in register tiles:
// advect_y (src/AdvectionHorz_DCU.f90:322-556) and advect_z / advect_sigma
// with settling and deposit (src/AdvectionVert_DCU.f90:100-323, :341-564).
//
// A wavefront takes 64 neighbouring lines (lanes along the contiguous
// index) and M consecutive cells of each; the cells and their +-2 stencil
// sit in registers, the bin-independent terms of the tile (interface
// speeds, dt/kappa) are formed once and serve every bin of the wave's bin
// group, and the next bin's cells are loaded while a bin is updated.  The
// sweep is bound by HBM latency and bandwidth; against the kernel that
// streams whole lines (advect.hip) a tile keeps M + 4 independent loads in
// flight per wave, shares the two divisions per cell among all bins, has no
// register window to shift, and cuts a line into N / M waves, so that small
// grids fill the chip.
//
// Neighbouring tiles read each other's edge cells, so the sweep runs out of
// place (cout != c0) with independent waves, or in place with a line's
// waves in one workgroup and a barrier per bin between its loads and its
// stores.  The arithmetic is the streamed kernel's, expression by
// expression, so the results are the same bits.
#include <algorithm>

#include "common.hpp"
#include "dcu.hpp"

namespace ash3d {

namespace {

constexpr int kTileBins = 8;  // most bins per group (their outflow increments wait in LDS)

struct TileArgs {
  AdvArgs A;
  int groups;   // bin groups (one wave each)
  int bins;     // bins per group
  bool plain;   // the whole grid and every bin: nothing to look up per wave
};

// Ghost cells along the lines read as zero: Set_BC(1) zeroes them in y and
// z before every sweep (src/Set_BC.f90:77-84).
template <int DIR, int M, int LIM, bool TOPO, bool INPL>
__device__ __forceinline__ void advect_tile_body(const TileArgs &T, const long long vb, const long long vn) {
  const AdvArgs &A = T.A;
  const Dims d = A.d;
  const LineGeom g = A.g;
  const int N = g.N, rmin = g.rmin, rmax = g.rmax;
  const int ntile = (g.Na + 63) / 64;
  const int S = (int)blockDim.y, LB = (N + M * S - 1) / (M * S);
  const TileGroup tg = xcd_tile_group(vb, T.groups, vn);
  if (tg.tile >= (long long)ntile * LB * g.Nb) return;  // padding workgroup (uniform)
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  // neighbouring lines first, then the line's tiles, then b: consecutive
  // workgroups touch consecutive addresses and share the tiles' edge cells
  // in the XCD's L2
  const int a0 = (int)(tg.tile % ntile) * 64 + 1;
  const long long rest = tg.tile / ntile;
  const int b = (int)(rest / LB) + 1;
  const int r0 = 1 + ((int)(rest % LB) * S + w) * M;  // first cell of the tile
  if (r0 > N) return;  // (in place S is the line's wave count: never)
  // lanes past the last line repeat it: the same loads, values and stores
  const int lane = (int)threadIdx.x;
  const unsigned al = (unsigned)min(lane, g.Na - a0);
  const bool repeat = a0 + lane > g.Na;
  const int a = a0 + (int)al;
  const bool line_on = a >= g.a0 && a <= g.a1 && b >= g.b0 && b <= g.b1;
  const bool plain = T.plain;
  const long long sL = line_stride(d, DIR), base = line_base(d, DIR, a0, b);
  auto row = [&](int r) { return base + sL * (long long)(r + 1); };  // uniform; + al
  double *junk = A.junk + lane + 64 * (int)(vb % (kJunk / 64));  // (of the wave with the line's last cells)
  const int nlo = tg.group * T.bins, nhi = min(nlo + T.bins, d.ns);
  const double *c = A.c0;
  double *co = A.cout;
  const int lim = A.limiter;
  const double dt = A.dt;
  const bool first = r0 == 1, last = r0 + M > N;  // the tile holds cell 1, cell N
  // A tile with no line or no cell of the box, and a bin that is not aloft,
  // are stored as zeros and not read (uniform; the outflow of an end of the
  // line belongs to a tile with cells of the box).  The 3x3x3 box of a
  // 360x240x50x15 step without diffusion: 641 us, 1057 us with every tile
  // read.  Bit n - nlo of run: bin n is swept here
  const unsigned group = (1u << (nhi - nlo)) - 1, on = plain ? group : A.aloft.bits(nlo, nhi);
  const bool in_box = a0 <= g.a1 && a0 + 63 >= g.a0 && b >= g.b0 && b <= g.b1 && r0 <= rmax && r0 + M > rmin;
  const unsigned run = in_box ? on : 0u;
  for (unsigned z = group & ~run; z; z &= z - 1) {
    const int u = __builtin_ctz(z);
    if (INPL && (on >> u & 1)) __syncthreads();  // (other waves read this tile's edge cells)
    double *cn = co + d.ncell * (long long)(nlo + u);
#pragma unroll
    for (int i = 0; i < M; ++i) (r0 + i <= N ? cn + row(r0 + i) + al : junk)[0] = 0.0;
  }
  if (!run) {
    if (DIR == 2 && first && !repeat)
      for (int n = nlo; n < nhi; ++n)
        A.dep[(long long)(a - 1) + (long long)d.nx * ((long long)(b - 1) + (long long)d.ny * n)] =
            A.of1[(long long)(a + 1) + (long long)(g.Na + 4) * ((long long)(b + 1) + (long long)(g.Nb + 4) * n)];
    return;
  }
  // ---- bin-independent terms.  Interface i of the tile is I = r0 + i
  // (0 <= i <= M), between cells I-1 and I
  double sg[M + 1], dtv[M + 1];
  double ub[M + 1];       // y: usig (:159-162); z: sigma of the interface
  double wv[M + 2];       // z: vz + vh of cells r0-1 .. r0+M
  double tf[M + 1], D[M + 1];  // topographic factor and D of cells r0-1 .. r0+M-1
  double um = 0.0, wm = 0.0, sg0 = 0.0, dtv0 = 0.0;  // interface 0 and cell 0, for the outflow at cell 0
  {
    double kp[M + 1], vl[M + 2], vh[M + 2];
#pragma unroll
    for (int i = 0; i <= M; ++i) {
      const long long o = row(min(r0 + i, N + 2));
      sg[i] = A.sig[o + al];
      kp[i] = A.kap[o + al];
    }
#pragma unroll
    for (int i = 0; i < M + 2; ++i) {
      const long long o = row(min(r0 - 1 + i, N + 2));
      vl[i] = A.vel[o + al];
      vh[i] = DIR == 2 ? A.vh[o + al] : 0.0;
    }
    double sgm = 0.0, kp0 = 0.0, vm = 0.0, vhm = 0.0;
    if (first || TOPO) sgm = A.sig[row(r0 - 1) + al];
    if (first) {
      kp0 = A.kap[row(0) + al];
      vm = A.vel[row(-1) + al];
      if (DIR == 2) vhm = A.vh[row(-1) + al];
    }
#pragma unroll
    for (int i = 0; i <= M; ++i) dtv[i] = dt / kp[i];  // (:155-156)
    if (first) dtv0 = dt / kp0;
    if constexpr (DIR == 2) {
#pragma unroll
      for (int i = 0; i < M + 2; ++i) wv[i] = vl[i] + vh[i];
#pragma unroll
      for (int i = 0; i <= M; ++i) ub[i] = sg[i];
      wm = vm + vhm;
      sg0 = sgm;
    } else {
#pragma unroll
      for (int i = 0; i <= M; ++i) ub[i] = 0.5 * (vl[i] + vl[i + 1]) * sg[i];
      um = 0.5 * (vm + vl[0]) * sgm;
    }
    if constexpr (TOPO) {
      // 0.5 * vel_c * (sig_c + sig_{c+1}) and DelD_c (:252-257), the latter
      // zero outside rmin-1 .. rmax+1
#pragma unroll
      for (int i = 0; i <= M; ++i) {
        const int cc = r0 - 1 + i;
        tf[i] = 0.5 * vl[i] * ((i == 0 ? sgm : sg[i > 0 ? i - 1 : 0]) + sg[i]);
        const double dd = A.deld[(long long)(a + 1) + (long long)(d.nx + 4) * (min(cc, N + 2) + 1)];
        D[i] = (cc >= rmin - 1 && cc <= rmax + 1) ? dd : 0.0;
      }
    }
  }
  // the outflow increments of the line ends wait in LDS, element (end, bin,
  // lane), and are added after the bins
  extern __shared__ double s_of[];
  const bool at_lo = first && rmin == 1, at_hi = last && rmax == N;

  // the cells r0-2 .. r0+M+1 of a bin (and the fall speeds of r0-1 .. r0+M)
  double qs[M + 4], vs[M + 2];
  auto fetch = [&](int n) {
    const double *cn = c + d.ncell * (long long)n;
#pragma unroll
    for (int i = 0; i < M + 4; ++i) qs[i] = (cn + row(min(max(r0 - 2 + i, 1), N)))[al];
    if constexpr (DIR == 2) {
      const double *fn = A.vf + d.ncell * (long long)n;
#pragma unroll
      for (int i = 0; i < M + 2; ++i) vs[i] = (fn + row(min(r0 - 1 + i, N + 2)))[al];
    }
  };
  fetch(nlo + __builtin_ctz(run));
  for (unsigned left = run; left; left &= left - 1) {
    const int n = nlo + __builtin_ctz(left);
    double q[M + 4], vc[M + 2];
#pragma unroll
    for (int i = 0; i < M + 4; ++i) q[i] = qs[i];
#pragma unroll
    for (int i = 0; i < M + 2; ++i) vc[i] = DIR == 2 ? wv[i] + vs[i] : 0.0;  // (:171-176)
    const double vf0 = DIR == 2 ? vs[0] : 0.0;
    const unsigned next = left & (left - 1);
    fetch(nlo + __builtin_ctz(next ? next : left));
    if (first) q[0] = q[1] = 0.0;
    if (r0 + M + 1 > N) {
#pragma unroll
      for (int i = 2; i < M + 4; ++i)
        if (r0 - 2 + i > N) q[i] = 0.0;
    }
    // interface i: the limited flux, whose interfaces rmin .. rmax+1
    // (:178-231) hold every interface of a cell that is stored or leaves the
    // grid, and the fluctuations (:238-259)
    double dq[M + 3], u[M + 1], fss[M + 1], up[M + 1], un[M + 1], res[M];
#pragma unroll
    for (int i = 0; i < M + 3; ++i) dq[i] = q[i + 1] - q[i];  // interface r0-1+i (:168-169)
#pragma unroll
    for (int i = 0; i <= M; ++i) {
      u[i] = DIR == 2 ? 0.5 * (vc[i] + vc[i + 1]) * ub[i] : ub[i];
      fss[i] = LIM == 0 ? 0.0 : limited_flux_flat<LIM>(lim, dq[i], dq[i + 1], dq[i + 2], u[i], dtv[i]);
      up[i] = fmax(0.0, u[i]);
      un[i] = fmin(0.0, u[i]);
    }
#pragma unroll
    for (int i = 0; i < M; ++i) {
      // cell r0 + i (:264-281)
      double fsl = un[i + 1] * dq[i + 2], fsr = up[i] * dq[i + 1];
      fsl = fsl + q[i + 2] * (up[i + 1] - up[i]);
      fsr = fsr + q[i + 2] * (un[i + 1] - un[i]);
      if (TOPO) {
        const double t = tf[i + 1] * q[i + 2] * D[i + 1];
        fsl = fsl - t;
        fsr = fsr + t;
      }
      const double upd = -dtv[i] * (fsl + fsr + fss[i + 1] - fss[i]);
      res[i] = q[i + 2] + upd;
    }
    if (!plain) {
#pragma unroll
      for (int i = 0; i < M; ++i) res[i] = (line_on && r0 + i >= rmin && r0 + i <= rmax) ? res[i] : 0.0;
    }
    if constexpr (INPL) __syncthreads();  // every load of the bin before its first store
    double *cn = co + d.ncell * (long long)n;
#pragma unroll
    for (int i = 0; i < M; ++i) (r0 + i <= N ? cn + row(r0 + i) + al : junk)[0] = res[i];
    if (at_lo) {
      // cell 0 (:289-291, :540-542; the deposit of z): interfaces 0 and 1
      const double ul = DIR == 2 ? 0.5 * ((wm + vf0) + vc[0]) * sg0 : um;
      double fsl = un[0] * dq[1], fsr = fmax(0.0, ul) * dq[0];
      fsr = fsr + q[1] * (un[0] - fmin(0.0, ul));
      fsl = fsl + q[1] * (up[0] - fmax(0.0, ul));
      if (TOPO) {
        const double t = tf[0] * q[1] * D[0];
        fsr = fsr + t;
        fsl = fsl - t;
      }
      s_of[(n - nlo) * 64 + lane] = -dtv0 * (fsl + fsr + fss[0] - 0.0);
    }
    if (at_hi) {
      // cell N+1 = r0 + i: interface N+2 is outside the sweep's range (zero)
#pragma unroll
      for (int i = 1; i <= M; ++i)
        if (r0 + i == N + 1) {
          double fsr = up[i] * dq[i + 1];
          fsr = fsr + q[i + 2] * (0.0 - un[i]);
          s_of[(T.bins + n - nlo) * 64 + lane] = -dtv[i] * (0.0 + fsr + 0.0 - fss[i]);
        }
    }
  }
  if (!first && !at_hi) return;
  const long long of0 = (long long)(a + 1) + (long long)(g.Na + 4) * (long long)(b + 1);
  const long long ofb = (long long)(g.Na + 4) * (g.Nb + 4);
  if (repeat) return;  // (the last line's increments once)
  for (int n = nlo; n < nhi; ++n) {
    const bool swept = line_on && (run >> (n - nlo) & 1);
    const long long of = of0 + ofb * (long long)n;
    if (at_hi && swept) A.of2[of] = A.of2[of] + s_of[(T.bins + n - nlo) * 64 + lane];
    if (!first) continue;
    if (DIR == 2 || (at_lo && swept)) {
      double v = A.of1[of];
      if (at_lo && swept) {
        v = v + s_of[(n - nlo) * 64 + lane];
        A.of1[of] = v;
      }
      // DepositGranularity = outflow_xy1 (src/AdvectionVert_DCU.f90:321)
      if (DIR == 2)
        A.dep[(long long)(a - 1) + (long long)d.nx * ((long long)(b - 1) + (long long)d.ny * n)] = v;
    }
  }
}

// most threads of a workgroup (in place: the waves of a line of 60, 48 or 64 cells)
template <int M, bool INPL>
constexpr int kTileThreads = !INPL ? 256 : M == 5 ? 768 : 512;

template <int DIR, int M, int LIM, bool TOPO, bool INPL>
__global__ __launch_bounds__((kTileThreads<M, INPL>)) void k_advect_tile(TileArgs T) {
  advect_tile_body<DIR, M, LIM, TOPO, INPL>(T, blockIdx.x, gridDim.x);
}
template <int DIR, int M, int LIM, bool TOPO, bool INPL>
__global__ __launch_bounds__((kTileThreads<M, INPL>)) void k_advect_tile_batch(
    const ASH3D_CONSTANT TileArgs *__restrict__ args, const ASH3D_CONSTANT int *__restrict__ member,
    const ASH3D_CONSTANT long long *__restrict__ first) {
  const int m = member[blockIdx.x];
  const TileArgs &T = *(const TileArgs *)(args + m);
  advect_tile_body<DIR, M, LIM, TOPO, INPL>(T, (long long)blockIdx.x - first[m], first[m + 1] - first[m]);
}

template <int DIR, int M, int LIM, bool TOPO, bool INPL>
hipError_t launch_tile(hipStream_t s, const AdvArgs &a, LaunchSpec *sp) {
  const int S = INPL ? (a.g.N + M - 1) / M : 4;
  const long long tiles = (long long)((a.g.Na + 63) / 64) * ((a.g.N + M * S - 1) / (M * S)) * a.g.Nb;
  // bin groups: enough waves to fill the chip (256 CUs x 4 SIMDs x 2; more
  // only form the bin-independent terms more often), and at most 8 bins, so
  // that the last round of waves is short (15 bins in one group: 5 % slower
  // on 360x240x50)
  const long long want = std::max<long long>((2048 + tiles * S - 1) / (tiles * S), (a.d.ns + kTileBins - 1) / kTileBins);
  TileArgs t{a, 1, a.d.ns, true};
  for (int n = 0; n < a.d.ns; ++n) t.plain = t.plain && a.aloft.on(n);
  const LineGeom &g = a.g;
  t.plain = t.plain && g.rmin == 1 && g.rmax == g.N && g.a0 == 1 && g.a1 == g.Na && g.b0 == 1 && g.b1 == g.Nb;
  t.groups = (int)std::min<long long>(a.d.ns, want);
  t.bins = (a.d.ns + t.groups - 1) / t.groups;
  t.groups = (a.d.ns + t.bins - 1) / t.bins;
  const size_t lds = sizeof(double) * 2 * 64 * kTileBins;  // one size, so that members of an ensemble share a launch
  const long long blocks = padded_tiles(tiles) * t.groups;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  return issue(s, sp, (const void *)k_advect_tile<DIR, M, LIM, TOPO, INPL>,
               (const void *)k_advect_tile_batch<DIR, M, LIM, TOPO, INPL>, dim3((unsigned)blocks), dim3(64, S), lds, t);
}

template <int DIR, int M, bool TOPO, bool INPL>
hipError_t tile_lim(hipStream_t s, const AdvArgs &a, LaunchSpec *sp) {
  switch (a.limiter) {
    case 0: return launch_tile<DIR, M, 0, TOPO, INPL>(s, a, sp);
    case 5: return launch_tile<DIR, M, 5, TOPO, INPL>(s, a, sp);  // superbee, the reference's default
    default: return launch_tile<DIR, M, -1, TOPO, INPL>(s, a, sp);
  }
}

}  // namespace

// The y or z sweep of a in register tiles: issued (or described in sp), or
// hipErrorInvalidValue where the streamed kernel runs it (advect_tile_applies).
//
// Out of place: five cells per wave, 162 VGPRs, three waves per SIMD (with
// topography 194, two).  Measured on 360x240x50x15 (64.8 M bin-cells,
// superbee): y 300 us, z 467 us against 331 and 481 streamed; 1440x720x80x4:
// 1.55 and 2.45 ms (4.7 and 4.3 TB/s of the compulsory bytes) against 2.33 (y
// streamed) and, for the fused second horizontal + z pass, 4.2 ms;
// 120x80x40x10: 18 and 24 us against 47 and 55.  Three, four or six cells: y
// 315, 304, 300 us, z 492, 472, 478 us on the first grid.  One, two or three
// waves per workgroup instead of four, tiles of 64 lines cut across the ends
// of the rows (no idle lanes, but neighbouring tiles further apart in time: y
// 335 us), non-temporal stores (y 343 us): no gain.
//
// In place a line's N / M waves are one workgroup, and as many workgroups as
// fit a CU overlap one's loads with another's barrier: five cells (12 waves
// per CU, up to 60 cells) unless eight (8 waves) let two workgroups in where
// the waves of five cells are as many and shorter (21 to 32 cells: z of
// 656x58x31x10 90 us against 105 with five and 122 with six), or lines of 41
// to 48 cells fill 7 or 8 waves of six (z of 565x28x45x20 118 us against 124
// with five and eight).  z of 46x26x53x2, 76x22x49x9, 240x160x50x9: 17, 21 and
// 158 us against 58, 58 and 193 streamed.
hipError_t advect_tile(hipStream_t s, const AdvArgs &a, LaunchSpec *sp) {
  const bool inpl = a.cout == a.c0;
  const int N = a.g.N;
  if (!advect_tile_applies(a.g, a.d.ns, inpl)) return hipErrorInvalidValue;
  if (!inpl) {
    if (a.g.dir == 2) return tile_lim<2, 5, false, false>(s, a, sp);
    return a.deld ? tile_lim<1, 5, true, false>(s, a, sp) : tile_lim<1, 5, false, false>(s, a, sp);
  }
  const bool six = N > 40 && N <= 48, eight = (N > 20 && N <= 32) || N > 60;
  if (a.g.dir == 2) {
    if (six) return tile_lim<2, 6, false, true>(s, a, sp);
    return eight ? tile_lim<2, 8, false, true>(s, a, sp) : tile_lim<2, 5, false, true>(s, a, sp);
  }
  // (with topography five cells take more than three waves' registers)
  if (a.deld) return N <= 48 ? tile_lim<1, 6, true, true>(s, a, sp) : tile_lim<1, 8, true, true>(s, a, sp);
  if (six) return tile_lim<1, 6, false, true>(s, a, sp);
  return eight ? tile_lim<1, 8, false, true>(s, a, sp) : tile_lim<1, 5, false, true>(s, a, sp);
}

// Streamed instead: the z box that ends at the top without starting at the
// bottom (its top outflow is the update of cell ncells+1, src/
// AdvectionVert_DCU.f90:309-311); in place lines of more than 64 cells (their
// waves would not fit one workgroup), and z lines with enough tiles to fill
// the chip either way, where a tile's set-up serves few bins (one, or two, four
// or eight, which the streamed kernel takes in whole pairs), or long lines have
// many bins.  Tile of five, six or eight cells against streamed: 497x387x54x2
// 271 and 236 us, 354x247x35x2 72 and 63, 334x221x50x4 163 and 149,
// 663x253x31x1 78 and 68, 607x194x51x1 104 and 82, 134x180x41x8 100 and 85,
// 240x160x50x8 137 and 131, 360x240x50x15 532 and 504, 426x189x63x15 603 and
// 563; below the bounds 552x94x60x2 73 and 89, 389x90x58x1 40 and 46,
// 41x253x45x8 49 and 59, 65x25x58x15 44 and 91.
bool advect_tile_applies(const LineGeom &g, int ns, bool in_place) {
  if (g.dir == 0 || (g.dir == 2 && g.rmax == g.N && g.rmin != 1)) return false;
  if (!in_place) return true;
  if (g.N > 64) return false;
  if (g.dir == 1) return true;
  const long long tiles = (long long)((g.Na + 63) / 64) * g.Nb;
  if (ns == 1 && g.N > 20 && tiles >= 768) return false;
  if ((ns == 2 || ns == 4) && g.N > 32 && tiles >= 1024) return false;
  if (ns == 8 && g.N > 32 && tiles >= 512) return false;
  return !(ns > 12 && g.N > 48 && tiles >= 1024);
}

}  // namespace ash3d
