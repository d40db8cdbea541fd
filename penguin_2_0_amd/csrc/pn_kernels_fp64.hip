// pn_kernels_fp64.hip -- FP64 directional sweeps (the drop-in path).
//
// Built with -ffp-contract=off so each operation rounds as the reference's does; the
// remaining differences to a CPU FP64 build are the last-ulp results of the device
// transcendentals (sqrt, exp, log, pow, sin, cos) and, in 2-D, of the series and reciprocal roots
// that stand for some of them.
//
// These sweeps are bound by the FP64 VALU, so what they cost is their instruction count.  The
// geometry's reciprocals, the Eulerian paraset and the star's pull at fixed radii come from a
// per-slot table instead of ~60 divisions a cell, the rest share reciprocals (div64), and in 2-D
// the angle to the planet is turned from a per-column cosine and sine instead of taken anew at
// three times: 1024 x 3072, inviscid, 5347 -> 2516 static VALU instructions a radial pass.  With the
// radial and theta sweeps staged through LDS and short windows packed two to a wavefront (below):
//   1024 x 3072 radial 197 -> 113 us, azimuthal 189 -> 114 us; 256 x 768 radial 29.2 -> 13.4 us;
//   96 x 288 x 32, whose sweeps round every operation as written, r / phi / theta 97 / 78 / 342 ->
//   58 / 56 / 101 us (timed back to back; the azimuthal ones carry the next step's CFL since).
#include "pn_launch.hpp"
#include "ppm_wave.hpp"

namespace pn {

namespace {

constexpr int kK = 2;              // cells per lane: 64 lanes x 2 = one 128-cell window
constexpr int kWavesPerBlock = 4;
constexpr double kTwoPi = 6.283185307179586476925286766559;

__device__ __forceinline__ int xcd_swizzle(int bid, int nblk) {
  const int nx = 8;
  int q = nblk / nx, rem = nblk % nx;
  int x = bid % nx, idx = bid / nx;
  return x * q + (x < rem ? x : rem) + idx;
}

__device__ __forceinline__ int wrapj(int j, int jmax) {
  if (j < 0) j += jmax;
  if (j >= jmax) j -= jmax;
  return j;
}

__device__ __forceinline__ int win_len(int len, int nwin, int l) {
  return (l < nwin - 1) ? kWin : (len - kReal * (nwin - 1) + 2 * kNpad);
}

__device__ __forceinline__ Planet load_planet(const StepScalars* ss, int bary) {
  Planet p;
  p.bary = bary;
  p.m = ss->planet.m;
  p.x = ss->planet.x;
  p.y = ss->planet.y;
  p.vx = ss->planet.vx;
  p.vy = ss->planet.vy;
  p.rs = ss->planet.rs;
  return p;
}

// Waves per SIMD asked for.  The isothermal sweeps settle at 166-190 VGPRs, two waves; at 168 they
// hold three for at most nine spilled registers a pass (1024 x 3072 azimuthal 115 -> 108 us, theta
// sweep of 96 x 288 x 32 190 -> 176 us).  The other closures need 210 and more: two waves.
template <class CF>
constexpr int waves64() {
  return CF::EOS == 0 ? 3 : 1;
}

// CFL term of one direction, (|v| + c_s) / width (timestep.cu:48-73), y = 1 / width: the rounded
// quotient, and infinity for an infinite speed (which div64 alone would lose)
__device__ __forceinline__ double cfl_term(double v, double cs, double width, double y) {
  const double a = fabs(v) + cs;
  return fmax(div64(a, width, y), 0.5 * (a * y));
}
// sqrt(gam p / r) of the CFL, rounded as written; anything but an ordinary positive quotient by the
// library's root (a negative pressure gives NaN, which the maximum passes over)
__device__ __forceinline__ double cfl_sound(double gp, double r) {
  const double y = rcp64(r);
  const double c2 = fmax(div64(gp, r, y), 0.5 * (gp * y));
  const double s = sqrt64_rn(c2);
  return c2 > 0.0 && c2 < 1.0e300 ? s : sqrt(c2);
}
__device__ __forceinline__ double wave_max(double v) {
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
  return v;
}

// ---------------------------------------------------------------------------------------
// radial and theta sweeps (sweepx, ppm.cu:26-160; the reference has no caller for the theta sweep,
// main.cu:376: it is assembled from the theta pieces it holds, forces.cu:298-372,
// states.cu:29-39, evolve.cu:26-29, 63-67, 110-124, remap.cu:50-54, init.cpp:415-541).
//
// A pencil crosses rings, so its cells lie jmax apart in HBM and a wavefront's load of one field
// touched 128 lines; the cells of neighbouring lab columns are contiguous.  A workgroup of four
// waves therefore takes one window of four consecutive columns, stages its fields in LDS with
// loads contiguous along phi, runs a pencil per wave from LDS, puts the results back in place and
// stores them contiguously (1024 x 3072 radial: 148 -> 125 us; two columns a wave, for 64-byte
// rows, lost more to the registers its loop holds: 192 us).  A window of at most 64 cells (a short
// last window, a short theta pencil) takes eight columns instead, two per wavefront, one in each
// half: every stage indexes cells within its own window, so a stencil across the seam sees what it
// sees past a window's end, and no kept cell depends on it.
template <int NF>
struct Tile64 {
  // [field][column][cell]: 4 columns of 130 or 8 of 66 (even strides: two-cell reads aligned)
  static constexpr int kField = 528;
  double f[NF][kField];
  int srot[kWin];   // rot_j of the window's slots
  double red[kWavesPerBlock];
};

// columns of a workgroup's window of lim cells
__host__ __device__ inline int tile_columns(int lim) { return lim <= kWin / 2 ? 2 * kWavesPerBlock : kWavesPerBlock; }

// With do_cfl (the theta sweep, a 3-D step's last) every thread returns the largest CFL term of the
// cells it stored.
template <class CF>
__device__ __forceinline__ double pencil64(const DevGrid& g, const DevParams& prm, const StepScalars* __restrict__ ss,
                                           int src, int grp, int l, int row, int do_cfl,
                                           Tile64<CF::GX == 2 ? 5 : 4>& T) {
  constexpr bool TH = CF::AXIS == 2;
  constexpr int NF = CF::GX == 2 ? 5 : 4, TPB = 64 * kWavesPerBlock, NIT = 2;
  const int jmax = g.jmax;
  const int lim = TH ? win_len(g.kmax, g.nwin_z, l) : win_len(g.imax, g.nwin_x, l);
  const int s0 = TH ? slot_of(g, row, kReal * l - kNpad) : slot_of(g, kReal * l - kNpad, row);
  const int step = TH ? g.sr : 1;
  const bool two = lim <= kWin / 2;   // workgroup-uniform: two columns per wavefront
  const int sh = two ? 3 : 2, nc = 1 << sh, ld = two ? kWin / 2 + 2 : kWin + 2;
  const int jb = grp * nc;
  static_assert(kWavesPerBlock == 4, "columns of a workgroup");
  // staging: this thread moves cells cs and cs + cstep of column qs; columns past jmax read column
  // jmax - 1, which is not stored
  const int cstep = TPB >> sh, qs = threadIdx.x & (nc - 1), cs = threadIdx.x >> sh;
  const int jl = jb + qs, jlc = jl < jmax ? jl : jmax - 1;
  for (int c = threadIdx.x; c < kWin; c += TPB) T.srot[c] = g.rot_j[s0 + step * (c < lim ? c : lim - 1)];
  __syncthreads();
  double v[NIT][NF];
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = cs + cstep * it;
    const long a = (long)(s0 + step * (c < lim ? c : lim - 1)) * jmax + wrapj(jlc - T.srot[c], jmax);
#pragma unroll
    for (int f = 0; f < NF; ++f) v[it][f] = g.f[src][f][a];
  }
#pragma unroll
  for (int it = 0; it < NIT; ++it)
#pragma unroll
    for (int f = 0; f < NF; ++f) T.f[f][qs * ld + cs + cstep * it] = v[it][f];
  __syncthreads();

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double dt = ss->dt, FrRot = ss->FrRot;
  const Planet pl = load_planet(ss, prm.bary);
  const RunFlags rf{prm.flat, prm.plnt > 0, 1, prm.has_w, prm.ndim};
  const int ll = two ? lane % 32 : lane, c0 = kK * ll;
  const int q = two ? 2 * wv + lane / 32 : wv;   // this lane's column
  if (jb + (two ? 2 * wv : wv) < jmax) {         // wave-uniform; the barriers below are outside
    const int j0 = jb + q < jmax ? jb + q : jmax - 1;
    // cells past the window read the table's next slots or its overhang (finite values no kept
    // cell depends on)
    const TabLane64 tx{TH ? g.tabz : g.tab, g.tstride,
                       8u * (unsigned)((TH ? kReal * l - kNpad + g.k0 + g.sk * (row + kNpad) : s0) + c0)};
    double* const tf = &T.f[0][q * ld + c0];   // this lane's cells of field 0
    constexpr int fs = Tile64<NF>::kField;
    Win<kK> W;
    const C<double, kK> radc = tx.get(kT64Rc);
    W.rad = tx.get(kT64Rad);
    W.xa0 = tx.get(TH ? kT64Za : kT64Xa);
    W.dx0 = tx.get(TH ? kT64Dz : kT64Dx);
    W.dvol0 = tx.get(TH ? kT64Volz : kT64Vol);
    W.azi = splat<double, kK>(g.yc[j0]);
    const double2 tr = g.ptrig[j0];
    W.ca = splat<double, kK>(tr.x);
    W.sa = splat<double, kK>(tr.y);
    long aw[kK];   // 2-D: w, carried only by a state that has one, comes straight from HBM
#pragma unroll
    for (int h = 0; h < kK; ++h) {
      const int c = c0 + h;
      const double r = tf[FR * fs + h], p = tf[FP * fs + h], fu = tf[FU * fs + h], fv = tf[FV * fs + h];
      double u, vv, w;
      if constexpr (TH) {   // sweep components: v_theta, v_r, angular momentum
        u = tf[FW * fs + h];
        vv = fu;
        w = fv * radc[h];
      } else {
        u = fu;
        vv = fv * radc[h];
        if constexpr (CF::GX == 2) {
          w = tf[FW * fs + h] * W.rad[h];
        } else {
          w = 0.0;
          if (prm.has_w) {
            const int cc = c < lim ? c : lim - 1;
            aw[h] = (long)(s0 + cc) * jmax + wrapj(j0 - T.srot[cc], jmax);
            w = g.f[src][FW][aw[h]];
          }
        }
      }
      W.r[h] = r; W.p[h] = p; W.u[h] = u; W.v[h] = vv; W.w[h] = w;
      W.e[h] = energy_of<CF>(p, r, u, vv, prm.gam);
    }

    ppmlr_wave<kK, CF>(W, tx, Ring64{}, c0, lim, dt, FrRot, pl, rf, prm.gam);
    const C<double, kK> irc = tx.get(kT64Irc), cs2 = tx.get(kT64Cs2);
    C<double, kK> vphi;
    if constexpr (TH) {
      // v_phi from the angular momentum the sweep carried; then device_viscosity_z
      // (viscosity.cu:474-518) on (v_r, v_phi, v_theta)
#pragma unroll
      for (int h = 0; h < kK; ++h) vphi[h] = div64(W.w[h], radc[h], irc[h]);
      if constexpr (CF::VISC) {
        C<double, kK> x;
#pragma unroll
        for (int h = 0; h < kK; ++h) x[h] = W.xa0[h] * W.rad[h];
        visc_z<kK, true>(W.r, c0, lim, dt, prm.vis_nu, x, W.v, vphi, W.u);
      }
    } else {
      if constexpr (CF::VISC) visc_r<kK, CF::GX == 2>(W, c0, lim, dt, radc, tx.get(kT64Nu), prm.ndim == 3);
#pragma unroll
      for (int h = 0; h < kK; ++h) vphi[h] = div64(W.v[h], radc[h], irc[h]);
    }
#pragma unroll
    for (int h = 0; h < kK; ++h) {
      const int c = c0 + h;
      if (c >= kNpad && c < lim - kNpad) {   // only this half's lanes hold column q
        const double r = W.r[h];
        double p;
        if constexpr (CF::EOS == 0) p = r * cs2[h];
        else if constexpr (CF::EOS == 1) p = cs2[h] * pow(r, prm.gam) / prm.gam;
        else p = W.p[h];
        tf[FR * fs + h] = r;
        tf[FP * fs + h] = p;
        tf[FU * fs + h] = TH ? W.v[h] : W.u[h];
        tf[FV * fs + h] = vphi[h];
        if constexpr (TH) tf[FW * fs + h] = W.u[h];
        else if constexpr (CF::GX == 2) tf[FW * fs + h] = W.w[h] / W.rad[h];
        else if (prm.has_w && jb + q < jmax) g.f[src ^ 1][FW][aw[h]] = W.w[h];
      }
    }
  }
  __syncthreads();
  double m = 0.0;
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = cs + cstep * it;
    if (jl < jmax && c >= kNpad && c < lim - kNpad) {
      const int s = s0 + step * c, j = wrapj(jl - T.srot[c], jmax);
      const long a = (long)s * jmax + j;
      double x[NF];
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        x[f] = T.f[f][qs * ld + c];
        g.f[src ^ 1][f][a] = x[f];
      }
      if constexpr (TH) {
        if (do_cfl) {   // k_cfl's terms of this cell
          const double* t = g.tab + s;
          const long ts = g.tstride;
          const double rc = t[kT64Rc * ts], snd = cfl_sound(prm.gam * x[FP], x[FR]);
          const double wy = g.dy[j] * rc, wz = t[kT64Dz * ts] * t[kT64Rad * ts];
          m = fmax(m, cfl_term(x[FU], snd, t[kT64Dx * ts], t[kT64Idx * ts]));
          m = fmax(m, cfl_term(x[FV] - g.rot_v[s] - FrRot * rc, snd, wy, rcp64(wy)));
          m = fmax(m, cfl_term(x[FW], snd, wz, rcp64(wz)));
        }
      }
    }
  }
  return m;
}

// the largest of a workgroup's values to *out; red: one double per wave
__device__ __forceinline__ void block_cfl(double m, double* red, double* out) {
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) *out = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// workgroups of one row's windows: every window but the last is full
__host__ __device__ inline int row_groups(int len, int nwin, int jmax, int* last) {
  const int nc = tile_columns(len - kReal * (nwin - 1) + 2 * kNpad);
  *last = (jmax + nc - 1) / nc;
  return (nwin - 1) * ((jmax + kWavesPerBlock - 1) / kWavesPerBlock) + *last;
}

// items: column group x window x row (radial: theta layer k; theta: ring i), column groups fastest,
// so that workgroups of one XCD share the lines of neighbouring columns
template <class CF>
__global__ __launch_bounds__(64 * kWavesPerBlock) __attribute__((amdgpu_waves_per_eu(waves64<CF>(), 8))) void k_pencil64(
    DevGrid g, DevParams prm, const StepScalars* __restrict__ ss, double* __restrict__ cflp, int src, int do_cfl) {
  __shared__ Tile64<CF::GX == 2 ? 5 : 4> T;
  const int nwin = CF::AXIS == 2 ? g.nwin_z : g.nwin_x, len = CF::AXIS == 2 ? g.kmax : g.imax;
  const int full = (g.jmax + kWavesPerBlock - 1) / kWavesPerBlock;
  int last;
  const int per = row_groups(len, nwin, g.jmax, &last);
  const int bid = xcd_swizzle(blockIdx.x, gridDim.x);
  const int row = bid / per, r = bid % per;
  const int l = r < (nwin - 1) * full ? r / full : nwin - 1;
  const double m = pencil64<CF>(g, prm, ss, src, r - l * full, l, row, do_cfl, T);
  if constexpr (CF::AXIS == 2) {
    if (do_cfl) block_cfl(m, T.red, &cflp[blockIdx.x]);   // kernel-uniform
  }
}

// ---------------------------------------------------------------------------------------
// azimuthal sweep (sweepy, ppm.cu:162-307): pencil = one periodic ring
template <class CF>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(waves64<CF>(), 8))) void k_sweep_y(DevGrid g, DevParams prm, const StepScalars* __restrict__ ss,
                                                 double* __restrict__ cflp, int src, int do_cfl) {
  __shared__ double red[kWavesPerBlock];
  double m = 0.0;
  const int lane = threadIdx.x & 63;
  const int gw = xcd_swizzle(blockIdx.x, gridDim.x) * kWavesPerBlock + (threadIdx.x >> 6);
  const int l = gw % g.nwin_y;
  const int n = gw / g.nwin_y;
  if (n < g.imax * g.kmax) {   // wave-uniform; the barrier is outside
  const int i = n % g.imax, k = n / g.imax;
  const int s = slot_of(g, i, k);
  const int jmax = g.jmax;

  const double dt = ss->dt, FrRot = ss->FrRot;
  const Planet pl = load_planet(ss, prm.bary);
  // sweep slots: u = v_phi, v = physical w, w = v_r (always carried)
  RunFlags rf{prm.flat, prm.plnt > 0, prm.has_w, 1, prm.ndim};
  const int lim = win_len(jmax, g.nwin_y, l);
  const int rot = g.rot_j[s];
  const double rc = g.radc[s];
  const double pol = (prm.ndim == 3) ? g.zc[s] : 0.0;
  const double vrot = g.res_v[s] / rc;
  const long base = (long)s * jmax;
  const double* __restrict__ fr = g.f[src][FR] + base;
  const double* __restrict__ fp = g.f[src][FP] + base;
  const double* __restrict__ fu = g.f[src][FU] + base;
  const double* __restrict__ fv = g.f[src][FV] + base;
  const double* __restrict__ fw = g.f[src][FW] + base;

  Win<kK> W;
  int jd[kK];
  const double sinpol = prm.ndim == 3 ? g.tab[kT64Sp * g.tstride + s] : 1.0;
  const Ring64 ring{vrot, 1.0 / rc, sinpol, pol, rc / sinpol, g.uniform_phi ? g.p0y : nullptr};
#pragma unroll
  for (int h = 0; h < kK; ++h) {
    const int c = kK * lane + h;
    int jref = kReal * l - kNpad + (c < lim ? c : lim - 1);
    const int j0 = wrapj(jref, jmax);
    const int j = wrapj(j0 - rot, jmax);
    jd[h] = j;
    double azi = g.yc[j0], xa0 = g.y[j0];
    double dvol0 = g.yvol[j0];
    if (jref < 0) { xa0 -= kTwoPi; azi -= kTwoPi; }
    if (jref >= jmax) { xa0 += kTwoPi; azi += kTwoPi; }
    if (CF::GY > 2) dvol0 *= rc;
    W.azi[h] = azi;
    W.xa0[h] = xa0;
    W.dx0[h] = g.dy[j0];
    W.dvol0[h] = dvol0;
    W.rad[h] = rc;
    const double2 tr = g.ptrig[j0];
    W.ca[h] = tr.x;
    W.sa[h] = tr.y;
    const double r = fr[j], p = fp[j], u = fv[j];
    const double v = prm.has_w ? fw[j] : 0.0;
    W.r[h] = r; W.p[h] = p; W.u[h] = u; W.v[h] = v; W.w[h] = fu[j];
    W.e[h] = energy_of<CF>(p, r, u, v, prm.gam);
  }

  ppmlr_wave<kK, CF>(W, TabLane64{}, ring, kK * lane, lim, dt, FrRot, pl, rf, prm.gam);
  if constexpr (CF::VISC) {
    C<double, kK> x;
#pragma unroll
    for (int h = 0; h < kK; ++h) x[h] = W.xa0[h] * rc;
    visc_p<kK, CF::GX == 2>(W, kK * lane, lim, dt, rc, g.nu[s], x, prm.ndim == 3);
  }

  double* __restrict__ dr = g.f[src ^ 1][FR] + base;
  double* __restrict__ dp = g.f[src ^ 1][FP] + base;
  double* __restrict__ du = g.f[src ^ 1][FU] + base;
  double* __restrict__ dv = g.f[src ^ 1][FV] + base;
  double* __restrict__ dw = g.f[src ^ 1][FW] + base;
  const double cs2 = g.cs2[s];
#pragma unroll
  for (int h = 0; h < kK; ++h) {
    const int c = kK * lane + h;
    if (c >= kNpad && c < lim - kNpad) {
      const int j = jd[h];
      const double r = W.r[h];
      double p;
      if constexpr (CF::EOS == 0) p = r * cs2;
      else if constexpr (CF::EOS == 1) p = cs2 * pow(r, prm.gam) / prm.gam;
      else p = W.p[h];
      dr[j] = r;
      dp[j] = p;
      du[j] = W.w[h];
      dv[j] = W.u[h];
      if (prm.has_w) dw[j] = W.v[h];
      if constexpr (CF::GY == 3) {
        if (do_cfl) {   // the next step's CFL terms of this cell, as k_cfl takes them (2-D)
          const double snd = cfl_sound(prm.gam * p, r), wy = g.dy[j] * rc;
          m = fmax(m, cfl_term(W.w[h], snd, g.tab[kT64Dx * g.tstride + s], g.tab[kT64Idx * g.tstride + s]));
          m = fmax(m, cfl_term(W.u[h] - g.rot_v[s] - FrRot * rc, snd, wy, rcp64(wy)));
        }
      }
    }
  }
  }
  if constexpr (CF::GY == 3) {
    if (do_cfl) block_cfl(m, red, &cflp[blockIdx.x]);   // kernel-uniform
  }
}

template <int AX, class CF>
void launch_one(const LaunchCtx& c, int src, int do_cfl) {
  if constexpr (AX == 1) {
    const long waves = (long)c.g.nwin_y * c.g.imax * c.g.kmax;
    k_sweep_y<CF><<<(unsigned)((waves + kWavesPerBlock - 1) / kWavesPerBlock), 64 * kWavesPerBlock, 0, c.stream>>>(
        c.g, c.p, c.ss, c.cflp, src, do_cfl);
  } else {
    int last;
    const long per = AX == 0 ? row_groups(c.g.imax, c.g.nwin_x, c.g.jmax, &last)
                             : row_groups(c.g.kmax, c.g.nwin_z, c.g.jmax, &last);
    const long rows = AX == 0 ? c.g.kmax : c.g.imax;
    k_pencil64<CF><<<(unsigned)(per * rows), 64 * kWavesPerBlock, 0, c.stream>>>(c.g, c.p, c.ss, c.cflp, src, do_cfl);
  }
}

template <int AX>
hipError_t dispatch(const LaunchCtx& c, int src, int do_cfl) {
  if (do_cfl && (AX != (c.p.ndim == 3 ? 2 : 1) || fp64_cfl_partials(c.g) > c.ncflp)) return hipErrorInvalidValue;
  const DevParams& p = c.p;
#define PN_LAUNCH(GX, GY, GZ, EOS, VISC) launch_one<AX, Cfg<AX, GX, GY, GZ, EOS, VISC>>(c, src, do_cfl)
  if constexpr (AX == 2) {   // only spherical disks have a theta sweep
    if (p.ngeomx == 1) return hipErrorInvalidValue;
  }
  if (p.ngeomx == 1 && p.ngeomy == 3 && p.ngeomz == 0) {
    if constexpr (AX != 2) switch (p.eos * 2 + (p.visc ? 1 : 0)) {
      case 0: PN_LAUNCH(1, 3, 0, 0, 0); break;
      case 1: PN_LAUNCH(1, 3, 0, 0, 1); break;
      case 2: PN_LAUNCH(1, 3, 0, 1, 0); break;
      case 3: PN_LAUNCH(1, 3, 0, 1, 1); break;
      case 4: PN_LAUNCH(1, 3, 0, 2, 0); break;
      case 5: PN_LAUNCH(1, 3, 0, 2, 1); break;
      case 6: PN_LAUNCH(1, 3, 0, 3, 0); break;
      case 7: PN_LAUNCH(1, 3, 0, 3, 1); break;
      default: return hipErrorInvalidValue;
    }
  } else if (p.ngeomx == 2 && p.ngeomy == 4 && p.ngeomz == 5) {
    switch (p.eos * 2 + (p.visc ? 1 : 0)) {
      case 0: PN_LAUNCH(2, 4, 5, 0, 0); break;
      case 1: PN_LAUNCH(2, 4, 5, 0, 1); break;
      case 4: PN_LAUNCH(2, 4, 5, 2, 0); break;
      case 5: PN_LAUNCH(2, 4, 5, 2, 1); break;
      default: return hipErrorInvalidValue;
    }
  } else {
    return hipErrorInvalidValue;
  }
#undef PN_LAUNCH
  return hipGetLastError();
}

}  // namespace

int fp64_cfl_partials(const DevGrid& g) {
  if (g.ndim == 3) {
    int last;
    return row_groups(g.kmax, g.nwin_z, g.jmax, &last) * g.imax;
  }
  return (g.nwin_y * g.imax + kWavesPerBlock - 1) / kWavesPerBlock;
}

hipError_t fp64_sweep_x(const LaunchCtx& c, int src) { return dispatch<0>(c, src, 0); }
hipError_t fp64_sweep_y(const LaunchCtx& c, int src, int do_cfl) { return dispatch<1>(c, src, do_cfl); }
hipError_t fp64_sweep_z(const LaunchCtx& c, int src, int do_cfl) { return dispatch<2>(c, src, do_cfl); }

}  // namespace pn
