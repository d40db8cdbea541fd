// pn_torque.hpp -- the disk's pull on a moving planet (modes 8 / 9 of output_lv1,
// device_func.cu:49-198) with the damping zones, one pass over a 2-D state.
#pragma once

#include "pn_launch.hpp"
#include "ppm_wave.hpp"

namespace pn {

// columns of one work item (a run of one ring)
constexpr int kTorqueCols = 256;

// rot_j of slot s after the step's integer roll (rotate_rings, ppm.cu:309-322).  A shift of more
// than a turn (a cold or coarse disk's step, or a loaded record's inc_j) rolls by what is left of
// it: every address of the ring is formed from rot_j in [0, jmax).
__device__ __forceinline__ int rolled(const DevGrid& g, int s) {
  int inc = g.inc_j[s];
  if (inc >= g.jmax || inc <= -g.jmax) inc %= g.jmax;
  int j = g.rot_j[s] + inc;
  if (j < 0) j += g.jmax;
  if (j >= g.jmax) j -= g.jmax;
  return j;
}

inline int torque_blocks(const DevGrid& g) {
  const long n = (long)g.imax * ((g.jmax + kTorqueCols - 1) / kTorqueCols);
  return (int)(n < kMaxPartials / 2 ? n : kMaxPartials / 2);
}

// Per workgroup of 256 threads the sums of both integrands over its items, in a fixed order, to
// partials[2 blockIdx], [2 blockIdx + 1].  cell(s, n, a, k) gives Sigma of cell a (slot s, ring n)
// after the step's damping by the fraction k (0 outside the zones, kill_wave.cu:3-43), which it
// applies to the state.  roll: the step's roll of rot_j is still to come (k_planet_finish).
// Bound by FP64 issue: the two forces share one sincos and one distance, the powers of the radius
// come from a table.
template <class Cell>
__device__ __forceinline__ void planet_torque(const DevGrid& g, const DevParams& prm,
                                              const StepScalars* __restrict__ ss, int roll, double* partials,
                                              Cell cell) {
  __shared__ double sh[8];
  const pn_body& b = ss->moved;
  const Planet pl{b.m, b.x, b.y, b.vx, b.vy, b.rs, prm.bary};
  const Grav G(pl, false);
  const int nseg = (g.jmax + kTorqueCols - 1) / kTorqueCols;
  const double d_kill = 0.5 * prm.sc_h;
  double a8 = 0.0, a9 = 0.0;
  for (int it = blockIdx.x; it < g.imax * nseg; it += gridDim.x) {
    const int n = it / nseg, s = slot_of(g, n, 0);
    const int j = (it % nseg) * kTorqueCols + threadIdx.x;
    if (j >= g.jmax) continue;
    const double rad = g.xc[s];
    double k = 0.0;
    if (prm.kill) {
      const double inner = prm.xmin + d_kill, outer = prm.xmax - d_kill;
      if (rad < inner) k = (inner - rad) / d_kill;
      else if (rad > outer) k = (rad - outer) / d_kill;
      if (k != 0.0) k *= ss->dt * g.rpow[s].y;
    }
    const int rot = roll ? rolled(g, s) : g.rot_j[s];
    int j0 = j + rot;
    j0 += (j0 < 0) ? g.jmax : 0;
    j0 -= (j0 >= g.jmax) ? g.jmax : 0;
    const double r = cell(s, n, (long)s * g.jmax + j, k);
    const double phi = g.yc[j0];
    const double dd = (rad - pl.x) * (rad - pl.x) + rad * rad * (phi - pl.y) * (phi - pl.y);
    if (!(dd > 0.0)) continue;
    const double dm = (r - g.rpow[s].x) * g.xvol[s] * g.yvol[j0];
    double sn, cs;
    sincos(phi - pl.y, &sn, &cs);
    a8 += -grav_rad_cyl(G, rad, cs) * dm;
    a9 += -grav_azi_cyl(G, rad, cs, sn) * (rad * dm);
  }
  for (int off = 32; off > 0; off >>= 1) {
    a8 += __shfl_xor(a8, off);
    a9 += __shfl_xor(a9, off);
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sh[w] = a8;
    sh[4 + w] = a9;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
    partials[2 * blockIdx.x + 1] = (sh[4] + sh[5]) + (sh[6] + sh[7]);
  }
}

}  // namespace pn
