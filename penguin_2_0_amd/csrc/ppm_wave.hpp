// ppm_wave.hpp -- one directional PPMLR update of a 128-cell window on one wavefront.
//
// Method: the reference's ppmlr (ppmlr.cu:2-56) -- flatten, states (paraset, parabola,
// characteristic averages, interface force), Riemann solve, Lagrangian evolve, PPM remap --
// followed by the explicit viscosity (viscosity.cu:370-472).  The statements are the reference's; which
// of them round as it writes them and which carry an ulp of their own is said at ppmlr_wave.
//
// Execution model (not the reference's): one 64-lane wavefront owns a whole window, each
// lane K consecutive cells (cell c = K*lane + h).  Every stencil access is to the cell
// itself or to c+-1 / c+-2, i.e. to the same lane or a neighbouring lane, so neighbour
// values move by DPP wave shifts (v_mov_b32_dpp wave_shr:1 / wave_shl:1) instead of LDS
// round trips, and the ~50 block barriers of the reference window disappear.  All shifts
// run in wave-uniform control flow; per-cell index ranges of the reference stages become
// selects.
#pragma once

#include "pn_device.hpp"

namespace pn {

// ---------------------------------------------------------------------------------------
// lane exchange

// wave_shr:1 / wave_shl:1 with bound_ctrl: the lane without a source (0, resp. 63) reads 0,
// and the destination needs no initial value (one instruction per shift)
__device__ __forceinline__ int lane_prev_i(int x) {   // lane l receives lane l-1's value
  return __builtin_amdgcn_mov_dpp(x, 0x138, 0xf, 0xf, true);
}
__device__ __forceinline__ int lane_next_i(int x) {   // lane l receives lane l+1's value
  return __builtin_amdgcn_mov_dpp(x, 0x130, 0xf, 0xf, true);
}
__device__ __forceinline__ float lane_prev(float x) { return __int_as_float(lane_prev_i(__float_as_int(x))); }
__device__ __forceinline__ float lane_next(float x) { return __int_as_float(lane_next_i(__float_as_int(x))); }
__device__ __forceinline__ double lane_prev(double x) {
  int lo = lane_prev_i(__double2loint(x));
  int hi = lane_prev_i(__double2hiint(x));
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_next(double x) {
  int lo = lane_next_i(__double2loint(x));
  int hi = lane_next_i(__double2hiint(x));
  return __hiloint2double(hi, lo);
}

// per-lane slice of a window quantity
template <typename T, int K>
struct C {
  T a[K];
  __device__ __forceinline__ T& operator[](int h) { return a[h]; }
  __device__ __forceinline__ T operator[](int h) const { return a[h]; }
};

template <typename T, int K>
__device__ __forceinline__ C<T, K> splat(T s) {
  C<T, K> o;
#pragma unroll
  for (int h = 0; h < K; ++h) o[h] = s;
  return o;
}

// value of cell c-1
template <typename T, int K>
__device__ __forceinline__ C<T, K> prev1(const C<T, K>& x) {
  C<T, K> o;
  o[0] = lane_prev(x[K - 1]);
#pragma unroll
  for (int h = 1; h < K; ++h) o[h] = x[h - 1];
  return o;
}
// value of cell c+1
template <typename T, int K>
__device__ __forceinline__ C<T, K> next1(const C<T, K>& x) {
  C<T, K> o;
#pragma unroll
  for (int h = 0; h < K - 1; ++h) o[h] = x[h + 1];
  o[K - 1] = lane_next(x[0]);
  return o;
}
// value of cell c-2
template <typename T, int K>
__device__ __forceinline__ C<T, K> prev2(const C<T, K>& x) {
  if constexpr (K == 1) {
    return prev1(prev1(x));
  } else {
    C<T, K> o;
#pragma unroll
    for (int h = 0; h < K; ++h) o[h] = (h >= 2) ? x[h - 2] : lane_prev(x[K - 2 + h]);
    return o;
  }
}
// value of cell c+2
template <typename T, int K>
__device__ __forceinline__ C<T, K> next2(const C<T, K>& x) {
  if constexpr (K == 1) {
    return next1(next1(x));
  } else {
    C<T, K> o;
#pragma unroll
    for (int h = 0; h < K; ++h) o[h] = (h + 2 < K) ? x[h + 2] : lane_next(x[h + 2 - K]);
    return o;
  }
}

// the limited slope of parabola.cu:87-96: sign(t1) min(|t1|, 2 |da_l|, 2 |da_r|), zero at an
// extremum: a minimum of magnitudes and the sign by copysign, the values of the reference's
// compare chain (a minimum and a sign change round nothing, doubling is exact)
__device__ __forceinline__ double limited_slope(double t1, double da_l, double da_r) {
  t1 = copysign(fmin(fabs(t1), 2.0 * fmin(fabs(da_l), fabs(da_r))), t1);
  return da_l * da_r < 0.0 ? 0.0 : t1;
}
template <typename T>
__device__ __forceinline__ T max3(T A, T B, T Cc) {   // simple_func.cu:16-28
  if (A > B) return (Cc > A) ? Cc : A;
  return (Cc > B) ? Cc : B;
}

// ---------------------------------------------------------------------------------------
// FP64 divisions, roots, exp and log of the windows.  A sweep divides by the same few numbers
// over and over (a radius three times in a row, a cell's density, the Lagrangian volume), and
// the compiler's division is 11 instructions each time.  Here a reciprocal is formed once and
// each quotient by it takes three: q = a y, r = a - q b (exact in an FMA), q + r y (Markstein 1990).
// With y within an ulp of 1 / b the sum lies within 2^-51 ulp of a / b before its one rounding, so
// it is the division's result unless a / b lies that close to the middle between two numbers (one
// quotient in 2^50; a divisor 2 - 2^-52 has such ones).  For finite, normal operands; a zero or
// non-finite divisor gives NaN where a division gives an infinity.

// 1 / b to an ulp: the hardware estimate (2^-24 or better) and one cubic step
__device__ __forceinline__ double rcp64(double b) {
  const double y = __builtin_amdgcn_rcp(b);
  const double e = __builtin_fma(-b, y, 1.0);
  return __builtin_fma(y, __builtin_fma(e, e, e), y);
}
// 1 / b rounded as the division (as above), from y = rcp64(b)
__device__ __forceinline__ double rcp64_rn(double b) {
  const double y = rcp64(b);
  return __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
}
// a / b rounded as the division (as above), y = 1 / b to an ulp
__device__ __forceinline__ double div64(double a, double b, double y) {
  const double q = a * y;
  return __builtin_fma(__builtin_fma(-q, b, a), y, q);
}
// 1 / sqrt(x), x > 0, to 1.5 ulp
__device__ __forceinline__ double rsq64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-(x * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
}
// sqrt(x) rounded as the root but for values within 2^-49 ulp of a middle, x zero or normal and
// positive
__device__ __forceinline__ double sqrt64_rn(double x) {
  const double y = rsq64(x);
  const double g = x * y;
  return x == 0.0 ? x : __builtin_fma(__builtin_fma(-g, g, x), 0.5 * y, g);
}
// exp(t) for |t| < 1/8: 1 + (t + t^2 / 2 + ... + t^10 / 10!); the one rounding that matters is
// the last addition's
__device__ __forceinline__ double exp_small(double t) {
  double q = __builtin_fma(t, 1.0 / 3628800.0, 1.0 / 362880.0);
  q = __builtin_fma(t, q, 1.0 / 40320.0);
  q = __builtin_fma(t, q, 1.0 / 5040.0);
  q = __builtin_fma(t, q, 1.0 / 720.0);
  q = __builtin_fma(t, q, 1.0 / 120.0);
  q = __builtin_fma(t, q, 1.0 / 24.0);
  q = __builtin_fma(t, q, 1.0 / 6.0);
  q = __builtin_fma(t, q, 0.5);
  return 1.0 + __builtin_fma(t * t, q, t);
}
// atanh(x) for |x| < 1/8: the odd series to x^17; 2 atanh((a - b) / (a + b)) = log(a / b)
__device__ __forceinline__ double atanh_small(double x) {
  const double z = x * x;
  double q = __builtin_fma(z, 1.0 / 17.0, 1.0 / 15.0);
  q = __builtin_fma(z, q, 1.0 / 13.0);
  q = __builtin_fma(z, q, 1.0 / 11.0);
  q = __builtin_fma(z, q, 1.0 / 9.0);
  q = __builtin_fma(z, q, 1.0 / 7.0);
  q = __builtin_fma(z, q, 1.0 / 5.0);
  q = __builtin_fma(z, q, 1.0 / 3.0);
  return __builtin_fma(x * z, q, x);
}
// true in every lane when the condition holds in any lane of the wavefront (wave-uniform)
__device__ __forceinline__ bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0; }

// ---------------------------------------------------------------------------------------
// planet + star gravity (forces.cu:4-182).  Without bary: the star at the origin (its -1/r^2
// added by the caller in cylindrical r, included in the spherical forms) and the planet's
// indirect term; with bary (bary_flag): star at -x m/(1+m) and planet at x/(1+m) about their
// barycentre, no indirect term.

struct Planet {
  double m, x, y, vx, vy, rs;
  int bary;
};

// the planet and star as the force forms take them: plm, plx the planet's mass and distance
// (about the star: m, x, the spherical forms with the reduced mass m/(1+m); barycentric: m/(1+m)
// and x/(1+m)), stm, stx the star's mass 1/(1+m) and distance from the barycentre, ix2 = 1/x^2
// of the indirect term.  Formed once per wavefront.
struct Grav {
  double plm, plx, rs2, ix2, stm, stx, iplx, plx2, iplx2;
  bool bary;
  __device__ __forceinline__ Grav(const Planet& p, bool sph) {
    stm = 1.0 / (1.0 + p.m);
    bary = p.bary != 0;
    plm = (bary || sph) ? p.m * stm : p.m;
    plx = bary ? p.x * stm : p.x;
    stx = p.x * (p.m * stm);
    ix2 = 1.0 / (p.x * p.x);
    rs2 = p.rs * p.rs;
    iplx = rcp64(plx);
    plx2 = plx * plx;
    iplx2 = rcp64(plx2);
  }
};

// The forces take the angle to the planet as its cosine and sine (and in 3-D the cell's sin and
// cos theta): a sweep forms those once per column and turns them by small angles, instead of
// a library cos and sin of every cell at each of three times.  The planet's 1/R^3 comes from a
// reciprocal root (the cylindrical forms; the spherical ones below round as written).
__device__ __forceinline__ double cube(double x) { return x * x * x; }
// a / R^3, R = sqrt(R2), rounded as written: the star's pull, which the disk's rotation nearly
// cancels, so its last bit is seen
__device__ __forceinline__ double over_cube(double a, double R2) {
  const double R = sqrt64_rn(R2), R3 = R * R * R;
  return div64(a, R3, rcp64(R3));
}
__device__ __forceinline__ double grav_rad_cyl(const Grav& g, double rad, double cosfac) {   // forces.cu:112-134
  const double ri3 = cube(rsq64(rad * rad + g.plx * g.plx - 2.0 * g.plx * rad * cosfac + g.rs2));
  const double f = -g.plm * (rad - g.plx * cosfac) * ri3;
  if (!g.bary) return f - g.plm * cosfac * g.ix2;
  return f - over_cube(g.stm * (rad + g.stx * cosfac), rad * rad + g.stx * g.stx + 2.0 * g.stx * rad * cosfac);
}
__device__ __forceinline__ double grav_azi_cyl(const Grav& g, double rad, double cosfac, double sinfac) {   // forces.cu:136-159
  const double ri3 = cube(rsq64(rad * rad + g.plx * g.plx - 2.0 * g.plx * rad * cosfac + g.rs2));
  const double f = -g.plm * g.plx * sinfac * ri3;
  if (!g.bary) return f + g.plm * sinfac * g.ix2;
  return f + over_cube(g.stm * g.stx * sinfac, rad * rad + g.stx * g.stx + 2.0 * g.stx * rad * cosfac);
}
// The spherical forms round every operation as written.  The theta sweep's area factor
// (cos x0 - cos x) / (x - x0) of an edge that hardly moves turns a last-bit change of x into a
// relative 1e-9 of the pressure force on v_theta, so a 3-D disk follows the reference's run only
// as long as its rounding is followed everywhere.  star2 = stm / rad^2, which the caller forms (not
// used in the barycentric frame).
__device__ __forceinline__ double grav_rad_sph(const Grav& g, double rad, double cosfac, double sinpol, double star2) {   // forces.cu:23-50
  const double f = over_cube(-g.plm * (rad - g.plx * cosfac * sinpol),
                             rad * rad + g.plx * g.plx - 2.0 * g.plx * rad * cosfac * sinpol + g.rs2);
  if (!g.bary) return f - star2 - div64(g.plm * sinpol * cosfac, g.plx2, g.iplx2);
  return f - over_cube(g.stm * (rad + g.stx * cosfac * sinpol),
                       rad * rad + g.stx * g.stx + 2.0 * g.stx * rad * cosfac * sinpol);
}
// rad: the spherical radius
__device__ __forceinline__ double grav_azi_sph(const Grav& g, double rad, double cosfac, double sinfac, double sinpol) {   // forces.cu:52-81
  const double f = over_cube(-g.plm * g.plx * sinfac,
                             rad * rad + g.plx * g.plx - 2.0 * g.plx * rad * cosfac * sinpol + g.rs2);
  if (!g.bary) return f + div64(div64(g.plm * sinpol * sinfac, g.plx, g.iplx), g.plx, g.iplx);
  return f + over_cube(g.stm * g.stx * sinfac, rad * rad + g.stx * g.stx + 2.0 * g.stx * rad * cosfac * sinpol);
}
__device__ __forceinline__ double grav_pol_sph(const Grav& g, double rad, double cosfac, double sinpol, double cospol) {   // forces.cu:83-110
  const double f = over_cube(g.plm * g.plx * cosfac * cospol,
                             rad * rad + g.plx * g.plx - 2.0 * g.plx * rad * cosfac * sinpol + g.rs2);
  if (!g.bary) {
    const double d = sinpol * g.plx * g.plx;
    return f - div64(g.plm * cosfac * cospol, d, rcp64(d));
  }
  return f - over_cube(g.stm * g.stx * cosfac * cospol, rad * rad + g.stx * g.stx + 2.0 * g.stx * rad * cosfac * sinpol);
}
// sin and cos of e: Taylor series for |e| < 1/2, past it (a coarse ring's shift over a long
// step) the library functions, in wavefronts that need them
__device__ __forceinline__ void sincos_small(double e, double& s, double& c) {
  const double z = e * e;
  double q = __builtin_fma(z, 1.0 / 6227020800.0, -1.0 / 39916800.0);
  q = __builtin_fma(z, q, 1.0 / 362880.0);
  q = __builtin_fma(z, q, -1.0 / 5040.0);
  q = __builtin_fma(z, q, 1.0 / 120.0);
  q = __builtin_fma(z, q, -1.0 / 6.0);
  s = __builtin_fma(e * z, q, e);
  double w = __builtin_fma(z, -1.0 / 87178291200.0, 1.0 / 479001600.0);
  w = __builtin_fma(z, w, -1.0 / 3628800.0);
  w = __builtin_fma(z, w, 1.0 / 40320.0);
  w = __builtin_fma(z, w, -1.0 / 720.0);
  w = __builtin_fma(z, w, 1.0 / 24.0);
  w = __builtin_fma(z, w, -0.5);
  c = __builtin_fma(z, w, 1.0);
  const bool big = !(fabs(e) < 0.5);
  if (wave_any(big)) {
    double sb, cb;
    sincos(e, &sb, &cb);
    s = big ? sb : s;
    c = big ? cb : c;
  }
}
// cos and sin of (a + b) from those of a and b
__device__ __forceinline__ void turn(double ca, double sa, double cb, double sb, double& c, double& s) {
  c = ca * cb - sa * sb;
  s = sa * cb + ca * sb;
}
template <typename T>
__device__ __forceinline__ T potential(bool planet_on, const Planet& p, T rad, T azi, T z) {   // forces.cu:4-21
  if (planet_on) {
    T cosfac = cos(azi - (T)p.y);
    T stm = T(1.0) / (T(1.0) + (T)p.m);
    T plm = (T)p.m * stm;
    T plx = (T)p.x * stm;
    T stx = (T)p.x * plm;
    T rs = (T)p.rs;
    T Rp = rad * rad + plx * plx - T(2.0) * plx * rad * cosfac + z * z;
    Rp = sqrt(Rp + rs * rs);
    T Rs = sqrt(rad * rad + stx * stx + T(2.0) * stx * rad * cosfac + z * z);
    return -plm / Rp - stm / Rs;
  }
  return T(-1.0) / sqrt(rad * rad + z * z);
}

// ---------------------------------------------------------------------------------------
// window configuration

template <int AXIS_, int GX_, int GY_, int GZ_, int EOS_, int VISC_>
struct Cfg {
  static constexpr int AXIS = AXIS_, GX = GX_, GY = GY_, GZ = GZ_, EOS = EOS_, VISC = VISC_;
};

// the FP64 slot table's entries of this lane's two cells: one 16-byte load per entry, the
// entry's address in scalar registers and the lane's byte offset in a vector one
typedef double f64x2_t __attribute__((ext_vector_type(2), aligned(8)));
struct TabLane64 {
  const double* tab;
  long stride;     // doubles per entry
  unsigned voff;   // byte offset of the slot of this lane's first cell
  __device__ __forceinline__ C<double, 2> get(int e) const {
    const f64x2_t v = *reinterpret_cast<const f64x2_t*>(reinterpret_cast<const char*>(tab + e * stride) + voff);
    C<double, 2> o;
    o[0] = v.x;
    o[1] = v.y;
    return o;
  }
};

// the energy a cell carries into the Lagrangian step from the window's p, rho, u and first
// transverse slot v: EOS 2 as ppm.cu:106-108 has it (v already scaled by r_cyl in the radial
// sweep), EOS 3 the internal energy plus the sweep direction's kinetic energy; 0 otherwise
template <class CF>
__device__ __forceinline__ double energy_of(double p, double r, double u, double v, double gam) {
  if constexpr (CF::EOS == 2) return p / (r * (gam - 1.0)) + 0.5 * ((u * u) + (v * v));
  else if constexpr (CF::EOS == 3) return p / (r * (gam - 1.0)) + 0.5 * (u * u);
  else return 0.0;
}

struct RunFlags {
  int flat;      // flattening on
  int planet;    // plnt_flag > 0
  int remap_v;   // the sweep's first transverse slot is carried (else it is identically 0)
  int remap_w;   // the sweep's second transverse slot is carried
  int ndim;
};

template <typename T, int K>
struct Para {
  C<T, K> c0, c1, c2, c3, c4;
};

// paraset (parabola.cu:138-176) on the index range [nmin, nmaxp); c0 = this lane's first cell
template <typename T, int K>
__device__ __forceinline__ Para<T, K> paraset(int c0, int nmin, int nmaxp, const C<T, K>& dx) {
  Para<T, K> P;
  C<T, K> dxp = next1(dx);
  C<T, K> an, ain, bn, bi, cc, ci;
#pragma unroll
  for (int h = 0; h < K; ++h) {
    an[h] = dx[h] + dxp[h];
    ain[h] = T(1.0) / an[h];
    bn[h] = an[h] + dx[h];
    bi[h] = T(1.0) / bn[h];
    cc[h] = an[h] + dxp[h];
    ci[h] = T(1.0) / cc[h];
  }
  C<T, K> anm = prev1(an), anp = next1(an), bnm = prev1(bn), ainm = prev1(ain);
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const int c = c0 + h;
    T k0 = T(0), c1 = T(0), c2 = T(0), c3 = T(0), c4 = T(0);
    if (c >= nmin + 1 && c < nmaxp - 2) {
      T d = T(1.0) / (anm[h] + anp[h]);
      k0 = dx[h] * ain[h] * (T(1.0) + T(2.0) * d * dxp[h] * (anm[h] * bi[h] - anp[h] * ci[h]));
      c1 = -d * dx[h] * anm[h] * bi[h];
      c2 = d * dxp[h] * anp[h] * ci[h];
    }
    if (c >= nmin + 1 && c < nmaxp - 1) {
      T d = dx[h] / (anm[h] + dxp[h]);
      c3 = d * bnm[h] * ain[h];
      c4 = d * cc[h] * ainm[h];
    }
    P.c0[h] = k0; P.c1[h] = c1; P.c2[h] = c2; P.c3[h] = c3; P.c4[h] = c4;
  }
  return P;
}

// paraset of the Lagrangian grid, FP64.  Its coefficients multiply differences of neighbouring
// cells, which enter the edge values far below their last bit, so 2-D sweeps share reciprocals
// (one estimate for 1/an, 1/bn, 1/cc, one for both sums); with EX every quotient rounds as
// written.  Coefficients are formed in every cell; those outside the reference's index ranges
// (parabola.cu:138-176) reach no parabola that a kept cell reads.
template <int K, bool EX>
__device__ __forceinline__ Para<double, K> paraset64(const C<double, K>& dx) {
  Para<double, K> P;
  C<double, K> dxp = next1(dx);
  C<double, K> an, ain, bn, bi, cc, ci;
#pragma unroll
  for (int h = 0; h < K; ++h) {
    an[h] = dx[h] + dxp[h];
    bn[h] = an[h] + dx[h];
    cc[h] = an[h] + dxp[h];
    if constexpr (EX) {
      ain[h] = rcp64_rn(an[h]);
      bi[h] = rcp64_rn(bn[h]);
      ci[h] = rcp64_rn(cc[h]);
    } else {
      const double ab = an[h] * bn[h];
      const double t = rcp64(ab * cc[h]), tc = t * cc[h];
      ain[h] = tc * bn[h];
      bi[h] = tc * an[h];
      ci[h] = t * ab;
    }
  }
  C<double, K> anm = prev1(an), anp = next1(an), bnm = prev1(bn), ainm = prev1(ain);
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const double s1 = anm[h] + anp[h], s2 = anm[h] + dxp[h];
    double e;
    if constexpr (EX) {
      const double d = rcp64_rn(s1);
      P.c0[h] = dx[h] * ain[h] * (1.0 + 2.0 * d * dxp[h] * (anm[h] * bi[h] - anp[h] * ci[h]));
      P.c1[h] = -d * dx[h] * anm[h] * bi[h];
      P.c2[h] = d * dxp[h] * anp[h] * ci[h];
      e = div64(dx[h], s2, rcp64(s2));
    } else {
      const double t = rcp64(s1 * s2), d = t * s2;
      const double wb = d * anm[h] * bi[h], wc = d * anp[h] * ci[h];
      P.c0[h] = dx[h] * ain[h] * __builtin_fma(2.0 * dxp[h], wb - wc, 1.0);
      P.c1[h] = -dx[h] * wb;
      P.c2[h] = dxp[h] * wc;
      e = dx[h] * (t * s1);
    }
    P.c3[h] = e * bnm[h] * ain[h];
    P.c4[h] = e * cc[h] * ainm[h];
  }
  return P;
}

template <typename T, int K>
struct Parab {
  C<T, K> al, da, a6;   // left value, jump, curvature; valid on [nmin+2, nmaxp-2)
};

// parabola (parabola.cu:70-136), valid on [nmin+2, nmaxp-2) for coefficients valid on the
// reference's ranges of [nmin, nmaxp); outside it holds values no kept cell reads.  omf = 1 -
// flat.  The differences come once per interface (da_l of a cell is da_r of the one before it,
// the same subtraction); everything else is the reference's, operation for operation, but for the
// flattened edges, whose product rounds apart only with EX.
template <int K, bool EX>
__device__ __forceinline__ Parab<double, K> parabola(const C<double, K>& flat, const C<double, K>& omf,
                                                     const C<double, K>& val, const Para<double, K>& P) {
  C<double, K> vp = next1(val);
  C<double, K> slope, dar;
#pragma unroll
  for (int h = 0; h < K; ++h) dar[h] = vp[h] - val[h];
  C<double, K> dal = prev1(dar);
#pragma unroll
  for (int h = 0; h < K; ++h)
    slope[h] = limited_slope(P.c3[h] * dar[h] + P.c4[h] * dal[h], dal[h], dar[h]);
  C<double, K> slp = next1(slope);
  C<double, K> ar;
#pragma unroll
  for (int h = 0; h < K; ++h)
    ar[h] = val[h] + P.c0[h] * dar[h] + P.c1[h] * slp[h] + P.c2[h] * slope[h];
  C<double, K> alv = prev1(ar);
  Parab<double, K> o;
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const double a = val[h];
    double t1 = flat[h] * a;
    double arr = EX ? t1 + omf[h] * ar[h] : __builtin_fma(omf[h], ar[h], t1);
    double la = EX ? t1 + omf[h] * alv[h] : __builtin_fma(omf[h], alv[h], t1);
    t1 = arr - la;
    const double t2 = t1 * t1;
    t1 = t1 * (6.0 * (a - 0.5 * (arr + la)));
    if ((arr - a) * (a - la) <= 0.0) {
      arr = a;
      la = a;
    }
    const double a3 = 3.0 * a;
    if (t2 < t1) la = a3 - 2.0 * arr;
    if (t2 < -t1) arr = a3 - 2.0 * la;
    o.da[h] = arr - la;
    o.a6[h] = 6.0 * (a - 0.5 * (arr + la));
    o.al[h] = la;
  }
  return o;
}

// Window state and per-cell geometry.
template <int K>
struct Win {
  C<double, K> r, p, u, v, w, e;
  C<double, K> xa0, dx0, dvol0, rad;   // left edge, width, volume, radius of the sweep's forces
  C<double, K> azi;                    // azimuth of the cell centre
  C<double, K> ca, sa;                 // cos, sin of its angle from the planet before the step
};

// What a sweep reads beside the window: tx (radial and theta sweeps, the slot table at this
// lane's cells) or the ring's numbers (azimuthal sweep: vrot, 1 / rad rounded, sin theta, theta,
// the spherical radius, and p0, the uniform grid's interpolation coefficients, null on a grid that is not uniform)
struct Ring64 {
  double vrot, irad, sinpol, pol, rsph;
  const double* p0;
};

// One PPMLR update of the window (ppmlr.cu:2-56).  c0 = this lane's first cell, nmax = window
// length, drift = vrot - v_y (azimuthal sweep).  On return the cells [6, nmax-6) hold the
// updated r, u, v, w (and p for EOS 1, 2).  What is kept of the reference's rounding: in 3-D every
// operation's (quotients and roots as said at div64).  In 2-D the states, the star's and the
// centrifugal force, the Lagrangian step and the mass update round as written; the planet's pull, the
// interface's logarithm, exponential and powers (EOS 0, 2, 3), the Lagrangian interpolation
// coefficients, the flattened edges, the average over a swept face and the viscous increment carry an
// ulp of their own (1e-12 to 2e-11 of a field after some ten steps).
template <int K, class CF>
__device__ __forceinline__ void ppmlr_wave(Win<K>& W, const TabLane64& tx, const Ring64& ring, int c0, int nmax,
                                           double dt, double FrRot, const Planet& pl, const RunFlags& rf, double gam) {
  using T = double;
  constexpr int AX = CF::AXIS;
  const T hdt = T(0.5) * dt;
  const T smallp = T(1.0e-15), smallr = T(1.0e-15);
  const T fourthd = T(1.3333333333333333333333333);
  const T third = T(0.3333333333333333333333333);
  const T gamm = gam - T(1.0);
  constexpr bool EX = CF::GX == 2;   // 3-D: every operation rounds as the reference's
  const Grav G(pl, CF::GX == 2);
  // 3-D: cos and sin of the angle to the planet a time t into the step (forces.cu:25, 55-57)
  auto angle = [&](T azi, T vrot, T t) { return azi + t * vrot - (pl.y + t * pl.vy); };

  // ---- flatten (flatten.cu:7-40)
  C<T, K> flat = splat<T, K>(T(0));
  if (rf.flat) {
    C<T, K> pm1 = prev1(W.p), pp1 = next1(W.p), pm2 = prev2(W.p), pp2 = next2(W.p);
    C<T, K> um1 = prev1(W.u), up1 = next1(W.u);
    C<T, K> steep;
#pragma unroll
    for (int h = 0; h < K; ++h) {
      const int c = c0 + h;
      T s = T(0.0);
      if (c >= 2 && c < nmax - 2) {
        T dp1 = pp1[h] - pm1[h];
        T dp2 = pp2[h] - pm2[h];
        if (fabs(dp2) < smallp) dp2 = smallp;
        const T lo = fmin(pp1[h], pm1[h]);
        // a jump from no pressure at all (an infinite quotient, NaN here) is a shock; without a jump
        // the steepness below is 0 either way
        bool shock = !(div64(fabs(dp1), lo, rcp64(lo)) <= T(0.33));
        if (um1[h] < up1[h]) shock = false;
        if (shock) s = fmax(T(0.0), (dp1 / dp2 - T(0.75)) * T(5.0));
      }
      steep[h] = s;
    }
    C<T, K> sm = prev1(steep), sp = next1(steep);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      const int c = c0 + h;
      flat[h] = (c >= 2 && c < nmax - 2) ? fmin(T(0.5), max3(sm[h], steep[h], sp[h])) : T(0.0);
    }
  }

  // ---- states (states.cu:3-73)
  Para<T, K> P0;
  C<T, K> irad, idx, idvol;   // rounded reciprocals
  C<T, K> hc, hs, vrot;       // the turn of the angle to the planet in half a step; 3-D: vrot
  if constexpr (AX == 1) {
    if (ring.p0) {
      P0.c0 = splat<T, K>(ring.p0[0]);
      P0.c1 = splat<T, K>(ring.p0[1]);
      P0.c2 = splat<T, K>(ring.p0[2]);
      P0.c3 = splat<T, K>(ring.p0[3]);
      P0.c4 = splat<T, K>(ring.p0[4]);
    } else {
      P0 = paraset<T, K>(c0, 0, nmax, W.dx0);
    }
    irad = splat<T, K>(ring.irad);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      idx[h] = rcp64_rn(W.dx0[h]);
      idvol[h] = rcp64_rn(W.dvol0[h]);
    }
  } else {
    constexpr int b = AX == 0 ? kT64P0 : kT64P0z;
    P0.c0 = tx.get(b);
    P0.c1 = tx.get(b + 1);
    P0.c2 = tx.get(b + 2);
    P0.c3 = tx.get(b + 3);
    P0.c4 = tx.get(b + 4);
    irad = tx.get(kT64Irad);
    idx = tx.get(AX == 0 ? kT64Idx : kT64Idz);
    if constexpr (EX) {
      vrot = tx.get(kT64Vrot);
    } else if (rf.planet) {
      hc = tx.get(kT64RotC);
      hs = tx.get(kT64RotS);
    }
  }
  // half a step of the force at the left edge (forces.cu:185-372).  Star and centrifugal force
  // nearly cancel, and their sum moves the interface through u*, so both round as written
  C<T, K> fh;
  if constexpr (AX == 0) {
    C<T, K> vm = prev1(W.v), wm, spol;
    const C<T, K> fst = tx.get(kT64Fst), ixa = tx.get(kT64Ixa);   // -1/x/x, 1/x
    if constexpr (CF::GX == 2) {
      wm = prev1(W.w);
      spol = tx.get(kT64Sp);
    }
#pragma unroll
    for (int h = 0; h < K; ++h) {
      const T lv = T(0.5) * (W.v[h] + vm[h]);
      const T x = W.xa0[h], y = ixa[h];
      T f = fst[h], c = T(0), s;
      if constexpr (CF::GX == 1) {
        if (rf.planet) turn(W.ca[h], W.sa[h], hc[h], hs[h], c, s);
        if (rf.planet) f = grav_rad_cyl(G, x, c) + (G.bary ? T(0) : f);
        f += div64(div64(div64(lv * lv, x, y), x, y), x, y);
      } else {
        const T lw = T(0.5) * (W.w[h] + wm[h]);
        const T x2 = x * x, sp = x * spol[h], sp2 = sp * sp;
        if (rf.planet) c = cos(angle(W.azi[h], vrot[h], hdt));
        if (rf.planet) f = grav_rad_sph(G, x, c, spol[h], div64(G.stm, x2, rcp64(x2)));
        f += div64(div64(div64(lw * lw, x, y), x, y), x, y);
        f += div64(div64(lv * lv, x, y), sp2, rcp64(sp2));
      }
      fh[h] = hdt * f;
    }
  } else if constexpr (AX == 1) {
    const T drift = ring.vrot - pl.vy;
    T c1 = T(1), s1 = T(0);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      T f = T(0);
      if (rf.planet) {
        if constexpr (EX) {
          const T ph = angle(W.xa0[h], ring.vrot, hdt);
          f = grav_azi_sph(G, ring.rsph, cos(ph), sin(ph), ring.sinpol);
        } else {
          // from the cell's left edge; on a uniform grid the same turn in every cell
          if (h == 0 || !ring.p0) sincos_small(hdt * drift - T(0.5) * W.dx0[h], s1, c1);
          T c, s;
          turn(W.ca[h], W.sa[h], c1, s1, c, s);
          f = grav_azi_cyl(G, W.rad[h], c, s);
        }
      }
      fh[h] = hdt * f;
    }
  } else {
    C<T, K> wm = prev1(W.w);
    const C<T, K> spl = tx.get(kT64Spl), cpl = tx.get(kT64Cpl);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      const T l = T(0.5) * (W.w[h] + wm[h]);
      const T rc = W.rad[h] * spl[h], y = rcp64(rc);
      T f = T(0);
      if (rf.planet) f = grav_pol_sph(G, W.rad[h], cos(angle(W.azi[h], vrot[h], hdt)), spl[h], cpl[h]);
      f += div64(div64(div64(l * l * cpl[h], rc, y), rc, y), rc, y);
      fh[h] = hdt * f;
    }
  }
  C<T, K> cs, csfac, omf;
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const T c2 = div64(gam * W.p[h], W.r[h], rcp64(W.r[h]));
    T s = div64(hdt * sqrt64_rn(c2), W.dx0[h], idx[h]);
    if constexpr (AX == 1 || (AX == 2 && CF::GZ == 5)) s = div64(s, W.rad[h], irad[h]);
    cs[h] = s;
    csfac[h] = T(1.0) - fourthd * s;
    omf[h] = T(1.0) - flat[h];
  }
  auto traced = [&](const Parab<T, K>& q, C<T, K>& re, C<T, K>& le) {
#pragma unroll
    for (int h = 0; h < K; ++h) {
      re[h] = q.al[h] + q.da[h] - cs[h] * (q.da[h] - csfac[h] * q.a6[h]);
      le[h] = q.al[h] + cs[h] * (q.da[h] + csfac[h] * q.a6[h]);
    }
  };
  // left state at interface c = right-edge average of cell c-1; right state = left-edge
  // average of cell c (states.cu:45-68)
  C<T, K> Spl, Spr, Srl, Srr, Sul, Sur;
  {
    C<T, K> re, le;
    traced(parabola<K, EX>(flat, omf, W.p, P0), re, le);
    C<T, K> rem = prev1(re);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      Spl[h] = fmax(smallp, rem[h]);
      Spr[h] = fmax(smallp, le[h]);
    }
  }
  {
    C<T, K> re, le;
    traced(parabola<K, EX>(flat, omf, W.r, P0), re, le);
    C<T, K> rem = prev1(re);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      Srl[h] = fmax(smallr, rem[h]);
      Srr[h] = fmax(smallr, le[h]);
    }
  }
  {
    C<T, K> re, le;
    traced(parabola<K, EX>(flat, omf, W.u, P0), re, le);
    C<T, K> rem = prev1(re);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      Sul[h] = rem[h] + fh[h];
      Sur[h] = le[h] + fh[h];
    }
  }

  // ---- riemann (riemann.cu:3-115)
  C<T, K> umid, pmid;
#pragma unroll
  for (int h = 0; h < K; ++h) {
    T pl_ = Spl[h], rl = Srl[h], ul = Sul[h], pr = Spr[h], rr = Srr[h], ur = Sur[h];
    T um, pm;
    if constexpr (CF::EOS == 0) {
      // t1 = (sqrt(pl/rl) + sqrt(pr/rr))/2, t2 = -(ur-ul)/(2 t1), p* = sqrt(pl pr) exp(t2),
      // u* = ul - t1 log(p*/pl).  t1 scales small differences, so its roots are taken as
      // pl rsq(pl rl); p* and the ratio under the logarithm keep the roundings of the closed form.
      // Jumps past the series (a Mach or pressure jump of 1/8 between two cells) take the library
      // functions, in wavefronts that hold one in a cell whose interface is used.
      if constexpr (EX) {
        const T t1 = T(0.5) * (sqrt64_rn(div64(pl_, rl, rcp64(rl))) + sqrt64_rn(div64(pr, rr, rcp64(rr))));
        const T t2 = div64(T(-0.5) * (ur - ul), t1, rcp64(t1));
        pm = sqrt64_rn(pl_ * pr) * exp(t2);
        um = ul - t1 * log(div64(pm, pl_, rcp64(pl_)));
      } else {
        const T t1 = T(0.5) * __builtin_fma(pl_, rsq64(pl_ * rl), pr * rsq64(pr * rr));
        const T t2 = T(-0.5) * (ur - ul) * rcp64(t1);
        pm = sqrt64_rn(pl_ * pr) * exp_small(t2);
        const T ratio = div64(pm, pl_, rcp64(pl_));
        const T x = (ratio - T(1.0)) * rcp64(ratio + T(1.0));   // log(ratio) = 2 atanh(x)
        um = ul - t1 * (T(2.0) * atanh_small(x));
        const int c = c0 + h;
        const bool big = c >= 3 && c < nmax - 2 && !(fabs(t2) < 0.125 && fabs(x) < 0.125);
        if (wave_any(big)) {
          const T pb = sqrt(pl_ * pr) * exp(t2);
          const T ub = ul - t1 * log(pb / pl_);
          pm = big ? pb : pm;
          um = big ? ub : um;
        }
      }
    } else if constexpr (CF::EOS == 2 || CF::EOS == 3) {
      // two rarefactions for p*, then a shock or a rarefaction on each side.  2-D sweeps take every
      // power relative to p_l -- log(p_r/p_l), log(p*/p_l) = log(N/D)/z with N - D formed without
      // cancellation -- by the series, which hold for jumps up to 1/8, and past that the closed form
      // with the library's powers, in wavefronts that hold such a jump in a cell whose interface is
      // used.  Five library powers were half of the sweep (192 x 576: 22.7 -> 14.7 radial, 15.3 -> 11.4
      // us azimuthal).
      const T gamfac2 = gam + T(1.0), gamz = gamm / gam / T(2.0);
      auto closed = [&]() {
        T cs_l = sqrt(gam * pl_ / rl);
        T cs_r = sqrt(gam * pr / rr);
        pm = pow((cs_l + cs_r - (gamm / T(2.0)) * (ur - ul)) / (cs_l * pow(pl_, -gamz) + cs_r * pow(pr, -gamz)),
                 T(1.0) / gamz);
        T t1, t2;
        if (pm > pr) t1 = (pm - pr) * sqrt(T(2.0) / (rr * (gamfac2 * pm + pr * gamm)));
        else t1 = T(2.0) * cs_r * (pow(pm / pr, gamz) - T(1.0)) / gamm;
        if (pm > pl_) t2 = (pm - pl_) * sqrt(T(2.0) / (rl * (gamfac2 * pm + pl_ * gamm)));
        else t2 = T(2.0) * cs_l * (pow(pm / pl_, gamz) - T(1.0)) / gamm;
        um = T(0.5) * (ur + ul) + T(0.5) * (t1 - t2);
      };
      if constexpr (EX) {
        closed();
      } else {
        const T gl = gam * pl_, gr = gam * pr;
        const T cs_l = gl * rsq64(gl * rl), cs_r = gr * rsq64(gr * rr);
        const T x = (pr - pl_) * rcp64(pr + pl_);
        const T lr = T(2.0) * atanh_small(x);   // log(p_r/p_l)
        const T e = exp_small(-gamz * lr);
        const T D = __builtin_fma(cs_r, e, cs_l), d = cs_r * (T(1.0) - e) - (T(0.5) * gamm) * (ur - ul);
        const T y = d * rcp64(T(2.0) * D + d);
        const T lm = (T(2.0) / gamz) * atanh_small(y);   // log(p*/p_l)
        pm = pl_ * exp_small(lm);
        const T sh1 = (pm - pr) * (T(1.4142135623730951) * rsq64(rr * (gamfac2 * pm + pr * gamm)));
        const T sh2 = (pm - pl_) * (T(1.4142135623730951) * rsq64(rl * (gamfac2 * pm + pl_ * gamm)));
        const T ra1 = (T(2.0) / gamm) * cs_r * (exp_small(gamz * (lm - lr)) - T(1.0));
        const T ra2 = (T(2.0) / gamm) * cs_l * (exp_small(gamz * lm) - T(1.0));
        um = T(0.5) * (ur + ul) + T(0.5) * ((pm > pr ? sh1 : ra1) - (pm > pl_ ? sh2 : ra2));
        const int c = c0 + h;
        const bool big = c >= 3 && c < nmax - 2 && !(fabs(x) < 0.125 && fabs(y) < 0.125 && fabs(lm) < 0.125);
        if (wave_any(big)) {
          const T ps = pm, us = um;
          closed();
          pm = big ? pm : ps;
          um = big ? um : us;
        }
      }
    } else {
      const T gamfac2 = gam + T(1.0), gamfac1 = gamfac2 / gam / T(2.0);
      T cs_l = sqrt(gam * pl_ * rl);
      T cs_r = sqrt(gam * pr * rr);
      rl = T(1.0) / rl;
      rr = T(1.0) / rr;
      pm = pr - pl_ - cs_r * (ur - ul);
      pm = pl_ + pm * cs_l / (cs_l + cs_r);
      pm = fmax(smallp, pm);
      T t1 = T(0), t2 = T(0);
      for (int it = 0; it < 10; ++it) {
        T dum = pm;
        t1 = T(1.0) + gamfac1 * (pm - pl_) / pl_;
        t2 = T(1.0) + gamfac1 * (pm - pr) / pr;
        t1 = cs_l * sqrt(t1);
        t2 = cs_r * sqrt(t2);
        T en_l = T(4.0) * rl * t1 * t1;
        T en_r = T(4.0) * rr * t2 * t2;
        en_l = -en_l * t1 / (en_l - gamfac2 * (pm - pl_));
        en_r = en_r * t2 / (en_r - gamfac2 * (pm - pr));
        T uml = ul - (pm - pl_) / t1;
        T umr = ur + (pm - pr) / t2;
        pm = pm + (umr - uml) * (en_r * en_l) / (en_r - en_l);
        pm = fmax(smallp, pm);
        if (fabs(pm - dum) / pm < T(1.0e-8)) break;
      }
      T uml = ul - (pm - pl_) / t1;
      T umr = ur + (pm - pr) / t2;
      um = T(0.5) * (uml + umr);
    }
    umid[h] = um;
    pmid[h] = fmax(smallp, pm);
  }

  // ---- evolve (evolve.cu:3-166)
  C<T, K> dtdm, vf, xa, dxl, dvol;
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const int c = c0 + h;
    T delx;
    if constexpr (AX == 0) {
      delx = dt * umid[h];
    } else if constexpr (AX == 1) {
      if constexpr (CF::GY > 2) delx = dt * (div64(umid[h], W.rad[h], irad[h]) - ring.vrot - FrRot);
      else delx = dt * umid[h];
    } else {
      delx = div64(dt * umid[h], W.rad[h], irad[h]);
    }
    const T m = W.r[h] * W.dvol0[h];
    dtdm[h] = div64(dt, m, rcp64(m));
    bool in = (c >= 3 && c < nmax - 2);
    vf[h] = in ? W.xa0[h] + delx : W.xa0[h] + T(0.5) * W.dx0[h];
  }
  {
    C<T, K> vfp = next1(vf);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      const int c = c0 + h;
      bool in = (c >= 3 && c < nmax - 3);
      dxl[h] = in ? vfp[h] - vf[h] : W.dx0[h];
      xa[h] = in ? vf[h] : W.xa0[h];
    }
  }
  C<T, K> fto1, fto2, xcl;
  C<T, K> spol, cpol, star, irc, rcyl;
  if constexpr (AX == 0) star = tx.get(kT64Star);
  if constexpr (AX == 0 && CF::GX == 2) spol = tx.get(kT64Sp);
  if constexpr (AX == 2) {
    spol = tx.get(kT64Sp);
    cpol = tx.get(kT64Cp);
    rcyl = tx.get(kT64Rc);
    irc = tx.get(kT64Irc);
  }
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const T xc_ = xa[h] + T(0.5) * dxl[h];
    xcl[h] = xc_;
    T f1 = T(0), f2 = T(0);
    if constexpr (AX == 0) {
      // at the cell centre before and at the moved centre after the step (forces.cu:185-232)
      const T rad = W.rad[h], y2 = rcp64_rn(xc_);
      f1 = star[h];                    // -1 / rad / rad
      f2 = -div64(y2, xc_, y2);
      T c2 = T(0), s2;
      if constexpr (CF::GX == 1) {
        if (rf.planet) {
          turn(W.ca[h], W.sa[h], T(1.0) - T(2.0) * hs[h] * hs[h], T(2.0) * hs[h] * hc[h], c2, s2);
          f1 = grav_rad_cyl(G, rad, W.ca[h]) + (G.bary ? T(0) : f1);
          f2 = grav_rad_cyl(G, xc_, c2) + (G.bary ? T(0) : f2);
        }
        const T l2 = W.v[h] * W.v[h];
        f1 += div64(div64(div64(l2, rad, irad[h]), rad, irad[h]), rad, irad[h]);
        f2 += div64(div64(div64(l2, xc_, y2), xc_, y2), xc_, y2);
      } else {
        if (rf.planet) {
          const T a = rad * rad, b = xc_ * xc_;
          c2 = cos(angle(W.azi[h], vrot[h], dt));
          f1 = grav_rad_sph(G, rad, cos(angle(W.azi[h], T(0), T(0))), spol[h], div64(G.stm, a, rcp64(a)));
          f2 = grav_rad_sph(G, xc_, c2, spol[h], div64(G.stm, b, rcp64(b)));
        }
        const T w2 = W.w[h] * W.w[h], v2 = W.v[h] * W.v[h];
        const T p1 = rad * spol[h], p2 = xc_ * spol[h], q1 = p1 * p1, q2 = p2 * p2;
        f1 += div64(div64(div64(w2, rad, irad[h]), rad, irad[h]), rad, irad[h]);
        f1 += div64(div64(v2, rad, irad[h]), q1, rcp64(q1));
        f2 += div64(div64(div64(w2, xc_, y2), xc_, y2), xc_, y2);
        f2 += div64(div64(v2, xc_, y2), q2, rcp64(q2));
      }
    } else if constexpr (AX == 1) {
      if (rf.planet) {
        if constexpr (EX) {
          const T p1 = angle(W.azi[h], T(0), T(0)), p2 = angle(xc_, ring.vrot, dt);
          f1 = grav_azi_sph(G, ring.rsph, cos(p1), sin(p1), ring.sinpol);
          f2 = grav_azi_sph(G, ring.rsph, cos(p2), sin(p2), ring.sinpol);
        } else {
          T c, s, ce, se;
          sincos_small((xc_ - W.azi[h]) + dt * (ring.vrot - pl.vy), se, ce);
          turn(W.ca[h], W.sa[h], ce, se, c, s);
          f1 = grav_azi_cyl(G, W.rad[h], W.ca[h], W.sa[h]);
          f2 = grav_azi_cyl(G, W.rad[h], c, s);
        }
      }
    } else {
      const T l2 = W.w[h] * W.w[h];
      T sx, cx;
      sincos(xc_, &sx, &cx);
      const T rc2 = W.rad[h] * sx, y2 = rcp64(rc2);
      if (rf.planet) {
        f1 = grav_pol_sph(G, W.rad[h], cos(angle(W.azi[h], T(0), T(0))), spol[h], cpol[h]);
        f2 = grav_pol_sph(G, W.rad[h], cos(angle(W.azi[h], vrot[h], dt)), sx, cx);
      }
      f1 += div64(div64(div64(l2 * cpol[h], rcyl[h], irc[h]), rcyl[h], irc[h]), rcyl[h], irc[h]);
      f2 += div64(div64(div64(l2 * cx, rc2, y2), rc2, y2), rc2, y2);
    }
    fto1[h] = f1;
    fto2[h] = f2;
  }
  C<T, K> umidp, cxa, cx0;   // theta: cos of the moved and of the unmoved left edge
  if constexpr (AX == 2) cx0 = tx.get(kT64Cpl);
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const T x_ = xa[h], x0 = W.xa0[h], d_ = dxl[h];
    umidp[h] = umid[h] * pmid[h];
    T dv, vv;
    if constexpr (AX == 0) {
      if constexpr (CF::GX == 0) { dv = d_; vv = T(1.0); }
      else if constexpr (CF::GX == 1) { dv = d_ * (x_ + T(0.5) * d_); vv = T(0.5) * (x_ + x0); }
      else { dv = d_ * (x_ * (x_ + d_) + d_ * d_ * third); vv = (x_ - x0) * (third * (x_ - x0) + x0) + (x0 * x0); }
    } else if constexpr (AX == 1) {
      if constexpr (CF::GY == 0) { dv = d_; vv = T(1.0); }
      else { dv = d_ * W.rad[h]; vv = T(1.0); }
    } else {
      const T delx = x_ - x0;
      cxa[h] = cos(x_);
      dv = (cxa[h] - cos(x_ + d_)) * W.rad[h];
      vv = (delx == T(0.0)) ? sin(x_) : (cx0[h] - cxa[h]) / delx;
    }
    dvol[h] = dv;
    vf[h] = vv;   // area factor at the left face
  }
  C<T, K> q;
  {
    C<T, K> pmp = next1(pmid), vfp = next1(vf), ump = next1(umidp);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      const int c = c0 + h;
      bool in = (c >= 3 && c < nmax - 3);
      T qh = T(0);
      if constexpr (CF::EOS == 0) qh = W.p[h] / W.r[h];
      else if constexpr (CF::EOS == 1) qh = W.p[h] / pow(W.r[h], gam);
      T rn = fmax(W.r[h] * div64(W.dvol0[h], dvol[h], rcp64(dvol[h])), smallr);
      T delx = T(0.5) * dt * (fto1[h] + fto2[h]);
      delx += -dtdm[h] * (pmp[h] - pmid[h]) * T(0.5) * (vfp[h] + vf[h]);
      T un = W.u[h] + delx;
      if constexpr (CF::EOS == 2) {
        T ef = W.e[h] - dtdm[h] * (vfp[h] * ump[h] - vf[h] * umidp[h]);
        T x_ = xcl[h];
        T pol = T(0);   // theta of the cell in 3-D (the 2-D table does not hold it)
        if constexpr (AX == 0 && CF::GX == 2) pol = tx.get(kT64Pol)[h];
        if constexpr (AX == 0)
          qh = ef - T(0.5) * ((un * un) + (W.v[h] * W.v[h] / x_ / x_)) - potential<T>(rf.planet, pl, x_, W.azi[h], pol);
        else if constexpr (AX == 1)
          qh = ef - T(0.5) * (un * un) - potential<T>(rf.planet, pl, W.rad[h], x_, ring.pol);
        else
          qh = ef - T(0.5) * (un * un) - potential<T>(rf.planet, pl, W.rad[h], W.azi[h], x_);
        qh = fmax(gamm * qh, smallp);
      } else if constexpr (CF::EOS == 3) {
        // the energy-consistent form (the commented line of evolve.cu:146): e = p / (gamm rho)
        // + u^2 / 2 gains the pressure work and the time-centred work of the forces that move
        // u; the internal energy is what remains after the new u^2 / 2
        T ef = W.e[h] - dtdm[h] * (vfp[h] * ump[h] - vf[h] * umidp[h]) +
               T(0.5) * dt * (W.u[h] * fto1[h] + un * fto2[h]);
        qh = fmax(gamm * (ef - T(0.5) * (un * un)), smallp);
      }
      q[h] = qh;
      if (in) {
        W.r[h] = rn;
        W.u[h] = un;
      }
    }
  }

  // ---- remap (remap.cu:14-226)
  if constexpr (AX != 1) idvol = tx.get(AX == 0 ? kT64Ivol : kT64Ivolz);
  Para<T, K> P1 = paraset64<K, EX>(dxl);
  C<T, K> dxf, dxf2, fr;
  C<bool, K> delC;
  C<T, K> dxm = prev1(dxl);
  C<T, K> lvol;
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const T x_ = xa[h], x0 = W.xa0[h];
    T lv;
    if constexpr (AX == 0) {
      if constexpr (CF::GX == 0) lv = x_ - x0;
      else if constexpr (CF::GX == 1) { lv = x_ - x0; lv *= (x0 + T(0.5) * lv); }
      else { lv = x_ - x0; lv *= x0 * x_ + third * (lv * lv); }
    } else if constexpr (AX == 1) {
      if constexpr (CF::GY == 0) lv = x_ - x0;
      else lv = (x_ - x0) * W.rad[h];
    } else {
      lv = (cx0[h] - cxa[h]) * W.rad[h];
    }
    lvol[h] = lv;
    const T d = x_ - x0;
    delC[h] = d >= T(0.0);
    // 1 - (4/3) d' for a face moving up, 1 + (4/3) d' for one moving down, d' < 0
    const T den = d >= T(0.0) ? dxm[h] : dxl[h];
    const T e = EX ? div64(T(0.5) * d, den, rcp64(den)) : T(0.5) * d * rcp64(den);
    dxf[h] = e;
    dxf2[h] = T(1.0) - fourthd * fabs(e);
  }
  // face average of a parabola swept through the face (remap.cu:59-90, get_flux :1-10)
  auto face = [&](const Parab<T, K>& Q, C<T, K>& out) {
    C<T, K> alm = prev1(Q.al), dam = prev1(Q.da), a6m = prev1(Q.a6);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      T up, dn;
      if constexpr (EX) {
        up = alm[h] + dam[h] - dxf[h] * (dam[h] - dxf2[h] * a6m[h]);
        dn = Q.al[h] - dxf[h] * (Q.da[h] + dxf2[h] * Q.a6[h]);
      } else {
        up = __builtin_fma(-dxf[h], __builtin_fma(-dxf2[h], a6m[h], dam[h]), alm[h] + dam[h]);
        dn = __builtin_fma(-dxf[h], __builtin_fma(dxf2[h], Q.a6[h], Q.da[h]), Q.al[h]);
      }
      out[h] = delC[h] ? up : dn;
    }
  };
  C<T, K> mass, invm;
  {
    Parab<T, K> Q = parabola<K, EX>(flat, omf, W.r, P1);
    C<T, K> fv;
    face(Q, fv);
#pragma unroll
    for (int h = 0; h < K; ++h) fr[h] = fv[h] * lvol[h];
    C<T, K> frp = next1(fr);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      const int c = c0 + h;
      T m = W.r[h] * dvol[h];
      T rn = fmax(smallr, div64(m + fr[h] - frp[h], W.dvol0[h], idvol[h]));
      mass[h] = m;
      invm[h] = rcp64_rn(rn * W.dvol0[h]);
      if (c >= 6 && c < nmax - 6) W.r[h] = rn;
    }
  }
  auto remap_field = [&](C<T, K>& X) {
    Parab<T, K> Q = parabola<K, EX>(flat, omf, X, P1);
    C<T, K> fl;
    face(Q, fl);
#pragma unroll
    for (int h = 0; h < K; ++h) fl[h] = fl[h] * fr[h];
    C<T, K> flp = next1(fl);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      const int c = c0 + h;
      if (c >= 6 && c < nmax - 6) X[h] = (X[h] * mass[h] + (fl[h] - flp[h])) * invm[h];
    }
  };
  remap_field(W.u);
  if (rf.remap_v) remap_field(W.v);
  if (rf.remap_w) remap_field(W.w);
  if constexpr (CF::EOS != 0) {
    remap_field(q);
#pragma unroll
    for (int h = 0; h < K; ++h) {
      const int c = c0 + h;
      if (c >= 6 && c < nmax - 6) {
        if constexpr (CF::EOS == 1) W.p[h] = fmax(smallp, pow(W.r[h], gam) * q[h]);
        else W.p[h] = fmax(smallp, W.r[h] * q[h]);
      }
    }
  }
}

// derivs (viscosity.cu:2-19) with the divisions by its three coordinate differences shared by
// every field of a cell.  quot<EX>: a / b from y = 1 / b to an ulp; the viscous update is a small
// increment, so in 2-D its quotients need not round as divisions do
template <bool EX>
__device__ __forceinline__ double quot(double a, double b, double y) {
  if constexpr (EX) return div64(a, b, y);
  else return a * y;
}
template <bool EX>
struct Fit64 {
  double x2, x3, i2, i3, i32;
  __device__ __forceinline__ Fit64(double xm, double x0, double xp) {
    x2 = x0 - xm;
    x3 = xp - xm;
    i2 = rcp64(x2);
    i3 = rcp64(x3);
    i32 = rcp64(x3 - x2);
  }
  __device__ __forceinline__ void operator()(double um, double u0, double up, double& first, double& second) const {
    const double h2 = quot<EX>(u0 - um, x2, i2), h3 = quot<EX>(up - um, x3, i3), x32 = x3 - x2;
    second = 2.0 * quot<EX>(h3 - h2, x32, i32);
    first = second * x2 + quot<EX>(x3 * h2 - x2 * h3, x32, i32);
  }
};

// device_viscosity_r (viscosity.cu:370-421); R = cylindrical radius per cell, x = left edges
template <int K, bool EX>
__device__ __forceinline__ void visc_r(Win<K>& W, int c0, int lim, double dt, const C<double, K>& R, const C<double, K>& nu, bool do_w) {
  C<double, K> nr, vv;
#pragma unroll
  for (int h = 0; h < K; ++h) {
    nr[h] = nu[h] * W.r[h];
    const double R2 = R[h] * R[h];
    vv[h] = div64(W.v[h], R2, rcp64(R2));
  }
  C<double, K> xm = prev1(W.xa0), xp = next1(W.xa0);
  C<double, K> nm = prev1(nr), np = next1(nr);
  C<double, K> um = prev1(W.u), up = next1(W.u);
  C<double, K> vm = prev1(vv), vp = next1(vv);
  C<double, K> wm, wp;
  if (do_w) {
    wm = prev1(W.w);
    wp = next1(W.w);
  }
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const int c = c0 + h;
    const double rho = W.r[h], n = nr[h], Ri = R[h], iR = rcp64(Ri), irho = rcp64(rho);
    double dn, d1, d2;
    const Fit64<EX> D(xm[h], W.xa0[h], xp[h]);
    D(nm[h], n, np[h], dn, d2);
    D(um[h], W.u[h], up[h], d1, d2);
    double ddu = 2.0 * n * d2 + 2.0 * dn * d1 + quot<EX>(2.0 * n * d1, Ri, iR) - quot<EX>(quot<EX>(2.0 * n * W.u[h], Ri, iR), Ri, iR);
    ddu = W.u[h] + quot<EX>(dt * ddu, rho, irho);
    D(vm[h], vv[h], vp[h], d1, d2);
    double ddv = Ri * n * d2 + Ri * dn * d1 + 3.0 * n * d1;
    ddv = vv[h] * Ri + quot<EX>(dt * ddv, rho, irho);
    double ddw = W.w[h];
    if (do_w) {
      D(wm[h], W.w[h], wp[h], d1, d2);
      double t = n * d2 + dn * d1 + quot<EX>(n * d1, Ri, iR);
      ddw = W.w[h] + quot<EX>(dt * t, rho, irho);
    }
    if (c >= kNpad && c < lim - kNpad) {
      W.u[h] = ddu;
      W.v[h] = ddv * Ri;
      if (do_w) W.w[h] = ddw;
    }
  }
}

// device_viscosity_p (viscosity.cu:423-472), called with (u, v, w) = (u_r, v_phi, w) of the
// azimuthal sweep, i.e. sweep fields (w, u, v); x = left edges times R
template <int K, bool EX>
__device__ __forceinline__ void visc_p(Win<K>& W, int c0, int lim, double dt, double R, double nu, const C<double, K>& x, bool do_w) {
  C<double, K> nr;
#pragma unroll
  for (int h = 0; h < K; ++h) nr[h] = nu * W.r[h];
  C<double, K> xm = prev1(x), xp = next1(x);
  C<double, K> nm = prev1(nr), np = next1(nr);
  // parameter v of the reference = sweep u (v_phi); parameter u = sweep w (u_r);
  // parameter w = sweep v
  C<double, K> pvm = prev1(W.u), pvp = next1(W.u);
  C<double, K> pum = prev1(W.w), pup = next1(W.w);
  C<double, K> pwm, pwp;
  if (do_w) {
    pwm = prev1(W.v);
    pwp = next1(W.v);
  }
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const int c = c0 + h;
    const double rho = W.r[h], n = nr[h], irho = rcp64(rho);
    double dn, d1, d2;
    const Fit64<EX> D(xm[h], x[h], xp[h]);
    D(nm[h], n, np[h], dn, d2);
    D(pvm[h], W.u[h], pvp[h], d1, d2);
    double ddv = 2.0 * n * d2 + 2.0 * dn * d1;
    double ddu = 0.0;
    ddv = W.u[h] + quot<EX>(dt * ddv, rho, irho);
    double ddw = W.v[h];
    if (do_w) {
      D(pwm[h], W.v[h], pwp[h], d1, d2);
      double t = n * d2 + dn * d1;
      ddw = W.v[h] + quot<EX>(dt * t, rho, irho);
    }
    D(pum[h], W.w[h], pup[h], d1, d2);
    ddu += n * d2 + dn * d1;
    ddu = W.w[h] + quot<EX>(dt * ddu, rho, irho);
    if (c >= kNpad && c < lim - kNpad) {
      W.u[h] = ddv;
      if (do_w) W.v[h] = ddw;
      W.w[h] = ddu;
    }
  }
}

// device_viscosity_z (viscosity.cu:474-518): nu rho with the constant vis_nu, the component
// along the pencil (the reference's w) taking 2 nu rho d2 + 2 dn d1 and the transverse ones
// nu rho d2 + dn d1, no curvature terms.  The theta sweep passes (u, v, w) = (v_r, v_phi,
// v_theta) and x = r times the theta left edges.
template <int K, bool EX>
__device__ __forceinline__ void visc_z(const C<double, K>& rho, int c0, int lim, double dt, double nu, const C<double, K>& x, C<double, K>& u,
                                       C<double, K>& v, C<double, K>& w) {
  C<double, K> nr;
#pragma unroll
  for (int h = 0; h < K; ++h) nr[h] = nu * rho[h];
  C<double, K> xm = prev1(x), xp = next1(x);
  C<double, K> nm = prev1(nr), np = next1(nr);
  C<double, K> um = prev1(u), up = next1(u);
  C<double, K> vm = prev1(v), vp = next1(v);
  C<double, K> wm = prev1(w), wp = next1(w);
#pragma unroll
  for (int h = 0; h < K; ++h) {
    const int c = c0 + h;
    const double n = nr[h], rh = rho[h], irho = rcp64(rh);
    double dn, d1, d2;
    const Fit64<EX> D(xm[h], x[h], xp[h]);
    D(nm[h], n, np[h], dn, d2);
    D(wm[h], w[h], wp[h], d1, d2);
    double ddw = 2.0 * n * d2 + 2.0 * dn * d1;
    D(um[h], u[h], up[h], d1, d2);
    double ddu = n * d2 + dn * d1;
    D(vm[h], v[h], vp[h], d1, d2);
    double ddv = n * d2 + dn * d1;
    ddw = w[h] + quot<EX>(dt * ddw, rh, irho);
    ddu = u[h] + quot<EX>(dt * ddu, rh, irho);
    ddv = v[h] + quot<EX>(dt * ddv, rh, irho);
    if (c >= kNpad && c < lim - kNpad) {
      w[h] = ddw;
      u[h] = ddu;
      v[h] = ddv;
    }
  }
}

}  // namespace pn
