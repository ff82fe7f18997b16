// lbm_point.hpp — the pointwise arithmetic of the RK3 stages of FP64 storage:
// moments, equilibria and relaxation of one cell, in a form that every kernel
// of the step evaluates with the same roundings (contraction off, every fused
// multiply-add explicit), whether it holds all thirteen directions of a cell
// or four wavefronts share them.
#pragma once

#include "lbm_device.hpp"

namespace uqlbm {

// The directions moving cells share between four wavefronts: wavefront w has
// one along x, one along y and one diagonal, all of x sign (w == 0 || w == 3)
// and y sign (w < 2). Sums over the directions of a cell are formed by
// wavefront, (x + y) + diagonal (+ the rest direction for w = 0), and then
// over the wavefronts in order.
__host__ __device__ constexpr int quad_x(int w) { return w == 0 ? 1 : w == 1 ? 3 : w == 2 ? 11 : 9; }
__host__ __device__ constexpr int quad_y(int w) { return w == 0 ? 2 : w == 1 ? 10 : w == 2 ? 4 : 12; }
__host__ __device__ constexpr int quad_d(int w) { return 5 + w; }

// Mass, x and y momentum (in units of c) and energy.
struct Sums {
  double m, px, py, e;
};

// Wavefront w's part of a cell's sums. (Products with the lattice velocities
// 1 and 2 are exact.)
__host__ __device__ __forceinline__ Sums quad_sums(double exx, double exd, double eyy, double eyd, double fx, double fy,
                                                   double fd, double hx, double hy, double hd) {
#pragma clang fp contract(off)
  Sums s;
  s.m = (fx + fy) + fd;
  s.px = fused(exx, fx, exd * fd);
  s.py = fused(eyy, fy, eyd * fd);
  s.e = (hx + hy) + hd;
  return s;
}
__host__ __device__ __forceinline__ Sums operator+(const Sums& a, const Sums& b) {
#pragma clang fp contract(off)
  return Sums{a.m + b.m, a.px + b.px, a.py + b.py, a.e + b.e};
}
__host__ __device__ __forceinline__ Sums operator-(const Sums& a, const Sums& b) {
#pragma clang fp contract(off)
  return Sums{a.m - b.m, a.px - b.px, a.py - b.py, a.e - b.e};
}

template <int W>
__host__ __device__ __forceinline__ Sums quad_sums_of(const double* f, const double* h) {
  constexpr int X = quad_x(W), Y = quad_y(W), D = quad_d(W);
  return quad_sums(lat_x(X), lat_x(D), lat_y(Y), lat_y(D), f[X], f[Y], f[D], h[X], h[Y], h[D]);
}
// Sums of all thirteen directions (rest: whether the rest direction counts).
__host__ __device__ __forceinline__ Sums cell_sums(const double* f, const double* h, bool rest) {
#pragma clang fp contract(off)
  Sums a = quad_sums_of<0>(f, h);
  if (rest) {
    a.m = a.m + f[0];
    a.e = a.e + h[0];
  }
  return ((a + quad_sums_of<1>(f, h)) + quad_sums_of<2>(f, h)) + quad_sums_of<3>(f, h);
}

// The functions below take the instance record as they are given it (In: the
// record, or the record in the constant address space) and its gas constants
// as part of it (KQ). A Macro of theirs is in lattice units: velocities in units
// of c, temperature in units of Tc.
//
// Constants of the gas, from its internal degrees of freedom K: b = K + 2.
enum { kqB, kqHalfB, kqInvB, kqCount };
static_assert(kqCount <= kPointConsts, "InstDev::kq holds the constants");

inline void point_consts(double K, double* kq) {
  kq[kqB] = K + 2;
  kq[kqHalfB] = 0.5 * (K + 2);
  kq[kqInvB] = 1 / (K + 2);
}

// x / d from the constant id = 1/d: rounded to nearest, where x * id alone errs
// by the same fraction in every cell and step.
__host__ __device__ __forceinline__ double over(double x, double d, double id) {
#pragma clang fp contract(off)
  const double q = x * id;
  return fused(fused(-d, q, x), id, q);
}

// Moments of a cell (reference macroProp, cpuLBM.cpp:916-970), T = (2 e/(rho R
// Tc) - u^2)/b.
template <typename In>
__host__ __device__ __forceinline__ void point_moments(const In& in, const Sums& s, Macro& m) {
#pragma clang fp contract(off)
  const double irho = recip(s.m), sc = s.m * in.RTc, q = irho * in.iRTc;
  const double isc = fused(fused(-sc, q, 1.0), q, q);
  m.rho = s.m;
  m.ux = s.px * irho;
  m.uy = s.py * irho;
  const double usq = fused(m.ux, m.ux, m.uy * m.uy);
  m.T = over(fused(2.0, s.e * isc, -usq), in.kq[kqB], in.kq[kqInvB]);
  m.p = sc * m.T;
}
template <typename In>
__device__ __forceinline__ void point_macro(const In& in, const InstDev& inst, const Sums& s, Macro& m) {
#pragma clang fp contract(off)
  point_moments(in, s, m);
  m.itf = in.visc_model == 0 ? m.p * in.imu : m.p / viscosity_of(inst, m.T * in.Tc);
  m.ith = m.itf * in.Pr;
  m.ithf = m.itf * in.Pr_m1;
}

// Equilibria: the closed forms of eq_dir (reference inlineFunctions.cpp:10-61)
// as the specific energy times f plus a rest in which K does not occur,
//   fe = rho F(u, v, t),  he = (b/2 t + (u^2 + v^2)/2) R Tc fe + rho R Tc t/3 G(u, v, t),
// the G of a cell's thirteen directions summing to zero: the sums over the
// directions give back the cell's mass, momentum and energy whatever the
// roundings of the factors. Each stage takes the conserved moments from the
// equilibria, so a constant that rounds to one side (a third, 10 (16 + 3 K),
// ...) shifts them by the same fraction in every cell and step. Such are kept
// out of the sums: rho/3 is rounded to nearest, the other factors are whole
// numbers or common to all directions. Mean error of a cell's energy in eps,
// nested forms with coefficients in K -> these: -0.60 -> 0.00 at gamma 1.4,
// -1.15 -> 0.01 at 5/3; pressure of a 200^2 Riemann solve after 60 steps against
// long double 6.4e-15 -> 2.7e-15, temperature 8.3e-15 -> 4.3e-15.
struct PointEq {
  double u, v, t;  // velocity / sqrt(R Tc), T / Tc
  double rho, r3;  // density, a third of it
  double rt3;      // rho R Tc t/3
  double en;       // specific energy
};

template <typename In>
__host__ __device__ __forceinline__ PointEq point_eq(const In& in, const Macro& m) {
#pragma clang fp contract(off)
  PointEq e;
  e.rho = m.rho;
  e.r3 = over(m.rho, 3.0, 1.0 / 3.0);
  e.u = m.ux;
  e.v = m.uy;
  e.t = m.T;
  e.rt3 = (e.r3 * in.RTc) * e.t;
  e.en = fused(in.kq[kqHalfB], e.t, 0.5 * fused(e.u, e.u, e.v * e.v)) * in.RTc;
  return e;
}

// The four kinds of directions at (a, b): rest, axis, diagonal, double axis.
__host__ __device__ __forceinline__ void eq_rest(const PointEq& e, double& fe, double& he) {
#pragma clang fp contract(off)
  const double u2 = e.u * e.u, v2 = e.v * e.v, uv = u2 * v2, t = e.t, s2 = u2 + v2;
  const double Z = fused(s2, s2 - 5.0, fused(2.0, uv, 4.0));
  fe = (e.rho * 0.25) * fused(10.0 * t, (t + s2) - 1.0, Z);
  const double G = fused(t, fused(25.0, t, fused(45.0, s2, -15.0)), 3.0 * fused(s2, fused(2.0, s2, -5.0), 4.0 * uv));
  he = fused(e.en, fe, (0.5 * e.rt3) * G);
}
__host__ __device__ __forceinline__ void eq_axis(const PointEq& e, double a, double b, double& fe, double& he) {
#pragma clang fp contract(off)
  const double a2 = a * a, b2 = b * b;
  const double t = e.t, q = fused(3.0, b2, a2), w = q - 4.0, x = fused(3.0, q, -4.0);
  fe = (e.r3 * -0.5) * fused(t, fused(6.0, t, fused(8.0, a2, fused(6.0, a, w))), (a + a2) * w);
  const double G = fused(t, fused(10.0, t, fused(12.0 * a, fused(2.0, a, 1.0), x)), a * fused(4.0 * a, q - 2.0, x));
  he = fused(e.en, fe, (-0.5 * e.rt3) * G);
}
__host__ __device__ __forceinline__ void eq_diag(const PointEq& e, double a, double b, double& fe, double& he) {
#pragma clang fp contract(off)
  const double a2 = a * a, b2 = b * b;
  const double t = e.t, ab = a * b, s = 3.0 * (a + b);
  fe = (e.rho * 0.25) * ((t + (a + a2)) * (t + (b + b2)));
  const double G = fused(t, fused(5.0, t, fused(9.0, a2 + b2, 2.0 * s)), (3.0 * ab) * fused(4.0, ab, s + 2.0));
  he = fused(e.en, fe, (0.25 * e.rt3) * G);
}
__host__ __device__ __forceinline__ void eq_axis2(const PointEq& e, double a, double& fe, double& he) {
#pragma clang fp contract(off)
  const double t = e.t, g = fused(a, a, a);
  fe = (e.r3 * 0.125) * fused(t, fused(3.0, t, fused(6.0, g, -1.0)), g * (g - 2.0));
  const double G = fused(t, fused(5.0, t, fused(a, fused(18.0, a, 12.0), -1.0)),
                         (2.0 * a) * fused(a, fused(a, fused(2.0, a, 3.0), -1.0), -1.0));
  he = fused(e.en, fe, (0.125 * e.rt3) * G);
}

// Direction I. (The gas enters by the moments alone.)
template <int I, typename KQ>
__host__ __device__ __forceinline__ void eq_point(const KQ&, const PointEq& e, double& fe, double& he) {
  constexpr int base = eq_base(I);
  const double a = eq_sa(I) * (eq_swap(I) ? e.v : e.u), b = eq_sb(I) * (eq_swap(I) ? e.u : e.v);
  if constexpr (base == 0) eq_rest(e, fe, he);
  else if constexpr (base == 1) eq_axis(e, a, b, fe, he);
  else if constexpr (base == 5) eq_diag(e, a, b, fe, he);
  else eq_axis2(e, a, fe, he);
}

// Stages 1 and 2 (cpuLBM.cpp:1819-1924) in closed form. With af = dt/(2 tf),
// ah = dt/(2 th), ahf = dt/(2 thf), r = 1/(1 + af), rh = 1/(1 + ah) the two
// implicit stages give (feq2 = feq1 = fe, heq2 = heq1 = he)
//   f2 = fe + q (f - fe),   q = (1 + 2 af) r^2
//   h2 = he + qh (h - he) + mu (e.u) (f - fe),
//        qh = (1 + 2 ah) rh^2, mu = ahf rh (q - rh r).
// e.u is R Tc (lat_x u + lat_y v) with the normalised velocity u, v of PointEq
// (c = sqrt(R Tc)): the coefficients of e.u carry the factor R Tc.
struct Relax12 {
  double q, qh, mu;
};
template <typename In>
__host__ __device__ __forceinline__ Relax12 make_relax12(const In& in, const Macro& m) {
#pragma clang fp contract(off)
  Relax12 R;
  const double hdt = in.dt * 0.5, af = hdt * m.itf, ah = hdt * m.ith, ahf = hdt * m.ithf;
  const double r = recip(1.0 + af), rh = recip(1.0 + ah);
  R.q = fused(2.0, af, 1.0) * (r * r);
  R.qh = fused(2.0, ah, 1.0) * (rh * rh);
  R.mu = ((ahf * rh) * fused(-rh, r, R.q)) * in.RTc;
  return R;
}
__host__ __device__ __forceinline__ void point_s12(const Relax12& R, const PointEq& e, double lx, double ly, double f,
                                                   double h, double fe, double he, double& f2, double& h2) {
#pragma clang fp contract(off)
  const double eu = fused(lx, e.u, ly * e.v), y = f - fe, x = h - he;
  f2 = fused(R.q, y, fe);
  h2 = fused(R.qh, x, fused(R.mu * eu, y, he));
}

// Stage 3 (cpuLBM.cpp:1926-1993) from the stage-2 distributions, which carry
// the moments and, through the closed forms above, the values of f and h: with
// D = fe - f2, E = he - h2, f = fe - D/q and h from h2 likewise,
//   P = f - dF2 + af D            = fe - ka D - dF2
//   Q = (h - dH2) - ahf eu D + ah E = he - kh E - la (e.u) D - dH2
//   ka = (1 + af - af^2)/(1 + 2 af), kh the same in ah,
//   la = ahf (ah + (1 + af)/(1 + 2 af))/(1 + 2 ah)
//   f3 = (P + af3 fe3)/(1 + af3)
//   h3 = (Q - ahf3 eu3 (fe3 - f3) + ah3 he3)/(1 + ah3),
// evaluated as the equilibrium plus a difference,
//   y = ((fe - fe3) - ka D - dF2)/(1 + af3),  f3 = fe3 + y, h3 likewise,
// so that only the last sum rounds at the size of the values: an error of the
// factors or of the reciprocals enters with y, whose conserved sums are none.
// So the state itself is not read again after stage 2. The rounding of f2
// enters f3 as ka eps/(1 + af3), at most af/(1 + af3) eps as in the form with
// f and af (fe - f2): bounded for stiff cells too. Root mean square errors
// against long double, with (P + af3 fe3)/(1 + af3) -> this: f3 0.19 -> 0.11
// eps, mass 0.50 -> 0.26 eps at weak relaxation, 0.13 -> 0.08 and 0.34 -> 0.20
// at stiff; the reference's formulas from the state itself 0.18 and 0.46, 0.25
// and 0.64.
struct Relax3 {
  double ka, kh, la;                  // stage-1 moments
  double af3, ah3, ahf3, iaf3, iah3;  // stage-3 moments
};
template <typename In>
__host__ __device__ __forceinline__ Relax3 make_relax3(const In& in, const Macro& m, const Macro& m3) {
#pragma clang fp contract(off)
  Relax3 R;
  const double hdt = in.dt * 0.5, af = hdt * m.itf, ah = hdt * m.ith, ahf = hdt * m.ithf;
  const double i1 = recip(fused(2.0, af, 1.0)), i2 = recip(fused(2.0, ah, 1.0));
  R.ka = fused(-af, af, 1.0 + af) * i1;
  R.kh = fused(-ah, ah, 1.0 + ah) * i2;
  R.la = ((ahf * fused(1.0 + af, i1, ah)) * i2) * in.RTc;
  R.af3 = hdt * m3.itf;
  R.ah3 = hdt * m3.ith;
  R.ahf3 = (hdt * m3.ithf) * in.RTc;
  R.iaf3 = recip(1.0 + R.af3);
  R.iah3 = recip(1.0 + R.ah3);
  return R;
}
__host__ __device__ __forceinline__ void point_s3(const Relax3& R, const PointEq& e, const PointEq& e3, double lx,
                                                  double ly, double f2, double h2, double dF, double dH, double fe,
                                                  double he, double fe3, double he3, double& f3, double& h3) {
#pragma clang fp contract(off)
  const double eu = fused(lx, e.u, ly * e.v), eu3 = fused(lx, e3.u, ly * e3.v);
  const double D = fe - f2, E = he - h2;
  const double y = (fused(-R.ka, D, fe - fe3) - dF) * R.iaf3;
  const double z = fused(-(R.la * eu), D, fused(-R.kh, E, he - he3)) - dH;
  f3 = fe3 + y;
  h3 = fused(fused(R.ahf3 * eu3, y, z), R.iah3, he3);
}

}  // namespace uqlbm
