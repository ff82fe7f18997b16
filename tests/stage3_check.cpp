// Host check of the rounding of stage 3 of FP64 storage, which takes the state
// back from the stage-2 distributions (point_s12, point_s3,
// uq_amd/csrc/lbm_point.hpp), against that of the reference's formulas
// (cpuLBM.cpp:1853-1993) evaluated in FP64 from the state itself: over random
// cells, for relaxation from dt/(2 tau) = 1e-6 to 1e5, the root mean square
// error of f3 and h3 (in units of the values that enter) and of their sums
// (mass, x momentum, energy) against long double must be no larger. Prints
// both, exits 1 otherwise.
#include <cmath>
#include <cstdio>
#include <random>
#include <utility>

#include "../uq_amd/csrc/lbm_point.hpp"

using namespace uqlbm;
typedef long double LD;

template <typename F, int... Is>
static void each_dir(F&& f, std::integer_sequence<int, Is...>) {
  (f(std::integral_constant<int, Is>{}), ...);
}
static const auto kDirs = std::make_integer_sequence<int, kQ>{};

// f3 and h3 by the reference's formulas, in the precision of T.
template <typename T>
static void reference_stages(const Macro& m, const Macro& m3, int I, T f, T h, T dF, T dH, T fe, T he, T fe3, T he3,
                             T& f3, T& h3) {
  const T hdt = T(0.5), af = hdt * T(m.itf), ah = hdt * T(m.ith), g = T(m.ithf);
  const T eu = T(lat_x(I)) * T(m.ux) + T(lat_y(I)) * T(m.uy), eu3 = T(lat_x(I)) * T(m3.ux) + T(lat_y(I)) * T(m3.uy);
  const T iaf = T(1) / (T(1) + af), iah = T(1) / (T(1) + ah);
  const T f1 = (f + af * fe) * iaf;
  const T h1 = (h - hdt * g * eu * (fe - f1) + ah * he) * iah;
  const T f2 = (f - af * (fe - f1) + af * fe) * iaf;
  const T h2 = (h - hdt * ((eu * g) * (fe - f2) - (eu * g) * (fe - f1)) - ah * (he - h1) + ah * he) * iah;
  const T P = (f - dF) + af * (fe - f2), Q = ((h - dH) - hdt * ((eu * g) * (fe - f2))) + ah * (he - h2);
  const T af3 = hdt * T(m3.itf), ah3 = hdt * T(m3.ith);
  f3 = (P + af3 * fe3) * (T(1) / (T(1) + af3));
  h3 = ((Q - hdt * ((eu3 * T(m3.ithf)) * (fe3 - f3))) + ah3 * he3) * (T(1) / (T(1) + ah3));
}

int main() {
  std::mt19937_64 rng(3);
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  const double eps = 2.2204460492503131e-16;
  bool ok = true;
  const double decades[][2] = {{-6, -4}, {-4, -2}, {-2, -1}, {-1, 0}, {0, 1}, {1, 3}, {3, 5}};
  for (const auto& range : decades) {
    double err[2][5] = {};  // form; f3, h3, mass, x momentum, energy
    const int n = 40000;
    for (int k = 0; k < n; k++) {
      InstDev in{};
      const double gamma = 1.2 + 0.45 * (0.5 + 0.5 * U(rng)), b = 2.0 / (gamma - 1.0);
      in.K = b - 2.0;
      in.Tc = in.iTc = in.RTc = in.isRTc = in.c = in.dt = in.R = in.imu = 1.0;
      in.ibR = 1.0 / b;
      in.Pr = 0.6 + 0.4 * (0.5 + 0.5 * U(rng));
      point_consts(in.K, in.kq);
      const double itf = 2.0 * std::pow(10.0, range[0] + (range[1] - range[0]) * (0.5 + 0.5 * U(rng)));
      auto moments = [&](const double* f, const double* h) {
        const Sums s = cell_sums(f, h, true);
        Macro m{};
        m.rho = s.m;
        m.ux = s.px / s.m;
        m.uy = s.py / s.m;
        m.T = (2.0 * (s.e / s.m) - (m.ux * m.ux + m.uy * m.uy)) * in.ibR;
        m.itf = itf;
        m.ith = itf * in.Pr;
        m.ithf = itf * (in.Pr - 1.0);
        return m;
      };
      Macro m{};
      m.rho = 1.0 + 0.3 * U(rng);
      m.T = 0.8 + 0.2 * U(rng);
      m.ux = 0.2 * U(rng);
      m.uy = 0.2 * U(rng);
      double f[kQ], h[kQ], dF[kQ], dH[kQ], g[kQ], gh[kQ];
      const PointEq near = point_eq(in, m);
      each_dir(
          [&](auto I) {
            double fe, he;
            eq_point<I>(in.kq, near, fe, he);
            f[I] = fe * (1 + 0.01 * U(rng));
            h[I] = he * (1 + 0.01 * U(rng));
            dF[I] = I ? 0.02 * fe * U(rng) : 0.0;
            dH[I] = I ? 0.02 * he * U(rng) : 0.0;
            g[I] = f[I] - dF[I];
            gh[I] = h[I] - dH[I];
          },
          kDirs);
      m = moments(f, h);
      const Macro m3 = moments(g, gh);
      const PointEq e = point_eq(in, m), e3 = point_eq(in, m3);
      const Relax12 r = make_relax12(in, m);
      const Relax3 r3 = make_relax3(in, m, m3);
      LD sums[2][3] = {};
      each_dir(
          [&](auto Ic) {
            constexpr int I = decltype(Ic)::value;
            double fe, he, fe3, he3, f2, h2, o[2][2];
            eq_point<I>(in.kq, e, fe, he);
            eq_point<I>(in.kq, e3, fe3, he3);
            point_s12(r, e, lat_x(I), lat_y(I), f[I], h[I], fe, he, f2, h2);
            point_s3(r3, e, e3, lat_x(I), lat_y(I), f2, h2, dF[I], dH[I], fe, he, fe3, he3, o[0][0], o[0][1]);
            reference_stages<double>(m, m3, I, f[I], h[I], dF[I], dH[I], fe, he, fe3, he3, o[1][0], o[1][1]);
            LD F3, H3;
            reference_stages<LD>(m, m3, I, f[I], h[I], dF[I], dH[I], fe, he, fe3, he3, F3, H3);
            const double sf = std::fabs(f[I]) + std::fabs(fe) + std::fabs(fe3);
            const double sh = std::fabs(h[I]) + std::fabs(he) + std::fabs(he3);
            for (int w = 0; w < 2; w++) {
              const LD df = o[w][0] - F3, dh = o[w][1] - H3;
              err[w][0] += std::pow((double)df / sf, 2) / kQ;
              err[w][1] += std::pow((double)dh / sh, 2) / kQ;
              sums[w][0] += df;
              sums[w][1] += df * lat_x(I);
              sums[w][2] += dh;
            }
          },
          kDirs);
      for (int w = 0; w < 2; w++)
        for (int j = 0; j < 3; j++) err[w][2 + j] += std::pow((double)sums[w][j] / m3.rho, 2);
    }
    const char* names[5] = {"f3", "h3", "mass", "x momentum", "energy"};
    std::printf("dt/(2 tau) 1e%g..1e%g, rms in eps (from the state):", range[0], range[1]);
    for (int j = 0; j < 5; j++) {
      const double a = std::sqrt(err[0][j] / n) / eps, b = std::sqrt(err[1][j] / n) / eps;
      std::printf(" %s %.3f (%.3f)", names[j], a, b);
      ok = ok && a <= b;
    }
    std::printf("\n");
  }
  return ok ? 0 : 1;
}
