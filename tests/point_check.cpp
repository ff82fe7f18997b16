// Host check of the pointwise arithmetic of FP64 storage
// (uq_amd/csrc/lbm_point.hpp): the nested equilibria against the closed form
// (eq_dir), and the closed-form stages against the reference's stage formulas
// (cpuLBM.cpp:1853-1993) in long double, over relaxation from dt/(2 tau) =
// 1e-6 to 1e4 and cells up to half the lattice speed. Errors are in units of
// eps times the size of the values that enter; prints the worst, exits 1
// beyond the bounds.
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

int main() {
  std::mt19937_64 rng(11);
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  const double eps = 2.2204460492503131e-16;
  double weq = 0, ws12 = 0, ws3 = 0, wsum = 0;
  for (int k = 0; k < 200000; k++) {
    InstDev in{};
    const double gamma = 1.2 + 0.45 * (0.5 + 0.5 * U(rng));
    in.K = 2.0 / (gamma - 1.0) - 2.0;
    in.Tc = 1.0;
    in.iTc = 1.0;
    in.RTc = 1.0;
    in.isRTc = 1.0;
    in.c = 1.0;
    in.dt = 1.0;
    point_consts(in.K, in.kq);
    const double amp = std::pow(10.0, -3.0 + 3.0 * (0.5 + 0.5 * U(rng)));
    auto cell = [&](double scale) {
      Macro m{};
      m.rho = 1.0 + 0.5 * scale * U(rng);
      m.T = 0.7 + 0.5 * scale * U(rng);
      m.ux = 0.5 * scale * U(rng);
      m.uy = 0.5 * scale * U(rng);
      return m;
    };
    Macro m = cell(amp), m3 = m;
    m3.rho *= 1 + 0.05 * U(rng);
    m3.ux += 0.02 * U(rng);
    m3.T *= 1 + 0.05 * U(rng);
    const double Pr = 0.6 + 0.4 * (0.5 + 0.5 * U(rng));
    const double af = std::pow(10.0, -6.0 + 10.0 * (0.5 + 0.5 * U(rng))), af3 = af * std::pow(2.0, U(rng));
    m.itf = 2 * af;
    m.ith = m.itf * Pr;
    m.ithf = m.itf * (Pr - 1.0);
    m3.itf = 2 * af3;
    m3.ith = m3.itf * Pr;
    m3.ithf = m3.itf * (Pr - 1.0);
    const PointEq e = point_eq(in, m), e3 = point_eq(in, m3);
    const EqIn<double> q = eq_inputs<double>(in, m);
    const Relax12 r = make_relax12(in, m);
    const Relax3 r3 = make_relax3(in, m, m3);
    double f2s[kQ], h2s[kQ], sm = 0;
    each_dir(
        [&](auto Ic) {
          constexpr int I = decltype(Ic)::value;
          double fe, he, fc, hc, fe3, he3;
          eq_point<I>(in.kq, e, fe, he);
          eq_point<I>(in.kq, e3, fe3, he3);
          eq_dir<I>(q, fc, hc);
          // the polynomials' terms at these cells are below 8 (f) and 200 (h)
          weq = std::fmax(weq, std::fmax(std::fabs(fe - fc) / (8 * eps), std::fabs(he - hc) / (200 * eps)));
          const double f = fe * (1 + 0.1 * amp * U(rng)), h = he * (1 + 0.1 * amp * U(rng));
          const double dF = 0.05 * fe * U(rng), dH = 0.05 * he * U(rng);
          double f2, h2, f3, h3;
          point_s12(r, e, lat_x(I), lat_y(I), f, h, fe, he, f2, h2);
          point_s3(r3, e, e3, lat_x(I), lat_y(I), f2, h2, dF, dH, fe, he, fe3, he3, f3, h3);
          const LD hdt = 0.5L, itf = m.itf, ith = m.ith, ithf = m.ithf, a = hdt * itf, b = hdt * ith;
          const LD eu = (LD)lat_x(I) * m.ux + (LD)lat_y(I) * m.uy;
          const LD f1 = (f + a * fe) / (1 + a), h1 = (h - hdt * ithf * eu * (fe - f1) + b * he) / (1 + b);
          const LD F2 = (f - a * (fe - f1) + a * fe) / (1 + a);
          const LD H2 = (h - hdt * (eu * ithf * (fe - F2) - eu * ithf * (fe - f1)) - b * (he - h1) + b * he) / (1 + b);
          const LD a3 = hdt * (LD)m3.itf, b3 = hdt * (LD)m3.ith, c3 = hdt * (LD)m3.ithf;
          const LD eu3 = (LD)lat_x(I) * m3.ux + (LD)lat_y(I) * m3.uy;
          const LD F3 = (f - dF + a * (fe - F2) + a3 * fe3) / (1 + a3);
          const LD H3 = (h - dH - hdt * ithf * eu * (fe - F2) - c3 * eu3 * (fe3 - F3) + b * (he - H2) + b3 * he3) / (1 + b3);
          const LD sf = std::fabs(f) + std::fabs(fe) + std::fabs(fe3), sh = std::fabs(h) + std::fabs(he) + std::fabs(he3) + sf;
          ws12 = std::fmax(ws12, (double)(std::fabs(f2 - F2) / (sf * eps)));
          ws12 = std::fmax(ws12, (double)(std::fabs(h2 - H2) / (sh * eps)));
          ws3 = std::fmax(ws3, (double)(std::fabs(f3 - F3) / (sf * eps)));
          ws3 = std::fmax(ws3, (double)(std::fabs(h3 - H3) / (sh * eps)));
          f2s[I] = f2;
          h2s[I] = h2;
          sm += std::fabs(f2) + std::fabs(h2);
        },
        std::make_integer_sequence<int, kQ>{});
    const Sums s = cell_sums(f2s, h2s, true);
    LD t[4] = {0, 0, 0, 0};
    for (int i = 0; i < kQ; i++) {
      t[0] += f2s[i];
      t[1] += (LD)f2s[i] * lat_x(i);
      t[2] += (LD)f2s[i] * lat_y(i);
      t[3] += h2s[i];
    }
    const double d = std::fmax(std::fmax(std::fabs((double)(s.m - t[0])), std::fabs((double)(s.px - t[1]))),
                               std::fmax(std::fabs((double)(s.py - t[2])), std::fabs((double)(s.e - t[3]))));
    wsum = std::fmax(wsum, d / (2 * sm * eps));
  }
  std::printf("worst error / (eps size): equilibria %.2f, stages 1-2 %.2f, stage 3 %.2f, sums %.2f\n", weq, ws12, ws3, wsum);
  // an equilibrium is some 20 roundings, a stage some 10 on top of its inputs
  // (stage 3: the stage-2 rounding times at most af/(1 + af3) <= 2), a sum 13
  return weq < 20 && ws12 < 16 && ws3 < 32 && wsum < 13 ? 0 : 1;
}
