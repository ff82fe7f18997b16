// Host check of the conserved sums of the equilibria of FP64 storage
// (point_moments, point_eq, eq_point, uq_amd/csrc/lbm_point.hpp): every stage
// takes a cell's mass, momentum and energy from its equilibria, so over random
// cells of several gases the sums over the directions must give back those that
// went in, without a mean error that would add up from step to step. Prints
// mean and root mean square of the relative errors (momentum relative to the
// mass) in eps, exits 1 beyond the bounds.
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
  const double eps = 2.2204460492503131e-16;
  const int n = 200000;
  bool ok = true;
  for (double gamma : {1.1, 1.3, 1.4, 5.0 / 3.0, 2.0})
    for (double Tc : {1.0, 750.0, 733.1}) {
      std::mt19937_64 rng(7);
      std::uniform_real_distribution<double> U(0.0, 1.0);
      InstDev in{};
      in.K = 2.0 / (gamma - 1.0) - 2.0;
      in.R = Tc == 1.0 ? 1.0 : 287.0;
      in.Tc = Tc;
      in.RTc = in.R * in.Tc;
      in.iRTc = 1.0 / in.RTc;
      point_consts(in.K, in.kq);
      LD mean[4] = {}, sq[4] = {};
      for (int k = 0; k < n; k++) {
        const double rho = 0.1 + 1.4 * U(rng), t = 0.3 + 0.7 * U(rng), u = U(rng) - 0.5, v = U(rng) - 0.5;
        const Sums s{rho, rho * u, rho * v, rho * in.RTc * ((in.K + 2.0) * t + u * u + v * v) / 2.0};
        Macro m{};
        point_moments(in, s, m);
        const PointEq e = point_eq(in, m);
        LD o[4] = {};
        each_dir(
            [&](auto Ic) {
              constexpr int I = decltype(Ic)::value;
              double fe, he;
              eq_point<I>(in.kq, e, fe, he);
              o[0] += fe;
              o[1] += (LD)fe * lat_x(I);
              o[2] += (LD)fe * lat_y(I);
              o[3] += he;
            },
            std::make_integer_sequence<int, kQ>{});
        const LD d[4] = {(o[0] - s.m) / s.m, (o[1] - s.px) / s.m, (o[2] - s.py) / s.m, (o[3] - s.e) / s.e};
        for (int j = 0; j < 4; j++) {
          mean[j] += d[j] / n;
          sq[j] += d[j] * d[j] / n;
        }
      }
      std::printf("gamma %.2f Tc %g: mean (rms) in eps:", gamma, Tc);
      const char* names[4] = {"mass", "x momentum", "y momentum", "energy"};
      for (int j = 0; j < 4; j++) {
        const double a = (double)mean[j] / eps, r = (double)std::sqrt(sq[j]) / eps;
        std::printf(" %s %+.3f (%.2f)", names[j], a, r);
        // the mean of n errors of 1 to 2 eps lies within 0.01 eps of none; a
        // constant rounded to one side brings up to half an eps
        ok = ok && std::fabs(a) <= 0.05 && r <= 2.0;
      }
      std::printf("\n");
    }
  return ok ? 0 : 1;
}
