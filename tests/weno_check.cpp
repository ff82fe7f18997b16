// Host check of the FP64 face reconstruction (weno5<double>,
// uq_amd/csrc/lbm_device.hpp) and of the reciprocal it and the pointwise stages
// take, against long double: lines of random values, smooth (differences 1e-4 to
// 1e-1), rough (0.5 to 1.5), or between 0.8 and 1.2 with a jump of ratio 4 to 1e6
// (up or down) at each place of the line, so that every candidate of the smooth
// side is above 0.3. The face value follows the smooth side of a jump, so its error is held
// to its own size, not to the jump's: root mean square below 1.5 eps (the last
// sum and the product with the speed round it twice, the correction, which is
// no larger than the differences of the smooth side, by less). Prints the worst
// of each kind, exits 1 beyond the bounds.
#include <cmath>
#include <cstdio>
#include <random>

#include "../uq_amd/csrc/lbm_device.hpp"

using namespace uqlbm;
typedef long double LD;

static LD exact(LD v, const LD* s) {
  LD q[5];
  for (int k = 0; k < 5; k++) q[k] = v * s[k];
  const LD b[3] = {13 / LD(12) * powl(q[0] - 2 * q[1] + q[2], 2) + powl(q[0] - 4 * q[1] + 3 * q[2], 2) / 4,
                   13 / LD(12) * powl(q[1] - 2 * q[2] + q[3], 2) + powl(q[1] - q[3], 2) / 4,
                   13 / LD(12) * powl(q[2] - 2 * q[3] + q[4], 2) + powl(3 * q[2] - 4 * q[3] + q[4], 2) / 4};
  const LD r[3] = {(2 * q[0] - 7 * q[1] + 11 * q[2]) / 6, (-q[1] + 5 * q[2] + 2 * q[3]) / 6,
                   (2 * q[2] + 5 * q[3] - q[4]) / 6};
  const LD d[3] = {LD(1) / 10, LD(6) / 10, LD(3) / 10};
  LD num = 0, den = 0;
  for (int k = 0; k < 3; k++) {
    const LD a = d[k] / powl(LD(1e-6) + b[k], 2);
    num += a * r[k];
    den += a;
  }
  return num / den;
}

int main() {
  std::mt19937_64 rng(5);
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  const double eps = 2.2204460492503131e-16;
  bool ok = true;
  // kind 0: smooth, 1: rough, 2: jump below line position `at`
  auto lines = [&](int kind, int at, double ratio, const char* what) {
    double sum = 0, most = 0;
    const int n = 20000;
    for (int k = 0; k < n; k++) {
      double s[5];
      const double amp = kind == 0 ? std::pow(10.0, -2.5 + 1.5 * U(rng)) : kind == 1 ? 0.5 : 0.2, base = 1.0 + (kind == 0 ? 0.4 * U(rng) : 0.0);
      for (int j = 0; j < 5; j++) {
        s[j] = base + amp * U(rng);
        if (kind == 2 && j >= at) s[j] *= ratio;
      }
      const double v = std::pow(10.0, 1.5 + 1.5 * U(rng));
      const LD t[5] = {s[0], s[1], s[2], s[3], s[4]};
      const LD e = exact(v, t);
      const double err = std::fabs((double)((weno5<double>(v, s[0], s[1], s[2], s[3], s[4]) - e) / e)) / eps;
      sum += err * err;
      most = std::fmax(most, err);
    }
    const double rms = std::sqrt(sum / n);
    std::printf("%-7s at %d ratio %8.2g: rms %.3g eps, most %.3g eps\n", what, at, ratio, rms, most);
    // a rough line's value may be small beside its points: no bound but for the smooth ones and jumps
    if (kind != 1) ok = ok && rms < 1.5;
  };
  lines(0, 0, 1, "smooth");
  lines(1, 0, 1, "rough");
  for (int at = 1; at < 5; at++)
    for (const double r : {4.0, 30.0, 400.0, 1e6}) {
      lines(2, at, r, "jump");
      lines(2, at, 1 / r, "jump");
    }
  // the device's reciprocal instruction is good to 2^-14 and better
  double worst = 0;
  for (int k = 0; k < 200000; k++) {
    const double x = std::pow(10.0, 24.0 * U(rng)), start = (1.0 / x) * (1.0 + U(rng) / 16384.0);
    worst = std::fmax(worst, std::fabs((double)(((LD)recip_steps(x, start) - 1 / (LD)x) * x)) / eps);
  }
  std::printf("reciprocal: most %.3g eps\n", worst);
  return ok && worst < 1.0 ? 0 : 1;
}
