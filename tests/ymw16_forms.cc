// Built and run by test_ymw16_forms.py: the short form of the YMW16 density
// (hamx_ymw16.h, compiled for the host with the device's helper functions
// restated below) against the literal one (hamx_models.h) over the parameters
// that ymw16_ordinary sends to it.
#include <cmath>
#include <cstdio>
#include <initializer_list>
#include <random>
#include <vector>

#define __device__
using std::fabs;
using std::fmax;
using std::fmin;

namespace hamx {
inline double rcp_f64(double x) { return 1. / x; }
inline double rsqrt_f64(double x) { return 1. / std::sqrt(x); }
inline double sqrt_pos(double x) { return std::sqrt(x); }
// the device's range: beyond it the reduction's remainder is meaningless
inline double exp_fast(double x) { return fabs(x) < 1e15 ? std::exp(x) : NAN; }
} // namespace hamx

#include "hamx_ymw16.h"
#include "hamx_models.h"

using namespace hamx;

int main(int, char **argv) {
  double p[73];
  std::FILE *f = std::fopen(argv[1], "rb");
  if (!f || std::fread(p, sizeof(double), 73, f) != 73)
    return 2;
  std::fclose(f);
  std::mt19937_64 gen(1);
  std::uniform_real_distribution<double> U(0, 1);
  struct Point {
    double x, y, z;
  };
  std::vector<Point> pts;
  const double kpc = cgs::kpc;
  auto around = [&](double x0, double lo, double decades, int n) {
    for (int i = 0; i < n; ++i) {
      const double s = std::pow(10., lo + decades * U(gen)) * kpc;
      const double x = x0 + (2 * U(gen) - 1) * s, y = (2 * U(gen) - 1) * s;
      pts.push_back({x, y, (2 * U(gen) - 1) * s});
    }
  };
  around(-8.3 * kpc, -3., 3.3, 6000); // the nebulae about the Sun
  around(0., -2., 2.5, 2000);         // the Galactic centre
  for (int i = 0; i < 6000; ++i) {
    const double x = (U(gen) * 40 - 20) * kpc, y = (U(gen) * 40 - 20) * kpc;
    pts.push_back({x, y, (U(gen) * 20 - 10) * kpc * std::pow(U(gen), 3)});
  }
  long sets = 0, bad = 0;
  auto run = [&](const double *q, const char *what, int i, double v) {
    if (!ymw16_ordinary(q))
      return;
    ++sets;
    const Ymw16 m = ymw16_fold(q);
    long finite = 0;
    double worst = 0.;
    for (const Point &t : pts) {
      const double r2 = t.x * t.x + t.y * t.y, inv = 1. / std::sqrt(r2);
      const double a = ymw16_density(m, t.x, t.y, t.z, r2 * inv, inv);
      const double b = tereg_ymw16_eval(q, t.x, t.y, t.z);
      if (std::isfinite(a) != std::isfinite(b))
        ++finite;
      else if (std::isfinite(a) && a != b)
        worst = fmax(worst, fabs(a - b) / fmax(fabs(b), 1e-250));
    }
    if (finite || worst > 1e-9) {
      ++bad;
      std::printf("%s %d = %g: worst %.2e, finite in one form only at %ld points\n", what, i, v,
                  worst, finite);
    }
  };
  run(p, "template", -1, 0.);
  std::vector<double> q(p, p + 73);
  for (int i = 0; i < 73; ++i)
    for (double v : {0., 1., 1e15, 3e16, 1e18, 1e20, 1e22, 1e24, -1e22, 1e-5, 1e-4, 1e-3, 1e-2, .1,
                     10., 1e2, -1e2, 1e3, -1e3, 1e4, -1e23, std::nan(""), HUGE_VAL}) {
      q[i] = v;
      run(q.data(), "parameter", i, v);
      q[i] = p[i];
    }
  // no disks: the bubble's smallest terms decide
  q[6] = 20 * cgs::pc;
  q[9] = 0.;
  for (int i = 12; i < 17; ++i)
    q[i] = 0.;
  for (int i : {61, 62, 66, 67})
    q[i] = 1.3 * cgs::pc;
  run(q.data(), "bubble", 0, 0.);
  std::printf("%ld parameter sets, %ld differ\n", sets, bad);
  return bad != 0;
}
