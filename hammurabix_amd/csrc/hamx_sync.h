// The synchrotron kernels of the CRE grid emissivities on the device,
// replacing gsl_sf_synchrotron_1 / _2 (integrator.cc:321,390):
//   F(x) = x int_x^inf K_5/3(t) dt,   G(x) = x K_2/3(x),   0 < x <= 100.
// F = exp(P(u) - x) and G = F R(u), with P(u) = ln F + x and R(u) = G / F in
// u = ln x.  From u = ln 100 down to ln 100 - 18 (x = 1.5e-6) both are degree-8
// polynomials on segments of width 1/4 (hamx_sync_fine.h), below that piecewise
// Chebyshev series (hamx_synchrotron.h: 12 segments of width 4, one Clenshaw
// loop for both series); below the last segment (x < 1.8e-23) F is its leading
// term 2^(2/3) Gamma(2/3) x^(1/3) and R = 1/2.
#pragma once

#include <hip/hip_runtime.h>

#include "hamx_math.h"
#include "hamx_sync_fine.h"
#include "hamx_synchrotron.h"

namespace hamx {

// The short segments' table in LDS, one {P, R} pair per coefficient.
constexpr int kSyncTab = sync_tab::kFineSeg * (sync_tab::kFineSegDeg + 1);

__device__ inline void load_sync_tab(double2 *dst) {
  const double *src = &sync_tab::kFineTab[0][0][0];
  for (int i = threadIdx.x; i < kSyncTab; i += blockDim.x)
    dst[i] = make_double2(src[2 * i], src[2 * i + 1]);
}

// Below the short segments: the Chebyshev tables, read where they lie (few
// samples come here; a call would cost the march its registers).  Their rows above
// u = ln 100 - 17, which the short segments took over, are those that the CPU test
// of the tables reads.
__device__ inline void sync_fg_low(double u, double x, double &F, double &G) {
  using namespace sync_tab;
  const double dtop = kUTop - u, fine_span = kFineN * kFineW;
  if (dtop >= fine_span + kCoarseN * kCoarseW) {
    F = exp_fast(kLnF0 + u / 3.);
    G = kR0 * F;
    return;
  }
  // the index is clamped in floating point (fmax drops a NaN), so every table
  // read stays inside the table whatever x is
  const int sc = static_cast<int>(fmin(fmax((dtop - fine_span) / kCoarseW, 0.), kCoarseN - 1.));
  const int s = kFineN + sc;
  const double lo = kUTop - fine_span - (sc + 1) * kCoarseW;
  const double t = 2. * (u - lo) / kCoarseW - 1.;
  // Clenshaw recurrences for sum_k c_k T_k(t), both series together
  double p1 = 0., p2 = 0., r1 = 0., r2 = 0.;
#pragma unroll 1
  for (int k = kCoarseDeg; k >= 1; --k) {
    const double p0 = kF[s][k] + 2. * t * p1 - p2;
    const double r0 = kR[s][k] + 2. * t * r1 - r2;
    p2 = p1;
    p1 = p0;
    r2 = r1;
    r1 = r0;
  }
  F = exp_fast(kF[s][0] + t * p1 - p2 - x);
  G = F * (kR[s][0] + t * r1 - r2);
}

// F(x) and G(x), x <= 100, with u = ln x given by the caller: the march forms
// it as a per-sample logarithm plus a per-bin constant instead of a logarithm
// per bin.  P changes by less than the error in u times 5/6, so u may carry a
// few ulps of error.  `tab` as load_sync_tab lays it out.
__device__ inline void sync_fg(const double2 *tab, double u, double x, double &F, double &G) {
  using namespace sync_tab;
  const double d = (kUTop - u) * (1. / kFineSegW);
  if (!(d < kFineSeg)) {
    sync_fg_low(u, x, F, G);
    return;
  }
  const int s = static_cast<int>(fmax(d, 0.)); // 0 for x a rounding above 100
  const double v = 2. * (static_cast<double>(s) - d) + 1.;
  const double2 *c = tab + s * (kFineSegDeg + 1);
  double P = c[kFineSegDeg].x, R = c[kFineSegDeg].y;
#pragma unroll
  for (int k = kFineSegDeg - 1; k >= 0; --k) {
    P = fma(P, v, c[k].x);
    R = fma(R, v, c[k].y);
  }
  F = exp_fast(P - x);
  G = F * R;
}

} // namespace hamx
