// The synchrotron emissivities of an imported CRE flux grid
// (sync_emissivity_t and _p, integrator.cc:286-325 and 355-394; the flux by
// CREfield::read_grid_num, cre.cc:144-199).
//
// Per sample, over the nE - 1 energy bins: the mean x of the bin's ends (above
// 100 the bin is skipped), the mean of flux / beta at its ends, F(x) and G(x)
// (hamx_sync.h), the midpoint sums, then the fore factor.  Bound by the three
// pipes together -- FP64, LDS (the coefficients) and the vector memory path
// (the flux) -- so each bin's share of each is kept small: about 60 FP64
// instructions, 8 16-byte LDS reads, 4 16-byte loads.
//
// * x = x_fact c_i and ln x = ln x_fact + ln c_i, with c_i and its logarithm
//   tabulated on the host; J_tot and J_pol share x (their x_fact differ in
//   rounding alone).  x falls with the energy, so a wavefront starts at the
//   first bin that any of its lanes keeps.
// * The eight corner weights are formed once per sample, and two energies are
//   loaded at a time from each corner.
#pragma once

#include "hamx_march.h"
#include "hamx_sync.h"

namespace hamx {

// Energy tables at gr.cre_tab, nE doubles each: per bin i the half mean of
// 1/E^2 at its ends, its logarithm and half the bin's width; per energy 1 / beta.
enum CreTab { kCreC = 0, kCreLnC = 1, kCreHalfDE = 2, kCreInvBeta = 3 };

// Two consecutive doubles, 8-byte aligned.
struct __attribute__((packed, aligned(8))) FluxPair {
  double a, b;
};

__device__ inline void cre_grid_emissivity(const Phys &ph, const Grids &gr, const Vec3 &pos,
                                           double b_per, const double2 *stab, double &jt,
                                           double &jp) {
  jt = 0.;
  jp = 0.;
  Cell c;
  const double ab = fabs(b_per);
  if (ab == 0. || !grid_cell(gr.g_cre, pos, c))
    return; // no field: every bin's x is infinite; outside the grid: no flux
  const uint32_t nE = static_cast<uint32_t>(gr.cre_nE);
  const double *tc = gr.cre_tab + kCreC * nE, *tl = gr.cre_tab + kCreLnC * nE;
  const double *td = gr.cre_tab + kCreHalfDE * nE, *tb = gr.cre_tab + kCreInvBeta * nE;
  const double xf = ph.xft_num / (ph.three_qe * ab);
  const double lx = log_pos(xf);
  // the first pair of bins that any lane keeps (uniform: the energy loop then
  // reads its tables with scalar loads)
  uint32_t q = 0;
  while (2 * q + 2 < nE && !__ballot(xf * tc[2 * q + 2 < nE - 1 ? 2 * q + 1 : nE - 2] <= 100.))
    ++q;
  const uint64_t sz = nE, sy = gr.g_cre.nz * sz, sx = gr.g_cre.ny * sy;
  const double *f0 = gr.cre + c.idx * sz, *f1 = f0 + sy, *f2 = f0 + sx, *f3 = f2 + sy;
  const double x1 = 1. - c.xd, y1 = 1. - c.yd, z1 = 1. - c.zd;
  const double w0 = x1 * y1, w1 = x1 * c.yd, w2 = c.xd * y1, w3 = c.xd * c.yd;
  const double wa[4] = {w0 * z1, w1 * z1, w2 * z1, w3 * z1};
  const double wb[4] = {w0 * c.zd, w1 * c.zd, w2 * c.zd, w3 * c.zd};
  const double *fp[4] = {f0, f1, f2, f3};
  double Jt = 0., Jp = 0.;
  auto bin = [&](uint32_t i, double flux2) { // flux2: the sum over the bin's ends
    const double x = xf * tc[i];
    double F, G;
    sync_fg(stab, lx + tl[i], x, F, G);
    const double m = !(x > 100.) ? flux2 * td[i] : 0.;
    Jt = fma(!(x > 100.) ? F : 0., m, Jt);
    Jp = fma(!(x > 100.) ? G : 0., m, Jp);
  };
  double last = 0.;
  bool have = false;
  for (uint32_t e = 2 * q; e < nE; e += 2) {
    double g0 = 0., g1 = 0.;
    if (e + 1 < nE) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const FluxPair a = *reinterpret_cast<const FluxPair *>(fp[k] + e);
        const FluxPair b = *reinterpret_cast<const FluxPair *>(fp[k] + sz + e);
        g0 = fma(b.a, wb[k], fma(a.a, wa[k], g0));
        g1 = fma(b.b, wb[k], fma(a.b, wa[k], g1));
      }
      g1 *= tb[e + 1];
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        g0 = fma(fp[k][sz + e], wb[k], fma(fp[k][e], wa[k], g0));
    }
    g0 *= tb[e];
    if (have)
      bin(e - 1, last + g0);
    if (e + 1 < nE)
      bin(e, g0 + g1);
    last = g1;
    have = true;
  }
  const double fore = ph.fore_num * ab / ph.fore_den;
  jt = Jt * fore;
  jp = Jp * fore;
}

} // namespace hamx
