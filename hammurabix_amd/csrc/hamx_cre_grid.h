// The synchrotron emissivities of an imported CRE flux grid
// (sync_emissivity_t and _p, integrator.cc:286-325 and 355-394; the flux by
// CREfield::read_grid_num, cre.cc:144-199).
//
// Per sample, over the nE - 1 energy bins: the mean x of the bin's ends (above
// 100 the bin is skipped), the mean of flux / beta at its ends, F(x) and G(x)
// (hamx_sync.h), the midpoint sums, then the fore factor.  Bound by FP64
// instructions (about half of the issue slots) and by the latency of the flux
// loads at three waves per SIMD; four waves spill (1.8 -> 2.3 ms).  Measured on
// 3 shells up to nside 64, 40x40x8 cells with 32 energies, ms per pass:
// literal form in the generic march 5.03; this file's 3.65; tables by scalar
// loads 2.9; loads ahead of the kernels 2.7; four wavefronts per ray 1.88.
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
  // in the constant address space (written before the launch, read by every
  // lane at one index): scalar loads, where a generic pointer's would be vector
  // loads, the march's stores after them possibly aliasing
  typedef const __attribute__((address_space(4))) double *ConstTab;
  const ConstTab tab = (ConstTab)gr.cre_tab;
  const ConstTab tc = tab + kCreC * nE, tl = tab + kCreLnC * nE;
  const ConstTab td = tab + kCreHalfDE * nE, tb = tab + kCreInvBeta * nE;
  const double xf = ph.xft_num / (ph.three_qe * ab);
  const double lx = log_pos(xf);
  // the first pair of bins that any lane keeps (uniform: the energy loop then
  // reads its tables with scalar loads)
  uint32_t q = 0;
  while (2 * q + 2 < nE && !__ballot(xf * tc[2 * q + 1] <= 100.))
    ++q;
  if (2 * q + 1 >= nE)
    return; // uniform: no bin is kept
  const uint64_t sz = nE, sy = gr.g_cre.nz * sz, sx = gr.g_cre.ny * sy;
  const double *f0 = gr.cre + c.idx * sz;
  const double *fp[4] = {f0, f0 + sy, f0 + sx, f0 + sx + sy};
  const double x1 = 1. - c.xd, y1 = 1. - c.yd, z1 = 1. - c.zd;
  const double w[4] = {x1 * y1, x1 * c.yd, c.xd * y1, c.xd * c.yd};
  const double wa[4] = {w[0] * z1, w[1] * z1, w[2] * z1, w[3] * z1};
  const double wb[4] = {w[0] * c.zd, w[1] * c.zd, w[2] * c.zd, w[3] * c.zd};
  // energies e and e + 1 from every corner; with an odd nE the last energy is
  // the second of the pair before it
  FluxPair ra[4], rb[4];
  auto load = [&](uint32_t e) {
    const uint32_t at = e + 1 < nE ? e : nE - 2;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      ra[k] = *reinterpret_cast<const FluxPair *>(fp[k] + at);
      rb[k] = *reinterpret_cast<const FluxPair *>(fp[k] + sz + at);
    }
  };
  double g0, g1;
  auto lerp = [&](uint32_t e) {
    const uint32_t at = e + 1 < nE ? e : nE - 2;
    g0 = g1 = 0.;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      g0 = fma(rb[k].a, wb[k], fma(ra[k].a, wa[k], g0));
      g1 = fma(rb[k].b, wb[k], fma(ra[k].b, wa[k], g1));
    }
    g0 *= tb[at];
    g1 *= tb[at + 1];
  };
  // F and G of a bin times half its width; false where the bin is skipped
  auto kernels = [&](uint32_t i, double &F, double &G) {
    const double x = xf * tc[i];
    sync_fg(stab, lx + tl[i], x, F, G);
    const double m = td[i];
    F *= m;
    G *= m;
    return !(x > 100.);
  };
  double Jt = 0., Jp = 0.;
  // a skipped bin's flux, which may be infinite or NaN, takes no part
  auto add = [&](bool on, double F, double G, double flux) {
    Jt = on ? fma(F, flux, Jt) : Jt;
    Jp = on ? fma(G, flux, Jp) : Jp;
  };
  double F, G;
  load(2 * q);
  bool on = kernels(2 * q, F, G);
  lerp(2 * q);
  add(on, F, G, g0 + g1);
  double last = g1;
  // the loads of a step are in flight while its two bins' kernels, which do
  // not depend on them, are evaluated
  for (uint32_t e = 2 * q + 2; e < nE; e += 2) {
    double F2 = 0., G2 = 0.;
    bool on2 = false;
    load(e);
    on = kernels(e - 1, F, G);
    if (e + 1 < nE)
      on2 = kernels(e, F2, G2);
    lerp(e);
    add(on, F, G, last + (e + 1 < nE ? g0 : g1));
    add(on2, F2, G2, g0 + g1);
    last = g1;
  }
  const double fore = ph.fore_num * ab / ph.fore_den;
  jt = Jt * fore;
  jp = Jp * fore;
}

} // namespace hamx
