// The YMW16 thermal electron density (tereg_ymw16.cc:10-333) as the marches
// evaluate it: the model of tereg_ymw16_eval (hamx_models.h, the same
// parameters, cuts and choice between components) in far fewer FP64
// instructions, which bound the march: with the literal form it took about
// 4500 VALU instructions per sample inside the limits.  Measured on 3 shells
// up to nside 128 with 200x200x40 random grids: generic march 12.7 -> 7.8 ms
// per pass with this evaluator, 4.8 ms in the specialised march.  Within 8e-14
// of the literal form at any of 8e6 random points (8e-15 rms), the difference
// largest where the Gum shell's angles cancelled.
//
// * sech^2 v = 4 e / (1 + e)^2 with e = exp(-2 |v|) in place of a cosh and a
//   division; factors of one product share the division.
// * cos(atan2(y, x)) = x / r in the warp; an arm's second winding is its
//   first times exp(2 pi tan pitch).
// * The Gum shell needs no angle: with Q = the squared distance from its axis,
//   Z = dz^2, S = k^2 Q + Z, its tan(theta)^2 = Z / Q construction
//   (zp, xyp, alpha in the model) gives
//     D^2 = (sqrt(S) - a k)^2 S / (k^4 Q + Z).
// * The Local Bubble's and Loop I's angles are evaluated only where their
//   other factors leave something: the bubble's components are dropped where
//   their exponents sum to more than 150 and what is left of them is below the
//   disks' density (`lb_floor`), the least that the bubble is compared with;
//   without disks, where the exponentials are 0.
#pragma once

#include "hamx_cgs.h"
#include "hamx_math.h"

namespace hamx {

// Parameters folded on the host (ymw16_fold), lengths in cm.
struct Ymw16 {
  double r_warp, gamma_w, r0;
  double bd, m2_ad, n1, z_thick, m2_h1; // m2_x: -2 / x
  double b2, m2_a2, n2, k2, m2_k2;
  double b2s, m2_aa, ka, m2_ka, arms_rmax, arms_amax;
  double ele[4], m2_w[4], smax[4], rref[4], phi[4], tp[4], cp[4], wind[4];
  double ncn, thetacn, inv_wcn, nsg, thetasg, inv_wsg;
  double ngc, gc_r2, inv_agc2, gc_zmax, m2_hgc;
  double ngn, gum_d2, inv_wgn2, k2g, k4g, akg; // k^2, k^4, a k
  double gum_x, gum_y, gum_z;
  double j_lb, lb_floor;
  double lb_n[2], lb_theta[2], lb_det[2], lb_w[2], lb_h[2];
  double nli, li_rmax, li_rli, inv_wli, li_tmax, inv_dli, li_cos, li_sin;
};

// The parameters for which the short forms below hold: finite, every scale
// positive and such that the exponents stay within exp_fast's range (|x| below
// 1e15), arms of a pitch short of a right angle, a Gum shell with a radius.
// Others (a scale height of 0 to switch a component off, say) take the literal
// form, in the generic march: there 1 / cosh(inf), the sign of a negative scale
// and a component's NaN have their own meaning.
inline bool ymw16_ordinary(const double *p) {
  auto in = [p](int i, double lo, double hi) { return p[i] >= lo && p[i] <= hi; };
  for (int i = 0; i < 73; ++i)
    if (!in(i, -1e25, 1e25))
      return false;
  for (int i : {3, 6, 7, 17, 18, 19, 20, 42, 51, 52, 54, 55, 61, 62, 66, 67, 70}) // lengths
    if (!in(i, 1e15, 1e24))
      return false;
  for (int i : {10, 43, 46, 49, 60, 65, 71}) // factors and angles
    if (!in(i, 1e-5, 1e5))
      return false;
  for (int i : {45, 48, 59, 64, 72}) // directions, in degrees
    if (!in(i, -1e6, 1e6))
      return false;
  for (int i = 0; i < 4; ++i)
    if (!in(27 + i, -1e3, 1e3) || !in(32 + i, -1e2, 1e2) || !in(37 + i, 1e-3, 1e3))
      return false;
  return in(1, -1e23, 1e23) && in(56, 1e-3, 1e3);
}

inline Ymw16 ymw16_fold(const double *p) {
  Ymw16 y;
  const double rad = cgs::rad, pc = cgs::pc;
  y.r_warp = p[0];
  y.r0 = p[1];
  y.gamma_w = p[2];
  y.bd = p[4];
  y.m2_ad = -2. / p[3];
  y.n1 = p[5];
  y.z_thick = 10. * p[6];
  y.m2_h1 = -2. / p[6];
  y.b2 = p[8];
  y.m2_a2 = -2. / p[7];
  y.n2 = p[9];
  y.k2 = p[10];
  y.m2_k2 = -2. / p[10];
  y.b2s = p[11];
  y.m2_aa = -2. / p[42];
  y.ka = p[43];
  y.m2_ka = -2. / p[43];
  y.arms_rmax = 10. * p[3];
  y.arms_amax = 10. * p[42];
  for (int i = 0; i < 4; ++i) {
    y.ele[i] = p[12 + i];
    y.m2_w[i] = -2. / p[17 + i];
    y.smax[i] = 10. * p[17 + i];
    y.rref[i] = p[22 + i];
    y.phi[i] = p[27 + i];
    y.tp[i] = p[32 + i];
    y.cp[i] = p[37 + i];
    y.wind[i] = std::exp(2. * cgs::pi * p[32 + i]);
  }
  y.ncn = p[44];
  y.thetacn = p[45];
  y.inv_wcn = 1. / p[46];
  y.nsg = p[47];
  y.thetasg = p[48];
  y.inv_wsg = 1. / p[49];
  y.ngc = p[50];
  y.gc_r2 = 10. * p[51] * p[51];
  y.inv_agc2 = 1. / (p[51] * p[51]);
  y.gc_zmax = 10. * p[52];
  y.m2_hgc = -2. / p[52];
  const double lc = 264. * rad, bc = -4. * rad, dc = 450. * pc;
  y.gum_x = dc * std::cos(bc) * std::sin(lc);
  y.gum_y = p[1] - dc * std::cos(bc) * std::cos(lc);
  y.gum_z = dc * std::sin(bc);
  y.ngn = p[53];
  y.gum_d2 = 10. * p[54] * p[54];
  y.inv_wgn2 = 1. / (p[54] * p[54]);
  y.k2g = p[56] * p[56];
  y.k4g = y.k2g * y.k2g;
  y.akg = p[55] * p[56];
  y.j_lb = p[57];
  // both components' sech^2 products at exponents of -150 and below
  y.lb_floor = 128. * std::exp(-150.) * std::fmax(std::fabs(p[58]), std::fabs(p[63]));
  for (int c = 0; c < 2; ++c) {
    const double *q = p + 58 + 5 * c;
    y.lb_n[c] = q[0];
    y.lb_theta[c] = q[1];
    y.lb_det[c] = q[2];
    y.lb_w[c] = q[3];
    y.lb_h[c] = q[4];
  }
  y.nli = p[68];
  y.li_rli = p[69];
  y.li_rmax = 10. * p[70];
  y.inv_wli = 1. / p[70];
  y.li_tmax = 10. * p[71];
  y.inv_dli = 1. / p[71];
  y.li_cos = std::cos(p[72] * rad);
  y.li_sin = std::sin(p[72] * rad);
  return y;
}

// 4 e / (1 + e)^2 = sech^2(log(e) / 2)
__device__ inline double sech2_of(double e) {
  const double d = 1. + e;
  return 4. * e * rcp_f64(d * d);
}

// The spiral arms (tereg_ymw16.cc:118-210): gd the radial factor shared with
// the thin disk, zh = z / h with h the thin disk's scale at r for k = 1.
__device__ inline double ymw16_arms(const Ymw16 &m, double x, double y, double r, double gd,
                                    double zh) {
  if ((r > m.bd && (r - m.bd) > m.arms_rmax) || zh > 10. * m.ka || (r - m.b2s) > m.arms_amax)
    return 0.;
  const double e1 = exp_fast(m.m2_ka * fabs(zh)), e2 = exp_fast(m.m2_aa * fabs(r - m.b2s));
  const double d = (1. + e1) * (1. + e2);
  const double scaling = gd * (16. * e1 * e2) * rcp_f64(d * d);
  double theta = atan2(y, x);
  if (theta < 0)
    theta += cgs::twopi;
  double ne = 0.;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    double dphi = theta - m.phi[i];
    if (dphi < 0)
      dphi += cgs::twopi;
    const double a = m.rref[i] * exp_fast(dphi * m.tp[i]);
    const double smin = fmin(fabs(a - r), fabs(a * m.wind[i] - r)) * m.cp[i];
    if (smin > m.smax[i])
      continue;
    double arm = m.ele[i] * sech2_of(exp_fast(m.m2_w[i] * smin));
    if (i == 2) {
      const double th = theta * cgs::rad;
      const double sg = (th - m.thetasg) * m.inv_wsg;
      const double cn = (th - m.thetacn) * m.inv_wcn;
      const double g_cn =
          (r > 6 * cgs::kpc && th > m.thetacn) ? m.ncn : m.ncn * exp_fast(fmax(-(cn * cn), -745.));
      arm *= (1. - m.nsg * exp_fast(fmax(-(sg * sg), -745.))) * (1. + g_cn);
    }
    ne += arm;
  }
  return ne * scaling;
}

// Galactocentric (px, py, pz); r and inv_r the cylindrical radius and its
// reciprocal (0 on the axis).
__device__ inline double ymw16_density(const Ymw16 &m, double px, double py, double pz, double r,
                                       double inv_r) {
  const double x = py, y = -px;
  double z = pz;
  if (r >= m.r_warp)
    z -= m.gamma_w * (r - m.r_warp) * (r > 0. ? x * inv_r : 1.);
  if (x * x + y * y + z * z > 625. * cgs::kpc * cgs::kpc)
    return 0.;
  const double az = fabs(z);
  const double gd = r > m.bd ? sech2_of(exp_fast(m.m2_ad * (r - m.bd))) : 1.;
  const double n_thick =
      z > m.z_thick ? 0. : m.n1 * gd * sech2_of(exp_fast(m.m2_h1 * az));
  // thin disk (tereg_ymw16.cc:97-115) and arms share the scale height
  const double zh = z * rcp_f64(32 * cgs::pc + 1.6e-3 * r + (4.e-7 / cgs::pc) * r * r);
  double n_thin = 0.;
  if (!(zh > 10. * m.k2)) {
    const double e1 = exp_fast(m.m2_a2 * fabs(r - m.b2)), e2 = exp_fast(m.m2_k2 * fabs(zh));
    const double d = (1. + e1) * (1. + e2);
    n_thin = m.n2 * gd * (16. * e1 * e2) * rcp_f64(d * d);
  }
  const double n_arm = ymw16_arms(m, x, y, r, gd, zh);
  // Galactic centre (tereg_ymw16.cc:213-229)
  double n_gc = 0.;
  {
    const double dx = x - 50. * cgs::pc, dz = z + 7. * cgs::pc, R2 = dx * dx + y * y;
    if (!(R2 > m.gc_r2) && !(fabs(dz) > m.gc_zmax))
      n_gc = m.ngc * exp_fast(-R2 * m.inv_agc2) * sech2_of(exp_fast(m.m2_hgc * fabs(dz)));
  }
  // Gum Nebula (tereg_ymw16.cc:232-270)
  double n_gum = 0.;
  if (!(y < 0 || x > 0)) {
    const double dx = x - m.gum_x, dy = y - m.gum_y, dz = z - m.gum_z;
    const double Q = dx * dx + dy * dy, Z = dz * dz, S = m.k2g * Q + Z;
    const double t = S * rsqrt_f64(S) - m.akg;
    const double D2 = t * t * S * rcp_f64(m.k4g * Q + Z);
    if (!(D2 > m.gum_d2))
      n_gum = m.ngn * exp_fast(-D2 * m.inv_wgn2);
  }
  // Local Bubble (tereg_ymw16.cc:46-48,273-307)
  const double Rlb = 110. * cgs::pc;
  const double u = (y - 8.34 * cgs::kpc) * 0.94 - 0.34 * z;
  const double rlb = sqrt_pos(u * u + x * x);
  const double n_disk = n_thin > n_arm ? n_thin : n_arm;
  const bool bubble = rlb < Rlb;
  const double n0 = (bubble ? m.j_lb * n_thick : n_thick) + n_disk;
  double n_lb = 0.;
  if (!(y < 0)) {
    const double dr = rlb - Rlb, skip = n0 > m.lb_floor ? 150. : 1500.;
    double ex[2];
    bool any = false;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      ex[c] = 2. * (fabs(dr) / m.lb_w[c] + az / m.lb_h[c]);
      any = any || !(ex[c] > skip);
    }
    if (any) {
      const double l = atan2(x, m.r0 - y) / cgs::rad;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const double dl = fmin(fabs(l + 360. - m.lb_theta[c]), fabs(m.lb_theta[c] - l));
        if (ex[c] > skip ||
            !(dl < 10. * m.lb_det[c] || dr < 10. * m.lb_w[c] || z < 10. * m.lb_h[c]))
          continue;
        n_lb += m.lb_n[c] * sech2_of(exp_fast(-2. * (dl / m.lb_det[c]))) *
                sech2_of(exp_fast(-2. * (fabs(dr) / m.lb_w[c]))) *
                sech2_of(exp_fast(-2. * (az / m.lb_h[c])));
      }
    }
  }
  // Loop I (tereg_ymw16.cc:310-333)
  double n_li = 0.;
  if (!(y < 0)) {
    const double dx = x + 10.156 * cgs::pc, dy = y - 8106.207 * cgs::pc, dz = z - 10.467 * cgs::pc;
    const double R2 = dx * dx + dy * dy + dz * dz;
    const double edge = m.li_rli + m.li_rmax;
    if (!(R2 > edge * edge * (1. + 1e-12))) {
      const double rLI = sqrt(R2);
      const double theta = acos((dx * m.li_cos + dz * m.li_sin) / rLI) / cgs::rad;
      if (!(theta > m.li_tmax || (rLI - m.li_rli) > m.li_rmax)) {
        const double a = (rLI - m.li_rli) * m.inv_wli, b = theta * m.inv_dli;
        n_li = m.nli * exp_fast(-(a * a) - b * b);
      }
    }
  }
  if (n_lb > n0 && (bubble || n_lb > n_gum))
    return n_lb;
  if (n_gum > n0)
    return n_gum;
  return n_li > n0 ? n_li : n0 + n_gc;
}

} // namespace hamx
