// 3D fast mode's arithmetic of the constitutive update and the kinematics.
//
// Ordered mode and 2D evaluate the reference's expressions in the reference's
// order (mpmx_device.h). The nodal sums of 3D fast mode differ from them, and
// from run to run, by rounding (atomics), so its stress kernels may regroup: fused multiply-adds,
// reciprocals and square roots by Newton steps on the hardware's estimates, the
// velocity gradient by interpolating axis by axis on box cells, and the
// Mohr-Coulomb gradients in the basis (identity, deviator, Lode direction)
// instead of two 6-vectors and a 6x6 product each. FP64 throughout. What the
// Lode angle is sensitive to (j2, j3 and the two ratios formed from them, whose
// rounding the angle magnifies by 1 / sin 3 theta) keeps the reference's
// expressions bit for bit; against the reference's arithmetic on 5e5 random
// states (stresses up to 2e4 Pa) the new stresses differ by 1e-12 Pa in the mean
// and 3e-8 Pa at most, where moving the start stress by an ulp moves the
// reference's own result by up to 6e-6 Pa (tests/test_fast_return_host.py).
// Collapse (2.1M particles, half of them yielding): stress update 364 + 180 us
// (deferred return mappings, 1450 instructions a correction) -> 345 us in one
// kernel; slope (5.2M, elastic) 702 + 19 -> 541 us, 4.3 TB/s of compulsory
// bytes where a copy reaches 4.7.
#pragma once

#include "mpmx_device.h"

namespace mpmx {
namespace fast {

// 1 / x and 1 / sqrt(x) for normal x > 0 or < 0 (rsqrt: > 0): Newton steps on
// v_rcp_f64 / v_rsq_f64, within 1 ulp (two: the estimates hold 2^-14 or better).
MPMX_DEV double rcp(double x) {
#pragma clang fp contract(fast)
  double r = __builtin_amdgcn_rcp(x);
  r = r + r * (1.0 - x * r);
  r = r + r * (1.0 - x * r);
  return r;
}
MPMX_DEV double rsqrt(double x) {
#pragma clang fp contract(fast)
  double y = __builtin_amdgcn_rsq(x);
  double e = 1.0 - (x * y) * y;
  y = y + y * (e * (0.5 + 0.375 * e));
  e = 1.0 - (x * y) * y;
  y = y + y * (0.5 * e);
  return y;
}

// c[0] + c[1] z + ... + c[5] z^5
MPMX_DEV double poly6(const double* c, double z) {
#pragma clang fp contract(fast)
  const double z2 = z * z;
  return (c[0] + c[1] * z) + z2 * ((c[2] + c[3] * z) + z2 * (c[4] + c[5] * z));
}

// acos v on [-1, 1], the half-angle form and polynomial of dmath::acos
MPMX_DEV double acos(double v) {
#pragma clang fp contract(fast)
  const double a = fabs(v);
  const bool far = a > 0.5;
  double z = v * v, y = v;
  if (far) {
    z = 0.5 - 0.5 * a;
    y = z > 0. ? z * rsqrt(z) : 0.;
  }
  const double* c = dmath::kAsin;
  const double z2 = z * z, z4 = z2 * z2;
  const double q0 = (c[0] + c[1] * z) + (c[2] + c[3] * z) * z2;
  const double q1 = (c[4] + c[5] * z) + (c[6] + c[7] * z) * z2;
  const double q2 = (c[8] + c[9] * z) + (c[10] + c[11] * z) * z2;
  const double s = y + (y * z) * (q0 + z4 * (q1 + z4 * (q2 + z4 * c[12])));
  if (!far) return dmath::kPio2Hi - (s - dmath::kPio2Lo);
  return v > 0. ? 2.0 * s : dmath::kPiHi - (2.0 * s - dmath::kPiLo);
}

// Invariants of a stress. s, c: sine and cosine of theta - pi/6, which lies in
// [-pi/6, pi/6] (no range reduction); all the angles of the yield functions
// and the potential are theta - pi/6 plus a constant.
struct Inv {
  double p, j2, j3, y;  // y = 1 / sqrt(j2) (1 where j2 is numerically zero)
  double rho, theta, s, c;
};
MPMX_DEV void invariants(const double* st, Inv& I) {
  I.p = mu_p(st);
  I.j2 = mu_j2(st);
  I.j3 = mu_j3(st);
  double v = 0.0;
  if (fabs(I.j2) > kDblEps) v = (3. * sqrt(3.) / 2.) * (I.j3 / dmath::pow_1p5(I.j2));
  if (v > 1.0) v = 1.0;
  if (v < -1.0) v = -1.0;
  {
#pragma clang fp contract(fast)
    I.theta = (1. / 3.) * acos(v);
    I.y = I.j2 > kDblEps ? rsqrt(I.j2) : 1.0;
    I.rho = I.j2 > kDblEps ? 1.4142135623730951 * (I.j2 * I.y) : sqrt(2. * I.j2);
    const double t = I.theta - 0.5235987755982989;
    const double z = t * t;
    I.s = t + (t * z) * poly6(dmath::kSin, z);
    I.c = 1.0 - z * (0.5 - z * poly6(dmath::kCos, z));
  }
}

// Constants of a friction / dilation angle pair (Material::fk for the peak
// angles).
struct Angles {
  double tphi;    // tan phi
  double kc;      // 1 / (sqrt(3) cos phi)
  double n, sn;   // n = (1 + sin phi) / (1 - sin phi), its square root
  double ap;      // sqrt(1 + n^2) + n
  double rmc;     // (3 - sin phi) / (6 cos phi)
  double e;       // eccentricity of the potential
  double tpsi;
};
MPMX_DEV Angles angles_of(const Material& m, double phi, double psi) {
  Angles A;
  if (phi == m.phi_peak && psi == m.psi_peak) {
    A.tphi = m.fk[0];
    A.kc = m.fk[1];
    A.n = m.fk[2];
    A.sn = m.fk[3];
    A.ap = m.fk[4];
    A.rmc = m.fk[5];
    A.e = m.fk[6];
    A.tpsi = m.fk[7];
    return A;
  }
  double fk[8];
  const McAngles a = mc_angles(phi, psi);
  fast_angle_constants(a.sphi, a.cphi, a.tpsi, fk);
  A.tphi = fk[0];
  A.kc = fk[1];
  A.n = fk[2];
  A.sn = fk[3];
  A.ap = fk[4];
  A.rmc = fk[5];
  A.e = fk[6];
  A.tpsi = fk[7];
  return A;
}

// compute_yield_state (mohr_coulomb.tcc:139-191)
MPMX_DEV int yield(double* yf, const Inv& I, const Angles& A, double cohesion, double tcut) {
#pragma clang fp contract(fast)
  constexpr double h3 = 0.8660254037844386, r23 = 0.816496580927726, r32 = 1.224744871391589;
  const double Tolerance = -1E-1;
  const double ct = h3 * I.c - 0.5 * I.s;  // cos theta; sin(theta + pi/3) = c
  yf[0] = r23 * ct * I.rho + (I.p - tcut);
  yf[1] = r32 * I.rho * (I.c * A.kc - I.s * (A.tphi * (1. / 3.))) + (I.p * A.tphi - cohesion);
  int t = FS_ELASTIC;
  if (yf[0] > Tolerance && yf[1] > Tolerance) {
    const double sigma_p = tcut * A.n - 2. * cohesion * A.sn;
    // cos(theta - 4 pi/3)
    const double h = yf[0] + A.ap * (r23 * (-h3 * I.c - 0.5 * I.s) * I.rho + (I.p - sigma_p));
    t = (h > kDblEps) ? FS_TENSILE : FS_SHEAR;
  }
  if (yf[0] < Tolerance && yf[1] > Tolerance) t = FS_SHEAR;
  if (yf[0] > Tolerance && yf[1] < Tolerance) t = FS_TENSILE;
  return t;
}

// compute_df_dp (mohr_coulomb.tcc:195-344) in the basis
//   df/dsigma = fp 1 + fr R + ft T,  dp/dsigma = gp 1 + gr R + gt T,
// R = d rho / d sigma = yr dev and T = d theta / d sigma (tensors; the Voigt
// gradients double the shears). The elastic tensor is isotropic: D applied to
// a tensor a 1 + A is 3K a 1 + 2G A + a2 tr(A) 1. Near a corner of the surface
// T is mostly rounding, neither traceless nor orthogonal to the deviator to
// better than 1 / sin 3 theta ulps, so its trace and products are formed, not
// taken as zero.
struct Grad {
  double fp, fr, ft, gp, gr, gt;
  double dev[6], tt[6];
  double yr;  // 1 / sqrt(2 j2), 0 where the deviator vanishes
};
// d theta / d sigma as a tensor, in the reference's arithmetic: near a corner
// of the surface (r = +-1) its two terms cancel and 1 / sqrt(1 - r^2)
// magnifies what rounding leaves of them.
MPMX_DEV void lode_direction(const Inv& I, const double* d, double* tt) {
  const double j2 = I.j2, j3 = I.j3;
  double dr_dj2 = -9.0 / 4.0 * sqrt(3.0) * j3;
  double dr_dj3 = 3.0 / 2.0 * sqrt(3.0);
  double dtheta_dr = -1.0 / 3.0;
  if (fabs(j2) > kDblEps) {
    const double r = j3 / 2.0 * dmath::pow_m1p5(j2 / 3.0);
    dr_dj2 *= dmath::pow_m2p5(j2);
    dr_dj3 *= dmath::pow_m1p5(j2);
    const double factor = (fabs(1 - r * r) < kDblEps) ? kDblEps : fabs(1 - r * r);
    dtheta_dr = -1.0 / (3.0 * sqrt(factor));
  }
  const double d1[3] = {d[0], d[3], d[5]};
  const double d2[3] = {d[3], d[1], d[4]};
  const double d3[3] = {d[5], d[4], d[2]};
  const double k = (2. / 3.) * j2;
  const double t[6] = {dot3(d1, d1) - k, dot3(d2, d2) - k, dot3(d3, d3) - k,
                       dot3(d1, d2),     dot3(d2, d3),     dot3(d1, d3)};
#pragma unroll
  for (int i = 0; i < 6; ++i) tt[i] = dtheta_dr * ((dr_dj2 * d[i]) + (dr_dj3 * t[i]));
}
MPMX_DEV void gradients(const Material& m, int yt, double tcut, const double* st, const Inv& I,
                        const Angles& A, Grad& g) {
#pragma clang fp contract(fast)
  mu_dev(st, g.dev);
  lode_direction(I, g.dev, g.tt);
  constexpr double h3 = 0.8660254037844386, r23 = 0.816496580927726, r32 = 1.224744871391589;
  const double rho = I.rho, y = I.y;
  const double ct = h3 * I.c - 0.5 * I.s, sn = h3 * I.s + 0.5 * I.c;
  if (I.j2 > kDblEps)
    g.yr = 0.7071067811865476 * y;
  else
    g.yr = sqrt(3. * I.j2) > kDblEps ? 1. / sqrt(2. * I.j2) : 0.;
  if (yt == FS_TENSILE) {
    g.fp = 1. / 3.;
    g.fr = r23 * ct;
    g.ft = -r23 * rho * sn;
    // Menetrey-Willam with eccentricity 0.6, xi 0.1 (mohr_coulomb.tcc:263-293)
    constexpr double e = 0.6, k = 1. - e * e, e21 = 2. * e - 1.;
    constexpr double q0 = 5. * e * e - 4. * e;
    double sq = 4. * k * ct * ct + q0;
    if (sq < kDblEps) sq = 1.E-5;
    const double ys = rsqrt(sq);
    double den = 2. * k * ct + e21 * (sq * ys);
    if (fabs(den) < kDblEps) den = 1.E-5;
    const double num = 4. * k * ct * ct + e21 * e21;
    const double id = rcp(den);
    const double rt = num * id * (1. / 3.);
    const double w = 0.01 * tcut * tcut + 1.5 * rt * rt * rho * rho;
    const double ic = w > 1.0e-30 ? rsqrt(w) : 1.0e15;
    const double dden = -2. * k * sn - e21 * 4. * k * ct * sn * ys;
    const double dnum = -8. * k * ct * sn;
    const double drt = (dnum * den - dden * num) * (id * id) * (1. / 3.);
    g.gp = 1. / 3.;
    g.gr = 1.5 * rho * rt * rt * ic;
    g.gt = 1.5 * rho * rho * rt * ic * drt;
  } else {
    g.fp = A.tphi * (1. / 3.);
    g.fr = r32 * (I.c * A.kc - I.s * (A.tphi * (1. / 3.)));
    g.ft = r32 * rho * (-I.s * A.kc - I.c * (A.tphi * (1. / 3.)));
    const double e = A.e, k = 1. - e * e, e21 = 2. * e - 1.;
    const double c2 = ct * ct;
    double sq = 4. * k * c2 + (5. * e * e - 4. * e);
    if (sq < kDblEps) sq = 1.E-5;
    const double ys = rsqrt(sq);
    double mm = 2. * k * ct + e21 * (sq * ys);
    if (fabs(mm) < kDblEps) mm = 1.E-5;
    const double l = 4. * k * c2 + e21 * e21;
    const double im = rcp(mm);
    const double rmw = l * im * A.rmc;
    const double u = 0.1 * m.c_peak * A.tpsi, v = rmw * r32 * rho;
    double omega = u * u + v * v;
    if (omega < kDblEps) omega = 1.E-5;
    const double dl = -8. * k * ct * sn;
    const double dm = -2. * k * sn + 0.5 * e21 * dl * ys;
    const double drmw = (mm * dl - l * dm) * (im * im);
    const double w = 1.5 * rho * rmw * rsqrt(omega);
    g.gp = A.tpsi * (1. / 3.);
    g.gr = w * rmw;
    g.gt = w * rho * A.rmc * drmw;
  }
}

// D (f 1 + r dev + t tt)
MPMX_DEV void elastic(const Material& m, const Grad& g, double f, double r, double t, double* y) {
#pragma clang fp contract(fast)
  const double g2 = m.a1 - m.a2;
  const double a = (m.a1 + 2. * m.a2) * f + m.a2 * t * (g.tt[0] + g.tt[1] + g.tt[2]);
  const double b = g2 * r, c = g2 * t;
#pragma unroll
  for (int i = 0; i < 3; ++i) y[i] = a + (b * g.dev[i] + c * g.tt[i]);
#pragma unroll
  for (int i = 3; i < 6; ++i) y[i] = b * g.dev[i] + c * g.tt[i];
}

// df . y for a stress-like y
MPMX_DEV double df_dot(const Grad& g, const double* y) {
#pragma clang fp contract(fast)
  const double r = g.fr * g.yr;
  double a = 0., b = 0.;
#pragma unroll
  for (int i = 0; i < 3; ++i) a = a + (g.fp + (r * g.dev[i] + g.ft * g.tt[i])) * y[i];
#pragma unroll
  for (int i = 3; i < 6; ++i) b = b + (r * g.dev[i] + g.ft * g.tt[i]) * y[i];
  return a + 2. * b;
}

// The softening modulus (mohr_coulomb.tcc:318-344)
MPMX_DEV double softening(const Material& m, double pdstrain, double phi, const Inv& I,
                          const Angles& A, const Grad& g) {
  if (!m.softening || !(pdstrain > m.pd_peak) || !(pdstrain < m.pd_res)) return 0.;
  const double icp = 1.7320508075688772 * A.kc;  // 1 / cos phi
  const double sphi = A.tphi / icp;
  const double dphi = (m.phi_res - m.phi_peak) / (m.pd_res - m.pd_peak);
  const double dc = (m.c_res - m.c_peak) / (m.pd_res - m.pd_peak);
  const double df_dphi =
      sqrt(1.5) * I.rho * ((sphi * I.c * A.kc * icp) + (-I.s * icp * icp / 3.)) +
      I.p * icp * icp;
  return (-1.) * ((df_dphi * dphi) - dc) * (g.gr * sqrt(2. / 3.));
}

// upd -= lam D dp; the plastic deviatoric strain's increment
MPMX_DEV double correct(double lam, const Grad& g, const double* y, double* upd) {
#pragma clang fp contract(fast)
#pragma unroll
  for (int i = 0; i < 6; ++i) upd[i] = upd[i] - lam * y[i];
  return lam * g.gr * 0.816496580927726;
}

// The plastic part of compute_stress (mohr_coulomb.tcc:412-512): mc_first and
// mc_iterate. s: the start-of-step stress, replaced by the returned one; ds:
// the strain increment; yt, y0: the trial state's yield type and function.
// sv: SV_PHI.. in, SV_EPS, SV_RHO, SV_THETA, SV_PDS out.
MPMX_DEV void plastic_return(const Material& m, double* s, const double* ds, int yt, double y0,
                             double* sv) {
  const Angles A = angles_of(m, sv[SV_PHI], sv[SV_PSI]);
  const double coh = sv[SV_COH], tcut = sv[SV_TCUT], pds0 = sv[SV_PDS];
  double trial[6], upd[6], yf[2];
  de_mul(m, ds, trial);
#pragma unroll
  for (int i = 0; i < 6; ++i) upd[i] = trial[i] = s[i] + trial[i];
  Inv I;
  Grad g;
  // first correction: from the current stress if it lies on the surface
  invariants(s, I);
  const int yc = yield(yf, I, A, coh, tcut);
  const double f = yc == FS_TENSILE ? yf[0] : yf[1];
  const bool use = yc != FS_ELASTIC && fabs(f) < 1E-1;
  if (!use) {
#pragma unroll
    for (int i = 0; i < 6; ++i) s[i] = trial[i];
    invariants(s, I);
  }
  gradients(m, use ? yc : yt, tcut, s, I, A, g);
  double y[6];
  double num = y0;
  if (use) {
    elastic(m, g, g.fp, g.fr * g.yr, g.ft, y);
    num = 0.;
    {
#pragma clang fp contract(fast)
#pragma unroll
      for (int i = 0; i < 6; ++i) num = num + y[i] * ds[i];
    }
  }
  elastic(m, g, g.gp, g.gr * g.yr, g.gt, y);
  double lam = num / (df_dot(g, y) + softening(m, pds0, sv[SV_PHI], I, A, g));
  double dpds = correct(lam, g, y, upd);
  double yv = y0;
#pragma nounroll
  for (int itr = 0;; ++itr) {
    invariants(upd, I);
    if (itr == 100) break;
    yt = yield(yf, I, A, coh, tcut);
    if (yf[0] < 1E-1 && yf[1] < 1E-1) break;
    if (yt == FS_TENSILE) yv = yf[0];
    if (yt == FS_SHEAR) yv = yf[1];
    gradients(m, yt, tcut, upd, I, A, g);
    elastic(m, g, g.gp, g.gr * g.yr, g.gt, y);
    lam = yv / (df_dot(g, y) + softening(m, pds0, sv[SV_PHI], I, A, g));
    dpds += correct(lam, g, y, upd);
  }
  sv[SV_EPS] = I.p * sqrt(3.);
  sv[SV_RHO] = I.rho;
  sv[SV_THETA] = I.theta;
  sv[SV_PDS] = pds0 + dpds;
#pragma unroll
  for (int i = 0; i < 6; ++i) s[i] = upd[i];
}

// The elastic predictor (mc_begin): true when the update is complete (elastic
// or separated; s and sv final), else yt and y0 describe the trial state and
// s keeps the start-of-step stress.
MPMX_DEV bool predictor(const Material& m, double* s, const double* ds, double density,
                        double* sv, int& yt, double& y0) {
  if (m.softening) {  // softened strength parameters (mohr_coulomb.tcc:356-384)
    const double pdstrain = sv[SV_PDS];
    if (pdstrain > m.pd_peak) {
      if (pdstrain < m.pd_res) {
        const double w = (pdstrain - m.pd_res) / (m.pd_peak - m.pd_res);
        sv[SV_PHI] = m.phi_res + (m.phi_peak - m.phi_res) * w;
        sv[SV_PSI] = m.psi_res + (m.psi_peak - m.psi_res) * w;
        sv[SV_COH] = m.c_res + (m.c_peak - m.c_res) * w;
      } else {
        sv[SV_PHI] = m.phi_res;
        sv[SV_PSI] = m.psi_res;
        sv[SV_COH] = m.c_res;
      }
      const double apex = sv[SV_COH] / dmath::tan(sv[SV_PHI]);
      if (sv[SV_TCUT] > apex) sv[SV_TCUT] = (apex > 1.0e-15 ? apex : 1.0e-15);
    }
  }
  double t[6];
  de_mul(m, ds, t);
#pragma unroll
  for (int i = 0; i < 6; ++i) t[i] = s[i] + t[i];
  sv[SV_YIELD] = 0;
  if (density <= m.critical_density) {
    sv[SV_PDS] += mu_q(t) / 3.0 / m.shear;
    sv[SV_YIELD] = 3;
#pragma unroll
    for (int i = 0; i < 6; ++i) s[i] = 0.;
    return true;
  }
  const Angles A = angles_of(m, sv[SV_PHI], sv[SV_PSI]);
  Inv I;
  invariants(t, I);
  double yf[2];
  yt = yield(yf, I, A, sv[SV_COH], sv[SV_TCUT]);
  if (yt == FS_ELASTIC) {
    sv[SV_EPS] = I.p * sqrt(3.);
    sv[SV_RHO] = I.rho;
    sv[SV_THETA] = I.theta;
#pragma unroll
    for (int i = 0; i < 6; ++i) s[i] = t[i];
    return true;
  }
  sv[SV_YIELD] = (yt == FS_TENSILE) ? 2 : 1;
  y0 = yt == FS_TENSILE ? yf[0] : yf[1];
  return false;
}

// ------------------------------ kinematics ----------------------------------
// Velocity gradient L (L[a][b] = d v_a / d x_b) at xi and divergence at the
// centroid on a box cell with sides len, axis by axis: differences and sums
// along x, interpolated over y and z. 24 node velocities, no node coordinates.
MPMX_DEV void box_gradient(const double* xi, const double* len, const double (*nv)[3],
                           double (*L)[3], double* div_c) {
#pragma clang fp contract(fast)
  double il[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) il[k] = rcp(len[k]);
  double dc = 0.;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    // rows along x at (y, z) = 00, 10, 01, 11
    const double d0 = nv[1][a] - nv[0][a], d1 = nv[2][a] - nv[3][a];
    const double d2 = nv[5][a] - nv[4][a], d3 = nv[6][a] - nv[7][a];
    const double s0 = nv[1][a] + nv[0][a], s1 = nv[2][a] + nv[3][a];
    const double s2 = nv[5][a] + nv[4][a], s3 = nv[6][a] + nv[7][a];
    const double m0 = s0 + xi[0] * d0, m1 = s1 + xi[0] * d1;
    const double m2 = s2 + xi[0] * d2, m3 = s3 + xi[0] * d3;
    const double a0 = (d0 + d1) + xi[1] * (d1 - d0), a1 = (d2 + d3) + xi[1] * (d3 - d2);
    const double b0 = m1 - m0, b1 = m3 - m2;
    const double c0 = (m0 + m1) + xi[1] * b0, c1 = (m2 + m3) + xi[1] * b1;
    L[a][0] = 0.25 * il[0] * ((a0 + a1) + xi[2] * (a1 - a0));
    L[a][1] = 0.25 * il[1] * ((b0 + b1) + xi[2] * (b1 - b0));
    L[a][2] = 0.25 * il[2] * (c1 - c0);
    const double w = a == 0   ? (d0 + d1) + (d2 + d3)
                     : a == 1 ? (s1 - s0) + (s3 - s2)
                              : (s2 + s3) - (s0 + s1);
    dc = dc + 0.25 * il[a] * w;
  }
  *div_c = dc;
}

// The same on a general cell from its Jacobian at xi and the stored centroid
// gradients.
MPMX_DEV void cell_gradient(const Mesh& M, int c, const double* xi, const double (*nv)[3],
                            double (*L)[3], double* div_c) {
#pragma clang fp contract(fast)
  constexpr int NN = Elem<3>::NN;
  double X[NN][3], Ji[3][3];
  load_cell_X<3>(M, c, X);
  jacobian_inverse<3>(xi, X, Ji);
  double G[3][3];  // sum_i v_i (x) grad_i, then L = G J^-T
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) G[a][b] = 0.;
  const double* dcp = M.dndx_c + (int64_t)c * NN * 3;
  double dc = 0.;
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    double g[3];
    grad_i<3>(xi, i, g);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      dc = dc + dcp[i * 3 + a] * nv[i][a];
#pragma unroll
      for (int b = 0; b < 3; ++b) G[a][b] = G[a][b] + nv[i][a] * g[b];
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      double t = G[a][0] * Ji[b][0];
#pragma unroll
      for (int k = 1; k < 3; ++k) t = t + G[a][k] * Ji[b][k];
      L[a][b] = t;
    }
  *div_c = dc;
}

// The particle fields the kinematics and the constitutive update read, loaded
// together before any store (a later load would wait for the stores' round
// trip: the compiler must assume they alias).
struct StressIn {
  double eps[6], F[9], s[6], vol, rho;
  int mat;
};
MPMX_DEV void load_stress_in(const Particles& P, int64_t p, StressIn& q) {
  const int64_t np = P.np;
#pragma unroll
  for (int k = 0; k < 6; ++k) q.eps[k] = stream_ld(&P.strain[k * np + p]);
  q.vol = stream_ld(&P.vol[p]);
  q.rho = stream_ld(&P.rho[p]);
#pragma unroll
  for (int k = 0; k < 9; ++k) q.F[k] = stream_ld(&P.F[k * np + p]);
#pragma unroll
  for (int k = 0; k < 6; ++k) q.s[k] = stream_ld(&P.stress[k * np + p]);
  q.mat = stream_ld(&P.mat[p]);
}

// The kinematics of the stress update (mpm_scheme.tcc:75-103; see kinematics
// in mpmx_kernels.hip) from the velocity gradient: strain increment ds, and
// strain, volume, density and F of particle p written.
MPMX_DEV void strain_update(const Particles& P, int64_t p, StressIn& q, const double (*L)[3],
                            double div_c, double dt, double* ds) {
#pragma clang fp contract(fast)
  const int64_t np = P.np;
  double R[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      double r = L[a][b] * dt;
      if (fabs(r) < 1.E-15) r = 0.;
      R[a][b] = a == b ? 1. + r : r;
    }
#pragma unroll
  for (int k = 0; k < 3; ++k) ds[k] = L[k][k];
  ds[3] = L[0][1] + L[1][0];
  ds[4] = L[1][2] + L[2][1];
  ds[5] = L[0][2] + L[2][0];
#pragma unroll
  for (int k = 0; k < 6; ++k) ds[k] = fabs(ds[k]) < 1.E-15 ? 0. : ds[k] * dt;
  const double dvol = dt * div_c;
  q.vol = q.vol * (1. + dvol);
  q.rho = q.rho * rcp(1. + dvol);
#pragma unroll
  for (int k = 0; k < 6; ++k)
    stream_st(&P.strain[k * np + p], q.eps[k] + ds[k]);
  stream_st(&P.vol[p], q.vol);
  stream_st(&P.rho[p], q.rho);
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double t = R[a][0] * q.F[j];
#pragma unroll
      for (int b = 1; b < 3; ++b) t = t + R[a][b] * q.F[b * 3 + j];
      stream_st(&P.F[(a * 3 + j) * np + p], t);
    }
}

// Return mappings of a workgroup of BS particles, compacted in LDS: the
// particles whose trial stress yields hand over their start-of-step stress,
// strain increment and trial yield value; shear returns fill the slots from
// the front, tensile ones from the back, so that the waves that complete them
// are full and mostly run one branch of the flow rule.
template <int BS>
struct Returns {
  double s[6][BS], ds[6][BS], y0[BS];
  int p[BS], mat[BS];
  int n[2];  // shear, tensile
};

template <int BS>
MPMX_DEV int push_return(Returns<BS>& q, int p, int mat, const double* s, const double* ds, int yt,
                         double y0) {
  const bool tensile = yt == FS_TENSILE;
  const unsigned long long t = __ballot(tensile), all = __ballot(1);
  const unsigned long long mine = tensile ? t : (all & ~t);
  const int lane = threadIdx.x & 63, leader = __ffsll((long long)mine) - 1;
  int base = 0;
  if (lane == leader) base = atomicAdd(&q.n[tensile ? 1 : 0], __popcll(mine));
  base = __shfl(base, leader, 64);
  const int k = base + __popcll(mine & ((1ull << lane) - 1ull));
  const int slot = tensile ? BS - 1 - k : k;
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    q.s[c][slot] = s[c];
    q.ds[c][slot] = ds[c];
  }
  q.y0[slot] = y0;
  q.p[slot] = p;
  q.mat[slot] = mat;
  return slot;
}

}  // namespace fast
}  // namespace mpmx
