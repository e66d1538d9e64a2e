// Host build of the 3D fast mode's constitutive update (mpm_amd/csrc/mpmx_fast.h)
// against the reference's arithmetic (mpmx_device.h, mc_stress) on random
// states: elastic, shear and tensile returns, corners of the surface, softening
// below, between and beyond the peak and residual strains, separation.
// The hardware's reciprocal estimates are stood in for by 32-bit ones.
// Arguments: seed, states, softening (0 or 1).
// Prints "states elastic shear tensile separated softened mismatches mean max
// nudge": particles of each yield state of the reference's arithmetic, those
// that have a softening modulus, differing yield states, mean and largest
// difference of a stress component in Pa, and the largest change that moving
// the start stress by one ulp makes to the reference's own result.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

static inline double rcp_estimate(double x) { return 1.f / (float)x; }
static inline double rsq_estimate(double x) { return 1.f / std::sqrt((float)x); }
#define __builtin_amdgcn_rcp rcp_estimate
#define __builtin_amdgcn_rsq rsq_estimate
static inline unsigned long long __ballot(int) { return 0; }  // push_return: not called
static inline int __shfl(int v, int, int) { return v; }
static inline int atomicAdd(int*, int) { return 0; }
static inline int __ffsll(long long) { return 0; }
static inline int __popcll(unsigned long long) { return 0; }
static struct { int x; } threadIdx;
#include "mpmx_fast.h"

using namespace mpmx;

static Material material(double E, double nu, double rho, double phi, double psi, double c,
                         double tcut, bool softening) {
  Material m;
  std::memset(&m, 0, sizeof(m));
  const double deg = M_PI / 180.;
  m.type = MC;
  m.density = rho;
  m.E = E;
  m.critical_density = 0.9 * rho;
  m.softening = softening;
  m.phi_peak = phi * deg;
  m.psi_peak = psi * deg;
  m.c_peak = c;
  m.phi_res = 0.8 * m.phi_peak;
  m.psi_res = 0.2 * m.psi_peak;
  m.c_res = 0.2 * c;
  m.pd_peak = 1e-3;
  m.pd_res = 1e-2;
  const double K = E / (3.0 * (1. - 2. * nu));
  m.shear = m.G = E / (2.0 * (1. + nu));
  m.a1 = K + (4.0 / 3.0) * m.G;
  m.a2 = K - (2.0 / 3.0) * m.G;
  dmath::sincos(m.phi_peak, &m.sphi, &m.cphi);
  m.tphi = m.sphi / m.cphi;
  m.tpsi = dmath::tan(m.psi_peak);
  fast_angle_constants(m.sphi, m.cphi, m.tpsi, m.fk);
  m.sv0[SV_PHI] = m.phi_peak;
  m.sv0[SV_PSI] = m.psi_peak;
  m.sv0[SV_COH] = c;
  m.sv0[SV_TCUT] = std::max(std::min(tcut, c / dmath::tan(m.phi_peak)), 1e-15);
  return m;
}

int main(int argc, char** argv) {
  if (argc < 4) return 2;
  std::mt19937_64 rng(std::atoi(argv[1]));
  const int states = std::atoi(argv[2]);
  const bool softening = std::atoi(argv[3]) != 0;
  std::uniform_real_distribution<double> U(-1, 1);
  auto unit = [&] { return 0.5 * (U(rng) + 1.); };
  const Material ms[3] = {material(5e6, 0.3, 1800., 30., 0., 0., 0., softening),
                          material(3e6, 0.2, 2000., 35., 5., 800., 300., softening),
                          material(4e6, 0.3, 1900., 32., 3., 500., 1e9, softening)};
  int count[4] = {0, 0, 0, 0}, softened = 0, mismatches = 0;
  double sum = 0., most = 0., nudge = 0.;
  for (int t = 0; t < states; ++t) {
    const Material& m = ms[t % 3];
    double s[6], ds[6], sv[NSV];
    const double p = -50. * std::pow(400., unit());
    for (int k = 0; k < 3; ++k) s[k] = p * (k == 2 ? 1. : 0.2 + 0.8 * unit());
    for (int k = 3; k < 6; ++k) s[k] = 0.2 * U(rng) * p;
    if (t % 5 == 0) {  // two equal principal stresses
      s[1] = s[0];
      s[3] = s[4] = s[5] = 0.;
    }
    if (t % 7 == 3)
      for (int k = 0; k < 6; ++k) s[k] = k < 3 ? 5. + 395. * unit() : 2. * U(rng);
    const double size = 1e-6 * std::pow(100., unit());
    for (int k = 0; k < 6; ++k) ds[k] = size * U(rng);
    for (int k = 0; k < NSV; ++k) sv[k] = m.sv0[k];
    const double pds[6] = {0., 5e-4, 2e-3, 9e-3, 1e-2, 3e-2};
    sv[SV_PDS] = pds[rng() % 6];
    const double density = t % 13 == 5 ? 0.8 * m.density : m.density;

    double a[6], va[NSV], b[6], vb[NSV], c[6], vc[NSV];
    std::memcpy(a, s, sizeof(s));
    std::memcpy(b, s, sizeof(s));
    std::memcpy(va, sv, sizeof(sv));
    std::memcpy(vb, sv, sizeof(sv));
    std::memcpy(vc, sv, sizeof(sv));
    mc_stress(m, a, ds, density, va);
    int yt = 0;
    double y0 = 0.;
    if (!fast::predictor(m, b, ds, density, vb, yt, y0)) fast::plastic_return(m, b, ds, yt, y0, vb);
    for (int k = 0; k < 6; ++k) c[k] = std::nextafter(s[k], 1e300);
    mc_stress(m, c, ds, density, vc);

    const int y = (int)va[SV_YIELD];
    ++count[y];
    if (softening && sv[SV_PDS] > m.pd_peak && sv[SV_PDS] < m.pd_res && (y == 1 || y == 2))
      ++softened;
    if (va[SV_YIELD] != vb[SV_YIELD]) ++mismatches;
    double d = 0.;
    for (int k = 0; k < 6; ++k) {
      d = std::fmax(d, std::fabs(a[k] - b[k]));
      if (va[SV_YIELD] == vc[SV_YIELD]) nudge = std::fmax(nudge, std::fabs(a[k] - c[k]));
    }
    for (int k : {SV_PHI, SV_PSI, SV_COH, SV_TCUT})
      if (!(std::fabs(va[k] - vb[k]) <= 1e-14 * std::fabs(va[k]))) ++mismatches;
    if (!(std::fabs(va[SV_PDS] - vb[SV_PDS]) <= 1e-12)) ++mismatches;
    sum += d;
    most = std::fmax(most, d);
  }
  std::printf("%d %d %d %d %d %d %d %.3e %.3e %.3e\n", states, count[0], count[1], count[2],
              count[3], softened, mismatches, sum / states, most, nudge);
  return 0;
}
