// Host build of the inverse hex8 map (mpm_amd/csrc/mpmx_device.h): fast mode's
// form against the general loop on random cells and points.
// Arguments: seed, points, cell size, distortion (0: parallelepipeds none;
// corners moved by up to half of it times the size, sheared by as much).
// Prints "points general differing worst octaves": points whose cell is valid,
// those that fast mode hands to the general loop, those that one form has in
// the cell and the other not (by more than 2e-10), the largest difference of
// the local coordinates inside the cell, and the most octaves that the search
// for the number of steps took at one point.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

static long octaves = 0;
inline float __log2f(float x) {  // called once per octave (and once per search)
  ++octaves;
  return std::log2(x);
}
#include "mpmx_device.h"

using namespace mpmx;

static bool inside(bool found, const double* xi) {
  for (int k = 0; k < 3; ++k) found = found && xi[k] >= -1. && xi[k] <= 1.;
  return found;
}

int main(int argc, char** argv) {
  if (argc < 5) return 2;
  std::mt19937_64 rng(std::atoi(argv[1]));
  std::uniform_real_distribution<double> U(-1, 1);
  const int points = std::atoi(argv[2]);
  const double h = std::atof(argv[3]), amp = std::atof(argv[4]);
  int n = 0, general = 0, differing = 0;
  double worst = 0.;
  long most = 0;
  for (int t = 0; t < points; ++t) {
    double X[8][3], A[3][3];
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) A[a][b] = (a == b ? 1. : 0.) + 0.5 * amp * U(rng);
    for (int i = 0; i < 8; ++i) {
      double p[3];
      for (int k = 0; k < 3; ++k) p[k] = 0.5 * h * (unit_vertex(i, k) + amp * U(rng));
      for (int k = 0; k < 3; ++k)
        X[i][k] = A[k][0] * p[0] + A[k][1] * p[1] + A[k][2] * p[2] + 3.7 * h * k + 0.3;
    }
    bool valid = true;  // a positive Jacobian determinant at every corner
    for (int i = 0; i < 8 && valid; ++i) {
      double xi[3], J[3][3] = {};
      for (int k = 0; k < 3; ++k) xi[k] = unit_vertex(i, k);
      for (int j = 0; j < 8; ++j) {
        double g[3];
        grad_i<3>(xi, j, g);
        for (int a = 0; a < 3; ++a)
          for (int b = 0; b < 3; ++b) J[a][b] += g[a] * X[j][b];
      }
      const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                         J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                         J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
      valid = det >= 1e-3 * h * h * h / 8;
    }
    if (!valid) continue;
    // half of the points inside, the others up to 1.02 and 2.5 half sides
    // away; some 1e-9 from a face
    double xt[3], N[8], p[3] = {0., 0., 0.}, a[3], b[3];
    const double far = t % 4 == 3 ? 2.5 : (t % 4 == 2 ? 1.02 : 0.999);
    for (int k = 0; k < 3; ++k) xt[k] = far * U(rng);
    if (t % 8 == 0) xt[t % 3] = U(rng) > 0 ? 1 - 1e-9 : -1 + 1e-9;
    shapefn<3>(xt, N);
    for (int i = 0; i < 8; ++i)
      for (int k = 0; k < 3; ++k) p[k] += N[i] * X[i][k];
    const bool ra = transform_real_to_unit_cell<3, false>(X, h, p, a);
    bool handed = false;
    octaves = 0;
    const bool rb = transform_real_to_unit_cell<3, true>(X, h, p, b, &handed);
    most = std::max(most, octaves);
    ++n;
    if (handed) {
      ++general;
      continue;
    }
    double d = 0.;
    for (int k = 0; k < 3; ++k) d = std::fmax(d, std::fabs(a[k] - b[k]));
    const bool ia = inside(ra, a), ib = inside(rb, b);
    if (ia != ib && !(d <= 2e-10)) ++differing;
    if (ia && ib) worst = std::fmax(worst, d);
  }
  std::printf("%d %d %d %.3e %ld\n", n, general, differing, worst, most);
  return 0;
}
