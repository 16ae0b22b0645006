// Host build of the Lax-Friedrichs face flux for tests/test_weno_lf.py.
#include "../../janc_amd/csrc/weno.hpp"

extern "C" {

// face flux of scaled split fluxes p0..p4 (H+) and m1..m5 (H-), unscaled
double host_weno_lf(const double* p, const double* m) {
  const double s = jh::LfScale<double>::value;
  double a[5], b[5];
  for (int k = 0; k < 5; ++k) {
    a[k] = s * p[k];
    b[k] = s * m[k];
  }
  return jh::weno5_lf(a[0], a[1], a[2], a[3], a[4], b[0], b[1], b[2], b[3], b[4]) / s;
}

// left- and right-biased values of a face over one reciprocal
void host_weno_LR(const double* v, double* out) {
  jh::weno5_LR(v[0], v[1], v[2], v[3], v[4], v[5], out[0], out[1]);
}

}  // extern "C"
