// riemanncheck.cpp -- host build of the bounded-state fluxes and face states
// (pip_riemann.h) beside the general ones (pip_phys.h), for
// tests/test_bounded_fluxes_cpu.py.  Test infrastructure; not used by
// libpipgpu.
#include "pip_riemann.h"

using namespace pip;

extern "C" {
// n faces, 9 variables a side; returns the number of faces the bounded
// function covered and writes both results (9 a face; uncovered: the general)
long rc_hlld(int nv, const double* vl, const double* vr, double gm, double ch, long n, double* gen, double* bnd) {
  long cov = 0;
  for (long i = 0; i < n; i++) {
    const double *l = vl + 9 * i, *r = vr + 9 * i;
    double *g = gen + 9 * i, *b = bnd + 9 * i;
    for (int k = 0; k < 9; k++) g[k] = b[k] = 0.0;
    if (nv == 9) hlld_flux<9>(l, r, gm, ch, g);
    else hlld_flux<8>(l, r, gm, ch, g);
    auto put = [&](int k, double x) { b[k] = x; };
    const bool ok = nv == 9 ? hlld_flux_b<9>(l, r, gm, 1.0 / (gm - 1.0), ch, put)
                            : hlld_flux_b<8>(l, r, gm, 1.0 / (gm - 1.0), ch, put);
    if (!ok)
      for (int k = 0; k < 9; k++) b[k] = g[k];
    cov += ok;
  }
  return cov;
}
long rc_hllc(const double* vl, const double* vr, double gm, long n, double* gen, double* bnd) {
  long cov = 0;
  for (long i = 0; i < n; i++) {
    const double *l = vl + 9 * i, *r = vr + 9 * i;
    double *g = gen + 9 * i, *b = bnd + 9 * i;
    for (int k = 0; k < 9; k++) g[k] = b[k] = 0.0;
    hllc_flux(l, r, gm, g);
    const bool ok = hllc_flux_b(l, r, gm, 1.0 / (gm - 1.0), [&](int k, double x) { b[k] = x; });
    if (!ok)
      for (int k = 0; k < 5; k++) b[k] = g[k];
    cov += ok;
  }
  return cov;
}
void rc_states(const double* a, long n, double* gen, double* bnd) {
  for (long i = 0; i < n; i++) {
    const double* c = a + 4 * i;
    gen[2 * i] = c[1] + 0.5 * minmod(c[0], c[1], c[2]);
    gen[2 * i + 1] = c[2] - 0.5 * minmod(c[1], c[2], c[3]);
    face_states(c[0], c[1], c[2], c[3], bnd[2 * i], bnd[2 * i + 1]);
  }
}
int rc_bounded(const double* v, int nv) { return bounded_cell(v, nv) ? 1 : 0; }
}
