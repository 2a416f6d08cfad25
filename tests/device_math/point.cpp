// The point routines of csrc/mcf_device.h and mcf_prec.h over arrays, for
// tests/test_device_math.py.
#include "mcf_prec.h"

using namespace mcf;

extern "C" {
void v_posfix(long n, const double *Q, const double *U, double *out) {
  for (long i = 0; i < n; ++i) out[i] = posfix(Q[i], U[i]);
}
void v_minmod2(long n, const double *a, const double *b, double *out) {
  for (long i = 0; i < n; ++i) out[i] = minmod2(a[i], b[i]);
}
void v_quot(long n, const double *num, const double *den, double *out) {
  for (long i = 0; i < n; ++i) out[i] = Quot(den[i])(num[i]);
}
void v_switch(long n, const double *u5, const double *rho, int *out) {
  for (long i = 0; i < n; ++i) out[i] = t_at_least_3(u5[i], rho[i]);
}
}
