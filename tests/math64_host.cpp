// math64_host.cpp -- the FP64 path's arithmetic (rt_math64.h, rt_physics.h)
// compiled for the host, element by element over arrays.
#include "rt_physics.h"

using namespace emma;

extern "C" {
void set_rcp_error(double e) { rcp_error = e; }
void div_all(int n, const double* a, const double* b, double* q) {
  for (int i = 0; i < n; i++) q[i] = div64(a[i], b[i]);
}
void log_all(int n, const double* x, double* h, double* l) {
  for (int i = 0; i < n; i++) {
    const Dd d = log_dd(x[i]);
    h[i] = d.h;
    l[i] = d.l;
  }
}
void exp_all(int n, const double* x, double* y) {
  for (int i = 0; i < n; i++) y[i] = exp64(x[i]);
}
void rates_all(int n, const double* t, double* out) {  // [n][6]
  for (int i = 0; i < n; i++) {
    const Rates r = rates_of(t[i]);
    const double v[6] = {r.A1, r.A3, r.A4, r.A6, r.alphab, r.beta};
    memcpy(out + 6 * i, v, sizeof(v));
  }
}
void closure_all(int n, const double* u, double c, double* out) {  // [n][4] -> [n][5]
  for (int i = 0; i < n; i++) {
    const double* s = u + 4 * i;
    const Closure<double> q = closure<double>(s[1], s[2], s[3], s[0], c);
    const double v[5] = {q.diag, q.arg, q.n[0], q.n[1], q.n[2]};
    memcpy(out + 5 * i, v, sizeof(v));
  }
}
}
