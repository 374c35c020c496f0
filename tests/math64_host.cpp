// math64_host.cpp -- the FP64 path's arithmetic (rt_math64.h, rt_physics.h)
// compiled for the host, element by element over arrays.  With PLAIN_DIVISION
// every quotient of rt_physics.h is a plain one.
#include "rt_math64.h"
#ifdef PLAIN_DIVISION
#define div64(a, b, ...) ((a) / (b))
#define quot64(a, b, ...) ((a) / (b))
#endif
#include "rt_physics.h"

using namespace emma;

extern "C" {
void set_rcp_error(double e) { rcp_error = e; }
void div_all(int n, const double* a, const double* b, double* q) {
  for (int i = 0; i < n; i++) q[i] = div64(a[i], b[i]);
}
// chem_cell of two groups: in [n][13] (e, fx, fy, fz, src of each group, x n_H,
// eint, n_H), out [n][13] (the first eight, x n_H, eint, T, status, sub-steps)
void chem_all(int n, const double* in, double dt, int chemonly, const double* unit, const double* group, double* out) {
  ChemConst K;
  memset(&K, 0, sizeof(K));
  K.static_cosmo = 1;
  K.fudgecool = 0.1;
  K.unit_l = unit[0], K.unit_t = unit[1], K.unit_N = unit[2], K.unit_n = unit[3], K.unit_d = unit[4];
  K.unit_v = unit[5];
  K.aexp = K.a2 = K.a3 = K.pa2 = K.pa3 = K.pa4 = K.pa5 = 1.;
  K.pv2 = K.unit_v * K.unit_v;
  K.pstar = K.unit_n * K.unit_d * K.pv2;
  K.dt = dt * K.unit_t;
  K.emin = kPmin / (kGamma - 1.) * K.unit_n * K.unit_d * K.pv2;
  K.r_a2 = K.r_a3 = K.r_pa3 = K.r_pa4 = K.r_pa5 = 1.;
  K.r_unit_N = 1. / K.unit_N, K.r_unit_l = 1. / K.unit_l, K.r_unit_t = 1. / K.unit_t;
  K.r_unit_n = 1. / K.unit_n, K.r_unit_d = 1. / K.unit_d, K.r_pv2 = 1. / K.pv2;
  for (int g = 0; g < 2; g++) {
    K.alphai[g] = group[3 * g];
    K.heat[g] = group[3 * g + 1];
    K.factgrp[g] = group[3 * g + 2];
    K.emin_grp[g] = kEmin * K.factgrp[g] / K.unit_N;
  }
  for (int i = 0; i < n; i++) {
    const double* u = in + 13 * i;
    double* o = out + 13 * i;
    double e[2] = {u[0], u[1]}, fx[2] = {u[2], u[3]}, fy[2] = {u[4], u[5]}, fz[2] = {u[6], u[7]};
    const double src[2] = {u[8], u[9]};
    double xn = u[10], eint = u[11], temp = 0.;
    int nit = 0;
    const int st = chem_cell<2>(K, 2, e, fx, fy, fz, src, xn, eint, u[12], temp, chemonly, nit);
    const double v[13] = {e[0], e[1], fx[0], fx[1], fy[0], fy[1], fz[0], fz[1], xn, eint, temp, (double)st, (double)nit};
    memcpy(o, v, sizeof(v));
  }
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
