// Launchers of the compressible step's helper kernels, shared by the
// pointwise-stage file and the native step driver (internal to
// libpadeops_hip).  Each launches on `s` and returns 0 or a library error
// code with the message recorded.
#pragma once

#include <hip/hip_runtime.h>

namespace pade {

int cg_fill(double *x, long long n, double v, hipStream_t s);

// mu = mu_ref (T / T_ref)^visc_n, bulk = 0, kap = mu * cp_by_pr
int cg_transport(long long n, const double *T, double mu_ref, double T_ref, double visc_n, double cp_by_pr,
                 double *mu, double *bulk, double *kap, hipStream_t s);

// e = p / (gam - 1) / rho, T = e (gam - 1) / Rgas
int cg_post_bc(long long n, const double *rho, const double *p, double gam, double Rgas, double *e, double *T,
               hipStream_t s);

// The four maxima of get_dt: max(|u|/dx + |v|/dy + |w|/dz + c sqrt(1/dx^2 +
// 1/dy^2 + 1/dz^2)), max(mu/rho), max(bulk/rho), max(kap T / (rho hmin^4)),
// into out[0..3] (synchronous: reduced on the device through dev4, read back
// through the pinned host words host4).
int cg_dt_maxima(long long n, const double *rho, const double *u, const double *v, const double *w, const double *p,
                 const double *mu, const double *bulk, const double *kap, const double *T, double dx, double dy,
                 double dz, double gam, double hmin, unsigned long long *dev4, unsigned long long *host4, double *out,
                 hipStream_t s);

// The three artificial properties before filtering (cgrid.F90:1083-1199) in
// one pass: fl holds grad(rho), grad(e) and the fourth derivatives of the
// strain magnitude, the dilatation and e (three planes each, in this order);
// mustar holds the bulk viscosity's switch on entry.
int cg_lad(long long n, double Cmu, double Cbeta, double Ckap, double gam, const double *h, const double *rho,
           const double *p, const double *T, const double *fl, double *mustar, double *bulkstar, double *kapstar,
           hipStream_t s);

// An RK45 stage of n values: Q = dt rhs + A Q, W += B Q.
int cg_rk_stage(long long n, double dt, double A, double B, const double *rhs, double *Q, double *W, hipStream_t s);

// The magnitude of the strain rate, the dilatation and the bulk viscosity's
// switch (cgrid.F90:1085-1087, :1140-1155) from the velocity gradients.
int cg_strain_switch(long long n, const double *du, double *func, double *dil, double *fsw, hipStream_t s);

// get_primitive and post_bc, then get_conserved of the result (the state
// between two substeps when nothing comes between them), with pade_cg_conserved's
// test of W.
int cg_primitive_conserved(long long n, double *W, double gam, double Rgas, double *rho, double *u, double *v,
                           double *w, double *e, double *p, double *T, unsigned long long *bad_index, hipStream_t s);

}  // namespace pade
