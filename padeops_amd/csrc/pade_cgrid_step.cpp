// The compressible solver's RK45 step, driven from native code: cgrid's
// advance_RK45 (src/compressible/cgrid.F90:663-717) with getRHS (:822-1056),
// getLAD (:1058-1257), filter (:1259-1336), get_dt (:719-762) and the
// primitive / conserved conversions (:764-820), for one ideal-gas species
// with the power-law viscosity model, periodic or bounded per axis.  It
// chains the library's operator applies (cd10 / cd06 derivatives, cf90 and
// Gaussian filters) with the fused pointwise kernels of pade_cgrid.hip, all
// on the caller's stream, with every work array allocated once at create.
// On one GPU the reference's y / x / z pencil transposes are identities:
// every field is one Fortran-ordered (nx, ny, nz) array, and groups of fields
// are consecutive planes of one allocation.
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "../../include/padeops_hip.h"
#include "pade_capi_internal.h"
#include "pade_cgrid.h"
#include "pade_err.h"

namespace {

// low-storage RK45 (src/utilities/RKCoeffs.F90:6-17)
const double kRkA[5] = {0.0, -6234157559845.0 / 12983515589748.0, -6194124222391.0 / 4410992767914.0,
                        -31623096876824.0 / 15682348800105.0, -12251185447671.0 / 11596622555746.0};
const double kRkB[5] = {494393426753.0 / 4806282396855.0, 4047970641027.0 / 5463924506627.0,
                        9795748752853.0 / 13190207949281.0, 4009051133189.0 / 8539092990294.0,
                        1348533437543.0 / 7166442652324.0};

constexpr double kMachineEps = 2.220446049250313e-16;   // epsilon(1.0_rkind), constants.F90:37

int err(int code, const std::string &msg) { return pade::set_error(code, msg.c_str()); }

}  // namespace

struct pade_cgrid_s {
    int n[3] = {0, 0, 0};
    long long N = 0;
    double h[3] = {1, 1, 1};
    double gam = 1.4, Rgas = 1.0, Cmu = 0.002, Cbeta = 1.75, Ckap = 0.01;
    double mu_ref = 1.0, T_ref = 1.0, visc_n = 0.75, Pr = 0.75;
    bool inviscid = true;
    bool periodic[3] = {true, true, true};
    int bc[3][2] = {{0, 0}, {0, 0}, {0, 0}};
    int der_kind = PADE_CD10;
    pade_op_t der[3] = {nullptr, nullptr, nullptr};
    pade_op_t fil[3] = {nullptr, nullptr, nullptr};
    pade_op_t gfil[3] = {nullptr, nullptr, nullptr};
    // fields (caller's or owned): rho u v w p T e mu bulk kap, and W (5 planes)
    double *f[PADE_CG_NFIELDS] = {};
    bool own[PADE_CG_NFIELDS] = {};
    // work: an intermediate (sizes without a partitioned kernel), du (9), gT
    // (3), fluxes (15, before them the gradients and fourth derivatives of the
    // LAD, and the filters' intermediates), rhs (5), Qtmp (5) and the three
    // LAD properties before filtering
    double *work = nullptr;
    double *t1 = nullptr, *du = nullptr, *gT = nullptr, *fl = nullptr, *rhs = nullptr, *Q = nullptr,
           *mustar = nullptr, *func = nullptr, *dil = nullptr;
    unsigned long long *dscal = nullptr;    // device: bad index, four maxima
    unsigned long long *hscal = nullptr;    // pinned host copy
    int step = 0;
    double tsim = 0.0, dt = 0.0, dtfixed = 0.0;
};

namespace {

double *F(pade_cgrid_t g, int k) { return g->f[k]; }
double *Wp(pade_cgrid_t g, int k) { return g->f[PADE_CG_W] + (long long)k * g->N; }

// A field of a batch: its arrays and the sign of the axis's bc pair (-1: odd
// at the walls).
struct Item {
    const double *f;
    double *out;
    int sign;
    double *Q = nullptr, *W = nullptr;   // of a Runge-Kutta stage
};

// One operator along `axis` (0, 1, 2) of several (nx, ny, nz) fields, in one
// launch where the sizes allow: out = op^times(f), or with acc out = alpha
// op^times(f) + out.
template <int N>
int apply(pade_cgrid_t g, pade_op_t op, int oper, int axis, const Item (&items)[N], int times, bool acc, double alpha,
          hipStream_t s, const pade::Stage *stage = nullptr)
{
    int na, nb;
    if (axis == 0) { na = g->n[1]; nb = g->n[2]; }
    else if (axis == 1) { na = g->n[0]; nb = g->n[2]; }
    else { na = g->n[0]; nb = g->n[1]; }
    pade::BatchField b[N];
    for (int k = 0; k < N; k++)
        b[k] = {items[k].f, items[k].out, items[k].sign * g->bc[axis][0], items[k].sign * g->bc[axis][1], items[k].Q,
                items[k].W};
    return pade::apply_fields(op, oper, axis + 1, N, b, na, nb, times, acc, alpha, 1.0, g->t1, s, stage);
}

// cgrid.F90:1259-1336: y, then x, then z, each `times` times, of the N planes
// src[k], through the work planes fl[0 .. 2N - 1] into dst[k], or added to
// them; the axis flips[k] takes field k's bc pair negated.
template <int N>
int filter(pade_cgrid_t g, const double *const (&src)[N], double *const (&dst)[N], const int (&flips)[N],
           pade_op_t const *ops, int times, bool add, hipStream_t s)
{
    Item y[N], x[N], z[N];
    for (int k = 0; k < N; k++) {
        double *a = g->fl + k * g->N, *b = g->fl + (N + k) * g->N;
        y[k] = {src[k], a, flips[k] == 1 ? -1 : 1};
        x[k] = {a, b, flips[k] == 0 ? -1 : 1};
        z[k] = {b, dst[k], flips[k] == 2 ? -1 : 1};
    }
    int rc = apply(g, ops[1], PADE_FILTER, 1, y, times, false, 1.0, s);
    if (!rc) rc = apply(g, ops[0], PADE_FILTER, 0, x, times, false, 1.0, s);
    if (!rc) rc = apply(g, ops[2], PADE_FILTER, 2, z, times, add, 1.0, s);
    return rc;
}

int transport(pade_cgrid_t g, hipStream_t s)
{
    // MixtureEOS.F90:175-229 (ns = 1) with PowerLawViscosity.F90:38-75
    if (g->inviscid) {
        for (int k : {PADE_CG_MU, PADE_CG_BULK, PADE_CG_KAP})
            if (int rc = pade::cg_fill(F(g, k), g->N, 0.0, s)) return rc;
        return 0;
    }
    const double Cp = g->gam * g->Rgas / (g->gam - 1.0);
    return pade::cg_transport(g->N, F(g, PADE_CG_T), g->mu_ref, g->T_ref, g->visc_n, Cp / g->Pr,
                              F(g, PADE_CG_MU), F(g, PADE_CG_BULK), F(g, PADE_CG_KAP), s);
}

// cgrid.F90:822-896 with getLAD (:1058-1257, no species diffusivity for one
// species), getRHS_x/y/z (:898-1056), get_tau (:1338-1390) and get_q
// (:1392-1444), into rhs (5 planes).
//
// Every operator pass takes all the fields that are ready for it in one
// launch, and the repeated operators (the fourth derivative, the second
// derivative twice, cgrid.F90:1089-1105; the Gaussian filter, twice per axis)
// one launch instead of two: 9 launches for 18 gradient passes, 9 fourth
// derivatives and 9 filter pairs, 3 for the 15 flux derivatives.  Before the
// fluxes fill them, the planes fl hold grad(rho) (0-2), grad(e) (3-5) and the
// fourth derivatives of the strain magnitude (6-8), the dilatation (9-11) and
// e (12-14), planes x, y, z each.  From 128^3 up the pointwise passes and the
// stage are bound by memory (5.4-5.7 TB/s), the twice-applied launches by
// their chain (3.1 TB/s along y and z); below, launch and latency of each pass
// bound all.  Per step, 256^3 and 96 x 80 x 65
// (walls in z): one launch per field and pass 39.0 and 4.0 ms, batched and
// fused 32.4 and 1.72 ms, with the stage in the last flux derivative, the
// bulk switch beside the strain and one pass for the state update 31.1 and
// 1.68 ms.
//
// With a stage the last flux derivative also advances Q and W (rhs then holds
// an unfinished sum).
int rhs_impl(pade_cgrid_t g, double *rhs, hipStream_t s, const pade::Stage *stage = nullptr)
{
    const long long N = g->N;
    int rc = 0;
    for (int a : {1, 0, 2}) {      // cgrid.F90:446-478: a velocity takes its own axis's bc pair negated
        const Item grads[6] = {{F(g, PADE_CG_U), g->du + a * N, a == 0 ? -1 : 1},
                               {F(g, PADE_CG_V), g->du + (3 + a) * N, a == 1 ? -1 : 1},
                               {F(g, PADE_CG_W_VEL), g->du + (6 + a) * N, a == 2 ? -1 : 1},
                               {F(g, PADE_CG_RHO), g->fl + a * N, 1},
                               {F(g, PADE_CG_E), g->fl + (3 + a) * N, 1},
                               {F(g, PADE_CG_T), g->gT + a * N, 1}};
        if (!rc) rc = apply(g, g->der[a], PADE_D1, a, grads, 1, false, 1.0, s);
    }
    // an inviscid grid's properties are the artificial ones alone, written below
    if (!rc && !g->inviscid) rc = transport(g, s);
    if (!rc) rc = pade::cg_strain_switch(N, g->du, g->func, g->dil, g->mustar, s);
    if (!rc && g->der_kind == PADE_CD06) return err(21, "CD06 is incomplete right now");   // derivatives.F90:524-525
    for (int a : {0, 2, 1}) {
        const Item d4[3] = {{g->func, g->fl + (6 + a) * N, 1},
                            {g->dil, g->fl + (9 + a) * N, 1},
                            {F(g, PADE_CG_E), g->fl + (12 + a) * N, 1}};
        if (!rc) rc = apply(g, g->der[a], PADE_D2, a, d4, 2, false, 1.0, s);
    }
    if (!rc)
        rc = pade::cg_lad(N, g->Cmu, g->Cbeta, g->Ckap, g->gam, g->h, F(g, PADE_CG_RHO), F(g, PADE_CG_P),
                          F(g, PADE_CG_T), g->fl, g->mustar, g->func, g->dil, s);
    if (!rc) {                                                                       // (:1113, :1161, :1199, :1252-1254)
        const double *const stars[3] = {g->mustar, g->func, g->dil};
        double *const props[3] = {F(g, PADE_CG_MU), F(g, PADE_CG_BULK), F(g, PADE_CG_KAP)};
        const int flips[3] = {-1, -1, -1};
        rc = filter(g, stars, props, flips, g->gfil, 2, !g->inviscid, s);
    }
    if (!rc)
        rc = pade_cg_fluxes(N, F(g, PADE_CG_W), F(g, PADE_CG_U), F(g, PADE_CG_V), F(g, PADE_CG_W_VEL),
                            F(g, PADE_CG_P), g->du, F(g, PADE_CG_MU), F(g, PADE_CG_BULK), F(g, PADE_CG_KAP), g->gT,
                            g->fl, s);
    // rhs = d(-fx)/dx (the x fluxes come negated), then rhs -= d(fy)/dy,
    // d(fz)/dz, accumulated inside the derivative kernel; every flux is odd at
    // the walls except the momentum flux along the derivative's own axis
    for (int a : {0, 1, 2}) {
        Item fx[5];
        for (int k = 0; k < 5; k++)
            fx[k] = {g->fl + (5LL * a + k) * N, rhs + k * N, k == 1 + a ? 1 : -1, g->Q + k * N, Wp(g, k)};
        if (!rc) rc = apply(g, g->der[a], PADE_D1, a, fx, 1, a != 0, a == 0 ? 1.0 : -1.0, s, a == 2 ? stage : nullptr);
    }
    return rc;
}

int post_bc_impl(pade_cgrid_t g, hipStream_t s)
{
    // cgrid.F90:813-820: e from p, then T (IdealGasEOS.F90:54-70)
    return pade::cg_post_bc(g->N, F(g, PADE_CG_RHO), F(g, PADE_CG_P), g->gam, g->Rgas, F(g, PADE_CG_E),
                            F(g, PADE_CG_T), s);
}

// The word that the kernels lower to the first bad index of W: all ones
// before, read back after them.
int reset_bad(pade_cgrid_t g, hipStream_t s)
{
    hipError_t e = hipMemsetAsync(g->dscal, 0xff, sizeof(unsigned long long), s);
    return e == hipSuccess ? 0 : err(1000 + int(e), "bad-index reset");
}

int read_bad(pade_cgrid_t g, long long *bad, hipStream_t s)
{
    hipError_t e = hipMemcpyAsync(g->hscal, g->dscal, sizeof(unsigned long long), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return err(1000 + int(e), "bad-index read");
    *bad = g->hscal[0] == ~0ull ? -1 : (long long)g->hscal[0];
    return 0;
}

int conserved_impl(pade_cgrid_t g, bool check, long long *bad, hipStream_t s)
{
    if (check)
        if (int rc = reset_bad(g, s)) return rc;
    int rc = pade_cg_conserved(g->N, F(g, PADE_CG_RHO), F(g, PADE_CG_U), F(g, PADE_CG_V), F(g, PADE_CG_W_VEL),
                               F(g, PADE_CG_E), F(g, PADE_CG_W), check ? g->dscal : nullptr, s);
    return rc || !check ? rc : read_bad(g, bad, s);
}

void release(pade_cgrid_t g)
{
    for (int a = 0; a < 3; a++) {
        pade_op_destroy(g->der[a]);
        pade_op_destroy(g->fil[a]);
        pade_op_destroy(g->gfil[a]);
    }
    for (int k = 0; k < PADE_CG_NFIELDS; k++)
        if (g->own[k] && g->f[k]) (void)hipFree(g->f[k]);
    if (g->work) (void)hipFree(g->work);
    if (g->dscal) (void)hipFree(g->dscal);
    if (g->hscal) (void)hipHostFree(g->hscal);
    delete g;
}

}  // namespace

extern "C" {

int pade_cgrid_create(int nx, int ny, int nz, double dx, double dy, double dz, int derivative, int filter_kind,
                      const double *params, int inviscid, const int *periodic, const int *bc, double *const *fields,
                      pade_cgrid_t *out)
{
    if (!out) return err(400, "null output handle");
    *out = nullptr;
    if (nx < 1 || ny < 1 || nz < 1) return err(400, "grid sizes must be positive");
    if (!(dx > 0.0) || !(dy > 0.0) || !(dz > 0.0)) return err(400, "grid spacings must be positive");
    if (derivative != PADE_CD10 && derivative != PADE_CD06) return err(1, "Invalid derivative method (cd10 or cd06)");
    if (filter_kind != PADE_CF90 && filter_kind != PADE_GAUSSIAN) return err(1, "Invalid filter (cf90 or gaussian)");
    pade_cgrid_t g = new pade_cgrid_s;
    g->n[0] = nx; g->n[1] = ny; g->n[2] = nz;
    g->N = (long long)nx * ny * nz;
    g->h[0] = dx; g->h[1] = dy; g->h[2] = dz;
    if (params) {
        g->gam = params[0]; g->Rgas = params[1]; g->Cmu = params[2]; g->Cbeta = params[3]; g->Ckap = params[4];
        g->mu_ref = params[5]; g->T_ref = params[6]; g->visc_n = params[7]; g->Pr = params[8];
    }
    g->inviscid = inviscid != 0;
    g->der_kind = derivative;
    for (int a = 0; a < 3; a++) {
        g->periodic[a] = periodic ? periodic[a] != 0 : true;
        const int b1 = (!g->periodic[a] && bc) ? bc[2 * a] : 0, bn = (!g->periodic[a] && bc) ? bc[2 * a + 1] : 0;
        auto okbc = [](int b) { return b == 0 || b == 1 || b == -1; };
        if (!okbc(b1) || !okbc(bn)) {
            release(g);
            return err(324, "Incorrect boundary specification (should be 0, 1 or -1)");
        }
        g->bc[a][0] = b1;
        g->bc[a][1] = bn;
        // derivatives.F90:276-389, filters.F90 init, cgrid.F90:321-340
        int rc = pade_op_create(derivative, g->n[a], g->h[a], g->periodic[a], 0, 0, &g->der[a]);
        if (rc) {
            release(g);
            return err(derivative == PADE_CD10 ? 11 : 12, "Initializing the derivative operator failed");
        }
        rc = pade_op_create(filter_kind, g->n[a], 0.0, g->periodic[a], 0, 0, &g->fil[a]);
        if (!rc) rc = pade_op_create(PADE_GAUSSIAN, g->n[a], 0.0, g->periodic[a], 0, 0, &g->gfil[a]);
        if (rc) {
            release(g);
            return err(51, "Initializing the filter failed");
        }
    }
    const size_t fb = sizeof(double) * (size_t)g->N;
    for (int k = 0; k < PADE_CG_NFIELDS; k++) {
        double *p = fields ? fields[k] : nullptr;
        if (!p) {
            hipError_t e = hipMalloc(&p, k == PADE_CG_W ? 5 * fb : fb);
            if (e != hipSuccess) {
                release(g);
                return err(1000 + int(e), "field allocation");
            }
            g->own[k] = true;
        }
        g->f[k] = p;
    }
    // t1 | du 9 | gT 3 | fl 15 | rhs 5 | Q 5 | mustar func dil
    const int nwork = 1 + 9 + 3 + 15 + 5 + 5 + 3;
    hipError_t e = hipMalloc(&g->work, fb * nwork);
    if (e == hipSuccess) e = hipMalloc(&g->dscal, 8 * sizeof(unsigned long long));
    if (e == hipSuccess) e = hipHostMalloc(&g->hscal, 8 * sizeof(unsigned long long), hipHostMallocDefault);
    if (e != hipSuccess) {
        release(g);
        return err(1000 + int(e), "work allocation");
    }
    double *w = g->work;
    auto take = [&](int k) { double *p = w; w += (long long)k * g->N; return p; };
    g->t1 = take(1); g->du = take(9); g->gT = take(3); g->fl = take(15); g->rhs = take(5);
    g->Q = take(5); g->mustar = take(1); g->func = take(1); g->dil = take(1);
    *out = g;
    return 0;
}

int pade_cgrid_destroy(pade_cgrid_t g)
{
    if (g) release(g);
    return 0;
}

int pade_cgrid_field(pade_cgrid_t g, int which, double **ptr)
{
    if (!g || !ptr || which < 0 || which >= PADE_CG_NFIELDS) return err(400, "bad field request");
    *ptr = g->f[which];
    return 0;
}

int pade_cgrid_state(pade_cgrid_t g, int *step, double *tsim, double *dt)
{
    if (!g) return err(400, "null grid");
    if (step) *step = g->step;
    if (tsim) *tsim = g->tsim;
    if (dt) *dt = g->dt;
    return 0;
}

int pade_cgrid_set_state(pade_cgrid_t g, int step, double tsim, double dtfixed)
{
    if (!g) return err(400, "null grid");
    g->step = step;
    g->tsim = tsim;
    g->dtfixed = dtfixed;
    return 0;
}

int pade_cgrid_post_bc(pade_cgrid_t g, void *stream)
{
    if (!g) return err(400, "null grid");
    return post_bc_impl(g, (hipStream_t)stream);
}

int pade_cgrid_get_conserved(pade_cgrid_t g, long long *bad_index, void *stream)
{
    if (!g) return err(400, "null grid");
    long long bad = -1;
    int rc = conserved_impl(g, bad_index != nullptr, &bad, (hipStream_t)stream);
    if (bad_index) *bad_index = bad;
    return rc;
}

int pade_cgrid_transport(pade_cgrid_t g, void *stream)
{
    if (!g) return err(400, "null grid");
    return transport(g, (hipStream_t)stream);
}

int pade_cgrid_get_primitive(pade_cgrid_t g, void *stream)
{
    if (!g) return err(400, "null grid");
    return pade_cg_primitive(g->N, F(g, PADE_CG_W), g->gam, g->Rgas, F(g, PADE_CG_RHO), F(g, PADE_CG_U),
                             F(g, PADE_CG_V), F(g, PADE_CG_W_VEL), F(g, PADE_CG_E), F(g, PADE_CG_P), F(g, PADE_CG_T),
                             (hipStream_t)stream);
}

int pade_cgrid_rhs(pade_cgrid_t g, double *rhs, void *stream)
{
    if (!g || !rhs) return err(400, "null grid or array");
    return rhs_impl(g, rhs, (hipStream_t)stream);
}

int pade_cgrid_get_dt(pade_cgrid_t g, double CFL, double *dt, int *stability, void *stream)
{
    if (!g || !dt) return err(400, "null grid or output");
    hipStream_t s = (hipStream_t)stream;
    if (CFL <= 0.0) {                                  // cgrid.F90:741-743
        g->dt = g->dtfixed;
        *dt = g->dt;
        if (stability) *stability = PADE_CG_DT_FIXED;
        return 0;
    }
    const double hmin = std::fmin(g->h[0], std::fmin(g->h[1], g->h[2]));
    double mx[4];
    int rc = pade::cg_dt_maxima(g->N, F(g, PADE_CG_RHO), F(g, PADE_CG_U), F(g, PADE_CG_V), F(g, PADE_CG_W_VEL),
                                F(g, PADE_CG_P), F(g, PADE_CG_MU), F(g, PADE_CG_BULK), F(g, PADE_CG_KAP),
                                F(g, PADE_CG_T), g->h[0], g->h[1], g->h[2], g->gam, hmin, g->dscal + 1, g->hscal + 1,
                                mx, s);
    if (rc) return rc;
    const double dtCFL = CFL / mx[0];
    const double dtmu = 0.2 * hmin * hmin / (mx[1] + kMachineEps);
    const double dtbulk = 0.2 * hmin * hmin / (mx[2] + kMachineEps);
    const double dtkap = 0.2 / (std::pow(mx[3], 1.0 / 3.0) + kMachineEps);
    int why = PADE_CG_DT_CONVECTIVE;
    double d = dtCFL;
    if (d > dtmu) { d = dtmu; why = PADE_CG_DT_SHEAR; }
    else if (d > dtbulk) { d = dtbulk; why = PADE_CG_DT_BULK; }
    else if (d > dtkap) { d = dtkap; why = PADE_CG_DT_CONDUCTIVE; }
    if (g->step <= 10) { d = d / 10.0; why = PADE_CG_DT_STARTUP; }
    g->dt = d;
    *dt = d;
    if (stability) *stability = why;
    return 0;
}

int pade_cgrid_advance_rk45(pade_cgrid_t g, double dt, pade_cgrid_hook hook_bc, void *user, int *bad_substep,
                            long long *bad_index, void *stream)
{
    if (!g) return err(400, "null grid");
    hipStream_t s = (hipStream_t)stream;
    if (bad_substep) *bad_substep = 0;
    if (bad_index) *bad_index = -1;
    if (dt > 0.0) g->dt = dt;
    int rc = 0;
    if (g->step == 0) rc = post_bc_impl(g, s);         // get_e_from_p, get_T (:675-679)
    if (!rc) rc = pade::cg_fill(g->Q, 5 * g->N, 0.0, s);
    double Qt = 0.0;
    for (int isub = 0; isub < 5 && !rc; isub++) {
        long long bad = -1;
        // (without a hook the state update of the substep before formed W and
        // its test already)
        rc = isub == 0 || hook_bc ? conserved_impl(g, true, &bad, s) : read_bad(g, &bad, s);
        if (rc) break;
        if (bad >= 0) {                                  // nancheck, :684-692
            if (bad_substep) *bad_substep = isub + 1;
            if (bad_index) *bad_index = bad;
            const long long l = bad / g->N, r = bad % g->N;
            const long long i = r % g->n[0], j = (r / g->n[0]) % g->n[1], k = r / ((long long)g->n[0] * g->n[1]);
            return err(999, "NaN encountered in solution at substep " + std::to_string(isub + 1) + " of step " +
                                std::to_string(g->step + 1) + " at Wcnsrv(" + std::to_string(i + 1) + "," +
                                std::to_string(j + 1) + "," + std::to_string(k + 1) + "," + std::to_string(l + 1) +
                                ")");
        }
        const pade::Stage stage = {g->dt, kRkA[isub], kRkB[isub]};
        rc = rhs_impl(g, g->rhs, s, &stage);
        Qt = g->dt + kRkA[isub] * Qt;
        g->tsim += kRkB[isub] * Qt;
        // the momentum component along an axis is odd at its walls (:701-706)
        const int flips[5] = {-1, 0, 1, 2, -1};
        double *const W[5] = {Wp(g, 0), Wp(g, 1), Wp(g, 2), Wp(g, 3), Wp(g, 4)};
        const double *const Wc[5] = {W[0], W[1], W[2], W[3], W[4]};
        if (!rc) rc = filter(g, Wc, W, flips, g->fil, 1, false, s);
        if (!rc && !hook_bc && isub < 4) {
            rc = reset_bad(g, s);
            if (!rc)
                rc = pade::cg_primitive_conserved(g->N, F(g, PADE_CG_W), g->gam, g->Rgas, F(g, PADE_CG_RHO),
                                                  F(g, PADE_CG_U), F(g, PADE_CG_V), F(g, PADE_CG_W_VEL),
                                                  F(g, PADE_CG_E), F(g, PADE_CG_P), F(g, PADE_CG_T), g->dscal, s);
        } else if (!rc) {
            rc = pade_cgrid_get_primitive(g, stream);
        }
        if (!rc && hook_bc) {
            hook_bc(g, user);
            rc = post_bc_impl(g, s);
        }
    }
    if (!rc) g->step += 1;
    return rc;
}

}  // extern "C"
