// Pointwise stages of the compressible solver's Runge-Kutta substep
// (src/compressible/cgrid.F90, one ideal-gas species): each kernel is one
// streaming pass over the fields that a group of the reference's array
// statements reads and writes, so that a substep moves each field a few
// times instead of once per statement.  Fields are FP64 arrays of N points;
// groups of fields (the five conserved variables, the nine velocity
// gradients, three gradient components, fifteen fluxes) are planes of one
// allocation, plane k at base + k * N.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "padeops_hip.h"
#include "pade_cgrid.h"
#include "pade_err.h"

namespace pade {
namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(long long n)
{
    const long long b = (n + kBlock - 1) / kBlock;
    return (unsigned)std::min<long long>(std::max<long long>(b, 1), 1LL << 20);
}

#define GRID_STRIDE(i, n) \
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (long long)gridDim.x * blockDim.x)

// Output stores.  The two kernels that write the most planes stream them past
// the caches (nontemporal) when the planes of a step, some fifty, cannot stay
// in the 256 MB last-level cache anyway; smaller grids keep them there for the
// next kernel.  256^3: k_fluxes 902 -> 862 us, k_lad 548 -> 527 us; 96 x 80 x 65
// (200 MB in all) is 1 % slower with streamed stores.
template <bool STREAM>
__device__ __forceinline__ void put(double *p, double v)
{
    if constexpr (STREAM) __builtin_nontemporal_store(v, p);
    else *p = v;
}
inline bool stream_planes(long long n) { return n >= 1LL << 20; }

// The test of nancheck (src/utilities/exits.F90:154,197): isnan(f) .OR.
// f + one == f, which also holds for +-Inf and for |f| >= 2^53 (the library
// is built without fast-math, so the comparison is IEEE).
__device__ __forceinline__ bool bad_value(double x) { return (x != x) | (x + 1.0 == x); }

// get_conserved, cgrid.F90:799-811, with the test of advance_RK45
// (:684-692) fused into the pass: bad_index is lowered (atomicMin) to the
// smallest plane-major linear index l * n + i of a W value that fails it,
// the first one nancheck_ind's Fortran-order loops find (exits.F90:188-210).
// Only lanes that saw such a value touch it.
__global__ __launch_bounds__(kBlock) void k_conserved(long long n, const double *__restrict__ rho,
                                                      const double *__restrict__ u, const double *__restrict__ v,
                                                      const double *__restrict__ w, const double *__restrict__ e,
                                                      double *__restrict__ W, unsigned long long *__restrict__ bad_index)
{
    unsigned long long first = ~0ull;
    GRID_STRIDE(i, n)
    {
        const double r = rho[i], uu = u[i], vv = v[i], ww = w[i];
        const double w1 = r * uu, w2 = r * vv, w3 = r * ww;
        const double w4 = r * (e[i] + 0.5 * (uu * uu + vv * vv + ww * ww));
        W[i] = r;
        W[n + i] = w1;
        W[2 * n + i] = w2;
        W[3 * n + i] = w3;
        W[4 * n + i] = w4;
        if (bad_value(r) | bad_value(w1) | bad_value(w2) | bad_value(w3) | bad_value(w4)) {
            const int l = bad_value(r) ? 0 : bad_value(w1) ? 1 : bad_value(w2) ? 2 : bad_value(w3) ? 3 : 4;
            const unsigned long long idx = (unsigned long long)(l * n + i);
            first = idx < first ? idx : first;
        }
    }
    if (bad_index && first != ~0ull) atomicMin(bad_index, first);
}

// get_primitive (cgrid.F90:764-797) followed by post_bc (:813-820):
// p from (rho, e), then e and T from (rho, p) (IdealGasEOS.F90:45-70)
__global__ __launch_bounds__(kBlock) void k_primitive(long long n, const double *__restrict__ W, double gam,
                                                      double Rgas, double *__restrict__ rho, double *__restrict__ u,
                                                      double *__restrict__ v, double *__restrict__ w,
                                                      double *__restrict__ e, double *__restrict__ p,
                                                      double *__restrict__ T)
{
    GRID_STRIDE(i, n)
    {
        const double r = W[i];
        const double onebyrho = 1.0 / r;
        const double uu = W[n + i] * onebyrho, vv = W[2 * n + i] * onebyrho, ww = W[3 * n + i] * onebyrho;
        const double ee = W[4 * n + i] * onebyrho - 0.5 * (uu * uu + vv * vv + ww * ww);
        const double pp = (gam - 1.0) * r * ee;
        const double e2 = pp / (gam - 1.0) / r;
        rho[i] = r;
        u[i] = uu;
        v[i] = vv;
        w[i] = ww;
        p[i] = pp;
        e[i] = e2;
        T[i] = e2 * ((gam - 1.0) / Rgas);
    }
}

// k_primitive, then k_conserved of its result, in one pass (5 fields read
// instead of 10).
__global__ __launch_bounds__(kBlock) void k_primitive_conserved(long long n, double *W, double gam, double Rgas,
                                                                double *__restrict__ rho, double *__restrict__ u,
                                                                double *__restrict__ v, double *__restrict__ w,
                                                                double *__restrict__ e, double *__restrict__ p,
                                                                double *__restrict__ T,
                                                                unsigned long long *__restrict__ bad_index)
{
    unsigned long long first = ~0ull;
    GRID_STRIDE(i, n)
    {
        const double r = W[i];
        const double onebyrho = 1.0 / r;
        const double uu = W[n + i] * onebyrho, vv = W[2 * n + i] * onebyrho, ww = W[3 * n + i] * onebyrho;
        const double ee = W[4 * n + i] * onebyrho - 0.5 * (uu * uu + vv * vv + ww * ww);
        const double pp = (gam - 1.0) * r * ee;
        const double e2 = pp / (gam - 1.0) / r;
        rho[i] = r;
        u[i] = uu;
        v[i] = vv;
        w[i] = ww;
        p[i] = pp;
        e[i] = e2;
        T[i] = e2 * ((gam - 1.0) / Rgas);
        const double w1 = r * uu, w2 = r * vv, w3 = r * ww;
        const double w4 = r * (e2 + 0.5 * (uu * uu + vv * vv + ww * ww));
        W[n + i] = w1;
        W[2 * n + i] = w2;
        W[3 * n + i] = w3;
        W[4 * n + i] = w4;
        if (bad_value(r) | bad_value(w1) | bad_value(w2) | bad_value(w3) | bad_value(w4)) {
            const int l = bad_value(r) ? 0 : bad_value(w1) ? 1 : bad_value(w2) ? 2 : bad_value(w3) ? 3 : 4;
            const unsigned long long idx = (unsigned long long)(l * n + i);
            first = idx < first ? idx : first;
        }
    }
    if (first != ~0ull) atomicMin(bad_index, first);
}

// LAD shear-viscosity sensor: magnitude of the strain rate (cgrid.F90:1085-1087);
// du planes: du/dx du/dy du/dz dv/dx ... dw/dz
__global__ __launch_bounds__(kBlock) void k_strain(long long n, const double *__restrict__ du,
                                                   double *__restrict__ func, double *__restrict__ dil)
{
    GRID_STRIDE(i, n)
    {
        const double ux = du[i], uy = du[n + i], uz = du[2 * n + i];
        const double vx = du[3 * n + i], vy = du[4 * n + i], vz = du[5 * n + i];
        const double wx = du[6 * n + i], wy = du[7 * n + i], wz = du[8 * n + i];
        func[i] = sqrt(ux * ux + 0.5 * (vx + uy) * (vx + uy) + 0.5 * (wx + uz) * (wx + uz) + vy * vy +
                       0.5 * (wy + vz) * (wy + vz) + wz * wz);
        dil[i] = ux + vy + wz;
    }
}

// mustar = Cmu rho |sum of h^6-weighted fourth derivatives| (cgrid.F90:1110)
__global__ __launch_bounds__(kBlock) void k_lad_mu(long long n, double Cmu, const double *__restrict__ rho,
                                                   double *__restrict__ mustar)
{
    GRID_STRIDE(i, n) { mustar[i] = Cmu * rho[i] * fabs(mustar[i]); }
}

// artificial bulk viscosity (cgrid.F90:1115-1158): g = grad(rho) planes,
// d4 = fourth derivatives of the dilatation along x, y, z
__global__ __launch_bounds__(kBlock) void k_lad_bulk(long long n, double Cbeta, double hx, double hy, double hz,
                                                     const double *__restrict__ rho, const double *__restrict__ g,
                                                     const double *__restrict__ d4, const double *__restrict__ du,
                                                     const double *__restrict__ dil, double *__restrict__ bulk)
{
    const double hx4 = hx * hx * hx * hx, hy4 = hy * hy * hy * hy, hz4 = hz * hz * hz * hz;
    GRID_STRIDE(i, n)
    {
        const double g1 = g[i] * g[i], g2 = g[n + i] * g[n + i], g3 = g[2 * n + i] * g[2 * n + i];
        const double den = g1 + g2 + g3 + 1.0e-32;
        const double ax = hx * g1 / den, ay = hy * g2 / den, az = hz * g3 / den;
        double b = d4[i] * hx4 * (ax * ax);
        b = b + d4[2 * n + i] * hz4 * (az * az);
        b = b + d4[n + i] * hy4 * (ay * ay);
        const double uy = du[n + i], uz = du[2 * n + i], vx = du[3 * n + i], vz = du[5 * n + i];
        const double wx = du[6 * n + i], wy = du[7 * n + i];
        const double c1 = wy - vz, c2 = uz - wx, c3 = vx - uy;
        const double curl2 = c1 * c1 + c2 * c2 + c3 * c3;
        const double f = dil[i];
        const double d2 = f * f;
        const double fsw = f >= 0.0 ? 0.0 : d2 / (d2 + curl2 + 1.0e-32);
        bulk[i] = Cbeta * rho[i] * fsw * fabs(b);
    }
}

// artificial conductivity (cgrid.F90:1163-1196): g = grad(e) planes, d4 =
// fourth derivatives of e along x, y, z
__global__ __launch_bounds__(kBlock) void k_lad_kap(long long n, double Ckap, double gam, double hx, double hy,
                                                    double hz, const double *__restrict__ rho,
                                                    const double *__restrict__ p, const double *__restrict__ T,
                                                    const double *__restrict__ g, const double *__restrict__ d4,
                                                    double *__restrict__ kap)
{
    const double hx4 = hx * hx * hx * hx, hy4 = hy * hy * hy * hy, hz4 = hz * hz * hz * hz;
    GRID_STRIDE(i, n)
    {
        const double g1 = g[i] * g[i], g2 = g[n + i] * g[n + i], g3 = g[2 * n + i] * g[2 * n + i];
        const double den = g1 + g2 + g3 + 1.0e-32;
        double k = d4[i] * hx4 * (hx * g1 / den);
        k = k + d4[2 * n + i] * hz4 * (hz * g3 / den);
        k = k + d4[n + i] * hy4 * (hy * g2 / den);
        const double sos = sqrt(gam * p[i] / rho[i]);
        kap[i] = Ckap * rho[i] * sos * fabs(k) / T[i];
    }
}

// k_strain with the bulk viscosity's switch, which reads the same velocity
// gradients: one plane written here instead of seven read by k_lad.
__global__ __launch_bounds__(kBlock) void k_strain_switch(long long n, const double *__restrict__ du,
                                                          double *__restrict__ func, double *__restrict__ dil,
                                                          double *__restrict__ fsw)
{
    GRID_STRIDE(i, n)
    {
        const double ux = du[i], uy = du[n + i], uz = du[2 * n + i];
        const double vx = du[3 * n + i], vy = du[4 * n + i], vz = du[5 * n + i];
        const double wx = du[6 * n + i], wy = du[7 * n + i], wz = du[8 * n + i];
        func[i] = sqrt(ux * ux + 0.5 * (vx + uy) * (vx + uy) + 0.5 * (wx + uz) * (wx + uz) + vy * vy +
                       0.5 * (wy + vz) * (wy + vz) + wz * wz);
        const double f = ux + vy + wz;
        dil[i] = f;
        const double c1 = wy - vz, c2 = uz - wx, c3 = vx - uy;
        const double curl2 = c1 * c1 + c2 * c2 + c3 * c3;
        const double d2 = f * f;
        fsw[i] = f >= 0.0 ? 0.0 : d2 / (d2 + curl2 + 1.0e-32);
    }
}

// k_lad_mu, k_lad_bulk and k_lad_kap in one pass: 19 fields read and 3
// written instead of 33 and 3 (and no accumulating passes for mustar).
template <bool STREAM>
__global__ __launch_bounds__(kBlock) void k_lad(long long n, double Cmu, double Cbeta, double Ckap, double gam,
                                                double hx, double hy, double hz, const double *__restrict__ rho,
                                                const double *__restrict__ p, const double *__restrict__ T,
                                                const double *__restrict__ fl, double *mustar,
                                                double *__restrict__ bulkstar, double *__restrict__ kapstar)
{
    const double hx4 = hx * hx * hx * hx, hy4 = hy * hy * hy * hy, hz4 = hz * hz * hz * hz;
    const double hx6 = hx4 * hx * hx, hy6 = hy4 * hy * hy, hz6 = hz4 * hz * hz;
    GRID_STRIDE(i, n)
    {
        const double r = rho[i], fsw = mustar[i];
        double m = hx6 * fl[6 * n + i];
        m = m + hz6 * fl[8 * n + i];
        m = m + hy6 * fl[7 * n + i];
        put<STREAM>(mustar + i, Cmu * r * fabs(m));
        double g1 = fl[i] * fl[i], g2 = fl[n + i] * fl[n + i], g3 = fl[2 * n + i] * fl[2 * n + i];
        double den = g1 + g2 + g3 + 1.0e-32;
        const double ax = hx * g1 / den, ay = hy * g2 / den, az = hz * g3 / den;
        double b = fl[9 * n + i] * hx4 * (ax * ax);
        b = b + fl[11 * n + i] * hz4 * (az * az);
        b = b + fl[10 * n + i] * hy4 * (ay * ay);
        put<STREAM>(bulkstar + i, Cbeta * r * fsw * fabs(b));
        g1 = fl[3 * n + i] * fl[3 * n + i];
        g2 = fl[4 * n + i] * fl[4 * n + i];
        g3 = fl[5 * n + i] * fl[5 * n + i];
        den = g1 + g2 + g3 + 1.0e-32;
        double k = fl[12 * n + i] * hx4 * (hx * g1 / den);
        k = k + fl[14 * n + i] * hz4 * (hz * g3 / den);
        k = k + fl[13 * n + i] * hy4 * (hy * g2 / den);
        const double sos = sqrt(gam * p[i] / r);
        put<STREAM>(kapstar + i, Ckap * r * sos * fabs(k) / T[i]);
    }
}

// get_tau (cgrid.F90:1338-1390), get_q (:1392-1444) and the fluxes of
// getRHS_x/y/z (:898-1056): f planes x (5), y (5), z (5); gT = grad(T).
// The x fluxes are stored negated: the right-hand side starts as d(-fx)/dx,
// which equals 0 - d(fx)/dx bit for bit (the operator is linear and
// negation exact), so it needs neither a cleared array nor an accumulate.
template <bool STREAM>
__global__ __launch_bounds__(kBlock) void k_fluxes(long long n, const double *__restrict__ W,
                                                   const double *__restrict__ u, const double *__restrict__ v,
                                                   const double *__restrict__ w, const double *__restrict__ p,
                                                   const double *__restrict__ du, const double *__restrict__ mu,
                                                   const double *__restrict__ bulk, const double *__restrict__ kap,
                                                   const double *__restrict__ gT, double *__restrict__ f)
{
    GRID_STRIDE(i, n)
    {
        const double ux = du[i], uy = du[n + i], uz = du[2 * n + i];
        const double vx = du[3 * n + i], vy = du[4 * n + i], vz = du[5 * n + i];
        const double wx = du[6 * n + i], wy = du[7 * n + i], wz = du[8 * n + i];
        const double m = mu[i], bk = bulk[i], kp = kap[i];
        const double bambda = (4.0 / 3.0) * m + bk;
        const double lam = bk - (2.0 / 3.0) * m;
        const double txy = m * (uy + vx), txz = m * (uz + wx), tyz = m * (vz + wy);
        const double txx = bambda * ux + lam * (vy + wz);
        const double tyy = bambda * vy + lam * (ux + wz);
        const double tzz = bambda * wz + lam * (ux + vy);
        const double qx = -kp * gT[i], qy = -kp * gT[n + i], qz = -kp * gT[2 * n + i];
        const double ru = W[n + i], rv = W[2 * n + i], rw = W[3 * n + i], TE = W[4 * n + i];
        const double uu = u[i], vv = v[i], ww = w[i], pp = p[i];
        put<STREAM>(f + i, -ru);
        put<STREAM>(f + n + i, -(ru * uu + pp - txx));
        put<STREAM>(f + 2 * n + i, -(ru * vv - txy));
        put<STREAM>(f + 3 * n + i, -(ru * ww - txz));
        put<STREAM>(f + 4 * n + i, -((TE + pp - txx) * uu - vv * txy - ww * txz + qx));
        put<STREAM>(f + 5 * n + i, rv);
        put<STREAM>(f + 6 * n + i, rv * uu - txy);
        put<STREAM>(f + 7 * n + i, rv * vv + pp - tyy);
        put<STREAM>(f + 8 * n + i, rv * ww - tyz);
        put<STREAM>(f + 9 * n + i, (TE + pp - tyy) * vv - uu * txy - ww * tyz + qy);
        put<STREAM>(f + 10 * n + i, rw);
        put<STREAM>(f + 11 * n + i, rw * uu - txz);
        put<STREAM>(f + 12 * n + i, rw * vv - tyz);
        put<STREAM>(f + 13 * n + i, rw * ww + pp - tzz);
        put<STREAM>(f + 14 * n + i, (TE + pp - tzz) * ww - uu * txz - vv * tyz + qz);
    }
}

// low-storage RK45 stage (cgrid.F90:697-699) over the five conserved planes
__global__ __launch_bounds__(kBlock) void k_rk(long long n5, double dt, double A, double B,
                                               const double *__restrict__ rhs, double *__restrict__ Q,
                                               double *__restrict__ W)
{
    GRID_STRIDE(i, n5)
    {
        const double q = dt * rhs[i] + A * Q[i];
        Q[i] = q;
        W[i] = W[i] + B * q;
    }
}

// fill (the cleared accumulators of the step)
__global__ __launch_bounds__(kBlock) void k_fill(double *__restrict__ x, long long n, double v)
{
    GRID_STRIDE(i, n) { x[i] = v; }
}

// transport properties, MixtureEOS.F90:175-229 (ns = 1) with the power-law
// viscosity of PowerLawViscosity.F90:38-75: mu = mu_ref (T / T_ref)^n,
// bulk = 0, kap = mu Cp / Pr
__global__ __launch_bounds__(kBlock) void k_transport(long long n, const double *__restrict__ T, double mu_ref,
                                                      double T_ref, double visc_n, double cp_by_pr,
                                                      double *__restrict__ mu, double *__restrict__ bulk,
                                                      double *__restrict__ kap)
{
    GRID_STRIDE(i, n)
    {
        const double m = pow(T[i] / T_ref, visc_n) * mu_ref;
        mu[i] = m;
        bulk[i] = 0.0;
        kap[i] = m * cp_by_pr;
    }
}

// post_bc, cgrid.F90:813-820: e from (rho, p), then T (IdealGasEOS.F90:54-70)
__global__ __launch_bounds__(kBlock) void k_post_bc(long long n, const double *__restrict__ rho,
                                                    const double *__restrict__ p, double gam, double Rgas,
                                                    double *__restrict__ e, double *__restrict__ T)
{
    GRID_STRIDE(i, n)
    {
        const double ee = p[i] / (gam - 1.0) / rho[i];
        e[i] = ee;
        T[i] = ee * ((gam - 1.0) / Rgas);
    }
}

// Order-preserving unsigned key of a double (larger double, larger key; NaN
// above +Inf, as a maximum that propagates NaN), and back.
__device__ __forceinline__ unsigned long long max_key(double x)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__host__ __device__ inline double key_value(unsigned long long k)
{
    const unsigned long long b = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    double x;
    __builtin_memcpy(&x, &b, 8);
    return x;
}

// the four maxima of get_dt (cgrid.F90:728-733): the convective rate, mu /
// rho, bulk / rho, kap T / (rho h^4); keys lowered per wave into out[0..3]
__global__ __launch_bounds__(kBlock) void k_dt_maxima(long long n, const double *__restrict__ rho,
                                                      const double *__restrict__ u, const double *__restrict__ v,
                                                      const double *__restrict__ w, const double *__restrict__ p,
                                                      const double *__restrict__ mu, const double *__restrict__ bulk,
                                                      const double *__restrict__ kap, const double *__restrict__ T,
                                                      double dx, double dy, double dz, double gam, double cfac,
                                                      double h4, unsigned long long *__restrict__ out)
{
    unsigned long long m[4] = {0, 0, 0, 0};
    GRID_STRIDE(i, n)
    {
        const double r = rho[i];
        const double cs = sqrt(gam * p[i] / r);
        const double c = fabs(u[i]) / dx + fabs(v[i]) / dy + fabs(w[i]) / dz + cs * cfac;
        const unsigned long long k[4] = {max_key(c), max_key(mu[i] / r), max_key(bulk[i] / r),
                                         max_key(kap[i] * T[i] / (r * h4))};
#pragma unroll
        for (int q = 0; q < 4; q++) m[q] = k[q] > m[q] ? k[q] : m[q];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        unsigned long long x = m[q];
        for (int off = 32; off >= 1; off >>= 1) {
            const unsigned long long y = __shfl_xor(x, off, 64);
            x = y > x ? y : x;
        }
        if ((threadIdx.x & 63) == 0 && x) atomicMax(out + q, x);
    }
}

// Status of the launch just made; callers clear stale errors of earlier,
// unrelated calls (hipGetLastError) before launching.
int launched(const char *what)
{
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) return 0;
    return set_error(1000 + int(e), what);
}

int bad_args(const char *what) { return set_error(400, what); }

}  // namespace

int cg_fill(double *x, long long n, double v, hipStream_t s)
{
    if (n < 1) return 0;
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(kBlock), 0, s, x, n, v);
    return launched("fill launch");
}

int cg_lad(long long n, double Cmu, double Cbeta, double Ckap, double gam, const double *h, const double *rho,
           const double *p, const double *T, const double *fl, double *mustar, double *bulkstar, double *kapstar,
           hipStream_t s)
{
    (void)hipGetLastError();
    hipLaunchKernelGGL((stream_planes(n) ? k_lad<true> : k_lad<false>), dim3(grid_for(n)), dim3(kBlock), 0, s, n, Cmu,
                       Cbeta, Ckap, gam, h[0], h[1], h[2], rho, p, T, fl, mustar, bulkstar, kapstar);
    return launched("artificial-property launch");
}

int cg_strain_switch(long long n, const double *du, double *func, double *dil, double *fsw, hipStream_t s)
{
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_strain_switch, dim3(grid_for(n)), dim3(kBlock), 0, s, n, du, func, dil, fsw);
    return launched("strain launch");
}

int cg_rk_stage(long long n, double dt, double A, double B, const double *rhs, double *Q, double *W, hipStream_t s)
{
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_rk, dim3(grid_for(n)), dim3(kBlock), 0, s, n, dt, A, B, rhs, Q, W);
    return launched("RK stage launch");
}

int cg_primitive_conserved(long long n, double *W, double gam, double Rgas, double *rho, double *u, double *v,
                           double *w, double *e, double *p, double *T, unsigned long long *bad_index, hipStream_t s)
{
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_primitive_conserved, dim3(grid_for(n)), dim3(kBlock), 0, s, n, W, gam, Rgas, rho, u, v, w, e,
                       p, T, bad_index);
    return launched("state update launch");
}

int cg_transport(long long n, const double *T, double mu_ref, double T_ref, double visc_n, double cp_by_pr,
                 double *mu, double *bulk, double *kap, hipStream_t s)
{
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_transport, dim3(grid_for(n)), dim3(kBlock), 0, s, n, T, mu_ref, T_ref, visc_n, cp_by_pr, mu,
                       bulk, kap);
    return launched("transport-property launch");
}

int cg_post_bc(long long n, const double *rho, const double *p, double gam, double Rgas, double *e, double *T,
               hipStream_t s)
{
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_post_bc, dim3(grid_for(n)), dim3(kBlock), 0, s, n, rho, p, gam, Rgas, e, T);
    return launched("post_bc launch");
}

int cg_dt_maxima(long long n, const double *rho, const double *u, const double *v, const double *w, const double *p,
                 const double *mu, const double *bulk, const double *kap, const double *T, double dx, double dy,
                 double dz, double gam, double hmin, unsigned long long *dev4, unsigned long long *host4, double *out,
                 hipStream_t s)
{
    const double cfac = sqrt(1.0 / (dx * dx) + 1.0 / (dy * dy) + 1.0 / (dz * dz));
    const double h4 = hmin * hmin * hmin * hmin;
    if (int rc = cg_fill(reinterpret_cast<double *>(dev4), 4, 0.0, s)) return rc;   // key 0: below every value
    // at most a few waves per CU: each wave reduces before one atomic per maximum
    const unsigned grid = std::min<unsigned>(grid_for(n), 2048);
    hipLaunchKernelGGL(k_dt_maxima, dim3(grid), dim3(kBlock), 0, s, n, rho, u, v, w, p, mu, bulk, kap, T, dx, dy, dz,
                       gam, cfac, h4, dev4);
    if (int rc = launched("get_dt reduction launch")) return rc;
    hipError_t e = hipMemcpyAsync(host4, dev4, 4 * sizeof(unsigned long long), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return set_error(1000 + int(e), "get_dt reduction read");
    for (int q = 0; q < 4; q++) out[q] = key_value(host4[q]);
    return 0;
}

}  // namespace pade

using namespace pade;

extern "C" {

int pade_cg_conserved(long long n, const double *rho, const double *u, const double *v, const double *w,
                      const double *e, double *W, unsigned long long *bad_index, void *stream)
{
    if (n < 1 || !rho || !u || !v || !w || !e || !W) return bad_args("pade_cg_conserved: n < 1 or a null array");
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_conserved, dim3(grid_for(n)), dim3(kBlock), 0, (hipStream_t)stream, n, rho, u, v, w, e, W,
                       bad_index);
    return launched("pade_cg_conserved launch");
}

int pade_cg_primitive(long long n, const double *W, double gam, double Rgas, double *rho, double *u, double *v,
                      double *w, double *e, double *p, double *T, void *stream)
{
    if (n < 1 || !W || !rho || !u || !v || !w || !e || !p || !T)
        return bad_args("pade_cg_primitive: n < 1 or a null array");
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_primitive, dim3(grid_for(n)), dim3(kBlock), 0, (hipStream_t)stream, n, W, gam, Rgas, rho,
                       u, v, w, e, p, T);
    return launched("pade_cg_primitive launch");
}

int pade_cg_strain(long long n, const double *du, double *func, double *dil, void *stream)
{
    if (n < 1 || !du || !func || !dil) return bad_args("pade_cg_strain: n < 1 or a null array");
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_strain, dim3(grid_for(n)), dim3(kBlock), 0, (hipStream_t)stream, n, du, func, dil);
    return launched("pade_cg_strain launch");
}

int pade_cg_lad_mu(long long n, double Cmu, const double *rho, double *mustar, void *stream)
{
    if (n < 1 || !rho || !mustar) return bad_args("pade_cg_lad_mu: n < 1 or a null array");
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_lad_mu, dim3(grid_for(n)), dim3(kBlock), 0, (hipStream_t)stream, n, Cmu, rho, mustar);
    return launched("pade_cg_lad_mu launch");
}

int pade_cg_lad_bulk(long long n, double Cbeta, double hx, double hy, double hz, const double *rho,
                     const double *grad_rho, const double *d4, const double *du, const double *dil, double *bulk,
                     void *stream)
{
    if (n < 1 || !rho || !grad_rho || !d4 || !du || !dil || !bulk)
        return bad_args("pade_cg_lad_bulk: n < 1 or a null array");
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_lad_bulk, dim3(grid_for(n)), dim3(kBlock), 0, (hipStream_t)stream, n, Cbeta, hx, hy, hz,
                       rho, grad_rho, d4, du, dil, bulk);
    return launched("pade_cg_lad_bulk launch");
}

int pade_cg_lad_kap(long long n, double Ckap, double gam, double hx, double hy, double hz, const double *rho,
                    const double *p, const double *T, const double *grad_e, const double *d4, double *kap,
                    void *stream)
{
    if (n < 1 || !rho || !p || !T || !grad_e || !d4 || !kap) return bad_args("pade_cg_lad_kap: n < 1 or a null array");
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_lad_kap, dim3(grid_for(n)), dim3(kBlock), 0, (hipStream_t)stream, n, Ckap, gam, hx, hy, hz,
                       rho, p, T, grad_e, d4, kap);
    return launched("pade_cg_lad_kap launch");
}

int pade_cg_fluxes(long long n, const double *W, const double *u, const double *v, const double *w, const double *p,
                   const double *du, const double *mu, const double *bulk, const double *kap, const double *grad_T,
                   double *fluxes, void *stream)
{
    if (n < 1 || !W || !u || !v || !w || !p || !du || !mu || !bulk || !kap || !grad_T || !fluxes)
        return bad_args("pade_cg_fluxes: n < 1 or a null array");
    (void)hipGetLastError();
    hipLaunchKernelGGL((stream_planes(n) ? k_fluxes<true> : k_fluxes<false>), dim3(grid_for(n)), dim3(kBlock), 0,
                       (hipStream_t)stream, n, W, u, v, w, p, du, mu,
                       bulk, kap, grad_T, fluxes);
    return launched("pade_cg_fluxes launch");
}

int pade_cg_rk_stage(long long n, double dt, double A, double B, const double *rhs, double *Q, double *W, void *stream)
{
    if (n < 1 || !rhs || !Q || !W) return bad_args("pade_cg_rk_stage: n < 1 or a null array");
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_rk, dim3(grid_for(5 * n)), dim3(kBlock), 0, (hipStream_t)stream, 5 * n, dt, A, B, rhs, Q, W);
    return launched("pade_cg_rk_stage launch");
}

}  // extern "C"
