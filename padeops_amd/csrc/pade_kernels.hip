// One-lane-per-pencil path of the compact-difference operators and the
// element-wise epilogue (the partitioned kernels are in pade_spike.h).
#include "pade_spike.h"

namespace pade {

// ------------------------------------------------------------------------
// Generic path: one lane per pencil, whole pencil as one partition (P = 1),
// the intermediate values kept in the output array (adjoint: in `work`).
template <typename T, bool ADJ>
__global__ __launch_bounds__(256) void generic_apply(ApplyArgs<T> a, T *__restrict__ work)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= a.npencils) return;
    const long long base = (q % a.A1) * a.B1 + (q / a.A1) * a.B2;
    const long long st = a.stride;
    const int n = a.n;
    const FieldArgs<T> &fd = a.fld[0];
    const T *__restrict__ tab = fd.tab;
    const T *__restrict__ lu = tab + kOffCoef;          // [n][6]
    const T *__restrict__ S = lu + 6 * n;               // [n][4]
    const T *__restrict__ Q = lu + 10 * n;              // [4][4]
    T *y = ADJ ? work : fd.out;

    // B applied to `src` (src_n points per pencil) at row i
    auto stencil_row = [&](const T *src, int src_n, int i) -> T {
        if (!a.periodic) {
            if (i < fd.nbl) {
                T s = T(0);
                for (int c = 0; c < kBColsDev && c < src_n; c++)
                    s += tab[kOffBl + i * kBColsDev + c] * src[base + (long long)c * st];
                return s;
            }
            if (i >= n - fd.nbr) {
                const int r = n - 1 - i;
                T s = T(0);
                for (int c = 0; c < kBColsDev && c < src_n; c++)
                    s += tab[kOffBr + r * kBColsDev + c] * src[base + (long long)(src_n - 1 - c) * st];
                return s;
            }
        }
        T s = T(0);
        for (int k = 0; k < 9; k++) {
            const T cf = tab[k];
            if (cf == T(0)) continue;
            const int j = wrap_index(i - 4 + k, src_n, a.periodic);
            s += cf * src[base + (long long)j * st];
        }
        return s;
    };

    // forward elimination; the forward operator forms each right-hand-side
    // row as it goes (f and the output never overlap)
    T zm1 = T(0), zm2 = T(0);
    for (int i = 0; i < n; i++) {
        const T r = ADJ ? fd.f[base + (long long)i * st] : stencil_row(fd.f, a.n_in, i);
        const T z = i == 0 ? r : r - lu[i * 6 + 0] * zm1 - lu[i * 6 + 1] * zm2;
        y[base + (long long)i * st] = z;
        zm2 = zm1;
        zm1 = z;
    }
    T gp1 = T(0), gp2 = T(0);
    for (int i = n - 1; i >= 0; i--) {
        T g = y[base + (long long)i * st] * lu[i * 6 + 2] - lu[i * 6 + 3] * gp1 - lu[i * 6 + 4] * gp2;
        y[base + (long long)i * st] = g;
        gp2 = gp1;
        gp1 = g;
    }
    if (a.periodic) {
        const T g0 = y[base], g1 = y[base + st], g2 = y[base + (long long)(n - 2) * st],
                g3 = y[base + (long long)(n - 1) * st];
        T u[4];
        for (int c = 0; c < 4; c++) u[c] = Q[c * 4 + 0] * g0 + Q[c * 4 + 1] * g1 + Q[c * 4 + 2] * g2 + Q[c * 4 + 3] * g3;
        for (int i = 0; i < n; i++) {
            const long long o = base + (long long)i * st;
            y[o] -= S[i * 4 + 0] * u[0] + S[i * 4 + 1] * u[1] + S[i * 4 + 2] * u[2] + S[i * 4 + 3] * u[3];
        }
    }
    if (ADJ) {
        for (int i = 0; i < n; i++) fd.out[base + (long long)i * st] = stencil_row(work, n, i);
    }
}

template <typename T>
hipError_t launch_generic(const ApplyArgs<T> &a, bool adj, T *work, hipStream_t s)
{
    const int bs = 256;
    const long long nblk = (a.npencils + bs - 1) / bs;
    if (adj)
        hipLaunchKernelGGL((generic_apply<T, true>), dim3((unsigned)nblk), dim3(bs), 0, s, a, work);
    else
        hipLaunchKernelGGL((generic_apply<T, false>), dim3((unsigned)nblk), dim3(bs), 0, s, a, work);
    return hipGetLastError();
}

template <typename T>
__global__ __launch_bounds__(256) void axpby_kernel(const T *__restrict__ x, T *__restrict__ y, T alpha, T beta,
                                                   long long count)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride)
        y[i] = (x ? alpha * x[i] : T(0)) + beta * y[i];
}

template <typename T>
hipError_t launch_axpby(const T *x, T *y, T alpha, T beta, long long count, hipStream_t s)
{
    if (count <= 0) return hipSuccess;
    const long long blocks = std::min<long long>((count + 255) / 256, 65536);
    hipLaunchKernelGGL((axpby_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, s, x, y, alpha, beta, count);
    return hipGetLastError();
}

template hipError_t launch_generic<double>(const ApplyArgs<double> &, bool, double *, hipStream_t);
template hipError_t launch_generic<float>(const ApplyArgs<float> &, bool, float *, hipStream_t);
template hipError_t launch_axpby<double>(const double *, double *, double, double, long long, hipStream_t);
template hipError_t launch_axpby<float>(const float *, float *, float, float, long long, hipStream_t);

}  // namespace pade
