// C ABI of libpadeops_hip: operator handles, plan tables, dispatch, errors.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/padeops_hip.h"
#include "pade_capi_internal.h"
#include "pade_cgrid.h"
#include "pade_dense.h"
#include "pade_err.h"
#include "pade_kernels.h"
#include "pade_plan.h"

namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string &msg)
{
    g_last_error = msg;
    return code;
}

int hip_fail(hipError_t e, const char *where)
{
    return fail(1000 + int(e), std::string(where) + ": " + hipGetErrorString(e));
}

// One factor variant (partition size M) of one plan, as laid out in the
// device table (see pade_kernels.h).
struct Variant {
    int M = 0, P = 0;
    int n = 0, n_in = 0;   // rows solved and input points per pencil
    bool rect = false;     // staggered system form (strided-row mode 2)
    int tail = 0;          // mode 2: one output row after the n solved
    long long off = 0;  // element offset of this variant's table in the plan buffer
    int nbl = 0, nbr = 0;
    int coef_len = 0, ncls = 0, kq = 0;
    int cls[pade::kMaxLongPartitions] = {0};
    int len = 0;
    bool uneven = false;   // partitions of `parts`
    pade::UnevenParts parts;
};

struct PlanKey {
    int oper, bc1, bcn, adj;
    bool operator<(const PlanKey &o) const
    {
        return std::tie(oper, bc1, bcn, adj) < std::tie(o.oper, o.bc1, o.bcn, o.adj);
    }
};

struct Plan {
    std::vector<Variant> spike;  // register-path variants: M of 16, 32, 64 (48) dividing the rows,
                                 // then the uneven ones
    Variant generic;             // whole pencil as one partition
    bool has_generic = false;
    // does a partition size divide the rows?
    bool even() const
    {
        return std::any_of(spike.begin(), spike.end(), [](const Variant &v) { return !v.uneven; });
    }
    pade::OpMatrices mats;       // for the dense form
};

// Assemble the table of one variant; returns 0 or an error code.
// parts: the uneven partitions to use (known: factors at hand), or null for an
// even split into M rows.
int build_variant(const pade::OpMatrices &m, int M, std::vector<double> &tab, Variant &v,
                  const pade::UnevenParts *parts = nullptr, std::vector<pade::PartFactors> *known = nullptr)
{
    pade::SpikeFactors sf;
    std::vector<pade::PartFactors> none;
    if (int rc = parts ? pade::spike_factor_uneven(m, *parts, known ? *known : none, sf) : pade::spike_factor(m, M, sf))
        return rc;
    if (parts) {
        v.uneven = true;
        v.parts = *parts;
    }
    const int P = sf.P;
    const bool periodic = m.periodic;
    const int m4 = 4 * P;
    v.M = M;
    v.P = P;
    v.n = m.n;
    v.n_in = m.n_in ? m.n_in : m.n;
    v.rect = m.rect;
    v.tail = m.tail ? 1 : 0;
    v.nbl = m.nbl;
    v.nbr = m.nbr;
    // coefficient classes: partitions with bit-identical (LU, S) blocks share one
    std::vector<int> reps;
    auto same = [&](int a, int b) {
        for (int r = 0; r < M; r++) {
            for (int c = 0; c < 5; c++)
                if (sf.lu[((size_t)a * M + r) * 5 + c] != sf.lu[((size_t)b * M + r) * 5 + c]) return false;
            for (int c = 0; c < 4; c++)
                if (sf.S[((size_t)a * M + r) * 4 + c] != sf.S[((size_t)b * M + r) * 4 + c]) return false;
        }
        return true;
    };
    for (int p = 0; p < P; p++) {
        int c = -1;
        for (int k = 0; k < (int)reps.size(); k++)
            if (same(reps[k], p)) { c = k; break; }
        if (c < 0) { c = (int)reps.size(); reps.push_back(p); }
        if (p < pade::kMaxLongPartitions) v.cls[p] = c;
    }
    if (periodic && !parts && reps.size() != 1) return 3;  // even periodic blocks are identical by construction
    v.ncls = (int)reps.size();
    // reduced-system window: farthest partition whose weight is not negligible
    double qmax = 0.0;
    for (double x : sf.Q) qmax = std::max(qmax, std::fabs(x));
    v.kq = 0;
    for (int p = 0; p < P; p++)
        for (int c = 0; c < 4; c++)
            for (int j = 0; j < m4; j++) {
                const double x = std::fabs(sf.Q[((size_t)p * 4 + c) * m4 + j]);
                if (x <= 1e-18 * qmax) continue;
                int d = std::abs(j / 4 - p);
                if (periodic) d = std::min(d, P - d);
                v.kq = std::max(v.kq, d);
            }
    const int window = std::min(2 * v.kq + 1, P);
    v.coef_len = v.ncls * 10 * M + (parts ? P * 16 * window : (periodic ? 4 * m4 : P * 4 * m4));
    v.len = (pade::kOffCoef + v.coef_len + 15) & ~15;
    v.off = (long long)tab.size();
    tab.resize(tab.size() + v.len, 0.0);
    double *t = &tab[v.off];
    for (int k = 0; k < 9; k++) t[k] = m.stencil[k];
    t[9] = m.tail_dn;      // system form of a staggered cell-to-edge operator
    t[10] = m.tail_idg;
    for (int r = 0; r < pade::kBRowsDev; r++)
        for (int c = 0; c < pade::kBColsDev; c++) {
            t[pade::kOffBl + r * pade::kBColsDev + c] = m.bl[r][c];
            t[pade::kOffBr + r * pade::kBColsDev + c] = m.br[r][c];
        }
    double *ca = t + pade::kOffCoef;
    for (int k = 0; k < v.ncls; k++) {
        const int p = reps[k];
        double *blk = ca + (size_t)k * 10 * M;
        for (int r = 0; r < M; r++) {
            for (int c = 0; c < 5; c++) blk[r * 6 + c] = sf.lu[((size_t)p * M + r) * 5 + c];
            for (int c = 0; c < 4; c++) blk[6 * M + r * 4 + c] = sf.S[((size_t)p * M + r) * 4 + c];
        }
    }
    double *qa = ca + (size_t)v.ncls * 10 * M;
    if (parts) {
        for (int p = 0; p < P; p++)
            for (int c = 0; c < 4; c++)
                for (int j = 0; j < window; j++) {
                    int q = window == P ? j : p - v.kq + j;
                    if (periodic) q = (q + P) % P;
                    if (q < 0 || q >= P) continue;
                    for (int k = 0; k < 4; k++)
                        qa[((size_t)p * 4 + c) * 4 * window + 4 * j + k] = sf.Q[((size_t)p * 4 + c) * m4 + 4 * q + k];
                }
        return 0;
    }
    const int nq = periodic ? 1 : P;
    for (int p = 0; p < nq; p++)
        for (int c = 0; c < 4; c++)
            for (int j = 0; j < m4; j++) qa[((size_t)p * 4 + c) * m4 + j] = sf.Q[((size_t)p * 4 + c) * m4 + j];
    return 0;
}

int operator_matrices(int kind, int oper, int n, double dx, bool periodic, int bc1, int bcn, bool adj,
                      pade::OpMatrices &out)
{
    pade::OpMatrices fwd;
    if (int rc = pade::build_operator(kind, oper, n, dx, periodic, bc1, bcn, fwd)) return rc;
    if (adj) pade::transpose_operator(fwd, out);
    else out = fwd;
    return 0;
}

bool oper_valid(int kind, int oper)
{
    if (kind == pade::CF90 || kind == pade::GAUSSIAN) return oper == pade::FILTER;
    if (kind == pade::CD06STAGG) return oper >= pade::D1_E2C && oper <= pade::D1_E2E;
    return oper == pade::D1 || oper == pade::D2;
}

// Staggered operations whose input / output lives on the n + 1 edge planes
// (periodic: the last a copy of the first, cd06stagg.F90:859,969,1036).
bool edge_output(int kind, int oper) { return kind == pade::CD06STAGG && pade::stagg_edge_out(oper); }
bool edge_input(int kind, int oper) { return kind == pade::CD06STAGG && pade::stagg_edge_in(oper); }

}  // namespace

int pade::set_error(int code, const char *msg) { return fail(code, msg); }

struct pade_op_s {
    int kind = 0, n = 0;
    double dx = 1.0;
    bool periodic = true;
    int init_bc1 = 0, init_bcn = 0;
    int device = 0;
    std::map<PlanKey, Plan> plans;
    double *dtab64 = nullptr;
    float *dtab32 = nullptr;
    long long tab_len = 0;
    std::mutex mu;
    pade::DenseCache dense;
};

namespace {

int plan_key_bc(const pade_op_s *op, int bc)
{
    return op->kind == pade::CD06 || op->kind == pade::CD06STAGG ? 0 : bc;
}

// Plan key of the complex z filter's mixed operator (bounded cf90): the
// right-hand side of boundary codes (bc1, bcn) solved with the (0, 0)
// left-hand side, as cf90.F90:1248-1249 does (ComputeZRHS_CMPLX with the
// caller's codes, then SolveZPenta_CMPLX with penta_nn).
constexpr int kFilterRhsBc = 100 + pade::FILTER;

// Partition sizes of the register path that serve this operator: those that
// divide its rows, or else the uneven splits.
// The bounded cf90 adjoint (inverse: A^-T before B^T) takes no uneven split
// that is less exact than what else serves the length: A is nearly singular at
// the shortest wave, which only B^T removes, so what a partition's ends add to
// its rounding stays (white noise, root mean square over the largest output,
// FP64 / FP32: n = 129 as one partition 6.0e-15 / 2.8e-6, in 32 slots 1.0e-14
// / 5.9e-6; n = 320 in 64 rows 8.6e-15 / 4.4e-6, in 40 slots 1.04e-14 /
// 4.8e-6; but n = 176 in 16 rows 1.8e-14 / 6.8e-6, in 32 slots 1.0e-14 /
// 5.3e-6).  It costs time (FP64, us, x / y / z, one lane per pencil and 32
// slots: n = 97, 128^2 pencils, 319 / 214 / 195 and 16 / 14 / 14; n = 129,
// 256^2 pencils, 677 / 352 / 335 and 53 / 46 / 46).
void add_spike_variants(const pade::OpMatrices &m, bool adj, bool inverse, std::vector<double> &tab,
                        std::vector<pade::PartFactors> &known, Plan &pl)
{
    // special rows the kernels hold
    const int rows = adj ? pade::kBRowsDev : (m.rect ? pade::kBRowsSys : pade::kBRowsFwd);
    for (int M : {16, 32, 64}) {
        if (m.n % M || m.n / M > pade::kMaxPartitions || m.nbl > rows || m.nbr > rows) continue;
        Variant v;
        if (build_variant(m, M, tab, v) == 0) pl.spike.push_back(v);
    }
    // Uneven partitions, of the sizes that pick_variant prefers: everywhere
    // that no size divides the rows, for lengths of 144 .. 240 that 16 alone
    // divides, and 40 or 48 slots from n = 257 to 384.
    const int n = m.n;
    const bool mid = n > 256 && n <= 384;
    if (mid && m.periodic && n == 8 * 48) {         // whole-pencil x waves
        Variant v;
        if (build_variant(m, 48, tab, v) == 0) pl.spike.push_back(v);
    }
    if (!pl.spike.empty() && !(n % 32 == 16 && n >= 144) && !mid) return;
    const bool none = pl.spike.empty();
    if (inverse && (none || n % 64 == 0)) return;
    for (int M : {16, 24, 32, 40, 48, 64}) {
        pade::UnevenParts parts;
        Variant v;
        bool want;
        if (mid) want = M == 48 || (M == 40 && n <= 320);
        else if (n <= 256) want = M == 32 || (none && (M == 16 || (M == 24 && n < 40)));
        else want = M == 64 || (M == 32 && m.periodic);
        if (!want || m.nbl > rows || m.nbr > rows) continue;
        if (!pade::uneven_parts(m.n, M, parts) || build_variant(m, M, tab, v, &parts, &known) != 0) continue;
        if (v.P > pade::kMaxPartitions && v.ncls > 8) continue;     // three bits per partition
        pl.spike.push_back(v);
    }
}

// One plan: the operator's matrices and the factor tables of the partition
// sizes that serve its rows, even and uneven (appended to `tab`), plus the
// one-lane-per-pencil form.  bc1 / bcn are the codes that build the
// operator (init-time for cd06 and cd06stagg).
int build_plan(int kind, int oper, int n, double dx, bool periodic, int bc1, int bcn, bool adj,
               std::vector<double> &tab, std::vector<pade::PartFactors> &known, Plan &pl)
{
    if (int rc = operator_matrices(kind, oper, n, dx, periodic, bc1, bcn, adj, pl.mats))
        return fail(rc, "operator construction failed");
    // rows of this operator (a staggered cell <-> edge operator has one more
    // or one fewer than n); the partitioned kernels need a square B
    const int m = pl.mats.n;
    // bounded staggered operators with an edge array: the partitioned
    // kernels run their system form (n rows)
    const bool sys_form = kind == pade::CD06STAGG && !periodic && (pade::stagg_edge_in(oper) || pade::stagg_edge_out(oper));
    pade::OpMatrices sys;
    if (sys_form) {
        if (int rc = pade::build_stagg_system(oper, n, dx, bc1, bcn, sys)) return fail(rc, "operator construction failed");
    }
    const pade::OpMatrices &pm = sys_form ? sys : pl.mats;
    add_spike_variants(pm, adj, kind == pade::CF90 && adj && !periodic, tab, known, pl);
    if (m >= 4 && build_variant(pl.mats, m, tab, pl.generic) == 0) pl.has_generic = true;
    return 0;
}

// All (oper, bc1, bcn, adj) plans an operator can be asked for.
int build_all_plans(pade_op_s *op)
{
    std::vector<double> tab;
    std::vector<pade::PartFactors> known;
    std::vector<int> opers;
    if (op->kind == pade::CF90 || op->kind == pade::GAUSSIAN) opers = {pade::FILTER};
    else if (op->kind == pade::CD06STAGG) {
        opers = {pade::D1_E2C, pade::D1_C2E, pade::D2_C2C, pade::D2_E2E, pade::INTERP_E2C, pade::INTERP_C2E};
        if (!op->periodic) opers.insert(opers.end(), {pade::D1_C2C, pade::D1_E2E});
    } else opers = {pade::D1, pade::D2};
    // init-time end codes choose cd06's and the staggered operators' closures
    const bool init_bc = op->kind == pade::CD06 || op->kind == pade::CD06STAGG;
    std::vector<std::pair<int, int>> bcs;
    if (op->periodic || init_bc) bcs = {{0, 0}};
    else
        for (int a = -1; a <= 1; a++)
            for (int b = -1; b <= 1; b++) bcs.push_back({a, b});
    for (int oper : opers) {
        if (op->kind == pade::CD06 && oper == pade::D2 && !op->periodic) continue;  // composed
        for (auto [b1, bn] : bcs)
            for (int adj = 0; adj < 2; adj++) {
                if (adj && op->n < 16) continue;  // adjoint needs n >= 16 (boundary rows of B^T)
                if (adj && op->kind == pade::CD06STAGG) continue;   // no staggered adjoint
                const int cb1 = init_bc ? op->init_bc1 : b1;
                const int cbn = init_bc ? op->init_bcn : bn;
                Plan pl;
                if (int rc = build_plan(op->kind, oper, op->n, op->dx, op->periodic, cb1, cbn, adj != 0, tab, known, pl))
                    return rc;
                op->plans[{oper, b1, bn, adj}] = std::move(pl);
            }
    }
    if (op->kind == pade::CF90 && !op->periodic) {
        pade::OpMatrices nn;
        if (int rc = operator_matrices(op->kind, pade::FILTER, op->n, op->dx, false, 0, 0, false, nn))
            return fail(rc, "operator construction failed");
        for (auto [b1, bn] : bcs) {
            if (b1 == 0 && bn == 0) continue;
            Plan pl;
            if (int rc = operator_matrices(op->kind, pade::FILTER, op->n, op->dx, false, b1, bn, false, pl.mats))
                return fail(rc, "operator construction failed");
            pl.mats.band = nn.band;      // (bc1, bcn) right-hand side, (0, 0) left-hand side
            add_spike_variants(pl.mats, false, false, tab, known, pl);
            if (op->n >= 4 && build_variant(pl.mats, op->n, tab, pl.generic) == 0) pl.has_generic = true;
            op->plans[{kFilterRhsBc, b1, bn, 0}] = std::move(pl);
        }
    }
    op->tab_len = (long long)tab.size();
    hipError_t e = hipMalloc(&op->dtab64, tab.size() * sizeof(double));
    if (e != hipSuccess) return hip_fail(e, "hipMalloc(tables)");
    e = hipMalloc(&op->dtab32, tab.size() * sizeof(float));
    if (e != hipSuccess) return hip_fail(e, "hipMalloc(tables)");
    std::vector<float> t32(tab.begin(), tab.end());
    e = hipMemcpy(op->dtab64, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_fail(e, "hipMemcpy(tables)");
    e = hipMemcpy(op->dtab32, t32.data(), t32.size() * sizeof(float), hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_fail(e, "hipMemcpy(tables)");
    return 0;
}

template <typename T>
__global__ void fill_kernel(T *dst, long long count, T v)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) dst[i] = v;
}

template <typename T>
int fill_zero(T *dst, long long count, hipStream_t s)
{
    const int bs = 256;
    const long long nb = (count + bs - 1) / bs;
    hipLaunchKernelGGL((fill_kernel<T>), dim3((unsigned)nb), dim3(bs), 0, s, dst, count, T(0));
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "fill");
}

int env_int(const char *name)
{
    const char *v = std::getenv(name);
    return v ? std::atoi(v) : 0;
}

// Largest thread count of one launch (grid size x workgroup size must stay
// below 2^32).
constexpr long long kMaxLaunchThreads = 0xffffffffLL;

// The strided-row kernels (modes 0 and 2) address the field with an SGPR base
// plus a 32-bit per-lane byte offset: the lane's pencil relative to its
// workgroup's first pencil plus its partition's offset within the wave
// ((PW - 1) M points along the pencil).  A variant whose offsets would reach
// 2^32 (e.g. z pencils of 4096 x 2048 planes with two 64-point partitions per
// wave) is not chosen; x pencils (mode 1) stay below 64 pencils x n points.
template <typename T>
bool offsets_fit(const pade::ApplyArgs<T> &a, int mode, int M, int PW)
{
    if (mode == 1) return true;
    const long long npen = 64 / PW, ts = (long long)sizeof(T);
    const long long rows = (npen + a.A1 - 2) / a.A1;    // pencil rows a workgroup spans beyond its first
    const long long lmax = ((npen - 1) * a.B1 + rows * a.B2) * ts;
    const long long part = (long long)(PW - 1) * M * a.stride * ts;
    return lmax + part < (1LL << 32);
}

// Fewest pencils that uneven partitions serve.  Below it these lengths run one
// lane per pencil, as pade_plan_variant reports for 100 x pencils of 100 points.
// Not a crossover: from 1 to 127 pencils (periodic cd10, FP64, x and z) one
// lane per pencil takes 44-54 us at n = 25, 106-136 at 65, 210-266 at 129,
// 418-530 at 257 and 1146-1397 at 700, uneven partitions 4-5, 7-8, 7-9,
// 10-11 and 17-19.
constexpr long long kUnevenPencils = 128;

// Choose (partition size M, partitions per wave PW) for this launch: two
// partitions per wave but for whole x pencils and more than sixteen
// partitions, M by type, axis, length and boundary as measured below, the
// smallest M for small problems.  PADE_SPIKE_M / PADE_SPIKE_PW override the
// choice (tuning).
template <typename T>
const Variant *pick_variant(const Plan &pl, const pade::ApplyArgs<T> &a, int mode, int *pw_out)
{
    static const int envM = env_int("PADE_SPIKE_M"), envPW = env_int("PADE_SPIKE_PW");
    const bool fp64 = std::is_same<T, double>::value;
    const long long npencils = a.npencils;
    const Variant *best = nullptr;
    int best_pw = 1, best_score = -1;
    // 64-point partitions for x and bounded pencils, 32 for periodic strided
    // rows (512^3 FP64: periodic z with 64 measured 323.7 -> 326.3-326.9 Gpts/s
    // but its accumulate-epilogue form 675 -> 945 us; y 355-357 -> 348-349)
    // Pencils up to n = 256 prefer 32 on every axis, periodic or bounded (512
    // x 512 pencils, two partitions per wave, FP64, 64 vs 32: periodic x n =
    // 64 223-231 vs 334-341, n = 128 329-334 vs 349, n = 192 312-314 vs
    // 341-343; bounded x / y / z n = 64 243-252 / 226-228 / 235-237 vs 270-272
    // / 330-331 / 330-332, n = 128 283 / 317-318 / 321 vs 325-329 / 364-368 /
    // 367-371, n = 256 306-308 / 311 / 293 vs 314-316 / 340-343 / 319-320;
    // bounded n = 512 337-338 / 322 / 303-304 vs 242 / 258 / 240).
    // From 257 to 384 points x takes 48 slots and strided rows 40 up to 320
    // and then 48: at most eight partitions, four waves per workgroup (512 x
    // 256 pencils, FP64, us, x / y / z, with 32, 40, 48, 64 slots: periodic n =
    // 260 223 / 138 / 138, 162 / 119 / 122, 153 / 116 / 121, 181 / 151 / 154;
    // n = 320 195 / 144 / 153, 164 / 130 / 136, 136 / 135 / 141, 140 / 146 /
    // 161; n = 384 215 / 164 / 175, 302 / 225 / 229, 157 / 153 / 160, 162 /
    // 164 / 184; bounded n = 288 202 / 153 / 157, 167 / 130 / 138, 145 / 139 /
    // 142, 172 / 173 / 175), but for bounded x that 64 divides (n = 320 152
    // with 64, 163 with 48; n = 384 169, 172).  Nine or more partitions of 40
    // or 48 rows lose a workgroup per CU, so longer pencils return to 64 and
    // 32.  (Even bounded rows of n = 512 measure 235 / 255 us with 64 and 230 /
    // 239 with 32 slots since those fit four waves per SIMD; they keep the
    // reported 64.)
    // FP32, whose even kernels have twice the waves in flight, stays with
    // these where they exist, but for bounded strided rows (512 x 512 pencils,
    // us, even and uneven: periodic n = 288 135 / 128 / 132 and 150 / 135 /
    // 138, n = 352 160 / 158 / 162 and 177 / 166 / 167; bounded 195 / 155 /
    // 158 and 172 / 140 / 140, n = 320 147 / 151 / 154 and 182 / 145 / 147).
    const int n = pl.mats.n;
    const bool beside = fp64 || !pl.even() || (mode != 1 && !pl.mats.periodic);
    const bool mid = n > 256 && n <= 384 && beside;
    const int pref_m = n <= 256 ? 32
                       : !mid   ? (mode == 1 || !pl.mats.periodic ? 64 : 32)
                       : mode == 1 ? (!pl.mats.periodic && n % 64 == 0 ? 64 : 48)
                                   : (n <= 320 ? 40 : 48);
    // Whole pencils per wave (x, 8 partitions of 32 or 64 points) read every
    // line once and stream their loads: preferred for periodic x when the
    // pencil fills all 8 partition slots of the wave (512^3: FP64 +1.5-2 %;
    // FP32 622-637 -> 667-684 Gpts/s once each memory instruction moved one
    // pencil and XCDs took runs of workgroups, 5-7 % slower before).  With
    // fewer partitions the idle slots cost more than the saved halo loads
    // (512 x 512 pencils, FP64 / FP32 Gpts/s, whole vs two per wave: n = 64,
    // one partition, 78 / 136 vs 222 / 386; n = 128 158 / 260 vs 334 / 637;
    // n = 256 263 / 467 vs 312 / 654; n = 320 308 / 549 vs 307-317 / 615-627);
    // filled with 8 partitions of 32 (n = 256) it wins again: 331-368 /
    // 541-671 against 307-309 / 505-648 for two 64-point partitions per wave.
    // Bounded tables are 4x larger, so one-wave workgroups copy 24 KiB of
    // coefficients per 8 pencils (bounded x 339 -> 223).
    const bool prefer_whole = mode == 1 && pl.mats.periodic;
    // eligible (variant, partitions per wave) pairs and their wave counts
    auto waves_of = [&](const Variant &v, int pw) -> long long {
        // uneven kernels take two partitions per wave, four of more than sixteen
        if (v.uneven && (pw != (v.P > pade::kMaxPartitions ? 4 : 2) || npencils < kUnevenPencils)) return -1;
        if ((v.P + pw - 1) / pw > 8) return -1;
        if (pw == 8 && (mode != 1 || v.P > 8 || (v.M != 32 && v.M != 48 && v.M != 64))) return -1;
        if (v.M == 48 && !v.uneven && (pw != 8 || !fp64)) return -1;        // whole pencils only
        // (FP32 x beside 16 from eleven partitions of 16 rows: n = 144 90 ->
        // 91 us, 176 116 -> 96, bounded 108 -> 113, 134 -> 108)
        if (v.uneven && !beside && !(mode == 1 && n > 160 && n <= 256)) return -1;
        // four partitions per wave: strided rows only, by request (tuning)
        if (pw == 4 && !v.uneven && (mode != 0 || envPW != 4 || (v.M != 32 && v.M != 64))) return -1;
        if (envM && v.M != envM) return -1;
        if (envPW && pw != envPW) return -1;
        if (!offsets_fit(a, v.rect ? 2 : mode, v.M, pw)) return -1;
        const long long groups = (npencils + 64 / pw - 1) / (64 / pw);
        const long long waves = groups * ((v.P + pw - 1) / pw);
        return waves * 64 > kMaxLaunchThreads ? -1 : waves;
    };
    // A latency-bound size (no variant reaches 4096 waves) takes the variant
    // with the most waves (the shortest partitions); otherwise the throughput
    // preferences below.  x above 256 points (FP32: 384) takes these as soon
    // as they give two waves per CU (9216 pencils of 512 points: FP64 21 us
    // with 64 rows, 31 with 32, FP32 15 and 19; of 288 FP64 17 with 48, 22
    // with 32, strided rows 15.9 and 15.4; of 384 FP32 13.8 with 64, 12.6).
    // And with the chip filled, more than ten partitions of 16 rows lose to 32
    // by their reduced system (FP64, 96^2 pencils, bounded x n = 192 19 -> 14
    // us, 176 20 -> 17, y 13.7 -> 12.6; 40^2 pencils 9.1 -> 10.1, kept, as is
    // periodic x beside uneven 32, 13.5 and 15.8).
    long long max_waves = -1, pref_waves = -1;
    for (const Variant &v : pl.spike)
        for (int pw : {1, 2, 4, 8}) {
            max_waves = std::max(max_waves, waves_of(v, pw));
            if (v.M == pref_m) pref_waves = std::max(pref_waves, waves_of(v, pw));
        }
    const bool small = max_waves < 4096 && !(mode == 1 && n > (fp64 ? 256 : 384) && pref_waves >= 512);
    auto small_rank = [&](const Variant &v) {
        const bool keep16 = mode == 1 && pl.mats.periodic && n % 32;
        return v.M == 16 && v.P > 10 && !keep16 && fp64 && max_waves >= 1024 ? 33 : v.M;
    };
    for (const Variant &v : pl.spike)
        for (int pw : {1, 2, 4, 8}) {
            if (waves_of(v, pw) < 0) continue;
            int score = (pw == 2 ? 100 : 0) + (pw == 8 && prefer_whole && v.P == 8 ? 300 : 0) +
                        (v.M == pref_m ? 50 : (v.M == 64 ? 30 : (v.M == 32 ? 20 : 10)));
            if (small) score = 1000 - 2 * small_rank(v) + (pw == 2 ? 1 : 0);
            if (score > best_score) { best_score = score; best = &v; best_pw = pw; }
        }
    *pw_out = best_pw;
    return best;
}

// Whole-pencil x waves (8 partitions per wave) per workgroup: the waves
// share one copy of the coefficient table.  PADE_SPIKE_GW overrides (tuning).
int whole_pencil_waves()
{
    static const int gw = [] {
        const int e = env_int("PADE_SPIKE_GW");
        return e >= 1 && e <= 8 ? e : 1;
    }();
    return gw;
}

// Optional epilogue of an apply: df = alpha * op(f) + beta * df.
template <typename T>
struct Epilogue {
    bool on = false;
    T alpha = T(1), beta = T(0);
};

// Device memory for the intermediates of an apply.  Off: the stream-ordered
// allocator.  On: carved from a region the caller provides, nothing
// allocated; a copy passed down to a nested apply holds what is left.
struct Workspace {
    bool on = false;
    char *ptr = nullptr;
    size_t bytes = 0;
    const char *owner = "the caller's region";   // named in the size error
};

template <typename T>
int scratch_get(Workspace &ws, size_t count, hipStream_t s, T **out, const char *what)
{
    if (ws.on) {
        const size_t bytes = (sizeof(T) * count + 255) & ~size_t(255);
        if (bytes > ws.bytes)
            return fail(400, std::string(what) + " needs " + std::to_string(bytes) + " bytes of scratch; " +
                                 ws.owner + " has " + std::to_string(ws.bytes) + " left");
        *out = reinterpret_cast<T *>(ws.ptr);
        ws.ptr += bytes;
        ws.bytes -= bytes;
        return 0;
    }
    hipError_t e = hipMallocAsync((void **)out, sizeof(T) * count, s);
    return e == hipSuccess ? 0 : hip_fail(e, what);
}

template <typename T>
void scratch_put(const Workspace &ws, T *p, hipStream_t s)
{
    if (!ws.on && p) (void)hipFreeAsync(p, s);
}

template <typename T>
int apply_impl(pade_op_t op, int oper, int axis, const T *f, T *df, int na, int nb, int bc1, int bcn,
               bool adj, hipStream_t s, Epilogue<T> epi = Epilogue<T>(), Workspace ws = Workspace());

// The launch an apply runs: kernel variant, partitions per wave, mode.
template <typename T>
struct LaunchPlan {
    const Variant *v = nullptr;
    int pw = 1, mode = 0;
    bool generic = false;
    pade::ApplyArgs<T> a{};
};

template <typename T>
void set_tables(const Variant &v, pade::FieldArgs<T> &fd)
{
    fd.nbl = v.nbl;
    fd.nbr = v.nbr;
    fd.coef_len = v.coef_len;
    fd.ncls = v.ncls;
    fd.kq = v.kq;
    fd.cls4 = 0;
    const int bits = v.P > pade::kMaxPartitions ? 3 : 4;
    for (int k = 0; k < v.P; k++) fd.cls4 |= (unsigned long long)v.cls[k] << (bits * k);
}

// Variant, partitions per wave and mode of an apply along `axis` over
// na x nb pencils; the table pointer of `a` is left to the caller.
template <typename T>
int plan_launch(const Plan &pl, bool periodic, int axis, const T *f, T *df, int na, int nb, LaunchPlan<T> &L)
{
    const int n = pl.mats.n;
    pade::ApplyArgs<T> &a = L.a;
    a = pade::ApplyArgs<T>{};
    a.nfields = 1;
    a.fld[0].f = f;
    a.fld[0].out = df;
    a.n = n;
    a.n_in = pl.mats.n_in ? pl.mats.n_in : n;
    a.periodic = periodic ? 1 : 0;
    a.npencils = (long long)na * nb;
    int mode = 0;
    if (axis == 1) {
        a.A1 = a.npencils; a.B1 = n; a.B2 = 0; a.stride = 1; mode = 1;
    } else if (axis == 2) {
        a.A1 = na; a.B1 = 1; a.B2 = (long long)na * n; a.stride = na;
    } else {
        a.A1 = a.npencils; a.B1 = 1; a.B2 = 0; a.stride = (long long)na * nb;
    }
    int pw = 1;
    const Variant *v = pick_variant<T>(pl, a, mode, &pw);
    L.generic = (v == nullptr);
    if (L.generic) {
        if (!pl.has_generic) return fail(21, "no solver variant for this size");
        if (a.npencils > kMaxLaunchThreads - 255) return fail(400, "too many pencils for one launch");
        v = &pl.generic;
    }
    a.n = v->n;
    a.n_in = v->n_in;
    a.tail = v->tail;
    if (v->rect) mode = 2;   // strided rows (axis 3) of a staggered system form
    a.M = v->M;
    a.P = v->P;
    set_tables(*v, a.fld[0]);
    a.ubase = v->parts.base;
    a.uextra = v->parts.extra;
    a.uunit = v->parts.unit;
    a.axpby = 0;
    a.alpha = T(1);
    a.beta = T(0);
    L.v = v;
    L.pw = pw;
    L.mode = mode;
    return 0;
}

template <typename T>
int apply_one(pade_op_t op, const Plan &pl, int axis, const T *f, T *df, int na, int nb, bool adj,
              hipStream_t s, Epilogue<T> epi, Workspace ws)
{
    LaunchPlan<T> L;
    if (int rc = plan_launch<T>(pl, op->periodic, axis, f, df, na, nb, L)) return rc;
    pade::ApplyArgs<T> &a = L.a;
    const T *tables = std::is_same<T, double>::value ? (const T *)op->dtab64 : (const T *)op->dtab32;
    a.fld[0].tab = tables + L.v->off;
    const Variant *v = L.v;
    const int pw = L.pw, mode = L.mode, n = v->n;
    const bool use_generic = L.generic;
    // Periodic operators are circulant, so A^T and B^T commute and the adjoint
    // B^T A^{-T} equals A^{-T} B^T: the transposed tables run through the
    // forward kernel (stencil first).  This avoids amplifying the Nyquist band
    // by A^{-T} before B^T damps it again.  Bounded operators use the adjoint
    // kernel (solve first, then B^T with the transposed closures).
    const bool kadj = adj && !op->periodic;
    hipError_t e;
    if (!use_generic) {
        if (epi.on) {
            a.axpby = 1;
            a.alpha = epi.alpha;
            a.beta = epi.beta;
        }
        if (v->uneven) {
            // The allocation-free entry point refuses accumulating applies
            // whose one-lane form would not fit its array; lengths that no
            // partition size divides keep that documented limit.
            if (ws.on && epi.on && !pl.even()) {
                T *unused = nullptr;
                if (int rc = scratch_get<T>(ws, (size_t)a.npencils * n, s, &unused, "accumulate temporary")) return rc;
            }
            e = pade::launch_uneven<T>(a, v->M, kadj, mode, s);
        } else {
            e = pade::launch_spike<T>(a, v->M, pw, pw == 8 ? whole_pencil_waves() : 1, kadj, mode, s);
        }
        if (e != hipSuccess) return hip_fail(e, "spike_apply launch");
        return 0;
    }
    // generic path: it keeps intermediates in its output, so an epilogue
    // goes through a temporary
    // (the adjoint keeps its intermediates in `work`)
    const size_t count = (size_t)a.npencils * n;
    T *work = nullptr, *tmp = nullptr;
    if (kadj) {
        if (int rc = scratch_get<T>(ws, count, s, &work, "generic adjoint work array")) return rc;
    }
    if (epi.on) {
        if (int rc = scratch_get<T>(ws, count, s, &tmp, "generic accumulate temporary")) {
            scratch_put<T>(ws, work, s);
            return rc;
        }
        a.fld[0].out = tmp;
    }
    e = pade::launch_generic<T>(a, kadj, work, s);
    if (e == hipSuccess && epi.on) e = pade::launch_axpby<T>(tmp, df, epi.alpha, epi.beta, (long long)count, s);
    scratch_put<T>(ws, work, s);
    scratch_put<T>(ws, tmp, s);
    if (e != hipSuccess) return hip_fail(e, "generic_apply launch");
    return 0;
}

// Does one launch apply this operator twice?  (Whole-pencil x waves, which a
// bounded pencil runs by request only, have no adjoint form.)
template <typename T>
bool twice_ok(const LaunchPlan<T> &L, bool adj)
{
    return std::is_same<T, double>::value && !L.generic && L.mode != 2 && (L.pw == 2 || (L.pw == 8 && !adj));
}

// Argument checks shared by every apply: 0 or the error code.
int check_apply(pade_op_t op, int oper, int axis, int na, int nb, int bc1, int bcn, bool adj)
{
    if (!op) return fail(400, "null operator");
    if (axis < 1 || axis > 3) return fail(400, "axis must be 1, 2 or 3");
    if (na < 1 || nb < 1) return fail(400, "na and nb must be positive");
    if (!oper_valid(op->kind, oper)) return fail(21, "operation not provided for this operator kind");
    if (op->kind == pade::CD06STAGG) {
        if (axis != 3) return fail(400, "the staggered operators act along z (axis 3)");
        if (adj) return fail(21, "no adjoint of the staggered operators");
        if (op->periodic && (oper == pade::D1_C2C || oper == pade::D1_E2E))
            return fail(21, "ddz_C2C and ddz_E2E are provided for the bounded staggered operators only");
    }
    if (op->kind != pade::CD06) {
        auto ok = [](int b) { return b == 0 || b == 1 || b == -1; };
        if (!ok(bc1) || !ok(bcn))
            return fail(324, "Incorrect boundary specification (should be 0, 1 or -1)");
    }
    return 0;
}

// Plan of (oper, bc1, bcn, adj), or null (error recorded).
const Plan *find_plan(pade_op_t op, int oper, int bc1, int bcn, bool adj)
{
    const int k1 = op->periodic ? 0 : plan_key_bc(op, bc1);
    const int kn = op->periodic ? 0 : plan_key_bc(op, bcn);
    auto it = op->plans.find({oper, k1, kn, adj ? 1 : 0});
    if (it == op->plans.end()) {
        fail(21, adj ? "adjoint needs n >= 16" : "no plan for this operation");
        return nullptr;
    }
    return &it->second;
}

template <typename T>
int apply_impl(pade_op_t op, int oper, int axis, const T *f, T *df, int na, int nb, int bc1, int bcn,
               bool adj, hipStream_t s, Epilogue<T> epi, Workspace ws)
{
    if (int rc = check_apply(op, oper, axis, na, nb, bc1, bcn, adj)) return rc;
    if (!f || !df) return fail(400, "null array");
    const long long count = (long long)na * nb * op->n;
    if (op->n == 1) {
        if (epi.on) {   // op(f) is f (filter) or 0 (derivatives)
            hipError_t e = oper == pade::FILTER ? pade::launch_axpby<T>(f, df, epi.alpha, epi.beta, count, s)
                                                : pade::launch_axpby<T>(nullptr, df, T(0), epi.beta, count, s);
            return e == hipSuccess ? 0 : hip_fail(e, "axpby");
        }
        if (oper == pade::FILTER) {
            hipError_t e = hipMemcpyAsync(df, f, sizeof(T) * count, hipMemcpyDeviceToDevice, s);
            return e == hipSuccess ? 0 : hip_fail(e, "copy");
        }
        return fill_zero(df, count, s);
    }
    if (op->kind == pade::CD06 && oper == pade::D2 && !op->periodic) {
        // bounded cd06 second derivative: the first derivative applied twice,
        // in one launch where the FP64 kernels for that serve the size.
        // Otherwise, without an epilogue and on the partitioned kernels, the second pass
        // runs in place on df: a workgroup holds every partition of its
        // pencils, and all of a pencil is loaded and consumed before any of
        // it is stored (a workgroup barrier between the two when a pencil
        // spans several waves; within a wave every stored value depends on
        // every loaded one), so no intermediate array is needed.  The
        // one-lane-per-pencil path overwrites its input as it sweeps and
        // keeps the intermediate.
        const Plan *p1 = find_plan(op, pade::D1, bc1, bcn, adj);
        if (!p1) return 21;
        LaunchPlan<T> L;
        if (int rc = plan_launch<T>(*p1, op->periodic, axis, f, df, na, nb, L)) return rc;
        if constexpr (std::is_same<T, double>::value) {
            if (twice_ok(L, adj)) {
                // (the allocation-free entry point keeps its size limit, see apply_one)
                if (ws.on && epi.on) {
                    const size_t fields = p1->even() ? 1 : 2;
                    T *unused = nullptr;
                    if (int rc = scratch_get<T>(ws, fields * (size_t)count, s, &unused,
                                                "cd06 second derivative intermediate"))
                        return rc;
                }
                L.a.fld[0].tab = op->dtab64 + L.v->off;
                L.a.axpby = epi.on ? 1 : 0;
                L.a.alpha = epi.alpha;
                L.a.beta = epi.beta;
                hipError_t e = pade::launch_twice(L.a, L.v->M, L.pw, L.pw == 8 ? whole_pencil_waves() : 1,
                                                  L.v->uneven, adj, L.mode, s);
                return e == hipSuccess ? 0 : hip_fail(e, "spike_apply launch");
            }
        }
        if (!epi.on) {
            if (!L.generic) {
                int rc = apply_one<T>(op, *p1, axis, f, df, na, nb, adj, s, Epilogue<T>(), ws);
                if (!rc) rc = apply_one<T>(op, *p1, axis, df, df, na, nb, adj, s, Epilogue<T>(), ws);
                return rc;
            }
        }
        T *tmp = nullptr;
        Workspace rest = ws;
        if (int rc = scratch_get<T>(rest, (size_t)count, s, &tmp, "cd06 second derivative intermediate")) return rc;
        int rc = apply_impl<T>(op, pade::D1, axis, f, tmp, na, nb, bc1, bcn, adj, s, Epilogue<T>(), rest);
        if (!rc) rc = apply_impl<T>(op, pade::D1, axis, tmp, df, na, nb, bc1, bcn, adj, s, epi, rest);
        scratch_put<T>(ws, tmp, s);
        return rc;
    }
    const Plan *pl = find_plan(op, oper, bc1, bcn, adj);
    if (!pl) return 21;
    const int rc = apply_one<T>(op, *pl, axis, f, df, na, nb, adj, s, epi, ws);
    if (!rc && op->periodic && edge_output(op->kind, oper)) {
        // an edge array's last plane repeats its first (cd06stagg.F90:859,969,1036)
        const size_t plane = (size_t)na * nb;
        hipError_t e = hipMemcpyAsync(df + plane * op->n, df, sizeof(T) * plane, hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) return hip_fail(e, "edge plane copy");
    }
    return rc;
}

// cf90 filter3 on complex(rkind) data (cf90.F90:1230-1251).  A complex
// (na, nb, n) array is a real (2 na, nb, n) one with the real and imaginary
// parts interleaved along its first axis, and the z filter treats both
// alike.  Bounded: the right-hand side of (bc1, bcn) when the caller passes
// them (has_bc), else of (0, 0), always solved with the (0, 0) left-hand side
// (penta_nn, cf90.F90:1249).  Periodic: the periodic filter (the reference
// solves with penta_nn there too, which a periodic cf90 never allocates).
int filter3_complex_impl(pade_op_t op, const double *f, double *df, int na, int nb, int bc1, int bcn, bool has_bc,
                         hipStream_t s)
{
    if (!op) return fail(400, "null operator");
    if (op->kind != pade::CF90) return fail(21, "filter3 on complex data is provided for cf90");
    if (!f || !df) return fail(400, "null array");
    if (na < 1 || nb < 1) return fail(400, "na and nb must be positive");
    if (na > (1 << 29)) return fail(400, "na too large");
    const int b1 = has_bc ? bc1 : 0, bn = has_bc ? bcn : 0;
    auto ok = [](int b) { return b == 0 || b == 1 || b == -1; };
    if (!ok(b1) || !ok(bn)) return fail(324, "Incorrect boundary specification (should be 0, 1 or -1)");
    if (op->periodic || op->n == 1 || (b1 == 0 && bn == 0))
        return apply_impl<double>(op, pade::FILTER, 3, f, df, 2 * na, nb, b1, bn, false, s);
    auto it = op->plans.find({kFilterRhsBc, b1, bn, 0});
    if (it == op->plans.end()) return fail(21, "no plan for this operation");
    return apply_one<double>(op, it->second, 3, f, df, 2 * na, nb, false, s, Epilogue<double>(), Workspace());
}

// Scratch of the allocation-free entry point (pade_op_apply_axpby_noalloc):
// one statically sized array per device, which each device holds until the
// process ends.  Host code uses the device address from hipGetSymbolAddress,
// looked up once per device with that device current; the array's own name
// is only a host-side handle.
constexpr size_t kNoAllocScratchBytes = size_t(PADE_NOALLOC_SCRATCH_BYTES);
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
char *g_scratch_ptr[kMaxDevices] = {};

// Device address of the current device's scratch array.
int noalloc_scratch(char **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return fail(400, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (!p) return fail(1000, "hipGetSymbolAddress(scratch) gave a null address");
        g_scratch_ptr[dev] = static_cast<char *>(p);
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

}  // namespace

extern "C" {

int pade_version(void) { return 100; }

const char *pade_last_error(void) { return g_last_error.c_str(); }

int pade_op_create(int kind, int n, double dx, int periodic, int bc1, int bcn, pade_op_t *out)
{
    if (!out) return fail(400, "null output handle");
    *out = nullptr;
    if (kind < pade::CD06 || kind > pade::GAUSSIAN) return fail(400, "unknown operator kind");
    if (n < 1) return fail(400, "n must be positive");
    const bool filter_kind = kind == pade::CF90 || kind == pade::GAUSSIAN;   // dx unused
    if (!filter_kind && !(dx > 0.0) && n > 1) return fail(400, "dx must be positive");
    if (int ierr = pade::init_error(kind, n, periodic != 0))
        return fail(ierr, "grid too small for this operator");
    if (kind == pade::CD06STAGG && !periodic) {
        auto ok = [](int b) { return b == 1 || b == -1 || b == 2 || b == -2; };
        if (!ok(bc1) || !ok(bcn))
            return fail(400, "bounded staggered ends: bc1 / bcn must be +-1 (even / odd) or "
                             "+-2 (one-sided closure, even / odd)");
    }
    auto op = std::make_unique<pade_op_s>();
    op->kind = kind;
    op->n = n;
    op->dx = filter_kind ? 1.0 : dx;
    op->periodic = periodic != 0;
    op->init_bc1 = bc1;
    op->init_bcn = bcn;
    hipError_t e = hipGetDevice(&op->device);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (n > 1) {
        if (int rc = build_all_plans(op.get())) {
            if (op->dtab64) hipFree(op->dtab64);
            if (op->dtab32) hipFree(op->dtab32);
            return rc;
        }
    }
    *out = op.release();
    return 0;
}

int pade_op_destroy(pade_op_t op)
{
    if (!op) return 0;
    if (op->dtab64) hipFree(op->dtab64);
    if (op->dtab32) hipFree(op->dtab32);
    pade::dense_release(op->dense);
    delete op;
    return 0;
}

int pade_op_size(pade_op_t op) { return op ? op->n : -1; }

int pade_op_apply(pade_op_t op, int oper, int axis, const double *f, double *df, int na, int nb,
                  int bc1, int bcn, void *stream)
{
    return apply_impl<double>(op, oper, axis, f, df, na, nb, bc1, bcn, false, (hipStream_t)stream);
}

int pade_op_apply_f32(pade_op_t op, int oper, int axis, const float *f, float *df, int na, int nb,
                      int bc1, int bcn, void *stream)
{
    return apply_impl<float>(op, oper, axis, f, df, na, nb, bc1, bcn, false, (hipStream_t)stream);
}

int pade_op_apply_adjoint(pade_op_t op, int oper, int axis, const double *f, double *df, int na,
                          int nb, int bc1, int bcn, void *stream)
{
    return apply_impl<double>(op, oper, axis, f, df, na, nb, bc1, bcn, true, (hipStream_t)stream);
}

int pade_op_apply_adjoint_f32(pade_op_t op, int oper, int axis, const float *f, float *df, int na,
                              int nb, int bc1, int bcn, void *stream)
{
    return apply_impl<float>(op, oper, axis, f, df, na, nb, bc1, bcn, true, (hipStream_t)stream);
}

int pade_op_apply_axpby(pade_op_t op, int oper, int axis, double alpha, const double *f, double beta, double *df,
                        int na, int nb, int bc1, int bcn, void *stream)
{
    Epilogue<double> epi;
    epi.on = true;
    epi.alpha = alpha;
    epi.beta = beta;
    return apply_impl<double>(op, oper, axis, f, df, na, nb, bc1, bcn, false, (hipStream_t)stream, epi);
}

int pade_op_apply_axpby_noalloc(pade_op_t op, int oper, int axis, double alpha, const double *f, double beta,
                                double *df, int na, int nb, int bc1, int bcn, void *stream)
{
    if (!op) return fail(400, "null operator");
    Workspace ws;
    ws.on = true;
    ws.bytes = kNoAllocScratchBytes;
    ws.owner = "the allocation-free entry point's scratch array (PADE_NOALLOC_SCRATCH_BYTES per device)";
    if (int rc = noalloc_scratch(&ws.ptr)) return rc;
    Epilogue<double> epi;
    epi.on = true;
    epi.alpha = alpha;
    epi.beta = beta;
    return apply_impl<double>(op, oper, axis, f, df, na, nb, bc1, bcn, false, (hipStream_t)stream, epi, ws);
}

int pade_op_apply_axpby_f32(pade_op_t op, int oper, int axis, float alpha, const float *f, float beta, float *df,
                            int na, int nb, int bc1, int bcn, void *stream)
{
    Epilogue<float> epi;
    epi.on = true;
    epi.alpha = alpha;
    epi.beta = beta;
    return apply_impl<float>(op, oper, axis, f, df, na, nb, bc1, bcn, false, (hipStream_t)stream, epi);
}

int pade_op_apply_host(pade_op_t op, int oper, int axis, const double *f, double *df, int na, int nb,
                       int bc1, int bcn)
{
    if (!op) return fail(400, "null operator");
    if (!f || !df) return fail(400, "null array");
    if (na < 1 || nb < 1) return fail(400, "na and nb must be positive");
    // staggered edge arrays hold one plane more than the pencil length
    const bool e_in = edge_input(op->kind, oper);
    const bool e_out = edge_output(op->kind, oper);
    const size_t plane = sizeof(double) * (size_t)na * nb;
    const size_t in_bytes = plane * (op->n + (e_in ? 1 : 0)), out_bytes = plane * (op->n + (e_out ? 1 : 0));
    double *df_d = nullptr, *f_d = nullptr;
    hipError_t e = hipMalloc(&f_d, in_bytes);
    if (e != hipSuccess) return hip_fail(e, "hipMalloc");
    e = hipMalloc(&df_d, out_bytes);
    if (e != hipSuccess) { hipFree(f_d); return hip_fail(e, "hipMalloc"); }
    int rc = 0;
    e = hipMemcpy(f_d, f, in_bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) rc = hip_fail(e, "hipMemcpy H2D");
    if (!rc) rc = apply_impl<double>(op, oper, axis, f_d, df_d, na, nb, bc1, bcn, false, nullptr);
    if (!rc) {
        e = hipMemcpy(df, df_d, out_bytes, hipMemcpyDeviceToHost);
        if (e != hipSuccess) rc = hip_fail(e, "hipMemcpy D2H");
    }
    hipFree(f_d);
    hipFree(df_d);
    return rc;
}

int pade_op_filter3_complex(pade_op_t op, const void *f, void *df, int na, int nb, int bc1, int bcn, int has_bc,
                            void *stream)
{
    return filter3_complex_impl(op, static_cast<const double *>(f), static_cast<double *>(df), na, nb, bc1, bcn,
                                has_bc != 0, (hipStream_t)stream);
}

int pade_op_filter3_complex_host(pade_op_t op, const void *f, void *df, int na, int nb, int bc1, int bcn,
                                 int has_bc)
{
    if (!op) return fail(400, "null operator");
    if (!f || !df) return fail(400, "null array");
    if (na < 1 || nb < 1) return fail(400, "na and nb must be positive");
    const size_t bytes = 2 * sizeof(double) * (size_t)na * nb * op->n;
    double *df_d = nullptr, *f_d = nullptr;
    hipError_t e = hipMalloc(&f_d, bytes);
    if (e != hipSuccess) return hip_fail(e, "hipMalloc");
    e = hipMalloc(&df_d, bytes);
    if (e != hipSuccess) { hipFree(f_d); return hip_fail(e, "hipMalloc"); }
    int rc = 0;
    e = hipMemcpy(f_d, f, bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) rc = hip_fail(e, "hipMemcpy H2D");
    if (!rc) rc = filter3_complex_impl(op, f_d, df_d, na, nb, bc1, bcn, has_bc != 0, nullptr);
    if (!rc) {
        e = hipMemcpy(df, df_d, bytes, hipMemcpyDeviceToHost);
        if (e != hipSuccess) rc = hip_fail(e, "hipMemcpy D2H");
    }
    hipFree(f_d);
    hipFree(df_d);
    return rc;
}

int pade_op_dense_apply(pade_op_t op, int oper, int axis, const void *f, int f_dtype, void *df,
                        int df_dtype, int na, int nb, int bc1, int bcn, int prec, void *stream)
{
    if (!op) return fail(400, "null operator");
    if (!f || !df) return fail(400, "null array");
    if (axis < 1 || axis > 3) return fail(400, "axis must be 1, 2 or 3");
    if (na < 1 || nb < 1) return fail(400, "na and nb must be positive");
    if (!oper_valid(op->kind, oper)) return fail(21, "operation not provided for this operator kind");
    if (op->kind != pade::CD06) {
        auto ok = [](int b) { return b == 0 || b == 1 || b == -1; };
        if (!ok(bc1) || !ok(bcn))
            return fail(324, "Incorrect boundary specification (should be 0, 1 or -1)");
    }
    if (op->kind == pade::CD06STAGG) return fail(21, "no dense form of the staggered operators");
    const bool full = (prec & PADE_DENSE_FULL) != 0;
    const int pbase = prec & ~PADE_DENSE_FULL;
    if (pbase != PADE_DENSE_F32 && pbase != PADE_DENSE_BF16X3) return fail(400, "unknown dense precision");
    if ((f_dtype != PADE_F64 && f_dtype != PADE_F32) || (df_dtype != PADE_F64 && df_dtype != PADE_F32))
        return fail(400, "unknown dtype");
    if (!op->periodic) return fail(21, "the dense form is provided for periodic operators");
    if (op->n < 64 || op->n % 64 != 0) return fail(21, "the dense form needs n a multiple of 64");
    auto it = op->plans.find({oper, 0, 0, 0});
    if (it == op->plans.end()) return fail(21, "no plan for this operation");
    const pade::DenseForm *D = nullptr;
    {
        std::lock_guard<std::mutex> lk(op->mu);
        int rc = pade::dense_get(op->dense, it->second.mats, oper, full, &D);
        if (rc) return fail(rc >= 1000 ? rc : 21, "dense operator construction failed");
    }
    hipError_t e = pade::dense_launch(*D, axis, f, f_dtype, df, df_dtype, na, nb, pbase, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e, "dense launch");
    return 0;
}

int pade_plan_variant(int kind, int oper, int n, double dx, int periodic, int bc1, int bcn, int adjoint, int axis,
                      int na, int nb, int dtype, int *info)
{
    if (!info) return fail(400, "null info");
    if (kind < pade::CD06 || kind > pade::GAUSSIAN) return fail(400, "unknown operator kind");
    if (!oper_valid(kind, oper)) return fail(21, "operation not provided for this operator kind");
    if (axis < 1 || axis > 3) return fail(400, "axis must be 1, 2 or 3");
    if (na < 1 || nb < 1) return fail(400, "na and nb must be positive");
    if (dtype != PADE_F64 && dtype != PADE_F32) return fail(400, "dtype must be PADE_F64 or PADE_F32");
    if (int ierr = pade::init_error(kind, n, periodic != 0)) return fail(ierr, "grid too small");
    if (adjoint && kind == pade::CD06STAGG) return fail(21, "no adjoint of the staggered operators");
    if (adjoint && n > 1 && n < 16) return fail(21, "adjoint needs n >= 16");
    for (int k = 0; k < 8; k++) info[k] = 0;
    info[5] = 1;
    if (n == 1) return 0;        // a copy or a fill, no solve
    if (kind == pade::CD06 && oper == pade::D2 && !periodic) {
        oper = pade::D1;         // the first derivative applied twice
        info[5] = 2;
    }
    std::vector<double> tab;
    std::vector<pade::PartFactors> known;
    Plan pl;
    const bool filter_kind = kind == pade::CF90 || kind == pade::GAUSSIAN;
    if (int rc = build_plan(kind, oper, n, filter_kind ? 1.0 : dx, periodic != 0, bc1, bcn, adjoint != 0, tab, known, pl))
        return rc;
    int rc;
    int M = 0, pw = 1, P = 0, generic = 0, mode = 0, uneven = 0;
    if (dtype == PADE_F64) {
        LaunchPlan<double> L;
        rc = plan_launch<double>(pl, periodic != 0, axis, nullptr, nullptr, na, nb, L);
        if (!rc) { M = L.v->M; pw = L.pw; P = L.v->P; generic = L.generic; mode = L.mode; uneven = L.v->uneven; }
    } else {
        LaunchPlan<float> L;
        rc = plan_launch<float>(pl, periodic != 0, axis, nullptr, nullptr, na, nb, L);
        if (!rc) { M = L.v->M; pw = L.pw; P = L.v->P; generic = L.generic; mode = L.mode; uneven = L.v->uneven; }
    }
    if (rc) return rc;
    info[0] = M;
    info[1] = generic ? 1 : pw;
    info[2] = P;
    info[3] = generic;
    info[4] = mode;
    info[6] = uneven;
    return 0;
}

int pade_op_dense_info(pade_op_t op, int oper, int prec, int axis, int f_dtype, int df_dtype, int *window,
                       int *halfwidth, int *products)
{
    if (!op || !window || !halfwidth || !products) return fail(400, "null argument");
    if (op->kind == pade::CD06STAGG) return fail(21, "no dense form of the staggered operators");
    if (axis < 1 || axis > 3) return fail(400, "axis must be 1, 2 or 3");
    if ((f_dtype != PADE_F64 && f_dtype != PADE_F32) || (df_dtype != PADE_F64 && df_dtype != PADE_F32))
        return fail(400, "dtype must be PADE_F64 or PADE_F32");
    if (!oper_valid(op->kind, oper)) return fail(21, "operation not provided for this operator kind");
    if (!op->periodic) return fail(21, "the dense form is provided for periodic operators");
    if (op->n < 64 || op->n % 64 != 0) return fail(21, "the dense form needs n a multiple of 64");
    auto it = op->plans.find({oper, 0, 0, 0});
    if (it == op->plans.end()) return fail(21, "no plan for this operation");
    const pade::DenseForm *D = nullptr;
    std::lock_guard<std::mutex> lk(op->mu);
    int rc = pade::dense_get(op->dense, it->second.mats, oper, (prec & PADE_DENSE_FULL) != 0, &D);
    if (rc) return fail(rc >= 1000 ? rc : 21, "dense operator construction failed");
    *window = 16 * D->S;
    *halfwidth = D->halfwidth;
    const int base_prec = prec & ~PADE_DENSE_FULL;
    *products = pade::dense_products(*D, axis, f_dtype, df_dtype, base_prec);
    return 0;
}

int pade_pencil_copy(const void *src, void *dst, long long nbytes, void *stream)
{
    if (!src || !dst) return fail(400, "null array");
    if (nbytes < 0) return fail(400, "negative size");
    hipError_t e = pade::pencil_copy_launch(src, dst, nbytes, (hipStream_t)stream);
    return e == hipSuccess ? 0 : hip_fail(e, "pencil copy");
}

int pade_permute3(const void *src, void *dst, int elem_size, int n1, int n2, int n3, int perm, void *stream)
{
    if (!src || !dst) return fail(400, "null array");
    if (elem_size != 4 && elem_size != 8) return fail(400, "elem_size must be 4 or 8");
    if (n1 < 1 || n2 < 1 || n3 < 1) return fail(400, "sizes must be positive");
    if (perm < 1 || perm > 3) return fail(400, "perm must be 1, 2 or 3");
    hipError_t e = pade::permute_launch(src, dst, elem_size, n1, n2, n3, perm, (hipStream_t)stream);
    return e == hipSuccess ? 0 : hip_fail(e, "permute");
}

int pade_plan_export(int kind, int oper, int n, double dx, int periodic, int bc1, int bcn, int adjoint,
                     int M, double *tab, long long tab_len, int *meta)
{
    if (!meta) return fail(400, "null meta");
    if (kind < pade::CD06 || kind > pade::GAUSSIAN) return fail(400, "unknown operator kind");
    if (!oper_valid(kind, oper)) return fail(21, "operation not provided for this operator kind");
    if (int ierr = pade::init_error(kind, n, periodic != 0)) return fail(ierr, "grid too small");
    if (n < 4) return fail(21, "no table for n < 4");
    pade::OpMatrices m;
    if (int rc = operator_matrices(kind, oper, n, kind == pade::CF90 || kind == pade::GAUSSIAN ? 1.0 : dx,
                                   periodic != 0, bc1, bcn,
                                   adjoint != 0, m))
        return fail(rc, "operator construction failed");
    // a bounded staggered operator with an edge array: M = 0 exports the
    // one-lane-per-pencil form, M > 0 the partitioned kernels' system form
    if (kind == pade::CD06STAGG && !periodic && M > 0 && (pade::stagg_edge_in(oper) || pade::stagg_edge_out(oper)))
        if (int rc = pade::build_stagg_system(oper, n, dx, bc1, bcn, m)) return fail(rc, "operator construction failed");
    const int rows = m.n, cols = m.n_in ? m.n_in : m.n;   // a staggered cell <-> edge operator: n +- 1
    if (M == 0) {
        M = rows;
        for (int c : {32, 64, 16})
            if (rows == cols && rows % c == 0 && rows / c <= pade::kMaxPartitions) { M = c; break; }
    }
    if (M != rows && ((rows != cols && !m.rect) || rows % M))
        return fail(400, "partition size must divide the rows of a square or system-form operator");
    std::vector<double> t;
    Variant v;
    if (int rc = build_variant(m, M, t, v)) return fail(rc == 1 ? 400 : rc, "factorisation failed");
    int vals[32] = {rows, v.M, v.P, periodic ? 1 : 0, v.nbl, v.nbr, pade::kOffBl, pade::kOffBr,
                    pade::kOffCoef, v.coef_len, v.ncls, v.kq, v.len, cols, m.rect ? 1 : 0, m.tail ? 1 : 0};
    for (int k = 0; k < pade::kMaxPartitions; k++) vals[16 + k] = v.cls[k];
    std::memcpy(meta, vals, sizeof(vals));
    if (tab) {
        if (tab_len < v.len) return fail(400, "table buffer too small");
        std::copy(t.begin(), t.end(), tab);
    }
    return 0;
}

int pade_plan_export_uneven(int kind, int oper, int n, double dx, int periodic, int bc1, int bcn, int adjoint, int M,
                            double *tab, long long tab_len, int *meta)
{
    if (!meta) return fail(400, "null meta");
    if (kind < pade::CD06 || kind > pade::GAUSSIAN) return fail(400, "unknown operator kind");
    if (!oper_valid(kind, oper)) return fail(21, "operation not provided for this operator kind");
    if (int ierr = pade::init_error(kind, n, periodic != 0)) return fail(ierr, "grid too small");
    pade::OpMatrices m;
    const bool filter_kind = kind == pade::CF90 || kind == pade::GAUSSIAN;
    if (int rc = operator_matrices(kind, oper, n, filter_kind ? 1.0 : dx, periodic != 0, bc1, bcn, adjoint != 0, m))
        return fail(rc, "operator construction failed");
    if (kind == pade::CD06STAGG && !periodic && (pade::stagg_edge_in(oper) || pade::stagg_edge_out(oper)))
        if (int rc = pade::build_stagg_system(oper, n, dx, bc1, bcn, m)) return fail(rc, "operator construction failed");
    pade::UnevenParts parts;
    if (M < 16 || M > 64 || M % 8 || M == 56 || !pade::uneven_parts(m.n, M, parts))
        return fail(21, "no uneven split of this length");
    std::vector<double> t;
    Variant v;
    if (int rc = build_variant(m, M, t, v, &parts)) return fail(rc == 1 ? 400 : rc, "factorisation failed");
    const int cols = m.n_in ? m.n_in : m.n;
    int vals[64] = {m.n, v.M, v.P, periodic ? 1 : 0, v.nbl, v.nbr, pade::kOffBl, pade::kOffBr,
                    pade::kOffCoef, v.coef_len, v.ncls, v.kq, v.len, cols, m.rect ? 1 : 0, m.tail ? 1 : 0};
    for (int k = 0; k < v.P; k++) vals[k < 16 ? 16 + k : 54 + k - 16] = v.cls[k];
    vals[32] = std::min(2 * v.kq + 1, v.P);
    for (int p = 0; p < v.P; p++) vals[33 + p] = parts.start(p);
    std::memcpy(meta, vals, sizeof(vals));
    if (tab) {
        if (tab_len < v.len) return fail(400, "table buffer too small");
        std::copy(t.begin(), t.end(), tab);
    }
    return 0;
}

}  // extern "C"

namespace pade {

// The stage of apply_fields as a pass of its own.
static int run_stage(pade_op_t op, int nf, const BatchField *flds, int na, int nb, const Stage *stage, hipStream_t s)
{
    for (int k = 0; stage && k < nf; k++)
        if (int rc = cg_rk_stage((long long)na * nb * op->n, stage->dt, stage->A, stage->B, flds[k].out, flds[k].Q,
                                 flds[k].W, s))
            return rc;
    return 0;
}

int apply_fields(pade_op_t op, int oper, int axis, int nf, const BatchField *flds, int na, int nb, int times, bool acc,
                 double alpha, double beta, double *tmp, hipStream_t s, const Stage *stage)
{
    if (nf < 1 || nf > kMaxFields || times < 1 || times > 2 || (stage && (!acc || times != 1)))
        return fail(400, "bad batch");
    for (int k = 0; k < nf; k++) {
        if (int rc = check_apply(op, oper, axis, na, nb, flds[k].bc1, flds[k].bcn, false)) return rc;
        if (!flds[k].f || !flds[k].out) return fail(400, "null array");
    }
    // one launch for all fields where they share a partitioned kernel
    const bool composed = op->kind == CD06 && oper == D2 && !op->periodic;
    if (op->n > 1 && !composed && op->kind != CD06STAGG) {
        LaunchPlan<double> L;
        bool one = true;
        for (int k = 0; k < nf && one; k++) {
            const Plan *pl = find_plan(op, oper, flds[k].bc1, flds[k].bcn, false);
            if (!pl) return 21;
            LaunchPlan<double> Lk;
            if (int rc = plan_launch<double>(*pl, op->periodic, axis, flds[k].f, flds[k].out, na, nb, Lk)) return rc;
            one = !Lk.generic && (times == 2 ? twice_ok(Lk, false)
                                             : nf == 1 || ((Lk.v->uneven || Lk.pw == 2 || Lk.pw == 8) && !(acc && Lk.mode == 1)));
            if (k == 0) L = Lk;
            else one = one && Lk.v->M == L.v->M && Lk.v->P == L.v->P && Lk.pw == L.pw && Lk.v->uneven == L.v->uneven;
            L.a.fld[k] = Lk.a.fld[0];
            L.a.fld[k].tab = op->dtab64 + Lk.v->off;
        }
        if (one) {
            L.a.nfields = nf;
            L.a.axpby = acc ? 1 : 0;
            L.a.alpha = alpha;
            L.a.beta = beta;
            const int gw = L.pw == 8 ? whole_pencil_waves() : 1;
            hipError_t e;
            if (stage && L.mode == 0 && L.pw == 2) {
                for (int k = 0; k < nf; k++) {
                    L.a.fld[k].stage_q = flds[k].Q;
                    L.a.fld[k].stage_w = flds[k].W;
                }
                L.a.stage_dt = stage->dt;
                L.a.stage_a = stage->A;
                L.a.stage_b = stage->B;
                e = launch_stage(L.a, L.v->M, L.v->uneven, s);
                return e == hipSuccess ? 0 : hip_fail(e, "spike_apply launch");
            }
            if (times == 2) e = launch_twice(L.a, L.v->M, L.pw, gw, L.v->uneven, false, L.mode, s);
            else if (nf > 1) e = launch_fields(L.a, L.v->M, L.pw, gw, L.v->uneven, L.mode, s);
            else if (L.v->uneven) e = launch_uneven<double>(L.a, L.v->M, false, L.mode, s);
            else e = launch_spike<double>(L.a, L.v->M, L.pw, gw, false, L.mode, s);
            if (e != hipSuccess) return hip_fail(e, "spike_apply launch");
            return run_stage(op, nf, flds, na, nb, stage, s);
        }
    }
    for (int k = 0; k < nf; k++) {
        Epilogue<double> epi;
        epi.on = acc;
        epi.alpha = alpha;
        epi.beta = beta;
        const double *src = flds[k].f;
        if (times == 2) {
            if (!tmp) return fail(400, "no intermediate for a repeated apply");
            if (int rc = apply_impl<double>(op, oper, axis, src, tmp, na, nb, flds[k].bc1, flds[k].bcn, false, s,
                                            Epilogue<double>(), Workspace()))
                return rc;
            src = tmp;
        }
        if (int rc = apply_impl<double>(op, oper, axis, src, flds[k].out, na, nb, flds[k].bc1, flds[k].bcn, false, s,
                                        epi, Workspace()))
            return rc;
    }
    return run_stage(op, nf, flds, na, nb, stage, s);
}

bool apply_in_place_ok(pade_op_t op, int oper, int axis, int na, int nb, int bc1, int bcn)
{
    if (!op || op->n == 1 || axis < 1 || axis > 3 || na < 1 || nb < 1) return false;
    if (op->kind == CD06 && oper == D2 && !op->periodic) return false;
    if (op->periodic && edge_output(op->kind, oper)) return false;
    const int k1 = op->periodic ? 0 : plan_key_bc(op, bc1);
    const int kn = op->periodic ? 0 : plan_key_bc(op, bcn);
    auto it = op->plans.find({oper, k1, kn, 0});
    if (it == op->plans.end()) return false;
    LaunchPlan<double> L;
    if (plan_launch<double>(it->second, op->periodic, axis, (const double *)nullptr, (double *)nullptr, na, nb, L))
        return false;
    return !L.generic;
}

}  // namespace pade
