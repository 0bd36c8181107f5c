// Compact-difference operator kernels for CDNA4 (gfx950).
//
// One operator application is  out = A^{-1} (B f)  (forward) or
// out = B^T (A^{-T} g)  (adjoint), applied to every pencil of a 3-D
// Fortran-ordered array along one axis.  A is a band matrix of half-width 2
// (cyclic when periodic), B a 9-point stencil with explicit boundary rows.
//
// Fast path (spike_apply): a pencil of n = P*M points is split into P
// partitions of M points.  A workgroup holds NPEN = 64/PW pencils and all P
// partitions of them; each wave serves PW partitions (PW = 1: 64 pencils x 1
// partition, PW = 2: 32 pencils x 2 partitions, PW = 8: 8 whole pencils of
// up to 8 partitions, x pencils only), one (pencil, partition) per lane with
// the M values in registers.  Each lane
//   1. loads its window (M points + 4-point halos) and evaluates the stencil,
//   2. solves its partition's band block (forward + backward sweep) with
//      coefficients staged once per workgroup in LDS,
//   3. publishes the four "tip" values (first two / last two) through LDS,
//   4. forms the neighbouring tips from the precomputed inverse of the reduced
//      tip system (only the partitions whose weights are not negligible), and
//   5. corrects its partition with the coupling columns.
// This is an exact partitioned (SPIKE-type) solve: every value of f is read
// once and every value of out written once, so the HBM traffic is the
// algorithmic 2 * sizeof(T) bytes per point.  PW = 2 halves the pencils per
// workgroup so that two workgroups fit on a CU and one's memory phase
// overlaps the other's arithmetic.
//
// Pencils along y and z are strided in memory: lanes are neighbouring pencils,
// so every load is a contiguous row.  Pencils along x are contiguous: each
// wave moves small tiles through LDS so that global loads/stores stay
// coalesced (MODE 1).
//
// Uneven partitions (UNE): where M does not divide n, partitions of at most M
// rows occupy M slots each (UnevenParts: padding slots with y_t = y_{t-2}).
// Windows of M points start at each partition's first row and overlap the
// next partition; right-hand sides of padding slots are zeroed and their
// results not stored, everything else is the even kernel, with a coefficient
// class per partition size and every partition's reduced-system rows over its
// window.  What bounds it is, as there, memory, and beside it the slots that
// carry no row (up to a third for short pencils) and lines shared between
// partitions or pencils.  The one-lane path that these lengths took before is
// a chain of n dependent loads per lane.  cd10 d1 with 33.5 M points, FP64, x
// / y / z Gpts/s: n = 129 (512^2 pencils) 229 / 300 / 297 periodic, 210 / 260
// / 245 bounded; n = 257 (361^2) 189 / 217 / 214; one lane per pencil ran a
// 257 x 193 x 129 bounded gradient in 1641 us, uneven partitions in 122 us.
//
// Generic path (generic_apply, pade_kernels.hip): one lane per pencil with
// the whole pencil as one partition in global memory -- for sizes the
// register path does not cover (n < 24 unless 16, n > 1344, or fewer than 128 pencils of an uneven length).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdlib>

#include <algorithm>
#include <cstdint>

#include "pade_kernels.h"

namespace pade {

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Workgroup barrier that orders LDS only: outstanding global loads stay in
// flight across it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ int wrap_index(int j, int n, int periodic)
{
    if (j < 0) return periodic ? j + n : 0;
    if (j >= n) return periodic ? j - n : n - 1;
    return j;
}

// Element at wave-uniform pointer `u` plus a per-lane byte offset `off`:
// written this way the address is an SGPR base plus one 32-bit VGPR, so the
// unrolled loads/stores do not each carry a 64-bit per-lane address.
template <typename T>
__device__ __forceinline__ T ld(const T *u, unsigned off)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(u) + off);
}
template <typename T>
__device__ __forceinline__ void st(T *u, unsigned off, T v)
{
    *reinterpret_cast<T *>(reinterpret_cast<char *>(u) + off) = v;
}

// Streaming (non-temporal) forms for the field.  Every output is written
// once, so the stores do not need to stay in L2: with the nt hint they stop
// evicting the lines that neighbouring partitions still read as halos (x
// reads fall from 1.09x to 1.05x of the field) and the solve runs 2-4 %
// faster on every axis.  The loads stay cached where other partitions read
// the same lines again as halos: nt loads slowed x (two partitions per wave)
// and z, whose halo lines are then fetched twice (x reads 1.05x -> 1.17x).
// Whole-pencil x waves read every line once, and stream their loads.  (A
// plain 1 GiB device copy goes from 5.6 to 6.4 TB/s with both.)
constexpr bool kNtStore = true;    // output stores
template <bool NT, typename T>
__device__ __forceinline__ T ld_s(const T *u, unsigned off)
{
    const T *p = reinterpret_cast<const T *>(reinterpret_cast<const char *>(u) + off);
    if constexpr (NT) return __builtin_nontemporal_load(p);
    return *p;
}
template <typename T>
__device__ __forceinline__ void st_s(T *u, unsigned off, T v)
{
    T *p = reinterpret_cast<T *>(reinterpret_cast<char *>(u) + off);
    if constexpr (kNtStore) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// Scheduling region length (rows): a compiler memory barrier every kRegion
// rows of the unrolled sweeps keeps the LDS coefficient reads next to their
// use; left alone the compiler issues all of them up front and spills them.
// (Field loads are all issued before the sweeps and stores come after, so the
// barrier does not reduce memory-level parallelism.)
constexpr int kRegion = 4;

// Rows per batch of the accumulate epilogue's loads on strided rows.
constexpr int kEpiRows = 8;
__device__ __forceinline__ void mem_region_fence() { asm volatile("" ::: "memory"); }
// Materialise a value here: keeps MachineSink from moving the arithmetic that
// produces it down into the (conditional) store block while the coefficient
// reads it consumed stay behind, alive in spilled registers.
template <typename T>
__device__ __forceinline__ void pin(T &x) { asm volatile("" : "+v"(x)); }
#define PADE_REGION_END(t) \
    do {                                         \
        if (((t) % kRegion) == kRegion - 1) mem_region_fence(); \
    } while (0)

// x-pencil transpose tile: XT points of a row per chunk (aligned segments
// of 64 bytes for FP64, 128 bytes for FP32 -- the widths that keep the FP64
// M = 64 kernel within 256 registers and the FP32 one within 128; partitions
// that those do not divide take 16 or 8 points); the halo
// chunk holds the 4 + 4 window points either side of the partition.
__host__ __device__ constexpr int xtile_points(int tsize, int M)
{
    const int xt = tsize == 8 ? 16 : 32;
    return M % xt == 0 ? xt : (M % 16 == 0 ? 16 : 8);
}
constexpr int kHaloChunk = 8;
// How the row segments of a strided-row workgroup (its pencils' values at one
// point) lie in memory:
//   kWholeLines  every segment is whole 128-byte lines: streamed (nontemporal)
//                stores, and loads on bounded pencils;
//   kHalfLines   whole 64-byte memory accesses, but lines shared with the
//                neighbouring workgroups: streamed stores, cached loads;
//   kShared      segments start anywhere: cached stores and loads, so that the
//                parts of a 64-byte access meet in L2 instead of being written
//                to memory one by one.
// Where lines are shared, runs of consecutive workgroups go to one XCD, whose
// L2 then holds both users of a line.  cd10 d1 n = 256, FP64, y / z Gpts/s
// (1 GB fields): planes of 720^2 (whole lines) 342 / 316; 721^2 streamed in
// launch order 179 / 161, streamed with runs 205 / 178, cached with runs 273
// / 243; 728-wide rows (half lines) 306, 332 and 310; bounded z at 721^2 148,
// 171 and 252; FP32 1025^2 230 / 213, 304 / 256 and 505 / 447.  (Windows that
// overlap so that every 32-byte sector is stored whole by one workgroup:
// 242 / 208.)
enum RowLayout { kWholeLines = 0, kHalfLines = 1, kShared = 2 };
// Epilogue: store op(f); alpha op(f) + beta out; a Runge-Kutta stage on that.
enum Epi { kStore = 0, kAxpby = 1, kStage = 2 };
// rows every partition has (UnevenParts keeps to it)
constexpr int kMinRows = 8;
// 16-byte lanes: VL elements per lane, XT / VL lanes per tile row; tile rows
// padded by one lane width (16-byte aligned)
__host__ __device__ constexpr int xtile_row(int tsize, int M) { return xtile_points(tsize, M) + 16 / tsize; }

// LDS layout (elements of T):
//   tips  [4P][NPEN]               (whole-pencil x waves: in their tile)
//   halo  [8P][NPEN]               adjoint, y/z pencils (partition end values)
//   bnd   [256]                    bounded only: boundary rows (left 128, right 128)
//   coef  [coef_len]               coefficient classes + reduced-system rows
//   xt    [waves][64][XT + VL]     x pencils only; the x adjoint's halo
//                                  exchange uses the start of this area (the
//                                  tiles are idle between the load and store
//                                  transposes), which keeps the M = 64 FP64
//                                  adjoint at two workgroups per CU
__host__ __device__ inline int lds_elems(int M, int P, int PW, bool adj, int mode, int coef_len, int tsize, bool bnd,
                                         int gw)
{
    const int npen = 64 / PW;
    const bool whole = mode == 1 && PW == 8;      // tips in the tile area
    const int waves = whole ? gw : (P + PW - 1) / PW;
    // (x pencils exchange the adjoint halo through their transpose tiles)
    int e = (whole ? 0 : (adj && mode != 1 ? 12 : 4) * P * npen) + (bnd ? 256 : 0) + coef_len;
    if (mode == 1) {
        const int vl = 16 / tsize;
        e = (e + vl - 1) / vl * vl;           // 16-byte aligned tile
        e += waves * 64 * xtile_row(tsize, M);
    }
    return e;
}

inline size_t spike_lds_bytes(size_t tsize, int M, int P, int PW, bool adj, int mode, int coef_len, bool bnd, int gw)
{
    return (size_t)lds_elems(M, P, PW, adj, mode, coef_len, (int)tsize, bnd, gw) * tsize;
}

// Right rows read the window from its last point (RS = 0: column c is point
// n - 1 - c) or from the first right-halo point (RS = 1: point n - c, the
// input of a staggered edge-to-cell operator has one point more).
template <typename T, int M, int NB, int RS = 0>
__device__ __forceinline__ void boundary_rows(const T (&w)[M + 8], const T *rows, int nrows, bool right,
                                              T (&res)[NB])
{
#pragma unroll
    for (int r = 0; r < NB; r++) {
        T s = T(0);
        if (r < nrows) {
#pragma unroll
            for (int c = 0; c < kBColsDev; c++)
                s += rows[r * kBColsDev + c] * (right ? w[M + 3 + RS - c] : w[4 + c]);
        }
        res[r] = s;
    }
}

// B (or B^T) applied in place on the window: w[t+4] is point t on entry,
// w[t] is row t on exit; special rows at the ends of a bounded pencil replace
// the interior stencil there.
template <typename T, int M, int NB, int RS = 0>
__device__ __forceinline__ void apply_stencil(T (&w)[M + 8], const T *__restrict__ tab, const T *bnd,
                                              bool edge_left, bool edge_right, int nbl, int nbr)
{
    T lb[NB], rb[NB];
    if (edge_left) boundary_rows<T, M, NB>(w, bnd, nbl, false, lb);
    if (edge_right) boundary_rows<T, M, NB, RS>(w, bnd + 128, nbr, true, rb);
    T cst[9];
#pragma unroll
    for (int k = 0; k < 9; k++) cst[k] = tab[k];
#pragma unroll
    for (int t = 0; t < M; t++) {
        T s = cst[0] * w[t];
#pragma unroll
        for (int k = 1; k < 9; k++) s += cst[k] * w[t + k];
        w[t] = s;
    }
    if (edge_left) {
#pragma unroll
        for (int r = 0; r < NB; r++)
            if (r < nbl) w[r] = lb[r];
    }
    if (edge_right) {
#pragma unroll
        for (int r = 0; r < NB; r++)
            if (r < nbr) w[M - 1 - r] = rb[r];
    }
}

// The fields of a launch, grid y.  A launch of one field has a kernel of its
// own (NF = 1), whose arguments are all at known places: a struct indexed by
// the field stays in memory as a whole, so it is an argument beside the others
// (one struct for both: FP64 x, M = 32, periodic, 132 registers instead of 128,
// three waves per SIMD instead of four), and the dependent read of its entries
// stands before the first load of every workgroup (FP64 cd06 64^3 x / z 5.7 /
// 5.6 us indexed, 5.5 / 5.3 not; cd10 512^3 z 421.9 and 417.4, FP32 x 187.5 and
// 186.0; uneven, 97 points, 192 x 144 pencils, z 12.3 and 11.5).
template <typename T, int NF>
struct FieldSet {
    SolveArgs<T> shared;   // the other argument once more, see spike_apply
    FieldArgs<T> fld[NF];
};

template <typename T, int M, int PW, bool ADJ, int MODE, bool BND, int EPI, bool UNE = false, int ROWS = kWholeLines,
          int REP = 1, int NF = 1>
__global__ __launch_bounds__(512) void spike_apply(SolveArgs<T> args, FieldSet<T, NF> fields)
{
    constexpr int NPEN = 64 / PW;
    // Strided kernels of several fields run out of scalar registers and read
    // the shared arguments from memory instead (129 points, 512 x 512 pencils,
    // periodic z 117.6 -> 113.5 us; the stage, M = 32, 133 -> 122 registers, 51
    // -> 0 spilled scalars)
    const SolveArgs<T> &a = NF > 1 && (MODE == 0 || PW == 8) ? fields.shared : args;
    const FieldArgs<T> &fd = fields.fld[NF > 1 ? blockIdx.y : 0];
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T *smem = reinterpret_cast<T *>(smem_raw);
    constexpr bool WHOLE = MODE == 1 && PW == 8;
    const int lane = threadIdx.x & 63;
    const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Waves of a workgroup serve consecutive partitions of the same NPEN
    // pencils; whole-pencil waves (all partitions in the wave) serve
    // consecutive groups of NPEN pencils instead, sharing the coefficient copy.
    const int wave = WHOLE ? 0 : wave_id;        // the wave's partition group
    const int half = PW == 1 ? 0 : lane / NPEN;  // this lane's partition within the wave
    const int pen = lane & (NPEN - 1);
    const int P = a.P;
    const int n = a.n;
    const int p = wave * PW + half;              // this lane's partition
    const bool active = p < P;
    const int pc = active ? p : P - 1;           // clamped for addressing
    // first point and rows of a partition (uneven: see UnevenParts)
    auto part_start = [&](int part) { return UNE ? part * a.ubase + min(part, a.uextra) * a.uunit : part * M; };
    auto part_rows = [&](int part) {
        return UNE && part < P - 1 ? a.ubase + (part < a.uextra ? a.uunit : 0) : M;
    };
    const int pM = part_start(pc);
    const int mrows = part_rows(pc);             // rows of this lane's partition
    const int pw0 = part_start(wave * PW);       // first point of this wave's first partition
    long long bid = blockIdx.x;
    if (a.remap) {
        // workgroup i runs on XCD i % 8 as that XCD's (i / 8)-th; each XCD
        // takes runs of C consecutive workgroups (C = remap, or an eighth of
        // the grid for remap < 0), the grid's tail beyond whole rounds of 8 C
        // in launch order
        const long long C = a.remap > 0 ? a.remap : gridDim.x / 8;
        const long long gc = C > 0 ? gridDim.x / (8 * C) * (8 * C) : 0;
        if (bid < gc) {
            const long long k = bid / 8;
            bid = (k / C) * (8 * C) + (bid % 8) * C + k % C;
        }
    }
    const long long q0 = WHOLE ? (bid * (blockDim.x >> 6) + wave_id) * NPEN : bid * NPEN;
    const long long q = q0 + pen;
    const bool inrange = q < a.npencils;
    const bool valid = active && inrange;
    // Base of the workgroup's first pencil and this lane's byte offset from it.
    // x and z pencils are one run of npencils; y pencils runs of A1, the
    // lane's run found from the first pencil's (32-bit: a launch has fewer
    // than 2^32 pencils).  The 64-bit divisions this replaces were several
    // hundred instructions before the first load.
    long long base0;
    unsigned loff = 0;
    if (MODE == 1 || a.A1 == a.npencils) {
        base0 = q0 * a.B1;
        if (MODE != 1 && inrange) loff = (unsigned)(pen * a.B1 * (long long)sizeof(T));
    } else {
        const unsigned run = (unsigned)a.A1, r0 = (unsigned)q0 / run, i0 = (unsigned)q0 - r0 * run;
        base0 = i0 * a.B1 + r0 * a.B2;
        const unsigned i = i0 + pen;
        const unsigned dr = run >= (unsigned)NPEN ? (i >= run ? 1u : 0u) : i / run;
        if (inrange)
            loff = (unsigned)((((long long)(i - dr * run) - i0) * a.B1 + (long long)dr * a.B2) * (long long)sizeof(T));
    }
    const long long stp = a.stride;
    const T *__restrict__ fb = fd.f + base0;
    T *__restrict__ ob = fd.out + base0;
    const T *__restrict__ tab = fd.tab;
    const bool edge_left = BND && p == 0;
    const bool edge_right = BND && p == P - 1;

    // x tile rows <-> (pencil, partition of the wave).  Partition-major rows
    // (partition * NPEN + pencil: lane l owns row l) put the per-lane row
    // accesses of the transposes on distinct LDS banks; pencil-major rows
    // (pencil * PW + partition) put consecutive lanes on rows PW apart, an
    // 8-way bank conflict at PW = 8.  Measured at 512^3: whole-pencil FP64
    // x +7-8 %, pair-wave FP64 +1-2 %, pair-wave FP32 -2-3 % (it keeps
    // pencil-major rows, whose load instructions span fewer pencils).
    constexpr bool PMAJ = sizeof(T) == 8 || PW >= 4;
    auto row_pen = [](int r) { return PMAJ ? r % NPEN : r / PW; };
    auto row_part = [](int r) { return PMAJ ? r / NPEN : r % PW; };
    auto tile_row = [](int pn, int pt) { return PMAJ ? pt * NPEN + pn : pn * PW + pt; };
    T *bnd = smem + (WHOLE ? 0 : ((ADJ || REP > 1) && MODE != 1 ? 12 : 4) * P * NPEN);   // [256] (bounded)
    T *coef = bnd + (BND ? 256 : 0);                    // [coef_len]
    constexpr int XT = xtile_points(sizeof(T), M), PAD = xtile_row(sizeof(T), M);
    constexpr int VL = 16 / sizeof(T);                  // elements per 16-byte lane
    constexpr int LPR = XT / VL;                        // lanes per tile row
    typedef T vec_t __attribute__((ext_vector_type(VL)));
    // global vectors of uneven pencils start at any element
    typedef T vec_g __attribute__((ext_vector_type(VL), aligned(UNE ? sizeof(T) : 16)));
    auto ldg = [](const T *u, unsigned off) -> vec_t {
        return *reinterpret_cast<const vec_g *>(reinterpret_cast<const char *>(u) + off);
    };
    auto ldg_nt = [](const T *u, unsigned off) -> vec_t {
        return __builtin_nontemporal_load(reinterpret_cast<const vec_g *>(reinterpret_cast<const char *>(u) + off));
    };
    constexpr bool STREAM = ROWS != kShared;
    auto stg = [](T *u, unsigned off, vec_t v) {
        vec_g *d = reinterpret_cast<vec_g *>(reinterpret_cast<char *>(u) + off);
        if constexpr (STREAM) __builtin_nontemporal_store(v, d);
        else *d = v;
    };
    auto put = [](T *u, unsigned off, T v) {
        if constexpr (STREAM) st_s(u, off, v);
        else st(u, off, v);
    };
    // Tile row that this lane of memory instruction s moves (16 bytes of
    // it).  Whole-pencil waves with one instruction per pencil and chunk take
    // pencil s, its partitions across the lane groups (8 lines of one pencil
    // per instruction: copies of 512^3 FP64 x pencils measured 6.1 TB/s that
    // way against 5.9 TB/s for one line of each of 8 pencils); other waves
    // take 64 / LPR consecutive tile rows.
    constexpr bool PINS = WHOLE && XT / VL == NPEN && 64 / LPR == PW;
    auto instr_row = [&](int s_) { return PINS ? tile_row(s_, lane / LPR) : s_ * (64 / LPR) + lane / LPR; };
    const int xt0 = ((int)(coef - smem) + fd.coef_len + VL - 1) / VL * VL;
    T *xt = smem + xt0 + wave_id * 64 * PAD;
    // [8P][NPEN] adjoint halo: 8P * NPEN <= waves * 64 * PAD since PAD >= 8
    // (a whole-pencil wave: in its own tile, 8P * NPEN <= 64 * PAD)
    T *halo = MODE == 1 ? (WHOLE ? xt : smem + xt0) : smem + 4 * P * NPEN;
    // [4P][NPEN] tips; a whole-pencil wave keeps them in its own tile, idle
    // between the load and store transposes
    T *tips = WHOLE ? xt : smem;

    // ----------------------------------------------- 0. coefficients -> LDS
    // (broadcast LDS reads measured faster than scalar loads of the same
    // wave-uniform coefficients, and this order -- table copy, then the
    // field loads -- faster than issuing the field loads first)
    // Batches of eight loads per thread before their LDS writes (sixteen for
    // bounded tables, whose per-partition reduced-system rows run to a few
    // thousand elements: one round trip instead of two at n = 512, bounded
    // y / z +1 %), so a table costs one memory round trip per U x blockDim
    // elements.
    {
        const T *g = tab + kOffCoef;
        const int len = fd.coef_len;
        const int nt = blockDim.x;
        constexpr int U = BND ? 16 : 8;
        for (int b0 = threadIdx.x; b0 < len; b0 += U * nt) {
            T v[U];
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = g[min(b0 + u * nt, len - 1)];   // unconditional loads
#pragma unroll
            for (int u = 0; u < U; u++)
                if (b0 + u * nt < len) coef[b0 + u * nt] = v[u];
        }
        if (BND)
            for (int idx = threadIdx.x; idx < 256; idx += nt) bnd[idx] = tab[kOffBl + idx];
    }

    T w[M + 8];

    // --------------------------------------------------------------- 1. load
    T hv[kHaloChunk];                                    // x halo chunk (forward)
    if constexpr (MODE != 1) {
        // main rows: uniform base of this wave's first partition + per-lane offset
        const unsigned hoff = loff + (unsigned)((long long)(UNE ? pM - pw0 : half * M) * stp * (long long)sizeof(T));
        // (nontemporal on bounded pencils: 512^3 FP64 bounded y / z 324 / 307
        // -> 329-331 / 312 Gpts/s; on periodic ones no gain on y, z 323.5 ->
        // 313 with them)
        if constexpr (!ADJ) {
            // halo rows (wrapped per partition, or clamped at the ends of a
            // bounded pencil, where the boundary rows replace the stencil):
            // before the main rows on periodic FP32 pencils (512^3 y / z 223.4
            // / 228.7 -> 218.9 / 221.6 us, 222.0 / 222.7 as the compiler ordered
            // them before the kernel served several fields).  (Written out
            // twice: as one lambda they held the main loads of every kernel
            // back by 180 instructions, the twice-applied strided one 174 ->
            // 179 us.)
            constexpr bool HALO_FIRST = sizeof(T) == 4 && !BND && EPI == kStore;
            if constexpr (HALO_FIRST) {
                const T *fq = fd.f + base0 + (long long)(loff / sizeof(T));
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int jl = wrap_index(pM - 4 + k, n, !BND);
                    const int jr = wrap_index(pM + M + k, MODE == 2 ? a.n_in : n, !BND);
                    w[k] = fq[(long long)jl * stp];
                    w[M + 4 + k] = fq[(long long)jr * stp];
                }
                mem_region_fence();
            }
#pragma unroll
            for (int t = 4; t < M + 4; t++) w[t] = ld_s<BND && ROWS == kWholeLines>(fb + (long long)(pw0 - 4 + t) * stp, active ? hoff : loff);
            if constexpr (!HALO_FIRST) {
                const T *fq = fd.f + base0 + (long long)(loff / sizeof(T));
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int jl = wrap_index(pM - 4 + k, n, !BND);
                    // a staggered operator's input may hold one point more than its rows
                    const int jr = wrap_index(pM + M + k, MODE == 2 ? a.n_in : n, !BND);
                    w[k] = fq[(long long)jl * stp];
                    w[M + 4 + k] = fq[(long long)jr * stp];
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < M; t++) w[t] = ld_s<BND && ROWS == kWholeLines>(fb + (long long)(pw0 + t) * stp, active ? hoff : loff);
        }
    } else {
        // x pencils: tile rows r = (pencil, half) of this wave.  Main chunks:
        // XT contiguous points of one row, 16 bytes per lane, so that every
        // load instruction covers G whole 128-byte rows.  Then the forward
        // halo chunk (issued last, so that its lines are mostly in flight or
        // in L2 already from the neighbouring partitions' main chunks),
        // wrapped, or clamped at the ends of a bounded pencil:
        //   PW == 2: one side per tile row -- the left halo of the pair's
        //     first partition and the right halo of its second (of the first
        //     when the pair has no second); the boundary inside the pair
        //     comes from the main chunks in LDS;
        //   PW == 1 or 4: both sides, 4 + 4 points;
        //   PW == 8 (whole pencils per wave, P <= 8): none -- every halo is
        //     in the wave's own tile.
        constexpr int G = 64 / LPR;                      // rows per load instruction
        constexpr int NCH = M / XT;
        constexpr int W0 = ADJ ? 0 : 4;                  // register slot of the first point
        static_assert(M % XT == 0, "chunking");
#pragma unroll
        for (int c = 0; c < NCH; c++) {
#pragma unroll
            for (int s = 0; s < XT / VL; s++) {
                const int r = instr_row(s);                  // tile row
                const int rp = row_pen(r), rh = row_part(r);
                const int part = wave * PW + rh;
                const bool ok = q0 + rp < a.npencils && part < P;
                const int j = part_start(ok ? part : 0) + c * XT + VL * (lane % LPR);
                const unsigned xo = ok ? (unsigned)((rp * (long long)n + j) * (long long)sizeof(T)) : 0u;
                const vec_t v = WHOLE ? ldg_nt(fb, xo) : ldg(fb, xo);
#pragma unroll
                for (int e = 0; e < VL; e++) w[W0 + c * XT + s * VL + e] = v[e];
            }
        }
        if constexpr (!ADJ && !WHOLE) {    // (whole-pencil waves need no halo loads)
            constexpr int HC = PW == 2 ? 4 : kHaloChunk;     // halo values per tile row
            constexpr int GH = 64 / HC;
#pragma unroll
            for (int s = 0; s < HC; s++) {
                const int r = s * GH + lane / HC;
                const int rp = row_pen(r), rh = row_part(r);
                const int part = wave * PW + rh;
                const int k = lane % HC;
                bool ok = q0 + rp < a.npencils;
                int j0;
                if constexpr (PW == 2) {
                    const int tp = min(part, P - 1);
                    j0 = rh == 0 ? part_start(tp) - 4 + k : part_start(tp) + M + k;
                } else {
                    ok = ok && part < P;
                    j0 = part_start(ok ? part : 0) + (k < 4 ? k - 4 : M + k - 4);
                }
                const int j = wrap_index(j0, n, !BND);
                const unsigned xo = ok ? (unsigned)((rp * (long long)n + j) * (long long)sizeof(T)) : 0u;
                hv[s] = ld(fb, xo);
            }
        }
    }

    if constexpr (MODE == 1) {
        // wave-local transposes: row-major tile -> one row per lane
        constexpr int G = 64 / LPR;
        constexpr int NCH = M / XT;
        constexpr int W0 = ADJ ? 0 : 4;
        const int myrow = tile_row(pen, half);
#pragma unroll
        for (int c = 0; c < NCH; c++) {
#pragma unroll
            for (int s = 0; s < XT / VL; s++) {
                vec_t v;
#pragma unroll
                for (int e = 0; e < VL; e++) v[e] = w[W0 + c * XT + s * VL + e];
                *reinterpret_cast<vec_t *>(xt + instr_row(s) * PAD + VL * (lane % LPR)) = v;
            }
            wave_lds_sync();
#pragma unroll
            for (int j = 0; j < XT / VL; j++) {
                const vec_t v = *reinterpret_cast<const vec_t *>(xt + myrow * PAD + VL * j);
#pragma unroll
                for (int e = 0; e < VL; e++) w[W0 + c * XT + j * VL + e] = v[e];
            }
            if constexpr (PW == 2 && !ADJ) {
                // the pair's shared boundary: the first partition's right halo
                // is the second's first four points, the second's left halo the
                // first's last four (uneven: the first partition has ma <= M
                // rows, so the second starts at its slot ma; of its right halo
                // only slots M .. ma + 3 are read by its rows)
                const int ma = UNE ? part_rows(min(wave * 2, P - 1)) : M;
                if (c == 0) {
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const T t = xt[tile_row(pen, 1) * PAD + (UNE ? min(M - ma + k, XT - 1) : k)];
                        if (half == 0) w[M + 4 + k] = t;
                    }
                }
                if constexpr (UNE) {
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const int t = ma - 4 + k - c * XT;       // column of this chunk
                        if (t >= 0 && t < XT) {                  // uniform over the wave
                            const T v = xt[tile_row(pen, 0) * PAD + t];
                            if (half == 1) w[k] = v;
                        }
                    }
                } else if (c == NCH - 1) {
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const T t = xt[tile_row(pen, 0) * PAD + XT - 4 + k];
                        if (half == 1) w[k] = t;
                    }
                }
            } else if constexpr (WHOLE && !ADJ) {
                // whole pencils in the wave (P <= PW): every halo is the end of
                // a neighbouring partition in the tile, across the periodic
                // wrap too (at the ends of a bounded pencil the boundary rows
                // replace the rows that would read the wrapped values)
                if (c == 0) {
                    const int hr = half + 1 < P ? half + 1 : 0;
#pragma unroll
                    for (int k = 0; k < 4; k++) w[M + 4 + k] = xt[tile_row(pen, hr) * PAD + k];
                }
                if (c == NCH - 1) {
                    const int hl = half >= 1 ? half - 1 : P - 1;
#pragma unroll
                    for (int k = 0; k < 4; k++) w[k] = xt[tile_row(pen, hl) * PAD + XT - 4 + k];
                }
            }
            wave_lds_sync();
        }
        if constexpr (!ADJ && !WHOLE) {
            constexpr int HC = PW == 2 ? 4 : kHaloChunk;
            constexpr int GH = 64 / HC;
#pragma unroll
            for (int s = 0; s < HC; s++)
                xt[(s * GH + lane / HC) * PAD + (lane % HC)] = hv[s];
            wave_lds_sync();
            if constexpr (PW == 2) {
                const bool pair = wave * 2 + 1 < P;      // uniform: the wave's second partition exists
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const T own = xt[myrow * PAD + k];
                    const T nxt = xt[tile_row(pen, 1) * PAD + k];
                    if (half == 0) {
                        w[k] = own;
                        if (!pair) w[M + 4 + k] = nxt;
                    } else {
                        w[M + 4 + k] = own;
                    }
                }
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    w[k] = xt[myrow * PAD + k];
                    w[M + 4 + k] = xt[myrow * PAD + 4 + k];
                }
            }
            wave_lds_sync();
        }
    }

    // coefficient blocks of this lane's partition
    // (four partitions per wave of a long uneven pencil: three bits each)
    constexpr int CB = UNE && PW == 4 ? 3 : 4;
    const int cls = BND || UNE ? (int)(fd.cls4 >> (CB * pc)) & ((1 << CB) - 1) : 0;
    const T *lu = coef + cls * 10 * M;      // [M][6]
    const T *S = lu + 6 * M;                // [M][4]
    const T *Qb = coef + fd.ncls * 10 * M;   // periodic: [4][4P] of partition 0; bounded: [P][4][4P];
                                            // uneven: [P][4][4W], W = min(2 kq + 1, P)

    lds_barrier();   // coefficients visible

    // staggered cell-to-edge operators: the system leaves out the last output
    // row, which follows from its own right-hand-side row (the last row of
    // the right-row table) and the solution next to it after the solve
    T rtail = T(0);
    if constexpr (MODE == 2) {
        if (edge_right && a.tail) {
#pragma unroll
            for (int c = 0; c < kBColsDev; c++)
                rtail += bnd[128 + (kBRowsDev - 1) * kBColsDev + c] * w[M + 4 - c];
        }
    }
    // REP > 1: the operator applied REP times, the intermediate never leaving
    // the registers (halos through LDS as in the adjoint).  (REP = 1: left at
    // the end, no loop.  As a loop of one pass some kernels took four registers
    // more, FP32 M = 64 system form accumulating 131 instead of 127; the stage
    // takes two less as one.)
    constexpr bool ONCE = REP == 1 && EPI != kStage;
#pragma unroll 1
    for (int rep = 0; ONCE || rep < REP; rep++) {
    if constexpr (!ADJ) apply_stencil<T, M, MODE == 2 ? kBRowsSys : kBRowsFwd, MODE == 2 ? 1 : 0>(w, tab, bnd, edge_left, edge_right, fd.nbl, fd.nbr);
    // the padding slots of an uneven partition have a zero right-hand side
    if constexpr (UNE) {
#pragma unroll
        for (int t = kMinRows; t < M; t++) w[t] = t < mrows ? w[t] : T(0);
    }

    // ---------------------------------------------- 2. local band LU solve
#pragma unroll
    for (int t = 1; t < M; t++) {
        T z = w[t] - lu[t * 6 + 0] * w[t - 1];
        if (t >= 2) z -= lu[t * 6 + 1] * w[t - 2];
        w[t] = z;
        PADE_REGION_END(t);
    }
    w[M - 1] = w[M - 1] * lu[(M - 1) * 6 + 2];
    w[M - 2] = w[M - 2] * lu[(M - 2) * 6 + 2] - lu[(M - 2) * 6 + 3] * w[M - 1];
#pragma unroll
    for (int t = M - 3; t >= 0; t--) {
        w[t] = w[t] * lu[t * 6 + 2] - lu[t * 6 + 3] * w[t + 1] - lu[t * 6 + 4] * w[t + 2];
        PADE_REGION_END(t);
    }

    // --------------------------------- 3-5. reduced system and correction
    if (!BND || P > 1) {
        if (active) {
            tips[(4 * p + 0) * NPEN + pen] = w[0];
            tips[(4 * p + 1) * NPEN + pen] = w[1];
            tips[(4 * p + 2) * NPEN + pen] = w[M - 2];
            tips[(4 * p + 3) * NPEN + pen] = w[M - 1];
        }
        // full barrier: the field has been consumed, and it also keeps the
        // coupling-column reads below from being hoisted above this point.
        // Whole-pencil waves hold their tips in their own tile: a wave-local
        // sync, so that the waves of a workgroup do not run in lockstep.
        if constexpr (WHOLE) {
            wave_lds_sync();
            mem_region_fence();
        } else {
            __syncthreads();
        }
        T u0 = T(0), u1 = T(0), u2 = T(0), u3 = T(0);
        const int m = 4 * P;
        const int kq = fd.kq;
        const bool all = 2 * kq + 1 >= P;
        const int d0 = all ? 0 : -kq;
        const int d1 = all ? P - 1 : kq;
        for (int d = d0; d <= d1; d++) {
            int qq = all ? d : pc + d;                 // source partition
            if (!all) {
                if (qq < 0) { if (BND) continue; qq += P; }
                if (qq >= P) { if (BND) continue; qq -= P; }
            }
            // periodic: the rows of partition pc are those of partition 0
            // rotated by pc partitions; bounded: each partition has its own
            int qrel = qq - pc;
            if (qrel < 0) qrel += P;
            const int mq = UNE ? 4 * (d1 - d0 + 1) : m;          // length of a stored row
            const T *Qr = UNE ? Qb + pc * 4 * mq + 4 * (d - d0)
                              : (BND ? Qb + (long long)pc * 4 * m + 4 * qq : Qb + 4 * qrel);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const T g = tips[(4 * qq + k) * NPEN + pen];
                u0 += Qr[0 * mq + k] * g;
                u1 += Qr[1 * mq + k] * g;
                u2 += Qr[2 * mq + k] * g;
                u3 += Qr[3 * mq + k] * g;
            }
        }
        mem_region_fence();
#pragma unroll
        for (int t = 0; t < M; t++) {
            w[t] -= S[t * 4 + 0] * u0 + S[t * 4 + 1] * u1 + S[t * 4 + 2] * u2 + S[t * 4 + 3] * u3;
            pin(w[t]);
            PADE_REGION_END(t);
        }
    }

    if (ADJ || rep + 1 < REP) {
        // ------------- the solved values with their halos (via LDS) as a window
        const bool exch = !BND || P > 1;
        if (exch) {
            if constexpr (WHOLE) wave_lds_sync();        // the tips, in the same place, have been read
            if (active) {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    halo[(8 * p + k) * NPEN + pen] = w[k];
                    if constexpr (!UNE) halo[(8 * p + 4 + k) * NPEN + pen] = w[M - 4 + k];
                }
                // an uneven partition's last four rows end at slot mrows - 1
                if constexpr (UNE) {
#pragma unroll
                    for (int t = kMinRows - 4; t < M; t++)
                        if (t >= mrows - 4 && t < mrows) halo[(8 * p + 8 + t - mrows) * NPEN + pen] = w[t];
                }
            }
            __syncthreads();
        }
        int pl = pc - 1, pr = pc + 1;
        bool hasl = true, hasr = true;
        if (pl < 0) { if (!BND) pl += P; else hasl = false; }
        if (pr >= P) { if (!BND) pr -= P; else hasr = false; }
#pragma unroll
        for (int t = M - 1; t >= 0; t--) w[t + 4] = w[t];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            w[k] = (exch && hasl) ? halo[(8 * pl + 4 + k) * NPEN + pen] : T(0);
            w[M + 4 + k] = (exch && hasr) ? halo[(8 * pr + k) * NPEN + pen] : T(0);
        }
        // uneven: the right halo follows the partition's last row, over the
        // padding slots
        if constexpr (UNE) {
#pragma unroll
            for (int t = kMinRows; t < M; t++)
                if (hasr && t >= mrows && t < mrows + 4) w[t + 4] = halo[(8 * pr + t - mrows) * NPEN + pen];
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (hasr && M + k >= mrows + 4) w[M + 4 + k] = T(0);
                else if (hasr) w[M + 4 + k] = halo[(8 * pr + M + k - mrows) * NPEN + pen];
        }
        // x: the halo lives in the transpose tiles, which the store phase
        // (whole-pencil waves: the next pass's tips) rewrites -- every wave
        // reads its halo first
        if constexpr (MODE == 1)
            if (exch) __syncthreads();
        if constexpr (ADJ) apply_stencil<T, M, kBRowsDev>(w, tab, bnd, edge_left, edge_right, fd.nbl, fd.nbr);
    }
    if (ONCE) break;
    }

    // ---------------------------------------------------------------- store
    if constexpr (MODE != 1) {
        const unsigned hoff = loff + (unsigned)((long long)(UNE ? pM - pw0 : half * M) * stp * (long long)sizeof(T));
        if (valid) {
            if constexpr (EPI == kStage) {
                // low-storage Runge-Kutta stage on the finished right-hand
                // side r = alpha op(f) + beta out: Q = dt r + A Q, W += B Q
                // (r itself is not written), in batches as below
                constexpr int KB = kEpiRows / 2;
                const long long qd = fd.stage_q - fd.out, wd = fd.stage_w - fd.out;
                T cur[3][KB], nxt[3][KB];
                auto load = [&](T (&o)[3][KB], int t0) {
#pragma unroll
                    for (int k = 0; k < KB; k++) {
                        T *row = ob + (long long)(pw0 + t0 + k) * stp;
                        o[0][k] = ld_s<ROWS == kWholeLines>(row, hoff);
                        o[1][k] = ld_s<ROWS == kWholeLines>(row + qd, hoff);
                        o[2][k] = ld_s<ROWS == kWholeLines>(row + wd, hoff);
                    }
                };
                load(cur, 0);
#pragma unroll
                for (int t0 = 0; t0 < M; t0 += KB) {
                    if (t0 + KB < M) load(nxt, t0 + KB);
#pragma unroll
                    for (int k = 0; k < KB; k++)
                        if (!UNE || t0 + k < mrows) {
                            T *row = ob + (long long)(pw0 + t0 + k) * stp;
                            const T r = a.alpha * w[t0 + k] + a.beta * cur[0][k];
                            const T q = a.stage_dt * r + a.stage_a * cur[1][k];
                            put(row + qd, hoff, q);
                            put(row + wd, hoff, cur[2][k] + a.stage_b * q);
                        }
#pragma unroll
                    for (int k = 0; k < KB; k++)
#pragma unroll
                        for (int j = 0; j < 3; j++) cur[j][k] = nxt[j][k];
                }
            } else if constexpr (EPI) {
                // Old values are loaded in batches of rows, the next batch
                // before the current one is stored: the compiler cannot show
                // that the store of row t and the load of row t + 1 touch
                // different addresses (the stride is a runtime value), and row
                // by row it waited for each load in turn -- M serial memory
                // round trips per wave.  The old values are read once, just
                // before they are overwritten: nontemporal loads (512^3 FP64
                // y / z 626 / 661 -> 588 / 620 us).
                constexpr int KB = kEpiRows;
                T cur[KB], nxt[KB];
#pragma unroll
                for (int k = 0; k < KB; k++) cur[k] = ld_s<ROWS == kWholeLines>(ob + (long long)(pw0 + k) * stp, hoff);
#pragma unroll
                for (int t0 = 0; t0 < M; t0 += KB) {
                    if (t0 + KB < M) {
#pragma unroll
                        for (int k = 0; k < KB; k++) nxt[k] = ld_s<ROWS == kWholeLines>(ob + (long long)(pw0 + t0 + KB + k) * stp, hoff);
                    }
#pragma unroll
                    for (int k = 0; k < KB; k++)
                        if (!UNE || t0 + k < mrows)
                            put(ob + (long long)(pw0 + t0 + k) * stp, hoff, a.alpha * w[t0 + k] + a.beta * cur[k]);
#pragma unroll
                    for (int k = 0; k < KB; k++) cur[k] = nxt[k];
                }
            } else {
#pragma unroll
                for (int t = 0; t < M; t++)
                    if (!UNE || t < kMinRows || t < mrows) put(ob + (long long)(pw0 + t) * stp, hoff, w[t]);
            }
        }
        if constexpr (MODE == 2) {
            // the left-out last row (table slots 9, 10: its sub-diagonal entry
            // and the inverse of its diagonal)
            if (valid && edge_right && a.tail) {
                T v = (rtail - tab[9] * w[M - 1]) * tab[10];
                T *dst = ob + (long long)(pw0 + M) * stp;
                if constexpr (EPI) v = a.alpha * v + a.beta * ld(dst, hoff);
                put(dst, hoff, v);
            }
        }
    } else {
        constexpr int G = 64 / LPR;
        const int myrow = tile_row(pen, half);
#pragma unroll
        for (int c = 0; c < M / XT; c++) {
#pragma unroll
            for (int j = 0; j < XT / VL; j++) {
                vec_t v;
#pragma unroll
                for (int e = 0; e < VL; e++) v[e] = w[c * XT + j * VL + e];
                *reinterpret_cast<vec_t *>(xt + myrow * PAD + VL * j) = v;
            }
            wave_lds_sync();
#pragma unroll
            for (int s = 0; s < XT / VL; s++) {
                const vec_t v = *reinterpret_cast<const vec_t *>(xt + instr_row(s) * PAD + VL * (lane % LPR));
#pragma unroll
                for (int e = 0; e < VL; e++) w[c * XT + s * VL + e] = v[e];
            }
            wave_lds_sync();
        }
        // every row of this wave's tile is stored (the common case): no
        // per-store conditions
        const bool full_tile = q0 + NPEN <= a.npencils && (wave + 1) * PW <= P;
        auto row_off = [&](int s) {
            const int r = instr_row(s);
            const int rp = row_pen(r), rh = row_part(r);
            const int ps = UNE ? part_start(min(wave * PW + rh, P - 1)) - pw0 : rh * M;
            return (unsigned)((rp * (long long)n + ps + VL * (lane % LPR)) * (long long)sizeof(T));
        };
        // elements of chunk c that this lane stores of its row
        auto row_left = [&](int s, int c) {
            return UNE ? part_rows(min(wave * PW + row_part(instr_row(s)), P - 1)) - c * XT - VL * (lane % LPR) : VL;
        };
        auto row_ok = [&](int s) {
            const int r = instr_row(s);
            return full_tile || (q0 + row_pen(r) < a.npencils && wave * PW + row_part(r) < P);
        };
        // accumulate: a chunk's old values are loaded together, the next
        // chunk's before the current one is stored (a memory round trip per
        // chunk, overlapped with the previous chunk's stores; nontemporal
        // loads, as on strided rows: 512^3 FP64 596 -> 545 us).  Rows that do
        // not exist load the first one's: with conditional loads, partitions
        // of one chunk (FP64 M = 16, FP32 M = 32) needed 230 registers, with
        // these 96 to 117 (whole-pencil waves of more chunks the other way
        // round: FP64 M = 48 182 and 166).
        vec_t cur[EPI ? XT / VL : 1], nxt[EPI ? XT / VL : 1];
        auto load_old = [&](int c, vec_t *o) {
#pragma unroll
            for (int s = 0; s < XT / VL; s++)
            {
                const bool ok = row_ok(s);
                if (WHOLE && M > XT && !ok) continue;
                const unsigned ro = ok ? row_off(s) : 0u;
                o[s] = STREAM ? ldg_nt(ob + pw0 + c * XT, ro) : ldg(ob + pw0 + c * XT, ro);
            }
        };
        if constexpr (EPI) load_old(0, cur);
#pragma unroll
        for (int c = 0; c < M / XT; c++) {
            if constexpr (EPI) {
                if (c + 1 < M / XT) load_old(c + 1, nxt);
            }
#pragma unroll
            for (int s = 0; s < XT / VL; s++) {
                if (!row_ok(s)) continue;
                vec_t v;
#pragma unroll
                for (int e = 0; e < VL; e++) v[e] = w[c * XT + s * VL + e];
                if constexpr (EPI) v = a.alpha * v + a.beta * cur[s];
                const int left = row_left(s, c);
                if (left >= VL) {
                    stg(ob + pw0 + c * XT, row_off(s), v);
                } else if constexpr (UNE) {
#pragma unroll
                    for (int e = 0; e + 1 < VL; e++)
                        if (e < left) put(ob + pw0 + c * XT + e, row_off(s), v[e]);
                }
            }
            if constexpr (EPI) {
#pragma unroll
                for (int s = 0; s < XT / VL; s++) cur[s] = nxt[s];
            }
        }
    }
}

// ------------------------------------------------------------------------
// launchers

// Bytes of x pencils per XCD run of workgroups.  Measured at 512^3 FP64 cd10
// ddx (one whole-pencil wave of 8 pencils, 32 KB, per workgroup): launch
// order (XCDs interleaved per workgroup) 342-348 Gpts/s; runs of 64 KB 316-318,
// 128 KB 347, 256 KB 341, 384 KB 356, 512 KB 363-367, 768 KB 353, 1 MB
// 370-371, 2 MB 360-362, 4 MB 355-357, 8 MB 355, a contiguous eighth of the
// field per XCD 350-355; FP32 whole-pencil x with 1 MB or 512 KB runs 667-684
// against 622-637 for pair waves in launch order.  (y and z pencils keep the
// launch order: every run length measured there was at best even, z up to
// 10 % slower.)  The
// PADE_XCD_RUN_BYTES environment variable overrides the run length (0: launch
// order).
inline long long xcd_run_bytes()
{
    static const long long v = [] {
        const char *e = std::getenv("PADE_XCD_RUN_BYTES");
        return e ? std::atoll(e) : (1LL << 20);
    }();
    return v;
}

// The split that the uneven kernels' addressing relies on (UnevenParts).
template <typename T>
bool uneven_layout_ok(const ApplyArgs<T> &a, int M)
{
    const int inner = (a.P - 1) * a.ubase + std::min(a.P - 1, a.uextra) * a.uunit;
    return a.P >= 2 && a.P <= (M == 64 ? kMaxLongPartitions : kMaxPartitions) && a.ubase >= kMinRows && a.ubase + (a.uextra ? a.uunit : 0) <= M &&
           a.uextra >= 0 && a.uextra < a.P && inner + M == a.n;
}

// Layout of the row segments of a strided-row launch.
template <typename T>
uintptr_t field_bits(const ApplyArgs<T> &a)
{
    uintptr_t bits = 0;
    for (int k = 0; k < a.nfields; k++)
        bits |= reinterpret_cast<uintptr_t>(a.fld[k].f) | reinterpret_cast<uintptr_t>(a.fld[k].out) |
                reinterpret_cast<uintptr_t>(a.fld[k].stage_q) | reinterpret_cast<uintptr_t>(a.fld[k].stage_w);
    return bits;
}

template <typename T>
RowLayout row_layout(const ApplyArgs<T> &a)
{
    const auto bits = field_bits(a) | (uintptr_t)(a.stride * (long long)sizeof(T)) | (uintptr_t)(a.B2 * (long long)sizeof(T));
    if (bits % 128 == 0) return kWholeLines;
    return bits % 64 == 0 ? kHalfLines : kShared;
}

// Workgroups per XCD run where neighbouring workgroups share lines.
constexpr int kSharedRun = 64;

template <typename T, int M, int PW, bool ADJ, int MODE, bool BND, int EPI, bool UNE, int REP, int NF>
hipError_t launch_kernel(const ApplyArgs<T> &a_in, int gw, hipStream_t s)
{
    constexpr int NPEN = 64 / PW;
    constexpr bool WHOLE = MODE == 1 && PW == 8;
    if (a_in.nfields < 1 || a_in.nfields > NF) return hipErrorInvalidValue;
    SolveArgs<T> a = a_in;
    FieldSet<T, NF> fields{};
    std::copy_n(a_in.fld, NF, fields.fld);
    const int waves = WHOLE ? gw : (a.P + PW - 1) / PW;
    int coef_len = 0;
    for (int k = 0; k < a.nfields; k++) coef_len = std::max(coef_len, fields.fld[k].coef_len);
    const size_t lds = spike_lds_bytes(sizeof(T), M, a.P, PW, ADJ || REP > 1, MODE, coef_len, BND, gw);
    const long long nblk = (a.npencils + (long long)NPEN * gw - 1) / ((long long)NPEN * gw);
    a.remap = 0;
    auto launch = [&](auto kernel) {
        fields.shared = a;
        hipLaunchKernelGGL(kernel, dim3((unsigned)nblk, (unsigned)a.nfields), dim3(64 * waves), lds, s,
                           a, fields);
        return hipGetLastError();
    };
    if constexpr (MODE == 1) {
        // Whole-pencil x waves and FP64 bounded x pencils: each XCD takes runs of
        // consecutive workgroups covering xcd_run_bytes() of the field (a
        // power-of-two number of workgroups; 512^3 bounded FP64 x pair waves
        // 331-333 -> 343 Gpts/s, FP32 pair waves measured 1-2 % slower with runs)
        if (WHOLE || (sizeof(T) == 8 && BND)) {
            const long long wg_bytes = (long long)NPEN * gw * a.n * (long long)sizeof(T);
            long long c = 1;
            while (2 * c * wg_bytes <= xcd_run_bytes()) c *= 2;
            if (c >= 2 && nblk >= 16 * c) a.remap = (int)c;
        }
        // uneven x partitions may start anywhere in a line: cached stores, as
        // for strided rows (129 x 512 x 512 FP64 x 155 -> 229 Gpts/s)
        if constexpr (UNE) {
            const auto bits = field_bits(a_in) | (uintptr_t)(a.n * sizeof(T)) |
                              (uintptr_t)(a.uunit * sizeof(T));
            if (bits % 128) return launch(spike_apply<T, M, PW, ADJ, MODE, BND, EPI, UNE, kShared, REP, NF>);
        }
        return launch(spike_apply<T, M, PW, ADJ, MODE, BND, EPI, UNE, kWholeLines, REP, NF>);
    } else {
        const RowLayout rows = row_layout(a_in);
        if (rows == kWholeLines) return launch(spike_apply<T, M, PW, ADJ, MODE, BND, EPI, UNE, kWholeLines, REP, NF>);
        int c = kSharedRun;
        while (c > 1 && nblk < 16LL * c) c /= 2;
        if (c >= 2) a.remap = c;
        if (rows == kShared) return launch(spike_apply<T, M, PW, ADJ, MODE, BND, EPI, UNE, kShared, REP, NF>);
        // without an epilogue periodic kernels load alike for whole and half lines
        return launch(spike_apply<T, M, PW, ADJ, MODE, BND, EPI, UNE, (BND || EPI ? kHalfLines : kWholeLines), REP, NF>);
    }
}

template <typename T, int M, int PW, bool ADJ, int MODE, bool UNE = false, int REP = 1,
          int NF = (REP > 1 && !(ADJ && MODE == 1) ? kMaxFields : 1)>
hipError_t launch_spike_t(const ApplyArgs<T> &a, int gw, hipStream_t s)
{
    constexpr bool WHOLE = MODE == 1 && PW == 8;
    // whole-pencil waves: no wave of a workgroup without pencils (its loads
    // would start behind the field)
    while (gw > 1 && (!WHOLE || (a.npencils + 7) / 8 % gw)) gw--;
    // the accumulate epilogue exists for the forward operator only
    if (ADJ && a.axpby) return hipErrorInvalidValue;
    const bool epi = !ADJ && a.axpby;
    if constexpr (MODE == 2) {
        // staggered operators: forward, bounded, strided rows only
        if (ADJ || a.periodic || a.n_in < a.n || a.n_in > a.n + 1) return hipErrorInvalidValue;
        return epi ? launch_kernel<T, M, PW, false, 2, true, kAxpby, UNE, REP, NF>(a, gw, s)
                   : launch_kernel<T, M, PW, false, 2, true, kStore, UNE, REP, NF>(a, gw, s);
    } else if constexpr (ADJ) {
        // (a periodic adjoint runs the forward kernel on the transposed tables)
        if (a.periodic) return hipErrorInvalidValue;
        return launch_kernel<T, M, PW, true, MODE, true, kStore, UNE, REP, NF>(a, gw, s);
    } else if constexpr (NF > 1 && REP == 1 && MODE == 1) {
        // several fields along x: without an epilogue
        if (epi) return hipErrorInvalidValue;
        return a.periodic ? launch_kernel<T, M, PW, false, MODE, false, kStore, UNE, REP, NF>(a, gw, s)
                          : launch_kernel<T, M, PW, false, MODE, true, kStore, UNE, REP, NF>(a, gw, s);
    } else {
        if (a.periodic)
            return epi ? launch_kernel<T, M, PW, false, MODE, false, kAxpby, UNE, REP, NF>(a, gw, s)
                       : launch_kernel<T, M, PW, false, MODE, false, kStore, UNE, REP, NF>(a, gw, s);
        return epi ? launch_kernel<T, M, PW, false, MODE, true, kAxpby, UNE, REP, NF>(a, gw, s)
                   : launch_kernel<T, M, PW, false, MODE, true, kStore, UNE, REP, NF>(a, gw, s);
    }
}

}  // namespace pade
