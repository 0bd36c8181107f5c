// Kernel-side argument block and launchers (internal to libpadeops_hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace pade {

constexpr int kBRowsDev = 8;
// Special rows of a forward operator at one end, and of a staggered system
// form (the transposes have up to 8).  Their results stay in registers while
// the stencil runs: with four rows instead of eight the FP64 M = 32 bounded
// kernels need 127 registers instead of 145 (four waves per SIMD instead of
// three: 256^3 bounded y / z 60 / 61 -> 55 / 57 us).
constexpr int kBRowsFwd = 4, kBRowsSys = 2;
constexpr int kBColsDev = 16;

// Device table layout of one plan (element offsets):
//   [0, 16)                     stencil (offsets -4..4, 1/dx^p folded in)
//   [16, 16+128)                left special rows (8 x 16)
//   [144, 144+128)              right special rows (8 x 16, stored reflected)
//   [272, 272+coef_len)         coefficient area, copied to LDS as a whole:
//       ncls blocks of 10M: M band-LU rows (l1, l2, 1/piv, u1/piv, u2/piv, 0)
//                           then M coupling rows S (4 each);
//       then the reduced-system rows: periodic -> the 4 rows (4P each) of
//       partition 0 (partition p uses them rotated by p); bounded -> the 4
//       rows of every partition ([P][4][4P]).
// Partition p uses block cls(p) of the launch arguments.  Uneven partitions store of every
// partition's reduced-system rows the entries of its window only
// ([P][4][4W], W = min(2 kq + 1, P); entry j belongs to partition p - kq + j,
// cyclic when periodic, or to partition j when W = P).
constexpr int kOffBl = 16;
constexpr int kOffBr = 144;
constexpr int kOffCoef = 272;
constexpr int kMaxPartitions = 16;
// Uneven partitions of 64 slots go on to 21, four per wave (three bits of class
// each in the 64 of FieldArgs): pencils of up to 1344 points.
constexpr int kMaxLongPartitions = 21;

// One field of a launch: its arrays, and the table of its operator (boundary
// codes may differ between the fields of a launch).
template <typename T>
struct FieldArgs {
    const T *f;
    T *out;
    const T *tab;
    unsigned long long cls4;   // block of partition p in bits 4p .. 4p + 3, 3p .. 3p + 2
                               // where P > 16 (shifted out of a scalar register:
                               // an array indexed per lane is a load from the
                               // argument segment)
    int nbl, nbr;
    int coef_len;          // length of the coefficient area
    int ncls;              // number of coefficient blocks
    int kq;                // reduced-system window: partitions p-kq..p+kq (2kq+1 >= P: all)
    T *stage_q, *stage_w;  // Runge-Kutta stage epilogue: register and state
};

constexpr int kMaxFields = 6;

// What the fields of a launch share.
template <typename T>
struct SolveArgs {
    int nfields;           // grid y
    long long npencils;
    long long A1, B1, B2;  // pencil q -> base offset (q % A1)*B1 + (q / A1)*B2
    long long stride;      // element distance between consecutive points of a pencil
    int n, M, P, periodic;
    int n_in;              // input points per pencil: n except for the
                           // staggered cell <-> edge operators (generic path:
                           // the right boundary rows read in[n_in - 1 - c];
                           // strided-row mode 2: in[n - c], n_in = n or n + 1)
    int tail;              // mode 2: one more output row after the n solved
    // uneven partitions: partition p < P - 1 has ubase + (p < uextra ? uunit : 0)
    // rows and starts at row p * ubase + min(p, uextra) * uunit, the last has M
    int ubase, uextra, uunit;
    int axpby;             // 0: out = op(f); 1: out = alpha * op(f) + beta * out
    int remap;             // workgroup order: 0 launch order; C > 0 each of the 8 XCDs
                           // (workgroup i runs on XCD i % 8) takes runs of C
                           // consecutive workgroups; < 0 a contiguous eighth
    T alpha, beta;
    T stage_dt, stage_a, stage_b;
};

template <typename T>
struct ApplyArgs : SolveArgs<T> {
    FieldArgs<T> fld[kMaxFields];
};

// mode 0: strided rows (y, z); 1: x pencils through LDS transposes; 2:
// strided rows of a bounded staggered operator in system form (forward only).
// GW: whole-pencil x waves (PW = 8) per workgroup (other variants: 1).
template <typename T>
hipError_t launch_spike(const ApplyArgs<T> &a, int M, int PW, int GW, bool adj, int mode, hipStream_t s);

// launch_spike and launch_uneven of several fields: forward, mode 0, or mode 1
// without an epilogue, two partitions per wave (uneven: four of more than
// sixteen) or whole-pencil x waves (FP64).
hipError_t launch_fields(const ApplyArgs<double> &a, int M, int PW, int GW, bool uneven, int mode, hipStream_t s);

// The same solve over uneven partitions (a pencil length that is no multiple
// of M), two partitions per wave; modes as above.
template <typename T>
hipError_t launch_uneven(const ApplyArgs<T> &a, int M, bool adj, int mode, hipStream_t s);

// The operator applied twice in one pass, even or uneven partitions, modes 0
// and 1, two partitions per wave or whole-pencil x waves (FP64).
hipError_t launch_twice(const ApplyArgs<double> &a, int M, int PW, int GW, bool uneven, bool adj, int mode,
                        hipStream_t s);

// The accumulating apply along z finished by a Runge-Kutta stage: r = alpha
// op(f) + beta out (not written), Q = stage_dt r + stage_a Q, W += stage_b Q.
// Mode 0, two partitions per wave.
hipError_t launch_stage(const ApplyArgs<double> &a, int M, bool uneven, hipStream_t s);

template <typename T>
hipError_t launch_generic(const ApplyArgs<T> &a, bool adj, T *work, hipStream_t s);

// y = alpha * x + beta * y over `count` elements (x == nullptr: y = beta * y).
template <typename T>
hipError_t launch_axpby(const T *x, T *y, T alpha, T beta, long long count, hipStream_t s);

}  // namespace pade
