/*
 * padeops_hip.h -- C ABI of the MI355X compact-difference operator library
 * (libpadeops_hip.so).
 *
 * This is the drop-in boundary for PadeOps' compact operators: the
 * cd06 / cd10 first and second derivatives and the cf90 compact filter,
 * applied along x, y or z of a Fortran-ordered 3-D array (i fastest).
 * Plain pointers, sizes and integer codes only; a Fortran iso_c_binding shim
 * (padeops_amd/fortran/) re-exports the reference's module surface on top.
 *
 * Conventions
 *   axis 1: f(n, na, nb)   derivative along the contiguous axis (dd1 / d2d1 / filter1)
 *   axis 2: f(na, n, nb)   (dd2 / d2d2 / filter2)
 *   axis 3: f(na, nb, n)   (dd3 / d2d3 / filter3)
 *   bc codes: 0 one-sided closure, 1 symmetric, -1 antisymmetric; an absent
 *   optional bc in the reference means 0, so callers pass 0.
 *   Device-pointer entry points are asynchronous on `stream` (a hipStream_t,
 *   NULL = default stream); f and df must not overlap.
 *
 * Return codes
 *   0      success
 *   2,3,7  init size errors, as the reference's init returns them
 *   21     operation not provided for this operator kind
 *   324    bc code outside {-1,0,1} (the reference's GracefulExit code)
 *   400    invalid argument (null pointer, size mismatch, bad axis)
 *   1000+e HIP runtime error e
 * pade_last_error() gives a message for the last non-zero code of the
 * calling thread.
 */
#ifndef PADEOPS_HIP_H
#define PADEOPS_HIP_H

#ifdef __cplusplus
extern "C" {
#endif

/* PADE_GAUSSIAN: the explicit Gaussian filter of width 4 dx
 * (src/filters/gaussian.F90:11-36, periodic stencil :137-185, bounded rows
 * :189-334 with the apply-time bc codes 0 / 1 / -1), n = 1 or n >= 9;
 * PADE_FILTER on any axis, dx ignored.  It is the compressible solver's
 * filter of its artificial transport properties (cgrid.F90:338,1113). */
enum pade_kind { PADE_CD06 = 1, PADE_CD10 = 2, PADE_CF90 = 3, PADE_CD06STAGG = 4, PADE_GAUSSIAN = 5 };
/* PADE_CD06STAGG (n > 4) takes the staggered operations, along z (axis 3)
 * only, on edge (E) arrays of n + 1 planes and cell (C) arrays of n:
 *   PADE_D1_E2C      ddz_E2C      (cd06stagg.F90:820)
 *   PADE_D1_C2E      ddz_C2E      (:850)
 *   PADE_D2_C2C      d2dz2_C2C    (:995)
 *   PADE_D2_E2E      d2dz2_E2E    (:1027)
 *   PADE_INTERP_E2C  InterpZ_E2C  (:928)
 *   PADE_INTERP_C2E  InterpZ_C2E  (:960)
 *   PADE_D1_C2C      ddz_C2C      (:883, bounded only)
 *   PADE_D1_E2E      ddz_E2E      (:905, bounded only)
 * through pade_op_apply / _f32 / _axpby (f and df sized by their grid).
 * Periodic (init_periodic, cd06stagg.F90:170-195): an E array's last plane
 * repeats its first, and E outputs get it copied, as the reference does.
 * Bounded (init_nonperiodic, cd06stagg.F90:197-232): create with
 * periodic = 0 and bc1 (the k = 1 end, "Bot") / bcn (the k = n end, "Top")
 * each +1 (isEven), -1 (odd), +2 (isSided, even) or -2 (isSided, odd); the
 * apply-time bc1 / bcn are ignored.  The first derivatives E2C, C2E, C2C
 * and both interpolations have one-sided closures; ddz_E2E and the second
 * derivatives use the parity only, as in the reference.  No adjoint and no
 * dense form. */
enum pade_oper {
    PADE_D1 = 1, PADE_D2 = 2, PADE_FILTER = 3,
    PADE_D1_E2C = 11, PADE_D1_C2E = 12, PADE_D2_C2C = 13, PADE_D2_E2E = 14,
    PADE_INTERP_E2C = 15, PADE_INTERP_C2E = 16, PADE_D1_C2C = 17, PADE_D1_E2E = 18
};
enum pade_dense_prec { PADE_DENSE_F32 = 1, PADE_DENSE_BF16X3 = 2, PADE_DENSE_FULL = 16 };
enum pade_dtype { PADE_F64 = 0, PADE_F32 = 1 };

typedef struct pade_op_s *pade_op_t;

/* Create an operator for pencils of n points.
 * Replaces cd06%init (src/derivatives/cd06.F90:129), cd10%init
 * (src/derivatives/cd10.F90:195) and, with dx ignored, cf90%init
 * (src/filters/cf90.F90:107).  bc1/bcn matter only for bounded cd06 (they
 * select its LHS closure at init, cd06.F90:264-327) and bounded cd06stagg
 * (the end codes listed with the staggered operations); cd10 / cf90 take the
 * bc at apply time.  Returns the reference's ierr (2, 3, 7; 21 for cd06stagg
 * with n <= 4) for too small n. */
int pade_op_create(int kind, int n, double dx, int periodic, int bc1, int bcn, pade_op_t *op);

/* Release device tables.  Replaces cd06/cd10/cf90 %destroy
 * (cd06.F90:203-219, cd10.F90:317-349, cf90.F90:177-196). */
int pade_op_destroy(pade_op_t op);

/* Pencil length.  Replaces %GetSize (cd06.F90:123-127, cd10.F90:189-193). */
int pade_op_size(pade_op_t op);

/* FP64 apply on device arrays.  oper PADE_D1 replaces dd1/dd2/dd3
 * (cd10.F90:2029,2099,2169; cd06.F90:775,797,819), PADE_D2 replaces
 * d2d1/d2d2/d2d3 (cd10.F90:2239,2309,2379; cd06 has no reference version,
 * see the operator definition in the library documentation), PADE_FILTER
 * replaces filter1/filter2/filter3 (cf90.F90:1020,1090,1160). */
int pade_op_apply(pade_op_t op, int oper, int axis, const double *f, double *df, int na, int nb,
                  int bc1, int bcn, void *stream);

/* FP32 banded apply (same operator, FP32 storage and arithmetic; factors
 * computed in FP64 and rounded).  No reference counterpart (precision study). */
int pade_op_apply_f32(pade_op_t op, int oper, int axis, const float *f, float *df, int na, int nb,
                      int bc1, int bcn, void *stream);

/* Adjoint apply: df = B^T A^{-T} f, including the transposed boundary
 * closures.  No reference counterpart (backward pass of the autograd entry
 * point). */
int pade_op_apply_adjoint(pade_op_t op, int oper, int axis, const double *f, double *df, int na,
                          int nb, int bc1, int bcn, void *stream);
int pade_op_apply_adjoint_f32(pade_op_t op, int oper, int axis, const float *f, float *df, int na,
                              int nb, int bc1, int bcn, void *stream);

/* Apply with an accumulate epilogue: df = alpha * op(f) + beta * df, in the
 * same pass over df (the composite operators gradient / divergence / curl of
 * src/utilities/operators.F90:18-156 sum derivatives along several axes;
 * this fuses each sum into the producing kernel instead of a separate array
 * add).  No reference counterpart. */
int pade_op_apply_axpby(pade_op_t op, int oper, int axis, double alpha, const double *f, double beta, double *df,
                        int na, int nb, int bc1, int bcn, void *stream);
/* Allocation-free pade_op_apply_axpby.  No reference counterpart: it is for
 * callers that cannot allocate device memory during an apply (code under HIP
 * graph capture, tight serving or time-stepping loops, harnesses that forbid
 * hipMalloc).  Same arguments, result and error codes as
 * pade_op_apply_axpby.  The intermediates some applies need come from one
 * static device array of PADE_NOALLOC_SCRATCH_BYTES per device instead of the
 * stream-ordered allocator.  An apply is refused with 400, before anything
 * is launched, when the array cannot hold what is reserved for it: one field
 * for an accumulating apply of n points that no even partition serves (even
 * ones are multiples of 16 up to 256, of 32 up to 512, of 64 up to 1024),
 * and for the bounded cd06 second derivative with an epilogue one field more
 * than its first derivative.  The limit depends on the call alone, not on
 * the kernel that runs: uneven partitions and the second derivative in one
 * launch keep it although they leave the array untouched.  Every call on a device shares that device's array, so calls
 * that overlap on one device (two streams, two threads) race; the array is
 * never read before it is written within a call. */
#define PADE_NOALLOC_SCRATCH_BYTES (64ull << 20)
int pade_op_apply_axpby_noalloc(pade_op_t op, int oper, int axis, double alpha, const double *f, double beta,
                                double *df, int na, int nb, int bc1, int bcn, void *stream);

int pade_op_apply_axpby_f32(pade_op_t op, int oper, int axis, float alpha, const float *f, float beta, float *df,
                            int na, int nb, int bc1, int bcn, void *stream);

/* Composite operators on device fields of (nx, ny, nz) points, Fortran
 * order, over three per-axis operator handles (x: n = nx, y: ny, z: nz; the
 * derivative handles cd06 / cd10, the filter handles cf90 / Gaussian).
 * Replace gradient, curl, divergence and filter3D of
 * src/utilities/operators.F90 (:18-53, :55-116, :118-156, :158-223).  bc[6]
 * = x_bc1, x_bcn, y_bc1, y_bcn, z_bc1, z_bcn (NULL: all 0, the reference's
 * absent optional arguments); divergence takes them negated, as the
 * reference does.  curl writes its three components as consecutive planes
 * of `curl` (3 nx ny nz values); filter3D filters y, then x, then z, each
 * numtimes times, in place on arr with `work` (a field of the same size) as
 * the other buffer.  Sums are accumulated by the producing kernels, and a
 * field of up to 256 MB is processed in slabs of z-planes with the y passes
 * on a second library stream beside the x passes, so that the second read
 * of each slab comes from cache; the call is ordered on `stream` as a whole.
 * Returns 234 (the reference's GracefulExit code) when a handle's length
 * does not match the grid. */
int pade_gradient(pade_op_t opx, pade_op_t opy, pade_op_t opz, const double *f, double *dfdx, double *dfdy,
                  double *dfdz, int nx, int ny, int nz, const int *bc, void *stream);
int pade_divergence(pade_op_t opx, pade_op_t opy, pade_op_t opz, const double *u, const double *v, const double *w,
                    double *div, int nx, int ny, int nz, const int *bc, void *stream);
int pade_curl(pade_op_t opx, pade_op_t opy, pade_op_t opz, const double *u, const double *v, const double *w,
              double *curl, int nx, int ny, int nz, const int *bc, void *stream);
int pade_filter3d(pade_op_t fx, pade_op_t fy, pade_op_t fz, double *arr, double *work, int nx, int ny, int nz,
                  int numtimes, const int *bc, void *stream);

/* Host-array apply for drop-in callers whose data lives in host memory:
 * copies in, applies on the device, copies out, synchronous.  Same meaning as
 * pade_op_apply (the reference's dd*, d2d*, filter* take host arrays). */
int pade_op_apply_host(pade_op_t op, int oper, int axis, const double *f, double *df, int na,
                       int nb, int bc1, int bcn);

/* cf90 filter3 on complex data: replaces filter3_CMPLX (cf90.F90:1230-1251),
 * the generic filter3's complex(rkind) binding.  f and df are complex128
 * arrays (na, nb, n) in Fortran order, real and imaginary parts interleaved
 * as Fortran stores complex(rkind); both parts are filtered along z.
 * has_bc != 0 stands for the optional bc1_/bcn_ being present (the reference
 * tests present(bcn_)); without them the codes are (0, 0).  As in the
 * reference, a bounded filter forms the right-hand side of (bc1, bcn) and
 * solves with the (0, 0) left-hand side (penta_nn).  A periodic cf90 applies
 * its periodic filter (the reference reads penta_nn there as well, which a
 * periodic cf90 never allocates).  Returns 21 for cd06/cd10 handles.
 * Device arrays, asynchronous on `stream`; the _host form copies host arrays
 * in and out and is synchronous. */
int pade_op_filter3_complex(pade_op_t op, const void *f, void *df, int na, int nb, int bc1, int bcn, int has_bc,
                            void *stream);
int pade_op_filter3_complex_host(pade_op_t op, const void *f, void *df, int na, int nb, int bc1, int bcn,
                                 int has_bc);

/* Dense-operator form of a periodic operator: df = D f with D = A^{-1} B
 * precomputed in FP64 (circulant) and applied as an MFMA GEMM over all
 * pencils.  prec PADE_DENSE_F32 (FP32 operands and accumulation) or
 * PADE_DENSE_BF16X3 (both operands split into three BF16 limbs, six limb
 * products, FP32 accumulation).  By default tiles of D beyond the operator's
 * decay band (entries summing to <= 2^-30 of a row's absolute sum) are
 * skipped; OR PADE_DENSE_FULL into prec to apply all n x n entries.
 * in/out dtype PADE_F64 or PADE_F32 (FP64 inputs are rounded to FP32 first).
 * Needs n a multiple of 64; returns 21 for bounded operators.
 * No reference counterpart (precision study). */
int pade_op_dense_apply(pade_op_t op, int oper, int axis, const void *f, int f_dtype, void *df,
                        int df_dtype, int na, int nb, int bc1, int bcn, int prec, void *stream);

/* Shape of the dense form that pade_op_dense_apply runs for (oper, prec) on
 * `axis` with the given dtypes: *window = input points per output block that
 * the GEMM visits (16 * slots; n for PADE_DENSE_FULL), *halfwidth = decay
 * half-width kept, *products = MFMA products per 32-point output block:
 * 32x32x16 products per 32-pencil tile, or -- x pencils in FP32 storage,
 * BF16x3, decay half-width <= 48 -- 16x16x32 products per 16-pencil tile
 * (BF16x3: up to 6 per window slot, fewer where the outer slots of a
 * decaying window drop limb products whose total stays within 2^-28 of a
 * row's absolute sum; FP32: one per slot).  MFMA flops per point are
 * 32 * products either way.  Builds and caches the form on first use.  No reference
 * counterpart. */
int pade_op_dense_info(pade_op_t op, int oper, int prec, int axis, int f_dtype, int df_dtype, int *window,
                       int *halfwidth, int *products);

/* Host-only query (no GPU needed): the kernel that an apply of (oper, axis)
 * over na x nb pencils runs on an operator created with (kind, n, dx,
 * periodic, bc1, bcn) -- the codes that build it: init-time for cd06 and
 * cd06stagg, else the apply-time ones -- for dtype PADE_F64 / PADE_F32 and
 * adjoint 0 / 1.  info[8] = {M, PW, P, generic, mode, launches, uneven, 0}: M
 * the partition length, PW the partitions per wave, P the partitions per
 * pencil, generic = 1 for the one-lane-per-pencil path (M = n, P = 1), mode
 * 0 strided rows (y, z), 1 x pencils through LDS transposes, 2 the
 * staggered system form, launches the solves of one apply (2: the bounded
 * cd06 second derivative, the first derivative twice, which the FP64
 * partitioned kernels run as one kernel launch), and
 * uneven = 1 when the kernel of padded slots runs: the partitions hold at
 * most M rows each.  M then mostly does not divide the rows; 40 and 48 slots
 * (257 to 384 rows), and 64 above 1024 rows, serve the lengths that they
 * divide as well.  The strided-row kernels address the field with 32-bit per-lane byte offsets (a
 * lane's pencil relative to its workgroup's first pencil plus (PW - 1) * M
 * points along the pencil); variants whose offsets would reach 2^32, or
 * whose launch would exceed 2^32 - 1 threads, are not chosen.  No reference
 * counterpart (tests and tuning). */
int pade_plan_variant(int kind, int oper, int n, double dx, int periodic, int bc1, int bcn, int adjoint, int axis,
                      int na, int nb, int dtype, int *info);

/* Pencil re-orientation on one GPU.  2DECOMP's transpose_x_to_y / y_to_z /
 * z_to_y / y_to_x (2decomp_fft/src/transpose_x_to_y.f90:14-91 and siblings)
 * keep (i,j,k) order and only move data between ranks, so on one rank they
 * are copies: pade_pencil_copy.  pade_permute3 is the axis-permuting
 * re-orientation dst(perm(i,j,k)) = src(i,j,k) for elem_size 4 or 8;
 * perm 1: (i,j,k)->(j,i,k), 2: (i,j,k)->(k,j,i), 3: (i,j,k)->(i,k,j). */
int pade_pencil_copy(const void *src, void *dst, long long nbytes, void *stream);
int pade_permute3(const void *src, void *dst, int elem_size, int n1, int n2, int n3, int perm,
                  void *stream);

/* Host-only planning export (no GPU needed): writes the FP64 table the
 * kernels consume for (kind, oper, n, dx, periodic, bc1, bcn, adjoint) with
 * partition size M (M = 0: library choice), and meta[32] =
 * {rows, M, P, periodic, nbl, nbr, off_bl, off_br, off_coef, coef_len, ncls,
 *  kq, len, cols, sys, tail, cls[0..15]}: rows = points solved per pencil,
 * cols = input points (both n except for the bounded staggered operators
 * with an edge array: M = 0 gives their one-lane-per-pencil form, rows =
 * outputs; M > 0 their system form, sys = 1: right rows read input point
 * rows - c, and with tail = 1 one more output row follows from right row 7
 * and the table's slots 9 (sub-diagonal) and 10 (inverse diagonal));
 * stencil at [0,9), left/right boundary rows (8 x 16, the right ones reading
 * input point cols - 1 - c) at off_bl/off_br, then at off_coef ncls blocks
 * of 10*M values
 * (M band-LU rows l1, l2, 1/pivot, u1/pivot, u2/pivot, 0 and M coupling rows
 * of 4) followed by the reduced-system rows (periodic: the 4 rows of 4P values
 * of partition 0, which partition p uses rotated by p; bounded: 4 rows for
 * every partition); partition p uses block cls[p]; kq is the reduced-system
 * window.  Pass tab = NULL to query len.  Used by tests to check the planner
 * on CPU. */
int pade_plan_export(int kind, int oper, int n, double dx, int periodic, int bc1, int bcn,
                     int adjoint, int M, double *tab, long long tab_len, int *meta);

/* The same for uneven partitions of M slots: 16 or 24 for a length between
 * one and two of them, 32 or 64 for one that M does not divide (64: or of more
 * than 1024 rows, up to 1344), 40 or 48 for any.  The table is that of the
 * padded slots (a staggered operator with an edge array: its system form).  meta[64]: as
 * pade_plan_export in [0, 32), [32] = W, the partitions of a reduced-system
 * row, [33 + p] = first row of partition p, [54 + p - 16] = class of p > 15.
 * Every partition occupies M slots: its rows, then padding slots with y_t =
 * y_{t-2} and a zero right-hand side; the last partition has M rows.  The
 * reduced-system rows hold, for every partition, 4 rows of 4 W values: entry
 * j for partition p - kq + j (cyclic when periodic), or partition j when W =
 * P.  Returns 21 when the length has no such split.  Used by tests. */
int pade_plan_export_uneven(int kind, int oper, int n, double dx, int periodic, int bc1, int bcn,
                            int adjoint, int M, double *tab, long long tab_len, int *meta);

/* Pointwise stages of the compressible solver's Runge-Kutta substep
 * (src/compressible/cgrid.F90, one ideal-gas species), each one streaming
 * pass on `stream` over FP64 arrays of n points; groups of fields are planes
 * of one allocation (plane k at base + k * n): W the five conserved
 * variables (rho, rho u, rho v, rho w, total energy), du the nine velocity
 * gradients (du/dx, du/dy, du/dz, dv/dx, ..., dw/dz), grad_* three gradient
 * components, d4 three fourth derivatives (x, y, z), fluxes the fifteen
 * x / y / z fluxes of the five equations (the x fluxes negated, so that the
 * first x derivative writes the right-hand side directly, -d(fx)/dx).  The
 * derivatives and filters
 * between them are the operator calls above.  Return 0 or 400 / 1000 + hip
 * error, with a message in pade_last_error(). */
/* get_conserved, cgrid.F90:799-811, with advance_RK45's check of W (:684-692):
 * bad_index (a device unsigned 64-bit value, may be NULL; the caller sets it
 * to all ones beforehand) is lowered to the smallest plane-major linear index
 * l * n + i (l = 0..4) of a W value for which nancheck's test
 * isnan(f) .OR. f + one == f holds (src/utilities/exits.F90:154,197: NaN,
 * +-Inf and |f| >= 2^53), the index nancheck_ind returns. */
int pade_cg_conserved(long long n, const double *rho, const double *u, const double *v, const double *w,
                      const double *e, double *W, unsigned long long *bad_index, void *stream);
int pade_cg_primitive(long long n, const double *W, double gam, double Rgas, double *rho, double *u, double *v,
                      double *w, double *e, double *p, double *T, void *stream);  /* :764-797, :813-820 */
int pade_cg_strain(long long n, const double *du, double *func, double *dil, void *stream);  /* :1085-1087, :1117 */
int pade_cg_lad_mu(long long n, double Cmu, const double *rho, double *mustar, void *stream);   /* :1110 */
int pade_cg_lad_bulk(long long n, double Cbeta, double hx, double hy, double hz, const double *rho,
                     const double *grad_rho, const double *d4, const double *du, const double *dil, double *bulk,
                     void *stream);                                                  /* :1115-1158 */
int pade_cg_lad_kap(long long n, double Ckap, double gam, double hx, double hy, double hz, const double *rho,
                    const double *p, const double *T, const double *grad_e, const double *d4, double *kap,
                    void *stream);                                                   /* :1163-1196 */
int pade_cg_fluxes(long long n, const double *W, const double *u, const double *v, const double *w, const double *p,
                   const double *du, const double *mu, const double *bulk, const double *kap, const double *grad_T,
                   double *fluxes, void *stream);                       /* :898-1056, :1338-1444 */
int pade_cg_rk_stage(long long n, double dt, double A, double B, const double *rhs, double *Q, double *W,
                     void *stream);                                                  /* :697-699 */

/* The compressible step driven from native code: a grid object that owns the
 * operators, filters and work arrays of cgrid's RK45 step and runs it on
 * `stream` through the kernels above.  One ideal-gas species, power-law
 * viscosity, periodic or bounded per axis.  Replaces, for a Fortran or C
 * host, cgrid%init's operator and array set-up (src/compressible/cgrid.F90
 * :150-445, &CINPUT parameters :160-199, per-axis bc :298-306, derivatives
 * and filters :321-340), advance_RK45 (:663-717), get_dt (:719-762),
 * get_primitive / get_conserved / post_bc (:764-820) and getRHS (:822-1056).
 *
 * Fields (enum pade_cg_field) are FP64 (nx, ny, nz) arrays in Fortran order
 * on the device; PADE_CG_W is the five conserved variables as consecutive
 * planes (rho, rho u, rho v, rho w, total energy).  `fields` gives the
 * caller's arrays (PADE_CG_NFIELDS pointers, any of them NULL, or fields
 * NULL: the grid allocates and frees them); pade_cgrid_field returns them.
 * params: gam, Rgas, Cmu, Cbeta, Ckap, mu_ref, T_ref, visc_n, Pr (NULL: the
 * defaults 1.4, 1, 0.002, 1.75, 0.01, 1, 1, 0.75, 0.75).  periodic[3]
 * (NULL: all periodic); bc[6] = x_bc1, x_bcn, y_bc1, ... (0, 1, -1; used on
 * bounded axes, NULL: 0).  derivative PADE_CD10 or PADE_CD06 (cd06 has no
 * second derivative: a viscous or LAD step returns 21 as
 * derivatives.F90:524-525 aborts), filter_kind PADE_CF90 or PADE_GAUSSIAN.
 * Errors: 324 bad bc, 11 / 12 / 51 operator set-up (derivatives.F90 and
 * filters.F90 GracefulExit codes), 400, 1000 + hip error.
 *
 * pade_cgrid_advance_rk45 runs the five substeps.  dt > 0 sets the time step
 * (else the last get_dt's).  hook_bc, if not NULL, runs after each
 * substep's primitive update with (grid, user) and the fields are then
 * brought back to consistency (post_bc), as cgrid.F90:709-710.  Before each
 * substep's right-hand side, W is tested as nancheck does (isnan(f) .OR.
 * f + 1 == f, src/utilities/exits.F90:154); on a failure it returns 999
 * (GracefulExit's code there) with the substep (1-5) in *bad_substep and the
 * plane-major index l * nx*ny*nz + i + nx (j + ny k) (0-based) of the first
 * failing W value in *bad_index, and the message of cgrid.F90:688-690.
 * Synchronises `stream` once per substep (the test).  pade_cgrid_get_dt
 * returns the step of cgrid.F90:719-762 (synchronous: device maxima) and the
 * limit that set it (enum pade_cg_dt); CFL <= 0 gives the fixed step of
 * pade_cgrid_set_state.  pade_cgrid_get_conserved with bad_index != NULL
 * applies the same test (-1: none). */
enum pade_cg_field {
    PADE_CG_RHO = 0, PADE_CG_U = 1, PADE_CG_V = 2, PADE_CG_W_VEL = 3, PADE_CG_P = 4, PADE_CG_T = 5, PADE_CG_E = 6,
    PADE_CG_MU = 7, PADE_CG_BULK = 8, PADE_CG_KAP = 9, PADE_CG_W = 10, PADE_CG_NFIELDS = 11
};
enum pade_cg_dt {
    PADE_CG_DT_CONVECTIVE = 0, PADE_CG_DT_SHEAR = 1, PADE_CG_DT_BULK = 2, PADE_CG_DT_CONDUCTIVE = 3,
    PADE_CG_DT_STARTUP = 4, PADE_CG_DT_FIXED = 5
};
typedef struct pade_cgrid_s *pade_cgrid_t;
typedef void (*pade_cgrid_hook)(pade_cgrid_t grid, void *user);
int pade_cgrid_create(int nx, int ny, int nz, double dx, double dy, double dz, int derivative, int filter_kind,
                      const double *params, int inviscid, const int *periodic, const int *bc, double *const *fields,
                      pade_cgrid_t *grid);
int pade_cgrid_destroy(pade_cgrid_t grid);
int pade_cgrid_field(pade_cgrid_t grid, int which, double **ptr);
int pade_cgrid_state(pade_cgrid_t grid, int *step, double *tsim, double *dt);
int pade_cgrid_set_state(pade_cgrid_t grid, int step, double tsim, double dtfixed);
int pade_cgrid_post_bc(pade_cgrid_t grid, void *stream);                            /* :813-820 */
int pade_cgrid_get_conserved(pade_cgrid_t grid, long long *bad_index, void *stream); /* :799-811 */
int pade_cgrid_get_primitive(pade_cgrid_t grid, void *stream);                      /* :764-797, :813-820 */
int pade_cgrid_rhs(pade_cgrid_t grid, double *rhs, void *stream);                   /* :822-1056 */
int pade_cgrid_transport(pade_cgrid_t grid, void *stream);   /* MixtureEOS.F90:175-229, ns = 1 */
int pade_cgrid_get_dt(pade_cgrid_t grid, double CFL, double *dt, int *stability, void *stream);
int pade_cgrid_advance_rk45(pade_cgrid_t grid, double dt, pade_cgrid_hook hook_bc, void *user, int *bad_substep,
                            long long *bad_index, void *stream);

/* Message for the last non-zero return code of this thread. */
const char *pade_last_error(void);

/* Library version (major*10000 + minor*100 + patch). */
int pade_version(void);

#ifdef __cplusplus
}
#endif

#endif /* PADEOPS_HIP_H */
