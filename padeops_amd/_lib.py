"""Loader for ``libpadeops_hip.so`` (ctypes over the C ABI in include/padeops_hip.h).

The product path always runs through this library; there is no CPU fallback.
If the library is missing the import of an operator fails loudly.
"""
from __future__ import annotations

import ctypes
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "lib", "libpadeops_hip.so")

PADE_CD06, PADE_CD10, PADE_CF90, PADE_CD06STAGG, PADE_GAUSSIAN = 1, 2, 3, 4, 5
PADE_D1, PADE_D2, PADE_FILTER = 1, 2, 3
PADE_D1_E2C, PADE_D1_C2E, PADE_D2_C2C, PADE_D2_E2E, PADE_INTERP_E2C, PADE_INTERP_C2E = 11, 12, 13, 14, 15, 16
PADE_D1_C2C, PADE_D1_E2E = 17, 18
PADE_DENSE_F32, PADE_DENSE_BF16X3, PADE_DENSE_FULL = 1, 2, 16
PADE_F64, PADE_F32 = 0, 1
PADE_NOALLOC_SCRATCH_BYTES = 64 << 20

# every symbol include/padeops_hip.h declares
EXPORTS = [
    "pade_op_create", "pade_op_destroy", "pade_op_size", "pade_op_apply", "pade_op_apply_f32",
    "pade_op_apply_adjoint", "pade_op_apply_adjoint_f32", "pade_op_apply_axpby", "pade_op_apply_axpby_f32",
    "pade_op_apply_axpby_noalloc",
    "pade_op_apply_host", "pade_gradient", "pade_divergence", "pade_curl", "pade_filter3d",
    "pade_op_filter3_complex", "pade_op_filter3_complex_host",
    "pade_op_dense_apply", "pade_op_dense_info", "pade_plan_variant", "pade_pencil_copy", "pade_permute3", "pade_plan_export",
    "pade_plan_export_uneven",
    "pade_last_error", "pade_version",
    "pade_cg_conserved", "pade_cg_primitive", "pade_cg_strain", "pade_cg_lad_mu", "pade_cg_lad_bulk",
    "pade_cg_lad_kap", "pade_cg_fluxes", "pade_cg_rk_stage",
    "pade_cgrid_create", "pade_cgrid_destroy", "pade_cgrid_field", "pade_cgrid_state", "pade_cgrid_set_state",
    "pade_cgrid_post_bc", "pade_cgrid_get_conserved", "pade_cgrid_get_primitive", "pade_cgrid_rhs",
    "pade_cgrid_get_dt", "pade_cgrid_advance_rk45", "pade_cgrid_transport",
]

# fields of a native compressible grid (enum pade_cg_field) and get_dt's limits
(PADE_CG_RHO, PADE_CG_U, PADE_CG_V, PADE_CG_W_VEL, PADE_CG_P, PADE_CG_T, PADE_CG_E, PADE_CG_MU, PADE_CG_BULK,
 PADE_CG_KAP, PADE_CG_W, PADE_CG_NFIELDS) = range(12)
PADE_CG_DT_NAMES = ("convective", "shear", "bulk", "conductive", "startup", "fixed")
CGRID_HOOK = ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_void_p)

_lib = None


class PadeError(RuntimeError):
    """Non-zero return code of the native library."""

    def __init__(self, code, msg):
        super().__init__(f"padeops_hip error {code}: {msg}")
        self.code = code


def load():
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise ImportError(
            f"{LIB_PATH} is not built; run `python -m padeops_amd._build` (or __graft_entry__.build())")
    lib = ctypes.CDLL(LIB_PATH)
    c_int, c_double, c_void_p, c_ll = ctypes.c_int, ctypes.c_double, ctypes.c_void_p, ctypes.c_longlong
    dp = ctypes.POINTER(ctypes.c_double)
    ip = ctypes.POINTER(ctypes.c_int)
    lib.pade_op_create.argtypes = [c_int, c_int, c_double, c_int, c_int, c_int, ctypes.POINTER(c_void_p)]
    lib.pade_op_destroy.argtypes = [c_void_p]
    lib.pade_op_size.argtypes = [c_void_p]
    apply_sig = [c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_void_p]
    for name in ("pade_op_apply", "pade_op_apply_f32", "pade_op_apply_adjoint", "pade_op_apply_adjoint_f32"):
        getattr(lib, name).argtypes = apply_sig
    lib.pade_op_apply_axpby.argtypes = [c_void_p, c_int, c_int, c_double, c_void_p, c_double, c_void_p, c_int,
                                        c_int, c_int, c_int, c_void_p]
    lib.pade_op_apply_axpby_noalloc.argtypes = lib.pade_op_apply_axpby.argtypes
    lib.pade_op_apply_axpby_f32.argtypes = [c_void_p, c_int, c_int, ctypes.c_float, c_void_p, ctypes.c_float,
                                            c_void_p, c_int, c_int, c_int, c_int, c_void_p]
    v3 = [c_void_p] * 3
    lib.pade_gradient.argtypes = v3 + [c_void_p] * 4 + [c_int] * 3 + [ctypes.POINTER(c_int), c_void_p]
    lib.pade_divergence.argtypes = v3 + [c_void_p] * 4 + [c_int] * 3 + [ctypes.POINTER(c_int), c_void_p]
    lib.pade_curl.argtypes = v3 + [c_void_p] * 4 + [c_int] * 3 + [ctypes.POINTER(c_int), c_void_p]
    lib.pade_filter3d.argtypes = v3 + [c_void_p] * 2 + [c_int] * 4 + [ctypes.POINTER(c_int), c_void_p]
    lib.pade_op_apply_host.argtypes = [c_void_p, c_int, c_int, dp, dp, c_int, c_int, c_int, c_int]
    lib.pade_op_filter3_complex.argtypes = [c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int,
                                            c_void_p]
    lib.pade_op_filter3_complex_host.argtypes = [c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int]
    lib.pade_op_dense_apply.argtypes = [c_void_p, c_int, c_int, c_void_p, c_int, c_void_p, c_int, c_int,
                                        c_int, c_int, c_int, c_int, c_void_p]
    lib.pade_op_dense_info.argtypes = [c_void_p, c_int, c_int, c_int, c_int, c_int, ctypes.POINTER(c_int),
                                       ctypes.POINTER(c_int), ctypes.POINTER(c_int)]
    lib.pade_plan_variant.argtypes = [c_int, c_int, c_int, c_double, c_int, c_int, c_int, c_int, c_int, c_int,
                                      c_int, c_int, ip]
    lib.pade_pencil_copy.argtypes = [c_void_p, c_void_p, c_ll, c_void_p]
    lib.pade_permute3.argtypes = [c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p]
    lib.pade_plan_export.argtypes = [c_int, c_int, c_int, c_double, c_int, c_int, c_int, c_int, c_int, dp,
                                     c_ll, ip]
    lib.pade_plan_export_uneven.argtypes = lib.pade_plan_export.argtypes
    v, d = c_void_p, c_double
    lib.pade_cg_conserved.argtypes = [c_ll, v, v, v, v, v, v, v, v]   # bad_index: device uint64
    lib.pade_cg_primitive.argtypes = [c_ll, v, d, d, v, v, v, v, v, v, v, v]
    lib.pade_cg_strain.argtypes = [c_ll, v, v, v, v]
    lib.pade_cg_lad_mu.argtypes = [c_ll, d, v, v, v]
    lib.pade_cg_lad_bulk.argtypes = [c_ll, d, d, d, d, v, v, v, v, v, v, v]
    lib.pade_cg_lad_kap.argtypes = [c_ll, d, d, d, d, d, v, v, v, v, v, v, v]
    lib.pade_cg_fluxes.argtypes = [c_ll, v, v, v, v, v, v, v, v, v, v, v, v]
    lib.pade_cg_rk_stage.argtypes = [c_ll, d, d, d, v, v, v, v]
    vp = ctypes.POINTER(c_void_p)
    lib.pade_cgrid_create.argtypes = [c_int, c_int, c_int, d, d, d, c_int, c_int, dp, c_int, ip, ip, vp,
                                      ctypes.POINTER(c_void_p)]
    lib.pade_cgrid_destroy.argtypes = [v]
    lib.pade_cgrid_field.argtypes = [v, c_int, vp]
    lib.pade_cgrid_state.argtypes = [v, ip, dp, dp]
    lib.pade_cgrid_set_state.argtypes = [v, c_int, d, d]
    lib.pade_cgrid_post_bc.argtypes = [v, v]
    lib.pade_cgrid_get_conserved.argtypes = [v, ctypes.POINTER(c_ll), v]
    lib.pade_cgrid_get_primitive.argtypes = [v, v]
    lib.pade_cgrid_rhs.argtypes = [v, v, v]
    lib.pade_cgrid_transport.argtypes = [v, v]
    lib.pade_cgrid_get_dt.argtypes = [v, d, dp, ip, v]
    lib.pade_cgrid_advance_rk45.argtypes = [v, d, CGRID_HOOK, v, ip, ctypes.POINTER(c_ll), v]
    lib.pade_last_error.restype = ctypes.c_char_p
    lib.pade_last_error.argtypes = []
    lib.pade_version.argtypes = []
    for name in EXPORTS:
        fn = getattr(lib, name)
        if fn.restype is ctypes.c_int or name not in ("pade_last_error",):
            if name != "pade_last_error":
                fn.restype = c_int
    _lib = lib
    return lib


def check(rc):
    if rc != 0:
        msg = load().pade_last_error().decode(errors="replace")
        raise PadeError(rc, msg)
    return rc


def plan_variant(kind, oper, n, dx, periodic, axis, na, nb, bc1=0, bcn=0, dtype=PADE_F64, adjoint=False):
    """Kernel an apply would run (host-only, pade_plan_variant): a dict with
    the partition length M, partitions per wave PW, partitions P, ``generic``
    (one lane per pencil), ``mode`` (0 strided rows, 1 x pencils, 2 staggered
    system form), ``launches`` per apply and ``uneven`` (partitions of at most M rows in padded slots; M may divide
    the rows where it is 40, 48, or 64 above 1024 rows).  bc1 / bcn: the codes that build the operator (init-time for cd06 / cd06stagg, else apply-time)."""
    info = (ctypes.c_int * 8)()
    check(load().pade_plan_variant(int(kind), int(oper), int(n), float(dx), int(bool(periodic)), int(bc1), int(bcn),
                                   int(bool(adjoint)), int(axis), int(na), int(nb), int(dtype), info))
    return {"M": info[0], "PW": info[1], "P": info[2], "generic": bool(info[3]), "mode": info[4],
            "launches": info[5], "uneven": bool(info[6])}
