"""Host-side mirror of the reference's operator types ``cd06``, ``cd10``, ``cf90``.

Same procedure names, argument meaning and error behaviour as
``src/derivatives/cd06.F90``, ``src/derivatives/cd10.F90`` and
``src/filters/cf90.F90``; the arithmetic runs in ``libpadeops_hip.so``.

Arrays are Fortran-ordered (i fastest): ``dd1`` takes ``f(n, na, nb)``,
``dd2`` ``f(na, n, nb)``, ``dd3`` ``f(na, nb, n)``.  Accepted arrays:

* torch tensors on the GPU, float64 or float32, whose memory is one dense
  block in Fortran order: a tensor of shape (n1, n2, n3) with strides
  (1, n1, n1*n2), e.g. from :func:`fortran_empty` or :func:`as_fortran`, or
  a flat contiguous tensor holding the elements in that order (a C-ordered
  multi-dimensional tensor raises ValueError);
* NumPy float64 arrays in host memory (copied to the device and back, the
  ``pade_op_apply_host`` path).
"""
from __future__ import annotations

import ctypes

import numpy as np

from . import _lib
from ._lib import PADE_CD06, PADE_CD10, PADE_CF90, PADE_GAUSSIAN, PADE_D1, PADE_D2, PADE_FILTER, PadeError
from ._lib import (PADE_CD06STAGG, PADE_D1_E2C, PADE_D1_C2E, PADE_D2_C2C, PADE_D2_E2E, PADE_INTERP_E2C,
                   PADE_INTERP_C2E, PADE_D1_C2C, PADE_D1_E2E)

try:  # torch is plumbing for device memory and streams
    import torch
except ImportError:  # pragma: no cover
    torch = None


def fortran_empty(shape, dtype=None, device="cuda"):
    """Uninitialised tensor of `shape` (n1, n2, n3[, ...]) with Fortran strides."""
    shape = tuple(int(s) for s in shape)
    nd = len(shape)
    return torch.empty(shape[::-1], dtype=dtype or torch.float64, device=device).permute(*range(nd - 1, -1, -1))


def as_fortran(t):
    """Copy of a torch tensor laid out in Fortran order (same shape)."""
    out = fortran_empty(tuple(t.shape), dtype=t.dtype, device=t.device)
    out.copy_(t)
    return out


def _is_complex(a):
    if isinstance(a, np.ndarray):
        return np.iscomplexobj(a)
    return torch is not None and isinstance(a, torch.Tensor) and a.is_complex()


def _is_dense_block(t):
    """A flat (1-D) contiguous tensor, or an N-D tensor with Fortran strides.
    A C-ordered (n1, n2, n3) tensor is refused: its memory read as Fortran
    order would put the derivative on the wrong axis."""
    shape, stride = t.shape, t.stride()
    # the usual case, three extents with exactly Fortran strides, without
    # building a view (the checks of a call on a 64^3 field cost as much host
    # time as its kernel runs)
    if len(shape) == 3 and stride == (1, shape[0], shape[0] * shape[1]):
        return True
    if len(shape) <= 1:
        return t.is_contiguous()
    return t.permute(*reversed(range(len(shape)))).is_contiguous()


def _stream_ptr():
    """The current stream of the current device, as the address ctypes passes."""
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def _check_device_arrays(f, df, count):
    dtype = f.dtype
    if dtype != df.dtype:
        raise TypeError("f and df must have the same dtype")
    if dtype != torch.float64 and dtype != torch.float32:
        raise TypeError("f must be float64 or float32")
    if not (f.is_cuda and df.is_cuda):
        raise TypeError("device arrays must live on the GPU")
    if f.numel() != count or df.numel() != count:
        raise ValueError(f"array size {f.numel()} does not match n*na*nb = {count}")
    if not (_is_dense_block(f) and _is_dense_block(df)):
        raise ValueError("arrays must be dense blocks in Fortran order")
    if f.data_ptr() == df.data_ptr():
        raise ValueError("f and df must not alias")


class _CompactOp:
    """Common plumbing: one native handle per initialised operator."""

    _kind = 0

    def __init__(self):
        self._h = ctypes.c_void_p()
        self._n = 0
        self._periodic = True

    # -- lifecycle -----------------------------------------------------------
    def _create(self, n, dx, periodic, bc1, bcn):
        lib = _lib.load()
        self.destroy()
        h = ctypes.c_void_p()
        rc = lib.pade_op_create(self._kind, int(n), float(dx), int(bool(periodic)), int(bc1), int(bcn),
                                ctypes.byref(h))
        if rc in (2, 3, 7):      # the reference's init ierr codes
            return rc
        _lib.check(rc)
        self._h = h
        self._n = int(n)
        self._periodic = bool(periodic)
        return 0

    def destroy(self):
        if self._h:
            _lib.load().pade_op_destroy(self._h)
            self._h = ctypes.c_void_p()

    def __del__(self):
        try:
            self.destroy()
        except Exception:
            pass

    def GetSize(self):
        return self._n

    @property
    def handle(self):
        return self._h

    # -- application -----------------------------------------------------------
    def _apply(self, oper, axis, f, df, na, nb, bc1=None, bcn=None, adjoint=False, alpha=None, beta=None):
        """df = op(f) (adjoint: op^T f); with alpha / beta given,
        df = alpha * op(f) + beta * df in the same pass (device arrays)."""
        if not self._h:
            raise PadeError(400, "operator used before init")
        b1 = 0 if bc1 is None else int(bc1)
        bn = 0 if bcn is None else int(bcn)
        lib = _lib.load()
        count = self._n * int(na) * int(nb)
        if isinstance(f, np.ndarray):
            if adjoint:
                raise TypeError("the adjoint is provided for device arrays")
            if f.dtype != np.float64 or df.dtype != np.float64:
                raise TypeError("host arrays must be float64")
            if f.size != count or df.size != count:
                raise ValueError(f"array size does not match n*na*nb = {count}")
            fa = np.asfortranarray(f) if f.ndim > 1 else np.ascontiguousarray(f)
            if not (df.flags.f_contiguous or df.ndim == 1):
                raise ValueError("df must be a Fortran-ordered array")
            dp = ctypes.POINTER(ctypes.c_double)
            _lib.check(lib.pade_op_apply_host(self._h, oper, axis, fa.ctypes.data_as(dp),
                                              df.ctypes.data_as(dp), int(na), int(nb), b1, bn))
            return df
        _check_device_arrays(f, df, count)
        if alpha is not None or beta is not None:
            if adjoint:
                raise TypeError("the accumulate form is provided for the forward operator")
            a = 1.0 if alpha is None else float(alpha)
            b = 0.0 if beta is None else float(beta)
            fn = lib.pade_op_apply_axpby if f.dtype == torch.float64 else lib.pade_op_apply_axpby_f32
            _lib.check(fn(self._h, oper, axis, a, f.data_ptr(), b, df.data_ptr(), int(na), int(nb), b1, bn,
                          _stream_ptr()))
            return df
        if f.dtype == torch.float64:
            fn = lib.pade_op_apply_adjoint if adjoint else lib.pade_op_apply
        else:
            fn = lib.pade_op_apply_adjoint_f32 if adjoint else lib.pade_op_apply_f32
        rc = fn(self._h, oper, axis, f.data_ptr(), df.data_ptr(), int(na), int(nb), b1, bn, _stream_ptr())
        if rc:
            _lib.check(rc)
        return df

    def dense_apply(self, oper, axis, f, df, na, nb, prec, bc1=None, bcn=None):
        """Dense-operator MFMA form (precision study); f/df float64 or float32."""
        if not self._h:
            raise PadeError(400, "operator used before init")
        lib = _lib.load()
        count = self._n * int(na) * int(nb)
        dt = {torch.float64: _lib.PADE_F64, torch.float32: _lib.PADE_F32}
        if f.dtype not in dt or df.dtype not in dt:
            raise TypeError("f and df must be float64 or float32")
        if not (f.is_cuda and df.is_cuda):
            raise TypeError("device arrays must live on the GPU")
        if f.numel() != count or df.numel() != count:
            raise ValueError(f"array size does not match n*na*nb = {count}")
        if not (_is_dense_block(f) and _is_dense_block(df)):
            raise ValueError("arrays must be dense blocks in Fortran order")
        if f.data_ptr() == df.data_ptr():
            raise ValueError("f and df must not alias")
        _lib.check(lib.pade_op_dense_apply(self._h, oper, axis, ctypes.c_void_p(f.data_ptr()), dt[f.dtype],
                                           ctypes.c_void_p(df.data_ptr()), dt[df.dtype], int(na), int(nb),
                                           0 if bc1 is None else int(bc1), 0 if bcn is None else int(bcn),
                                           int(prec), _stream_ptr()))
        return df

    def dense_info(self, oper, prec, axis=1, f_dtype=_lib.PADE_F32, df_dtype=_lib.PADE_F32):
        """(window, halfwidth, products) of the dense form applied along
        ``axis`` with these dtypes: input points visited per output block, the
        decay half-width kept, and the MFMA products per 32-point output block
        (32x32x16 products per 32 pencils, or 16x16x32 products per 16
        pencils: MFMA flops per point = 32 * products either way)."""
        lib = _lib.load()
        w, h, p = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
        _lib.check(lib.pade_op_dense_info(self._h, int(oper), int(prec), int(axis), int(f_dtype), int(df_dtype),
                                          ctypes.byref(w), ctypes.byref(h), ctypes.byref(p)))
        return w.value, h.value, p.value


class cd06(_CompactOp):
    """6th-order compact first derivative (src/derivatives/cd06.F90:70-119).

    ``dd1/dd2/dd3`` take no boundary codes (cd06.F90:775-839).  The second
    derivative ``d2d1/d2d2/d2d3`` has no reference implementation
    (cd06.F90:330-343,492-513,745-773,841-853); this library provides the
    periodic sixth-order tridiagonal scheme (alpha = 2/11) and, when bounded,
    the first derivative applied twice.
    """

    _kind = PADE_CD06

    def init(self, n, dx, periodic, bc1=0, bcn=0):
        """Returns ierr: 3 periodic n < 6, 2 bounded n < 8 (cd06.F90:129-201)."""
        return self._create(n, dx, periodic, bc1, bcn)

    def dd1(self, f, df, na, nb):
        return self._apply(PADE_D1, 1, f, df, na, nb)

    def dd2(self, f, df, na, nb):
        return self._apply(PADE_D1, 2, f, df, na, nb)

    def dd3(self, f, df, na, nb):
        return self._apply(PADE_D1, 3, f, df, na, nb)

    def d2d1(self, f, df, na, nb):
        return self._apply(PADE_D2, 1, f, df, na, nb)

    def d2d2(self, f, df, na, nb):
        return self._apply(PADE_D2, 2, f, df, na, nb)

    def d2d3(self, f, df, na, nb):
        return self._apply(PADE_D2, 3, f, df, na, nb)


class cd10(_CompactOp):
    """10th-order compact first and second derivatives (src/derivatives/cd10.F90:108-183)."""

    _kind = PADE_CD10

    def init(self, n, dx, periodic, bc1=0, bcn=0):
        """Returns ierr: 2 for 1 < n < 8 (cd10.F90:195-315)."""
        return self._create(n, dx, periodic, bc1, bcn)

    def dd1(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_D1, 1, f, df, na, nb, bc1, bcn)

    def dd2(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_D1, 2, f, df, na, nb, bc1, bcn)

    def dd3(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_D1, 3, f, df, na, nb, bc1, bcn)

    def d2d1(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_D2, 1, f, df, na, nb, bc1, bcn)

    def d2d2(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_D2, 2, f, df, na, nb, bc1, bcn)

    def d2d3(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_D2, 3, f, df, na, nb, bc1, bcn)


class cf90(_CompactOp):
    """8th-order compact filter with 90% truncation (src/filters/cf90.F90:54-101)."""

    _kind = PADE_CF90

    def init(self, n, periodic):
        """Returns ierr: 7 for 1 < n < 10 (cf90.F90:107-175)."""
        return self._create(n, 1.0, periodic, 0, 0)

    def filter1(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_FILTER, 1, f, df, na, nb, bc1, bcn)

    def filter2(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_FILTER, 2, f, df, na, nb, bc1, bcn)

    def filter3(self, f, df, na, nb, bc1=None, bcn=None):
        """Real data: filter along z.  Complex data (torch.complex128 on the
        GPU or numpy complex128 on the host): the reference's filter3_CMPLX
        (cf90.F90:1230-1251) -- both parts filtered; a bounded filter takes
        the right-hand side of (bc1, bcn) when bcn is given, else of (0, 0),
        and always solves with the (0, 0) left-hand side, as the reference
        does."""
        if _is_complex(f) or _is_complex(df):
            return self._filter3_complex(f, df, na, nb, bc1, bcn)
        return self._apply(PADE_FILTER, 3, f, df, na, nb, bc1, bcn)

    def _filter3_complex(self, f, df, na, nb, bc1, bcn):
        if not self._h:
            raise PadeError(400, "operator used before init")
        lib = _lib.load()
        count = self._n * int(na) * int(nb)
        has_bc = bcn is not None
        b1 = int(bc1) if (has_bc and bc1 is not None) else 0
        bn = int(bcn) if has_bc else 0
        if isinstance(f, np.ndarray):
            if f.dtype != np.complex128 or df.dtype != np.complex128:
                raise TypeError("complex host arrays must be complex128")
            if f.size != count or df.size != count:
                raise ValueError(f"array size does not match n*na*nb = {count}")
            fa = np.asfortranarray(f) if f.ndim > 1 else np.ascontiguousarray(f)
            if not (df.flags.f_contiguous or df.ndim == 1):
                raise ValueError("df must be a Fortran-ordered array")
            _lib.check(lib.pade_op_filter3_complex_host(self._h, ctypes.c_void_p(fa.ctypes.data),
                                                        ctypes.c_void_p(df.ctypes.data), int(na), int(nb),
                                                        b1, bn, int(has_bc)))
            return df
        if f.dtype != torch.complex128 or df.dtype != torch.complex128:
            raise TypeError("complex device arrays must be complex128")
        if not (f.is_cuda and df.is_cuda):
            raise TypeError("device arrays must live on the GPU")
        if f.numel() != count or df.numel() != count:
            raise ValueError(f"array size {f.numel()} does not match n*na*nb = {count}")
        if not (_is_dense_block(f) and _is_dense_block(df)):
            raise ValueError("arrays must be dense blocks in Fortran order")
        if f.data_ptr() == df.data_ptr():
            raise ValueError("f and df must not alias")
        _lib.check(lib.pade_op_filter3_complex(self._h, ctypes.c_void_p(f.data_ptr()), ctypes.c_void_p(df.data_ptr()),
                                               int(na), int(nb), b1, bn, int(has_bc), _stream_ptr()))
        return df


class gaussian(_CompactOp):
    """Explicit Gaussian filter of width 4 dx (src/filters/gaussian.F90:
    coefficients :11-36, periodic stencil :137-185, bounded rows for bc 0 /
    1 / -1 :189-334); the compressible solver's artificial-property filter."""

    _kind = PADE_GAUSSIAN

    def init(self, n, periodic):
        """Returns 0, or 21 for 1 < n < 9 (the stencil spans 9 points)."""
        return self._create(n, 1.0, periodic, 0, 0)

    def filter1(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_FILTER, 1, f, df, na, nb, bc1, bcn)

    def filter2(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_FILTER, 2, f, df, na, nb, bc1, bcn)

    def filter3(self, f, df, na, nb, bc1=None, bcn=None):
        return self._apply(PADE_FILTER, 3, f, df, na, nb, bc1, bcn)


class cd06stagg(_CompactOp):
    """Sixth-order staggered compact z operators (src/derivatives/cd06stagg.F90).
    Cell (C) arrays are (n1, n2, n), edge (E) arrays (n1, n2, n + 1); every
    operation acts along z.  Periodic form (init_periodic :170-195): an E
    array's last plane repeats its first.  Bounded form (init_nonperiodic
    :197-232): each end is even or odd, optionally with the one-sided
    closure.  Real (float64 / float32) and complex128 arrays."""

    _kind = PADE_CD06STAGG

    def init(self, nx, dx, isTopEven=None, isBotEven=None, isTopSided=False, isBotSided=False):
        """``init(nx, dx)``: periodic.  ``init(nx, dx, isTopEven, isBotEven
        [, isTopSided, isBotSided])``: bounded ("Bot" is the k = 1 end, "Top"
        the k = n end).  Raises PadeError(21) for nx <= 4 (GracefulExit 21,
        cd06stagg.F90:182-184,215-217)."""
        if (isTopEven is None) != (isBotEven is None):
            raise ValueError("give both isTopEven and isBotEven (bounded) or neither (periodic)")
        if isTopEven is None:
            rc = self._create(nx, dx, True, 0, 0)
        else:
            bc1 = (1 if isBotEven else -1) * (2 if isBotSided else 1)
            bcn = (1 if isTopEven else -1) * (2 if isTopSided else 1)
            rc = self._create(nx, dx, False, bc1, bcn)
        if rc:
            raise PadeError(rc, "cd06stagg init")
        return 0

    def _stagg(self, oper, f, df, n1, n2, e_in, e_out):
        if not self._h:
            raise PadeError(400, "operator used before init")
        n = self._n
        cin, cout = n1 * n2 * (n + e_in), n1 * n2 * (n + e_out)
        host = isinstance(f, np.ndarray)
        cplx = _is_complex(f)
        if cplx != _is_complex(df):
            raise TypeError("f and df must both be real or both complex")
        # a complex (n1, n2, m) array is a real (2 n1, n2, m) one
        na = 2 * int(n1) if cplx else int(n1)
        if host:
            if f.size != cin or df.size != cout:
                raise ValueError(f"array sizes must be n1*n2*{n + e_in} and n1*n2*{n + e_out}")
            lib = _lib.load()
            want = np.complex128 if cplx else np.float64
            fa = np.asfortranarray(f, dtype=want)
            if df.dtype != want or not (df.flags.f_contiguous or df.ndim == 1):
                raise ValueError(f"df must be a Fortran-ordered {np.dtype(want).name} array")
            dp = ctypes.POINTER(ctypes.c_double)
            _lib.check(lib.pade_op_apply_host(self._h, oper, 3, fa.ctypes.data_as(dp), df.ctypes.data_as(dp),
                                              na, int(n2), 0, 0))
            return df
        if cplx:
            if f.dtype != torch.complex128 or df.dtype != torch.complex128:
                raise TypeError("complex arrays must be complex128")
        elif f.dtype != df.dtype or f.dtype not in (torch.float64, torch.float32):
            raise TypeError("f and df must both be float64 or both float32")
        if not (f.is_cuda and df.is_cuda):
            raise TypeError("device arrays must live on the GPU")
        if f.numel() != cin or df.numel() != cout:
            raise ValueError(f"array sizes must be n1*n2*{n + e_in} and n1*n2*{n + e_out}")
        if not (_is_dense_block(f) and _is_dense_block(df)):
            raise ValueError("arrays must be dense blocks in Fortran order")
        if f.data_ptr() == df.data_ptr():
            raise ValueError("f and df must not alias")
        lib = _lib.load()
        fn = lib.pade_op_apply_f32 if f.dtype == torch.float32 else lib.pade_op_apply
        _lib.check(fn(self._h, oper, 3, ctypes.c_void_p(f.data_ptr()), ctypes.c_void_p(df.data_ptr()),
                      na, int(n2), 0, 0, _stream_ptr()))
        return df

    def ddz_E2C(self, fE, dfC, n1, n2):
        """cd06stagg.F90:820-833."""
        return self._stagg(PADE_D1_E2C, fE, dfC, n1, n2, 1, 0)

    def ddz_C2E(self, fC, dfE, n1, n2):
        """cd06stagg.F90:850-864."""
        return self._stagg(PADE_D1_C2E, fC, dfE, n1, n2, 0, 1)

    def d2dz2_C2C(self, fC, d2fC, n1, n2):
        """cd06stagg.F90:995-1009."""
        return self._stagg(PADE_D2_C2C, fC, d2fC, n1, n2, 0, 0)

    def d2dz2_E2E(self, fE, d2fE, n1, n2):
        """cd06stagg.F90:1027-1042."""
        return self._stagg(PADE_D2_E2E, fE, d2fE, n1, n2, 1, 1)

    def InterpZ_E2C(self, fE, IfC, n1, n2):
        """cd06stagg.F90:928-942."""
        return self._stagg(PADE_INTERP_E2C, fE, IfC, n1, n2, 1, 0)

    def InterpZ_C2E(self, fC, IfE, n1, n2):
        """cd06stagg.F90:960-975."""
        return self._stagg(PADE_INTERP_C2E, fC, IfE, n1, n2, 0, 1)

    def ddz_C2C(self, fC, dfC, n1, n2):
        """cd06stagg.F90:883-892 (bounded form only)."""
        return self._stagg(PADE_D1_C2C, fC, dfC, n1, n2, 0, 0)

    def ddz_E2E(self, fE, dfE, n1, n2):
        """cd06stagg.F90:905-914 (bounded form only)."""
        return self._stagg(PADE_D1_E2E, fE, dfE, n1, n2, 1, 1)
