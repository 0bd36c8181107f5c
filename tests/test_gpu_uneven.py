"""Uneven partitions on the GPU (pencil lengths that no partition size
divides): forward, accumulating and adjoint applies along every axis against
the dense oracle, at the edges of the splits (shortest partitions, odd and
even padding, one and two partitions in the last wave) with pencil counts
that leave the last workgroup partly empty.  FP64 to 1e-12, FP32 to the
suite's banded tolerance."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import pade_dense as pd
import padeops_amd as po
from padeops_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
KIND = {"cd06": po.cd06, "cd10": po.cd10, "cf90": po.cf90, "gaussian": po.gaussian}
OPER = {"d1": _lib.PADE_D1, "d2": _lib.PADE_D2, "filter": _lib.PADE_FILTER}


def setup(kind, n, periodic, axis, seed, dtype=torch.float64, pencils=(67, 5)):
    op = KIND[kind]()
    assert (op.init(n, periodic) if kind in ("cf90", "gaussian") else op.init(n, 0.05, periodic, 0, 0)) == 0
    shape = list(pencils)
    shape.insert(axis - 1, n)
    f = np.random.default_rng(seed).standard_normal(shape)
    ft = po.as_fortran(torch.tensor(f, device=DEV, dtype=dtype))
    return op, ft, ft.cpu().double().numpy()


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


CASES = [("cd10", "d1", True, (0, 0)), ("cd10", "d2", True, (0, 0)), ("cf90", "filter", True, (0, 0)),
         ("cd06", "d1", True, (0, 0)), ("cd10", "d1", False, (0, 0)), ("cd10", "d2", False, (1, -1)),
         ("cf90", "filter", False, (-1, 1)), ("cd06", "d1", False, (0, 0)), ("gaussian", "filter", False, (0, 1))]


@pytest.mark.parametrize("kind,which,periodic,bc", CASES)
@pytest.mark.parametrize("n", [24, 25, 37, 75, 129, 200, 257, 301, 1025, 1100])
@pytest.mark.parametrize("axis", [1, 2, 3])
def test_uneven_matches_oracle(kind, which, periodic, bc, n, axis):
    op, f, fh = setup(kind, n, periodic, axis, n + axis)
    v = _lib.plan_variant(op._kind, OPER[which], n, 0.05, periodic, axis, 67, 5, *bc)
    assert v["uneven"], v
    h = 1.0 if which == "filter" else 0.05
    D = pd.dense_operator(kind, which, n, h, periodic, *bc)
    ref = pd.apply_axis(D, fh, axis - 1)
    out = po.fortran_empty(f.shape, device=DEV)
    print(f"uneven {kind} {which} periodic {periodic} bc {bc} n {n} axis {axis}", flush=True)
    op._apply(OPER[which], axis, f, out, 67, 5, *bc)
    assert rel(out.cpu().numpy(), ref) < 1e-12
    acc = f.clone()
    op._apply(OPER[which], axis, f, acc, 67, 5, *bc, alpha=-0.75, beta=1.5)
    assert rel(acc.cpu().numpy(), -0.75 * ref + 1.5 * fh) < 1e-12
    op._apply(OPER[which], axis, f, out, 67, 5, *bc, adjoint=True)
    assert rel(out.cpu().numpy(), pd.apply_axis(D.T, fh, axis - 1)) < 1e-12


@pytest.mark.parametrize("n,pencils", [(129, (150, 130)), (176, (70, 65)), (300, (150, 130)), (320, (41, 40)),
                                       (384, (41, 40)), (513, (64, 33)), (1023, (40, 33)), (1088, (40, 33)),
                                       (1343, (25, 21))])
@pytest.mark.parametrize("axis", [1, 2, 3])
@pytest.mark.parametrize("periodic", [True, False])
def test_uneven_throughput_sizes(n, pencils, axis, periodic):
    """Enough pencils for the throughput partition sizes; FP64 and FP32."""
    D = pd.dense_operator("cd10", "d1", n, 0.05, periodic, 0, 0)
    for dtype, tol in ((torch.float64, 1e-12), (torch.float32, 1e-4)):
        op, f, fh = setup("cd10", n, periodic, axis, n, dtype, pencils)
        out = po.fortran_empty(f.shape, dtype=dtype, device=DEV)
        print(f"uneven throughput n {n} axis {axis} periodic {periodic} {dtype}", flush=True)
        op._apply(_lib.PADE_D1, axis, f, out, *pencils)
        assert rel(out.cpu().double().numpy(), pd.apply_axis(D, fh, axis - 1)) < tol


@pytest.mark.parametrize("oper", ["ddz_E2C", "ddz_C2E", "InterpZ_C2E", "d2dz2_E2E", "ddz_C2C"])
@pytest.mark.parametrize("n", [25, 70, 129, 1041])
def test_uneven_staggered_bounded(oper, n):
    name = {"ddz_E2C": "d1_e2c", "ddz_C2E": "d1_c2e", "InterpZ_C2E": "interp_c2e", "d2dz2_E2E": "d2_e2e",
            "ddz_C2C": "d1_c2c"}[oper]
    e_in = 1 if oper in ("ddz_E2C", "d2dz2_E2E") else 0
    e_out = 1 if oper in ("ddz_C2E", "InterpZ_C2E", "d2dz2_E2E") else 0
    f = np.random.default_rng(n).standard_normal((19, 11, n + e_in))
    ft = po.as_fortran(torch.tensor(f, device=DEV))
    for top, bot, tops, bots in ((True, False, False, False), (False, True, True, False), (True, True, True, True)):
        op = po.cd06stagg()
        op.init(n, 0.1, top, bot, tops, bots)
        out = po.fortran_empty((19, 11, n + e_out), device=DEV)
        print(f"uneven staggered {oper} n {n}", flush=True)
        getattr(op, oper)(ft, out, 19, 11)
        D = pd.stagg_bounded_operator(name, n, 0.1, (bot, bots), (top, tops))
        assert rel(out.cpu().numpy(), pd.apply_axis(D, f, 2)) < 1e-12


def test_uneven_in_place_filter3d():
    """filter3D's last z pass runs in place on uneven partitions too."""
    from padeops_amd import composite
    s = (33, 50, 97)
    fil = po.filters()
    fil.init(*s, True, True, False, "cf90", "cf90", "cf90")
    f = np.random.default_rng(1).standard_normal(s)
    ft = po.as_fortran(torch.tensor(f, device=DEV))
    print("uneven filter3D", flush=True)
    composite.filter3D(None, fil, ft)
    ref = f
    for a in (1, 0, 2):
        ref = pd.apply("cf90", "filter", ref, a, 1.0, a < 2, 0, 0)
    assert rel(ft.cpu().numpy(), ref) < 1e-12


@pytest.mark.parametrize("kind,which,n,side,periodic", [("cd10", "d1", 320, 165, True), ("cd10", "d1", 240, 190, False),
                                                        ("cd06", "d2", 320, 130, False)])
def test_noalloc_limit_of_divided_lengths(kind, which, n, side, periodic):
    """Lengths that a partition size divides need no scratch array to
    accumulate (cd06's bounded second derivative one field of it), also where
    they run uneven partitions: fields above that limit are taken."""
    op, f, _ = setup(kind, n, periodic, 3, n, pencils=(side, side))
    v = _lib.plan_variant(op._kind, OPER[which], n, 0.05, periodic, 3, side, side, 0, 0)
    assert f.numel() * 8 * (2 if which == "d2" else 1) > _lib.PADE_NOALLOC_SCRATCH_BYTES
    ref, out = f.clone(), f.clone()
    op._apply(OPER[which], 3, f, ref, side, side, alpha=0.5, beta=-2.0)
    print(f"noalloc {kind} {which} n {n} {v}", flush=True)
    rc = _lib.load().pade_op_apply_axpby_noalloc(op._h, OPER[which], 3, 0.5, ctypes.c_void_p(f.data_ptr()), -2.0,
                                                 ctypes.c_void_p(out.data_ptr()), side, side, 0, 0,
                                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    assert torch.equal(ref, out)


# FP32 bounds: the same calls in FP64 are within 14 (cd06, cd10), 40 (the first
# derivative twice) and 900 (cf90) rounding errors of the largest output; as
# many of 6e-8, doubled.
FP32_CASES = [("cd10", "d1", True, (0, 0), 2e-6), ("cd06", "d1", False, (0, 0), 2e-6), ("cd10", "d1", False, (1, -1), 2e-6),
              ("cd06", "d2", False, (0, 0), 5e-6), ("cf90", "filter", True, (0, 0), 1.1e-4),
              ("cf90", "filter", False, (0, 0), 1.1e-4)]


@pytest.mark.parametrize("kind,which,periodic,bc,tol", FP32_CASES)
@pytest.mark.parametrize("n,pencils", [(25, (67, 5)), (39, (67, 5)), (129, (67, 5)), (300, (67, 5)), (383, (150, 30)),
                                       (701, (67, 5)), (1025, (67, 5))])
@pytest.mark.parametrize("axis", [1, 2, 3])
def test_uneven_fp32(kind, which, periodic, bc, tol, n, pencils, axis):
    """Forward, accumulating and adjoint; cf90's bounded adjoint keeps the
    one-lane path, cd06's second derivative runs twice, in place."""
    op, f, fh = setup(kind, n, periodic, axis, n + axis, torch.float32, pencils)
    v = _lib.plan_variant(op._kind, OPER[which], n, 0.05, periodic, axis, *pencils, *bc, dtype=_lib.PADE_F32)
    assert v["uneven"], v
    D = pd.dense_operator(kind, "d1" if which == "d2" else which, n, 1.0 if which == "filter" else 0.05, periodic, *bc)
    if which == "d2":
        D = D @ D
    ref = pd.apply_axis(D, fh, axis - 1)
    out = po.fortran_empty(f.shape, dtype=torch.float32, device=DEV)
    print(f"uneven FP32 {kind} {which} periodic {periodic} bc {bc} n {n} axis {axis}", flush=True)
    op._apply(OPER[which], axis, f, out, *pencils, *bc)
    assert rel(out.cpu().double().numpy(), ref) < tol
    acc = f.clone()
    op._apply(OPER[which], axis, f, acc, *pencils, *bc, alpha=-0.75, beta=1.5)
    assert rel(acc.cpu().double().numpy(), -0.75 * ref + 1.5 * fh) < tol
    op._apply(OPER[which], axis, f, out, *pencils, *bc, adjoint=True)
    assert rel(out.cpu().double().numpy(), pd.apply_axis(D.T, fh, axis - 1)) < tol


@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 2e-6)])
@pytest.mark.parametrize("n", [128, 129, 132])
@pytest.mark.parametrize("axis", [1, 2, 3])
@pytest.mark.parametrize("periodic", [True, False])
def test_element_aligned_arrays(dtype, tol, n, axis, periodic):
    """Fields that start one element behind a 16-byte boundary."""
    op, f, fh = setup("cd10", n, periodic, axis, n, dtype)
    D = pd.dense_operator("cd10", "d1", n, 0.05, periodic, 0, 0)
    flat = torch.zeros(f.numel() + 1, dtype=dtype, device=DEV)[1:]
    out = torch.zeros(f.numel() + 1, dtype=dtype, device=DEV)[1:]
    flat.copy_(f.permute(2, 1, 0).reshape(-1))
    assert flat.data_ptr() % 16 and out.data_ptr() % 16

    def array(t):
        return t.cpu().double().numpy().reshape(tuple(f.shape), order="F")
    ref = pd.apply_axis(D, fh, axis - 1)
    print(f"element-aligned {dtype} n {n} axis {axis} periodic {periodic}", flush=True)
    op._apply(_lib.PADE_D1, axis, flat, out, 67, 5)
    assert rel(array(out), ref) < tol
    out.copy_(flat)
    op._apply(_lib.PADE_D1, axis, flat, out, 67, 5, alpha=2.0, beta=-0.5)
    assert rel(array(out), 2.0 * ref - 0.5 * fh) < tol
    op._apply(_lib.PADE_D1, axis, flat, out, 67, 5, adjoint=True)
    assert rel(array(out), pd.apply_axis(D.T, fh, axis - 1)) < tol
