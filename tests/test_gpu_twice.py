"""An operator applied twice in one launch, and several fields in one launch.

The bounded cd06 second derivative (the first derivative twice) is the public
call that runs the twice-applied kernels directly: forward, accumulating and
adjoint, even and uneven partitions, every axis, against the dense operator
squared (FP64, 1e-12).  The compressible step runs both through its batched
passes; its grids here cover the one-launch path on even and uneven sizes and
the one-field-at-a-time path of an axis without a partitioned kernel, viscous
(properties added to) and inviscid (properties written), at the tolerance and
step of the suite's other step tests."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from oracle import cgrid_step as cg
from oracle import pade_dense as pd
import padeops_amd as po
from padeops_amd import _lib
from padeops_amd import cgrid as gcg

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("n", [16, 24, 37, 64, 75, 96, 129, 257, 336, 512])
@pytest.mark.parametrize("axis", [1, 2, 3])
def test_bounded_cd06_second_derivative(n, axis):
    op = po.cd06()
    assert op.init(n, 0.05, False, 0, 0) == 0
    shape = [67, 5]
    shape.insert(axis - 1, n)
    f = po.as_fortran(torch.tensor(np.random.default_rng(n).standard_normal(shape), device=DEV))
    fh = f.cpu().numpy()
    D = pd.dense_operator("cd06", "d1", n, 0.05, False, 0, 0)
    D2 = D @ D
    ref = pd.apply_axis(D2, fh, axis - 1)
    out = po.fortran_empty(f.shape, device=DEV)
    print(f"cd06 d2 bounded n {n} axis {axis}", flush=True)
    op._apply(_lib.PADE_D2, axis, f, out, 67, 5)
    assert rel(out.cpu().numpy(), ref) < 1e-12
    acc = f.clone()
    op._apply(_lib.PADE_D2, axis, f, acc, 67, 5, alpha=0.5, beta=-2.0)
    assert rel(acc.cpu().numpy(), 0.5 * ref - 2.0 * fh) < 1e-12
    op._apply(_lib.PADE_D2, axis, f, out, 67, 5, adjoint=True)
    assert rel(out.cpu().numpy(), pd.apply_axis(D2.T, fh, axis - 1)) < 1e-12


@pytest.mark.parametrize("n,axis,pencils", [(512, 1, (66, 63)), (512, 2, (129, 128)), (512, 3, (129, 128)),
                                            (1024, 1, (33, 8)), (1024, 3, (33, 8)), (400, 1, (67, 5)), (400, 2, (67, 5)),
                                            (700, 1, (67, 5)), (700, 3, (67, 5)), (1001, 1, (67, 5)), (1001, 2, (67, 5))])
def test_bounded_cd06_second_derivative_64(n, axis, pencils):
    """64 rows or slots per partition, even and uneven: 512 points with the
    pencils from which these are chosen, the other lengths always."""
    v = _lib.plan_variant(_lib.PADE_CD06, _lib.PADE_D2, n, 0.05, False, axis, *pencils)
    assert v["M"] == 64 and v["PW"] == 2 and v["uneven"] == (n % 64 != 0), v
    op = po.cd06()
    assert op.init(n, 0.05, False, 0, 0) == 0
    shape = list(pencils)
    shape.insert(axis - 1, n)
    f = po.as_fortran(torch.tensor(np.random.default_rng(n).standard_normal(shape), device=DEV))
    fh = f.cpu().numpy()
    D = pd.dense_operator("cd06", "d1", n, 0.05, False, 0, 0)
    D2 = D @ D
    ref = pd.apply_axis(D2, fh, axis - 1)
    out = po.fortran_empty(f.shape, device=DEV)
    print(f"cd06 d2 bounded, 64 per partition, n {n} axis {axis}", flush=True)
    op._apply(_lib.PADE_D2, axis, f, out, *pencils)
    assert rel(out.cpu().numpy(), ref) < 1e-12
    acc = f.clone()
    op._apply(_lib.PADE_D2, axis, f, acc, *pencils, alpha=0.5, beta=-2.0)
    assert rel(acc.cpu().numpy(), 0.5 * ref - 2.0 * fh) < 1e-12
    op._apply(_lib.PADE_D2, axis, f, out, *pencils, adjoint=True)
    assert rel(out.cpu().numpy(), pd.apply_axis(D2.T, fh, axis - 1)) < 1e-12


def _state(shape, seed):
    rng = np.random.default_rng(seed)
    h = tuple(2 * np.pi / n for n in shape)
    X = np.meshgrid(*[np.arange(n) * hh for n, hh in zip(shape, h)], indexing="ij")

    def wave(amp, mean):
        k, ph = rng.integers(1, 3, size=(4, 3)), rng.uniform(0, 2 * np.pi, 4)
        return mean + amp * sum(np.cos(k[m, 0] * X[0] + k[m, 1] * X[1] + k[m, 2] * X[2] + ph[m]) for m in range(4)) / 4
    return dict(rho=wave(0.1, 1.0), u=wave(0.3, 0.1), v=wave(0.3, -0.2), w=wave(0.3, 0.15), p=wave(0.1, 1.0)), h


@pytest.mark.parametrize("shape,periodic,bc", [
    ((32, 40, 25), (True, True, True), ((0, 0),) * 3),
    ((48, 24, 33), (True, True, False), ((0, 0), (0, 0), (0, 0))),
    ((16, 24, 300), (True, True, True), ((0, 0),) * 3),
    ((384, 64, 64), (True, True, True), ((0, 0),) * 3),
    ((16, 24, 336), (True, True, True), ((0, 0),) * 3),
    ((16, 24, 1041), (True, True, True), ((0, 0),) * 3)])
@pytest.mark.parametrize("inviscid", [True, False])
def test_batched_step_matches_oracle(shape, periodic, bc, inviscid):
    s0, h = _state(shape, sum(shape))
    h = tuple(1.0 / (n - 1) if not p else hh for n, p, hh in zip(shape, periodic, h))
    kw = dict(gam=1.4, Rgas=1.0, inviscid=inviscid, mu_ref=0.01, T_ref=1.0, visc_n=0.75, Pr=0.7, periodic=periodic, bc=bc)
    og = cg.Grid(shape, h, **kw)
    s1 = og.advance(s0, 1e-4)
    g = gcg.cgrid(*shape, *h, **kw)
    for c in ("rho", "u", "v", "w", "p"):
        getattr(g, c).copy_(torch.tensor(s0[c], device=DEV))
    g.mu.fill_(7.0)              # an inviscid grid overwrites what its properties held
    g.post_bc()
    g.get_conserved()
    print(f"batched step {shape} periodic {periodic} inviscid {inviscid}", flush=True)
    g.advance_RK45(1e-4)
    torch.cuda.synchronize()
    vscale = max(np.abs(s1[c]).max() for c in ("u", "v", "w"))
    for c in ("rho", "u", "v", "w", "p", "T", "e"):
        scale = vscale if c in ("u", "v", "w") else np.abs(s1[c]).max()
        err = np.abs(getattr(g, c).cpu().numpy() - s1[c]).max() / scale
        assert err < 1e-12, (c, err)
    g.destroy()


@pytest.mark.parametrize("shape,periodic,bc", [
    ((20, 64, 37), (False, True, False), ((0, 0), (0, 0), (1, -1))),
    ((129, 16, 40), (False, False, True), ((1, 1), (-1, 0), (0, 0))),
    ((24, 336, 384), (True, True, True), ((0, 0),) * 3)])
@pytest.mark.parametrize("inviscid", [True, False])
def test_batched_rhs_matches_oracle(shape, periodic, bc, inviscid):
    """Bounded axes with mixed closures (the fields of a batch then differ in
    their tables), one of them without a partitioned kernel (x = 20)."""
    s0, h = _state(shape, sum(shape))
    h = tuple(1.0 / (n - 1) if not p else hh for n, p, hh in zip(shape, periodic, h))
    kw = dict(gam=1.4, Rgas=1.0, inviscid=inviscid, mu_ref=0.01, T_ref=1.0, visc_n=0.75, Pr=0.7, periodic=periodic, bc=bc)
    og = cg.Grid(shape, h, **kw)
    s = og.from_p(dict(s0))
    ref = og.rhs(og.conserved(s), s)
    g = gcg.cgrid(*shape, *h, **kw)
    for c in ("rho", "u", "v", "w", "p"):
        getattr(g, c).copy_(torch.tensor(s0[c], device=DEV))
    g.post_bc()
    g.get_conserved()
    rhs = po.fortran_empty((*shape, 5), device=DEV)
    print(f"batched rhs {shape} inviscid {inviscid}", flush=True)
    g.getRHS(rhs)
    got = rhs.cpu().numpy()
    for k in range(5):
        assert rel(got[..., k], ref[..., k]) < 1e-12, k
    g.destroy()


@pytest.mark.parametrize("shape,periodic,bc,tol", [
    ((512, 64, 64), (True, True, True), ((0, 0),) * 3, 4e-12),          # x: whole pencils of 64 rows
    ((1024, 16, 16), (True, True, True), ((0, 0),) * 3, 7e-12),
    ((700, 16, 24), (True, True, True), ((0, 0),) * 3, 8e-12),          # 64 slots
    ((16, 700, 24), (True, False, True), ((0, 0), (1, -1), (0, 0)), 2e-12),
    ((400, 16, 700), (False, True, False), ((0, 0),) * 3, 1.5e-9)])
def test_batched_rhs_64(shape, periodic, bc, tol):
    """64 rows and slots per partition in the batched passes and the operators
    applied twice.  The artificial properties' fourth derivatives amplify
    rounding on long axes, most with walls: the bounds are ten times what the
    oracle's right-hand sides differ by with operators from a 64-bit solve and
    with the same refined in extended precision (512 points: between those of
    384 and 700)."""
    s0, h = _state(shape, sum(shape))
    h = tuple(1.0 / (n - 1) if not p else hh for n, p, hh in zip(shape, periodic, h))
    kw = dict(gam=1.4, Rgas=1.0, inviscid=True, mu_ref=0.01, T_ref=1.0, visc_n=0.75, Pr=0.7, periodic=periodic, bc=bc)
    og = cg.Grid(shape, h, **kw)
    s = og.from_p(dict(s0))
    ref = og.rhs(og.conserved(s), s)
    g = gcg.cgrid(*shape, *h, **kw)
    for c in ("rho", "u", "v", "w", "p"):
        getattr(g, c).copy_(torch.tensor(s0[c], device=DEV))
    g.post_bc()
    g.get_conserved()
    rhs = po.fortran_empty((*shape, 5), device=DEV)
    print(f"batched rhs, 64 per partition {shape} periodic {periodic}", flush=True)
    g.getRHS(rhs)
    got = rhs.cpu().numpy()
    for k in range(5):
        assert rel(got[..., k], ref[..., k]) < tol, k
    g.destroy()


@pytest.mark.parametrize("shape,periodic,tol", [
    ((16, 16, 1024), (True, True, True), 2e-12), ((16, 16, 1024), (True, True, False), 1.2e-11),
    ((16, 24, 700), (True, True, True), 2e-12), ((16, 24, 700), (True, True, False), 2e-12)])
def test_stage_64_matches_oracle(shape, periodic, tol):
    """The Runge-Kutta stage in the last flux derivative with 64 rows and slots
    per partition of z.  On grids a tenth of these the oracle's step and the
    library's are each 5e-13 to 7e-13 from extended precision (the cf90
    filter's rounding); the largest of ten times the values is a tenth more,
    and the two add up to less than 2e-12.  At the walls of 1024 points the
    fourth derivatives' rounding is larger (see test_batched_rhs_64, whose rule
    gives that bound: 1.2e-12 between the two oracles)."""
    v = _lib.plan_variant(_lib.PADE_CD10, _lib.PADE_D1, shape[2], 0.1, periodic[2], 3, *shape[:2])
    assert v["M"] == 64 and v["PW"] == 2, v
    s0, h = _state(shape, sum(shape))
    h = tuple(1.0 / (n - 1) if not p else hh for n, p, hh in zip(shape, periodic, h))
    kw = dict(gam=1.4, Rgas=1.0, inviscid=True, periodic=periodic, bc=((0, 0),) * 3)
    s1 = cg.Grid(shape, h, mu_ref=0.01, T_ref=1.0, visc_n=0.75, Pr=0.7, **kw).advance(s0, 1e-5)
    g = gcg.cgrid(*shape, *h, mu_ref=0.01, T_ref=1.0, visc_n=0.75, Pr=0.7, **kw)
    for c in ("rho", "u", "v", "w", "p"):
        getattr(g, c).copy_(torch.tensor(s0[c], device=DEV))
    g.post_bc()
    g.get_conserved()
    print(f"stage of 64 per partition {shape} periodic {periodic}", flush=True)
    g.advance_RK45(1e-5)
    torch.cuda.synchronize()
    vscale = max(np.abs(s1[c]).max() for c in ("u", "v", "w"))
    for c in ("rho", "u", "v", "w", "p", "T", "e"):
        scale = vscale if c in ("u", "v", "w") else np.abs(s1[c]).max()
        err = np.abs(getattr(g, c).cpu().numpy() - s1[c]).max() / scale
        assert err < tol, (c, err)
    g.destroy()


def test_whole_pencil_waves_by_request():
    """PADE_SPIKE_PW=8 on bounded x pencils (read once per process): the cd06
    second derivative and its adjoint, which has no twice-applied form."""
    code = """
import numpy as np, torch, padeops_amd as po
from padeops_amd import _lib
from oracle import pade_dense as pd
n = 256
assert _lib.plan_variant(1, 2, n, 0.05, False, 1, 67, 5, adjoint=True)["PW"] == 8
op = po.cd06(); op.init(n, 0.05, False, 0, 0)
f = po.as_fortran(torch.tensor(np.random.default_rng(3).standard_normal((n, 67, 5)), device="cuda:0"))
D = pd.dense_operator("cd06", "d1", n, 0.05, False, 0, 0)
for adj in (False, True):
    out = po.fortran_empty(f.shape, device="cuda:0")
    print("whole-pencil cd06 d2, adjoint", adj, flush=True)
    op._apply(_lib.PADE_D2, 1, f, out, 67, 5, adjoint=adj)
    ref = pd.apply_axis((D @ D).T if adj else D @ D, f.cpu().numpy(), 0)
    assert np.abs(out.cpu().numpy() - ref).max() < 1e-12 * np.abs(ref).max(), adj
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", code], cwd=root, env={**os.environ, "PADE_SPIKE_PW": "8", "PYTHONPATH": root},
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
