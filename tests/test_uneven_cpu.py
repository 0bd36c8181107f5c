"""Uneven partitions (a pencil length that no partition size divides), on the
CPU: the tables the library exports for them, run the way the kernels run
them (padding slots with y_t = y_{t-2} and a zero right-hand side, windows
that overlap the next partition, windowed reduced-system rows), against the
dense oracle, over every operator, boundary pair and split."""
import ctypes

import numpy as np
import pytest

import spike_emulator as se
from oracle import pade_dense as pd
from padeops_amd import _lib
from padeops_amd._lib import PADE_CD10, PADE_CF90, PADE_D1, PADE_FILTER


def export(kind, oper, n, dx, periodic, bc1, bcn, adjoint, M):
    lib = _lib.load()
    meta = (ctypes.c_int * 64)()
    args = (kind, oper, n, dx, int(periodic), bc1, bcn, int(adjoint), M)
    rc = lib.pade_plan_export_uneven(*args, None, 0, meta)
    if rc == 21:
        return None, None
    _lib.check(rc)
    tab = np.zeros(meta[12])
    _lib.check(lib.pade_plan_export_uneven(*args, tab.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), tab.size, meta))
    keys = ["n", "M", "P", "periodic", "nbl", "nbr", "off_bl", "off_br", "off_coef", "coef_len", "ncls", "kq", "len",
            "n_in", "sys", "tail"]
    m = dict(zip(keys, list(meta)[:16]))
    m["cls"], m["W"], m["start"] = list(meta)[16:32] + list(meta)[54:59], meta[32], list(meta)[33:33 + m["P"]]
    m["rows"] = [b - a for a, b in zip(m["start"], m["start"][1:] + [m["n"]])]
    return tab, m


def solve(tab, m, r):
    """The partitioned solve of right-hand side r, slot by slot."""
    n, M, P, W, kq = m["n"], m["M"], m["P"], m["W"], m["kq"]
    assert m["rows"][-1] == M and all(8 <= k <= M for k in m["rows"]) and m["start"][0] == 0
    ca = tab[m["off_coef"]:m["off_coef"] + m["coef_len"]]
    blocks = ca[:m["ncls"] * 10 * M].reshape(m["ncls"], 10 * M)
    Q = ca[m["ncls"] * 10 * M:].reshape(P, 4, 4 * W)
    g = np.zeros((P, M))
    for p in range(P):
        lu = blocks[m["cls"][p], :6 * M].reshape(M, 6)
        w = g[p]
        w[:m["rows"][p]] = r[m["start"][p]:m["start"][p] + m["rows"][p]]
        for t in range(1, M):
            w[t] -= lu[t, 0] * w[t - 1] + (lu[t, 1] * w[t - 2] if t >= 2 else 0.0)
        w[M - 1] *= lu[M - 1, 2]
        w[M - 2] = w[M - 2] * lu[M - 2, 2] - lu[M - 2, 3] * w[M - 1]
        for t in range(M - 3, -1, -1):
            w[t] = w[t] * lu[t, 2] - lu[t, 3] * w[t + 1] - lu[t, 4] * w[t + 2]
    tips = np.stack([g[:, 0], g[:, 1], g[:, M - 2], g[:, M - 1]], axis=1)
    out = np.zeros(n)
    for p in range(P):
        u = np.zeros(4)
        for j in range(W):
            q = j if W == P else p - kq + j
            if not 0 <= q < P:
                if not m["periodic"]:
                    continue
                q %= P
            u += Q[p][:, 4 * j:4 * j + 4] @ tips[q]
        S = blocks[m["cls"][p], 6 * M:].reshape(M, 4)
        y = g[p] - S @ u
        k = m["rows"][p]
        scale = max(np.abs(y).max(), 1e-300)
        assert all(abs(y[t] - y[t - 2]) <= 1e-10 * scale for t in range(k, M))      # padding repeats the last rows
        out[m["start"][p]:m["start"][p] + k] = y[:k]
    return out


LENGTHS = [(24, 16), (25, 16), (30, 16), (31, 16), (33, 24), (36, 24), (39, 24), (40, 32), (41, 32), (63, 32), (97, 32),
           (129, 32), (200, 32), (511, 32), (72, 64), (73, 64), (257, 64), (300, 64), (1023, 64), (544, 64),
           (257, 40), (300, 40), (320, 40), (258, 48), (321, 48), (336, 48), (383, 48), (384, 48),
           (1025, 64), (1088, 64), (1100, 64), (1344, 64)]


@pytest.mark.parametrize("kind,which", [("cd06", "d1"), ("cd06", "d2"), ("cd10", "d1"), ("cd10", "d2"),
                                        ("cf90", "filter"), ("gaussian", "filter")])
@pytest.mark.parametrize("n,M", LENGTHS)
def test_uneven_tables_match_dense_oracle(kind, which, n, M):
    v = np.random.default_rng(n + M).standard_normal(n)
    cases = [(True, 0, 0)]
    if not (kind == "cd06" and which == "d2"):
        cases += [(False, 0, 0), (False, 1, 1)] if kind == "cd06" else \
            [(False, a, b) for a in (0, 1, -1) for b in (0, 1, -1)]
    if n > 300:
        cases = cases[:2]
    for periodic, b1, bn in cases:
        D = pd.dense_operator(kind, which, n, 0.3 if which != "filter" else 1.0, periodic, b1, bn)
        for adj in (False, True):
            tab, m = export(se.KIND[kind], se.OPER[which], n, 0.3, periodic, b1, bn, adj, M)
            pad = "wrap" if periodic else "clamp"
            if adj and not periodic:
                out = se._stencil(tab, m, solve(tab, m, v), pad)
            else:
                out = solve(tab, m, se._stencil(tab, m, v, pad))
            ref = (D.T if adj else D) @ v
            err = np.abs(out - ref).max() / np.abs(ref).max()
            assert err < 1e-12, (kind, which, periodic, b1, bn, adj, n, M, err)


STAGG = {"d1_e2c": 11, "d1_c2e": 12, "d2_c2c": 13, "d2_e2e": 14, "interp_e2c": 15, "interp_c2e": 16, "d1_c2c": 17,
         "d1_e2e": 18}
ENDS = {1: (True, False), -1: (False, False), 2: (True, True), -2: (False, True)}


@pytest.mark.parametrize("op", sorted(STAGG))
@pytest.mark.parametrize("n,M", [(25, 16), (70, 32), (97, 32), (129, 64)])
def test_uneven_staggered_system_form(op, n, M):
    rng = np.random.default_rng(n)
    v = rng.standard_normal(n + (1 if pd.STAGG_EDGE_IN.get(op, op == "d1_e2e") else 0))
    for bc1 in ENDS:
        for bcn in ENDS:
            tab, m = export(4, STAGG[op], n, 0.3, False, bc1, bcn, False, M)
            y = solve(tab, m, se.stagg_rhs(tab, m, v))
            if m["tail"]:
                br = tab[m["off_br"]:m["off_br"] + 128].reshape(8, 16)
                y = np.append(y, (se._sys_right(br[7], v, m["n"]) - tab[9] * y[-1]) * tab[10])
            ref = pd.stagg_bounded_operator(op, n, 0.3, ENDS[bc1], ENDS[bcn]) @ v
            assert y.size == ref.size
            assert np.abs(y - ref).max() / np.abs(ref).max() < 1e-12, (op, bc1, bcn, n, M)


def test_splits_keep_their_bounds():
    """Every length: rows per partition, the last partition full, starts a
    multiple of the widest vector that divides the length."""
    for n in range(17, 1360):
        for M in (16, 24, 32, 40, 48, 64):
            tab, m = export(PADE_CD10, PADE_D1, n, 0.1, True, 0, 0, False, M)
            if tab is None:
                P = -(-n // M)
                assert n <= M or (n % M == 0 and M not in (40, 48)) or P > (21 if M == 64 else 16) or (n - M) // (P - 1) < 8 + 3 or (M < 32 and n > 2 * M), (n, M)
                continue
            unit = 16 if M in (48, 64) and n % 16 == 0 else 4 if n % 4 == 0 else 2 if n % 2 == 0 else 1
            assert all(s % unit == 0 for s in m["start"]) and m["rows"][-1] == M
            assert all(8 <= k <= M for k in m["rows"]) and sum(m["rows"]) == n
            assert all(s + M <= n for s in m["start"])          # windows stay inside the pencil


def test_variant_choice():
    """Lengths without a dividing partition size take uneven partitions on
    every axis; few pencils, and lengths without a split, one lane per pencil."""
    def pv(n, axis, na, nb, **kw):
        return _lib.plan_variant(PADE_CD10, PADE_D1, n, 0.1, kw.pop("periodic", True), axis, na, nb, **kw)
    for axis in (1, 2, 3):
        for periodic in (True, False):
            v = pv(129, axis, 200, 200, periodic=periodic)
            assert v["uneven"] and not v["generic"] and v["PW"] == 2
            assert not pv(128, axis, 200, 200, periodic=periodic)["uneven"]
    assert pv(129, 2, 8, 16)["uneven"] and pv(129, 2, 127, 1)["generic"]
    assert pv(23, 1, 64, 64)["generic"] and pv(1345, 1, 64, 64)["generic"]
    assert pv(1025, 1, 64, 64)["PW"] == 4 and pv(1344, 2, 64, 64)["PW"] == 4 and pv(1024, 3, 64, 64)["PW"] == 2
    assert _lib.plan_variant(PADE_CF90, PADE_FILTER, 272, 1.0, False, 3, 64, 64)["uneven"]


def extended(A, b):
    """A^-1 b to the 64-bit mantissas of long double, by refinement."""
    x = np.linalg.solve(A, b.astype(float)).astype(np.longdouble)
    for _ in range(3):
        x += np.linalg.solve(A, (b - A.astype(np.longdouble) @ x).astype(float))
    return x


def rms_error(kind, which, n, periodic, bc, adj, M, v, ref):
    """Of the kernels' arithmetic in 64 bits; M = n: one partition."""
    dx, k, o = 0.3 if which != "filter" else 1.0, se.KIND[kind], se.OPER[which]
    tab, m = (se.export(kind, which, n, dx, periodic, *bc, adj, n) if M == n
              else export(k, o, n, dx, periodic, *bc, adj, M))
    run = se._solve if M == n else solve
    pad, sq = "wrap" if periodic else "clamp", 0.0
    for j in range(v.shape[1]):
        y = (se._stencil(tab, m, run(tab, m, v[:, j]), pad) if adj and not periodic
             else run(tab, m, se._stencil(tab, m, v[:, j].copy(), pad)))
        sq += float(((y - ref[:, j]) ** 2).sum())
    return sq ** 0.5


@pytest.mark.parametrize("kind,which,periodic,bc,adj", [
    ("cd10", "d1", True, (0, 0), False), ("cd10", "d1", False, (1, -1), False), ("cd10", "d2", False, (1, -1), False),
    ("cd10", "d2", False, (1, -1), True), ("cd06", "d1", False, (0, 0), False), ("cf90", "filter", True, (0, 0), False),
    ("cf90", "filter", False, (0, 0), False)])
@pytest.mark.parametrize("n,M", [(65, 32), (129, 32), (321, 48)])
def test_error_is_that_of_one_partition(kind, which, periodic, bc, adj, n, M):
    """FP64 against long double: the partitioned solve adds one rounding per
    value (the correction) to the five or more of the stencil and the two
    sweeps, a tenth in the root mean square; with the sampling error of a few
    thousand correlated values, less than 1.2 times one partition's error."""
    A, B = (x.astype(float) for x in pd.assemble(kind, which, n, 0.3 if which != "filter" else 1.0, periodic, *bc)[:2])
    v = np.random.default_rng(n).standard_normal((n, 48))
    vl, Bl = v.astype(np.longdouble), B.astype(np.longdouble)
    ref = Bl.T @ extended(A.T, vl) if adj else extended(A, Bl @ vl)
    one = rms_error(kind, which, n, periodic, bc, adj, n, v, ref)
    parts = rms_error(kind, which, n, periodic, bc, adj, M, v, ref)
    assert parts < 1.2 * one, parts / one


def test_bounded_cf90_adjoint_keeps_the_more_exact_form():
    """Lengths that no partition size divides, and those that 64 divides, run
    the bounded cf90 adjoint as before uneven partitions, on every axis; the
    forward filter and the other adjoints take them."""
    def pv(n, axis, adjoint, kind=PADE_CF90, oper=PADE_FILTER, periodic=False, dtype=_lib.PADE_F64):
        return _lib.plan_variant(kind, oper, n, 0.1, periodic, axis, 200, 200, adjoint=adjoint, dtype=dtype)
    for axis in (1, 2, 3):
        for dtype in (_lib.PADE_F64, _lib.PADE_F32):
            for n in (25, 39, 65, 129, 257, 321, 700, 1025):
                assert pv(n, axis, True, dtype=dtype)["generic"] and pv(n, axis, False, dtype=dtype)["uneven"]
                assert pv(n, axis, True, PADE_CD10, PADE_D1, dtype=dtype)["uneven"]
                assert pv(n, axis, True, periodic=True, dtype=dtype)["uneven"]
            for n in (320, 384):
                v = pv(n, axis, True, dtype=dtype)
                assert v["M"] == 64 and not v["uneven"] and not v["generic"]
