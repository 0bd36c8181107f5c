"""The framework's work as its users call it, as measurable cases.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same
ranges, ``prepare`` makes what a program holds before the call (fields,
operators, output arrays), ``run`` is one pass through the public entry
points, ``work`` the bytes and operations that pass cannot do without and
``exact`` its outputs in 64 bits from dense matrices built here.

Every grid is [0, 2 pi) on a periodic axis and [0, 2 pi] on one with walls;
fields are sums of Fourier modes with a k^(-5/3) energy spectrum.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import padeops_amd as po
from padeops_amd import autograd as pag
from padeops_amd import cgrid as cg
from padeops_amd import composite
from padeops_amd._lib import PADE_D1, PADE_DENSE_BF16X3

DEV = "cuda:0"


# --------------------------------------------------------------------- cases
def listed():
    return [
        # first derivatives of one field along all three axes through the
        # facade: a small box (launch-bound), the benchmark's box, an FP32
        # field whose sizes are no powers of two, and a wall-bounded grid
        # with 2^k + 1 points on an axis
        {"name": "gradient_64", "family": "gradient", "kind": "cd06", "n1": 64, "n2": 64, "n3": 64,
         "w1": False, "w2": False, "w3": False, "f32": False},
        {"name": "gradient_512", "family": "gradient", "kind": "cd10", "n1": 512, "n2": 512, "n3": 512,
         "w1": False, "w2": False, "w3": False, "f32": False},
        {"name": "gradient_f32_360x300x200", "family": "gradient", "kind": "cd10", "n1": 360, "n2": 300, "n3": 200,
         "w1": False, "w2": False, "w3": False, "f32": True},
        {"name": "gradient_walls_257x193x129", "family": "gradient", "kind": "cd10", "n1": 257, "n2": 193, "n3": 129,
         "w1": True, "w2": True, "w3": True, "f32": False},
        # second derivatives and compact filters along all three axes
        {"name": "second_filter_256", "family": "second", "n1": 256, "n2": 256, "n3": 256,
         "w1": False, "w2": False, "w3": False},
        # the composite filter of a channel-like box, in place
        {"name": "filter3d_192x144x97", "family": "filter3d", "n1": 192, "n2": 144, "n3": 97,
         "w1": False, "w2": False, "w3": True},
        # loss and gradients of 0.5 |div u|^2 through autograd
        {"name": "adjoint_256", "family": "adjoint", "n1": 256, "n2": 256, "n3": 256, "f32": False},
        # one RK3 step of linear advection-diffusion with walls in z, and its
        # gradient with respect to the initial field
        {"name": "advdiff_384x384x256", "family": "advdiff", "n1": 384, "n2": 384, "n3": 256},
        # the compressible solver's time step: a periodic box and one with
        # one-sided closures in z
        {"name": "cgrid_256", "family": "cgrid", "n1": 256, "n2": 256, "n3": 256, "w3": False},
        {"name": "cgrid_walls_96x80x65", "family": "cgrid", "n1": 96, "n2": 80, "n3": 65, "w3": True},
        # staggered z operators of a spectral solver: complex planes of
        # 192 / 2 + 1 by 192 wavenumbers, walls in z
        {"name": "staggered_97x192x128", "family": "staggered", "n1": 97, "n2": 192, "n3": 128, "walls": True,
         "top": 1, "bot": -1, "cplx": True},
        # the matrix-core form of the benchmark's derivative
        {"name": "dense_512", "family": "dense", "n1": 512, "n2": 512, "n3": 512, "axis": 1},
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of lo..hi; one in three a multiple of 16."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(16, (n + 8) // 16 * 16) if rng.random() < 1 / 3 else n


def _box(rng, lo, hi, most):
    """Three sizes of at most `most` points in all."""
    s = [_size(rng, lo, hi) for _ in range(3)]
    while s[0] * s[1] * s[2] > most:
        k = s.index(max(s))
        s[k] = max(lo, int(s[k] * rng.uniform(0.6, 0.95)))
    return {"n1": s[0], "n2": s[1], "n3": s[2]}


def draw(rng):
    family = rng.choice(["gradient", "gradient", "gradient", "second", "filter3d", "adjoint", "advdiff", "cgrid",
                         "staggered", "dense"])
    c = {"family": family}
    if family == "gradient":
        c["kind"] = rng.choice(["cd06", "cd10"])
        c.update(_box(rng, 24, 1100, 1 << 25))
        for w in ("w1", "w2", "w3"):
            c[w] = rng.random() < 0.4
        c["f32"] = rng.random() < 0.25
    elif family in ("second", "filter3d"):
        c.update(_box(rng, 24, 512, 1 << 24))
        for w in ("w1", "w2", "w3"):
            c[w] = rng.random() < 0.4
    elif family == "adjoint":
        c.update(_box(rng, 32, 384, 1 << 24))
        c["f32"] = rng.random() < 0.5
    elif family == "advdiff":
        c.update(_box(rng, 32, 256, 1 << 22))
    elif family == "cgrid":
        c.update(_box(rng, 24, 160, 1 << 20))
        c["w3"] = rng.random() < 0.5
    elif family == "staggered":
        c.update(_box(rng, 24, 256, 1 << 23))
        c.update(walls=rng.random() < 0.6, top=rng.choice([1, -1]), bot=rng.choice([1, -1]), cplx=rng.random() < 0.5)
    else:
        c.update(n1=64 * rng.randint(1, 8), n2=_size(rng, 32, 384), n3=_size(rng, 32, 384), axis=rng.randint(1, 3))
        if c["axis"] != 1:
            c["n1"], c["n%d" % c["axis"]] = c["n%d" % c["axis"]], c["n1"]
    return c


# ------------------------------------------------------------------- inputs
def _shape(c):
    return c["n1"], c["n2"], c["n3"]


def _walls(c):
    return [bool(c.get(w)) for w in ("w1", "w2", "w3")]


def _spacing(n, wall):
    return 2 * math.pi / (n - 1 if wall else n)


def _gen(seed, k):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000 * int(seed) + k)
    return g


def _field(shape, walls, seed, k, modes=40, kmax=None, dtype=torch.float64):
    """Sum of random Fourier modes, E(k) ~ k^(-5/3), unit RMS: a Fortran-ordered (n1, n2, n3) tensor."""
    g = _gen(seed, k)
    dirs = torch.randn((modes, 3), generator=g, device=DEV, dtype=torch.float64)
    dirs = dirs / dirs.norm(dim=1, keepdim=True)
    top = kmax or max(2.0, min(shape) / 3)
    mag = torch.exp(torch.rand(modes, generator=g, device=DEV, dtype=torch.float64) * math.log(top))
    kk = torch.round(dirs * mag[:, None])
    amp = mag ** (-1 / 3) * torch.randn(modes, generator=g, device=DEV, dtype=torch.float64)
    ph = torch.rand(modes, generator=g, device=DEV, dtype=torch.float64) * (2 * math.pi)
    e = []
    for a in range(3):
        x = torch.arange(shape[a], device=DEV, dtype=torch.float64) * _spacing(shape[a], walls[a])
        e.append(torch.exp(1j * kk[:, a, None] * x[None, :]))
    head = (torch.exp(1j * ph) * amp)[:, None] * e[0]                      # (m, n1)
    yz = (e[2][:, :, None] * e[1][:, None, :]).reshape(modes, -1).t()      # (n3 n2, m)
    f = yz.real.contiguous() @ head.real.contiguous() - yz.imag.contiguous() @ head.imag.contiguous()
    f = f.reshape(shape[2], shape[1], shape[0])
    f /= f.square().mean().sqrt().clamp_min(1e-12)
    return f.to(dtype).permute(2, 1, 0)


def _inputs(c, seed):
    """The fields of a case, made from the seed alone."""
    s, w, fam = _shape(c), _walls(c), c["family"]
    if fam == "gradient":
        return [_field(s, w, seed, 0, dtype=torch.float32 if c["f32"] else torch.float64)]
    if fam in ("second", "filter3d"):
        return [_field(s, w, seed, 0)]
    if fam == "adjoint":
        return [_field(s, w, seed, k, dtype=torch.float32 if c["f32"] else torch.float64) for k in range(3)]
    if fam == "advdiff":
        return [_field(s, [False, False, True], seed, 0, kmax=8.0)]
    if fam == "cgrid":      # smooth density, velocity and pressure of a subsonic flow
        r, u, v, q, p = (_field(s, w, seed, k, modes=12, kmax=4.0) for k in range(5))
        return [1.0 + 0.05 * r, 0.3 * u, 0.3 * v, 0.3 * q, 10.0 + 0.2 * p]
    if fam == "staggered":
        out = []
        for k, extra in ((0, 0), (2, 1)):     # a cell field and an edge field (n3 + 1 planes)
            z = (s[0], s[1], s[2] + extra)
            parts = [_field(z, [False, False, c["walls"]], seed, k + j) for j in range(2 if c["cplx"] else 1)]
            t = torch.complex(*[x.permute(2, 1, 0) for x in parts]) if c["cplx"] else parts[0].permute(2, 1, 0)
            if extra and not c["walls"]:
                t[-1] = t[0]                  # a periodic edge array's last plane repeats its first
            out.append(t.permute(2, 1, 0))
        return out
    return [_field(s, w, seed, 0, dtype=torch.float32)]


# ------------------------------------------------------------------ prepare
def _facade(c, kind):
    s, w = _shape(c), _walls(c)
    d = po.derivatives()
    d.init(*s, *[_spacing(n, q) for n, q in zip(s, w)], *[not q for q in w], kind, kind, kind)
    return d


def _filters(c):
    s, w = _shape(c), _walls(c)
    f = po.filters()
    f.init(*s, *[not q for q in w], "cf90", "cf90", "cf90")
    return f


def prepare(case, seed):
    c = case
    s, fam = _shape(c), c["family"]
    st = {"case": c, "f": _inputs(c, seed)}

    def outs(k, dtype=torch.float64):
        return [po.fortran_empty(s, dtype=dtype, device=DEV) for _ in range(k)]

    if fam == "gradient":
        st["der"] = _facade(c, c["kind"])
        st["out"] = outs(3, st["f"][0].dtype)
    elif fam == "second":
        st["der"], st["fil"], st["out"] = _facade(c, "cd10"), _filters(c), outs(6)
    elif fam == "filter3d":
        st["fil"], st["work"] = _filters(c), outs(1)[0]
    elif fam == "adjoint":
        st["der"] = _facade(c, "cd06")
        st["f"] = [f.requires_grad_(True) for f in st["f"]]
    elif fam == "advdiff":
        h = _advdiff_spacing(c)
        st["d"] = [po.cd06() for _ in range(3)]
        st["cf"] = [po.cf90() for _ in range(3)]
        for a in range(3):
            if st["d"][a].init(s[a], h[a], a < 2, 0, 0) or st["cf"][a].init(s[a], a < 2):
                raise ValueError("operator init")
        st["f"][0].requires_grad_(True)
    elif fam == "cgrid":
        w = _walls(c)
        g = cg.cgrid(*s, *[_spacing(n, q) for n, q in zip(s, w)], periodic=tuple(not q for q in w), device=DEV)
        for name, f in zip(("rho", "u", "v", "w", "p"), st["f"]):
            getattr(g, name).copy_(f)
        g.post_bc()
        st["grid"], st["dt"] = g, _cgrid_dt(c)
    elif fam == "staggered":
        o = po.cd06stagg()
        h = _spacing(s[2] + (1 if c["walls"] else 0), c["walls"])
        if c["walls"]:
            o.init(s[2], h, c["top"] == 1, c["bot"] == 1)
        else:
            o.init(s[2], h)
        dt = torch.complex128 if c["cplx"] else torch.float64
        st["op"] = o
        st["out"] = [po.fortran_empty((s[0], s[1], s[2] + e), dtype=dt, device=DEV) for e in (0, 1, 0, 1, 0, 1)]
    else:
        o = po.cd10()
        o.init(s[c["axis"] - 1], _spacing(s[c["axis"] - 1], False), True)
        st["op"], st["out"] = o, outs(1, torch.float32)
    return st


# ---------------------------------------------------------------------- run
def run(state):
    c, f = state["case"], state["f"]
    fam = c["family"]
    if fam == "gradient":
        d, o = state["der"], state["out"]
        d.ddx(f[0], o[0])
        d.ddy(f[0], o[1])
        d.ddz(f[0], o[2])
        return o
    if fam == "second":
        d, q, o = state["der"], state["fil"], state["out"]
        d.d2dx2(f[0], o[0])
        d.d2dy2(f[0], o[1])
        d.d2dz2(f[0], o[2])
        q.filterx(f[0], o[3])
        q.filtery(f[0], o[4])
        q.filterz(f[0], o[5])
        return o
    if fam == "filter3d":
        composite.filter3D(None, state["fil"], f[0], work=state["work"])
        return f[0]
    if fam == "adjoint":
        ops = [state["der"].operator(a) for a in "xyz"]
        r = pag.ddx(ops[0], f[0]) + pag.ddy(ops[1], f[1]) + pag.ddz(ops[2], f[2])
        loss = 0.5 * (r * r).sum()
        return [loss.detach(), *torch.autograd.grad(loss, f)]
    if fam == "advdiff":
        dx, dy, dz = (lambda u, k=k, fn=fn: fn(state["d"][k], u) for k, fn in enumerate((pag.ddx, pag.ddy, pag.ddz)))
        d2 = [lambda u, k=k, fn=fn: fn(state["d"][k], u) for k, fn in enumerate((pag.d2dx2, pag.d2dy2, pag.d2dz2))]
        cf = [lambda u, k=k, fn=fn: fn(state["cf"][k], u) for k, fn in enumerate((pag.filterx, pag.filtery, pag.filterz))]
        u1 = _rk3(f[0], (dx, dy, dz), d2, cf, _advdiff_dt(c))
        (g,) = torch.autograd.grad(torch.linalg.vector_norm(u1), f[0])
        return [u1.detach(), g]
    if fam == "cgrid":
        g = state["grid"]
        g.advance_RK45(state["dt"])
        return [g.W, g.p, g.T]
    if fam == "staggered":
        o, x, (cell, edge) = state["op"], state["out"], f
        n1, n2 = c["n1"], c["n2"]
        o.ddz_E2C(edge, x[0], n1, n2)
        o.ddz_C2E(cell, x[1], n1, n2)
        o.InterpZ_E2C(edge, x[2], n1, n2)
        o.InterpZ_C2E(cell, x[3], n1, n2)
        o.d2dz2_C2C(cell, x[4], n1, n2)
        o.d2dz2_E2E(edge, x[5], n1, n2)
        return x
    n = list(_shape(c))
    n.pop(c["axis"] - 1)
    state["op"].dense_apply(PADE_D1, c["axis"], f[0], state["out"][0], n[0], n[1], PADE_DENSE_BF16X3)
    return state["out"][0]


# shared by run() and exact(): the user's own program around the operators
def _advdiff_spacing(c):
    return [_spacing(c["n1"], False), _spacing(c["n2"], False), _spacing(c["n3"], True)]


def _advdiff_dt(c):
    return 0.5 * min(h / v for h, v in zip(_advdiff_spacing(c), (1.0, 0.5, 0.25)))


def _rk3(u, d1, d2, fil, dt, nu=1e-3, vel=(1.0, 0.5, 0.25)):
    """One Shu-Osher RK3 step of u_t + vel . grad u = nu lap u, then the filter."""
    def rhs(v):
        adv = vel[0] * d1[0](v) + vel[1] * d1[1](v) + vel[2] * d1[2](v)
        return -adv + nu * (d2[0](v) + d2[1](v) + d2[2](v))
    u1 = u + dt * rhs(u)
    u2 = 0.75 * u + 0.25 * u1 + 0.25 * dt * rhs(u1)
    u3 = u / 3.0 + (2.0 / 3.0) * u2 + (2.0 / 3.0) * dt * rhs(u2)
    return fil[2](fil[1](fil[0](u3)))


def _cgrid_dt(c):
    return 0.1 * min(_spacing(n, q) for n, q in zip(_shape(c), _walls(c))) / 5.0


# --------------------------------------------------------------------- work
def work(case):
    """Each input read once and each output written once; the operations of the stencils and of one band solve per point."""
    c = case
    n, fam = float(c["n1"]) * c["n2"] * c["n3"], c["family"]
    ts = 4 if c.get("f32") or fam == "dense" else 8
    solve = 30.0                                   # stencil, two sweeps
    if fam == "gradient":
        return {"bytes": 4 * ts * n, "flops": 3 * solve * n}
    if fam == "second":
        return {"bytes": 7 * ts * n, "flops": 6 * solve * n}
    if fam == "filter3d":
        return {"bytes": 2 * ts * n, "flops": 3 * solve * n}
    if fam == "adjoint":
        return {"bytes": 6 * ts * n, "flops": 6 * solve * n}
    if fam == "advdiff":
        return {"bytes": 3 * ts * n, "flops": 42 * solve * n}
    if fam == "cgrid":
        return {"bytes": 12 * ts * n, "flops": 5 * 84 * solve * n}
    if fam == "staggered":
        ts = 16 if c["cplx"] else 8
        return {"bytes": 8 * ts * n, "flops": 6 * ts / 8 * 20 * n}
    return {"bytes": 2 * ts * n, "flops": 2 * 64.0 * n}


# -------------------------------------------------------------------- exact
# Operators as dense matrices: A y = B f row by row from the schemes' own
# coefficients, solved in 64 bits.
_SCHEMES = {       # kind: (A offsets 1, 2), centre, B offsets 1.., parity, derivative order
    "cd06_1": ((1 / 3, 0.0), 0.0, (7 / 9, 1 / 36), -1, 1),
    "cd06_2": ((2 / 11, 0.0), None, (12 / 11, 3 / 44), 1, 2),
    "cd10_1": ((1 / 2, 1 / 20), 0.0, (17 / 24, 101 / 600, 1 / 600), -1, 1),
    "cd10_2": ((334 / 899, 43 / 1798), None, (1065 / 1798, 1038 / 3596, 79 / 16182), 1, 2),
    "cf90": ((0.66624, 0.16688), 0.99965, (0.66652, 0.16674, 4e-5, -5e-6), 1, 0),
    "gauss": ((0.0, 0.0), 3565 / 10368, (3091 / 12960, 1997 / 25920, 149 / 12960, 107 / 103680), 1, 0),
}


def _closures(kind):
    """One-sided rows at the left end: [(A entries around the diagonal from
    column 0, B entries from column 0)] for rows 0, 1, ..."""
    if kind == "cd06_1":
        q, r, s, ah = 1.5, 1.5, -1 / 6, 1 / 3
        app = ((40 * ah - 1) * q + 7 * (4 * ah - 1) * s) / (16 * (ah + 2) * q + 8 * (1 - 4 * ah) * s)
        qpp, rpp = (app + 2) / 3, (4 * app - 1) / 12
        w1 = (2 * ah + 1) / (2 * (q + s))
        w2 = ((8 * ah + 7) * q - 6 * (2 * ah + 1) * r + (8 * ah + 7) * s) / (9 * (q + s))
        w3 = (4 * (ah + 2) * q + 2 * (1 - 4 * ah) * s) / (9 * (q + s))
        return [([w1, 3 * w1], [-17 / 6 * w1, q * w1, r * w1, s * w1]),
                ([w2 / 4, w2, w2 / 4], [-0.75 * w2, 0, 0.75 * w2]),
                ([0, w3 * app, w3, w3 * app], [-w3 * rpp, -w3 * qpp, 0, w3 * qpp, w3 * rpp])]
    if kind == "cd10_1":
        q, r, s, qp = 1.5, 1.5, -1 / 6, 0.75
        qh, rh, sh = _SCHEMES[kind][2]
        a4 = (8 * rh - 175 * sh) / (18 * rh - 550 * sh)
        b4, q4 = (8 * a4 - 3) / 20, (12 - 7 * a4) / 12
        r4, s4 = (568 * a4 - 183) / 600, (9 * a4 - 4) / 300
        t = s * (rh + 2 * sh) - q * (qh + rh + sh)
        u = (q + s) * (qh + rh - sh * (q4 / s4 - 1))
        a3 = (17 * t / (72 * u) - 8 / 9) / (19 * t / (24 * u) - 1 / 3)
        b3, q3, r3 = (3 * a3 - 1) / 12, (8 - 3 * a3) / 9, (57 * a3 - 17) / 72
        w1 = (qh + 2 * rh + 3 * sh) / (q + s)
        w2 = (rh + sh * (1 + q4 / s4) - r * w1) / qp
        w3, w4 = (qh + rh + sh * (1 - q4 / s4)) / r3, sh / s4
        return [([w1, 3 * w1], [-17 / 6 * w1, q * w1, r * w1, s * w1]),
                ([w2 / 4, w2, w2 / 4], [-qp * w2, 0, qp * w2]),
                ([w3 * b3, w3 * a3, w3, w3 * a3, w3 * b3], [-w3 * r3, -w3 * q3, 0, w3 * q3, w3 * r3]),
                ([0, w4 * b4, w4 * a4, w4, w4 * a4, w4 * b4],
                 [-w4 * s4, -w4 * r4, -w4 * q4, 0, w4 * q4, w4 * r4, w4 * s4])]
    if kind == "cd10_2":
        a3 = 344 / 1179
        b3, qa, qb = (38 * a3 - 9) / 214, (696 - 1191 * a3) / 428, (2454 * a3 - 294) / 2140
        return [([1, 11], [13, -27, 15, -1, 0]), ([0.1, 1, 0.1], [1.2, -2.4, 1.2]),
                ([b3, a3, 1, a3, b3], [qb, qa, -2 * (qa + qb), qa, qb])]
    if kind == "cf90":
        return [([1], [1]), ([0.4997, 1, 0.4997], [0.49985, 0.9997, 0.49985]),
                ([0.16688, 0.66624, 1, 0.66624, 0.16688], [0.1668, 0.66656, 0.99952, 0.66656, 0.1668]),
                ([0, 0.16688, 0.66624, 1, 0.66624, 0.16688],
                 [4e-5, 0.16672, 0.66652, 0.99968, 0.66652, 0.16672, 4e-5])]
    if kind == "gauss":
        return [([1], [5 / 6, 1 / 6]), ([0, 1], [1 / 6, 2 / 3, 1 / 6]),
                ([0, 0, 1], [5 / 128, 7 / 32, 31 / 64, 7 / 32, 5 / 128]),
                ([0, 0, 0, 1], [1 / 64, 7 / 96, 15 / 64, 17 / 48, 15 / 64, 7 / 96, 1 / 64])]
    raise ValueError(kind)


@functools.lru_cache(maxsize=64)
def _matrix(kind, n, h, wall):
    """Dense operator of one axis as a 64-bit tensor on the GPU."""
    if kind == "cd06_2" and wall:        # the first derivative applied twice
        d = _matrix("cd06_1", n, h, True)
        return d @ d
    (a1, a2), centre, taps, par, order = _SCHEMES[kind]
    A, B = np.eye(n), np.zeros((n, n))
    i = np.arange(n)

    def put(M, off, v):
        j = i + off
        keep = np.ones(n, bool) if not wall else (j >= 0) & (j < n)
        np.add.at(M, (i[keep], j[keep] % n), v)

    for off, v in ((1, a1), (2, a2)):
        put(A, off, v)
        put(A, -off, v)
    put(B, 0, -2 * sum(taps) if centre is None else centre)
    for k, v in enumerate(taps):
        put(B, k + 1, v)
        put(B, -k - 1, par * v)
    if wall:
        for r, (ra, rb) in enumerate(_closures(kind)):
            for M, row, sg in ((A, ra, 1), (B, rb, par)):
                M[r], M[n - 1 - r] = 0, 0
                M[r, : len(row)] = row
                M[n - 1 - r, n - len(row):] = sg * np.array(row[::-1])
    return torch.from_numpy(np.linalg.solve(A, B / h ** order)).to(DEV)


def _along(M, f, a):
    """M along axis a of a Fortran-ordered (n1, n2, n3) tensor."""
    t = f.permute(2, 1, 0)
    if a == 0:
        t = t @ M.t()
    elif a == 1:
        t = M @ t
    else:
        t = (M @ t.reshape(t.shape[0], -1)).reshape(M.shape[0], t.shape[1], t.shape[2])
    return t.permute(2, 1, 0)


def _cgrid_exact(c, f):
    """advance_RK45 of one inviscid ideal-gas species with the artificial properties."""
    s, w, dt = _shape(c), _walls(c), _cgrid_dt(c)
    h = [_spacing(n, q) for n, q in zip(s, w)]
    gam, cmu, cbeta, ckap = 1.4, 0.002, 1.75, 0.01

    def op(kind, x, a):
        return _along(_matrix(kind, s[a], h[a] if kind.startswith("cd") else 1.0, w[a]), x, a)

    def grad(x):
        return [op("cd10_1", x, a) for a in range(3)]

    def d4(x, a):
        return op("cd10_2", op("cd10_2", x, a), a)

    def smooth(x, kind, times):
        for a in (1, 0, 2):
            for _ in range(times):
                x = op(kind, x, a)
        return x

    rk_a = (0.0, -6234157559845.0 / 12983515589748.0, -6194124222391.0 / 4410992767914.0,
            -31623096876824.0 / 15682348800105.0, -12251185447671.0 / 11596622555746.0)
    rk_b = (494393426753.0 / 4806282396855.0, 4047970641027.0 / 5463924506627.0, 9795748752853.0 / 13190207949281.0,
            4009051133189.0 / 8539092990294.0, 1348533437543.0 / 7166442652324.0)
    rho, u, v, q, p = f
    Q = [torch.zeros_like(rho) for _ in range(5)]
    for sub in range(5):
        e = p / (gam - 1.0) / rho
        T = e * (gam - 1.0)
        vel = (u, v, q)
        W = [rho, rho * u, rho * v, rho * q, rho * (e + 0.5 * (u * u + v * v + q * q))]
        du = [grad(x) for x in vel]
        strain = torch.sqrt(du[0][0] ** 2 + 0.5 * (du[1][0] + du[0][1]) ** 2 + 0.5 * (du[2][0] + du[0][2]) ** 2
                            + du[1][1] ** 2 + 0.5 * (du[2][1] + du[1][2]) ** 2 + du[2][2] ** 2)
        mu = smooth(cmu * rho * sum(d4(strain, a) * h[a] ** 6 for a in range(3)).abs(), "gauss", 2)
        dil = du[0][0] + du[1][1] + du[2][2]
        g = [x * x for x in grad(rho)]
        den = g[0] + g[1] + g[2] + 1e-32
        b = sum(d4(dil, a) * h[a] ** 4 * (h[a] * g[a] / den) ** 2 for a in range(3))
        curl2 = (du[2][1] - du[1][2]) ** 2 + (du[0][2] - du[2][0]) ** 2 + (du[1][0] - du[0][1]) ** 2
        sw = torch.where(dil >= 0, torch.zeros_like(dil), dil * dil / (dil * dil + curl2 + 1e-32))
        bulk = smooth(cbeta * rho * sw * b.abs(), "gauss", 2)
        g = [x * x for x in grad(e)]
        den = g[0] + g[1] + g[2] + 1e-32
        k = sum(d4(e, a) * h[a] ** 4 * (h[a] * g[a] / den) for a in range(3))
        kap = smooth(ckap * rho * torch.sqrt(gam * p / rho) * k.abs() / T, "gauss", 2)
        del g, den, k, sw, curl2, b
        gT = grad(T)
        lam = bulk - (2.0 / 3.0) * mu
        R = [torch.zeros_like(rho) for _ in range(5)]
        for a in range(3):
            tau = [mu * (du[a][m] + du[m][a]) + (lam * dil if m == a else 0.0) for m in range(3)]
            flux = [W[1 + a]] + [W[1 + a] * vel[m] - tau[m] + (p if m == a else 0.0) for m in range(3)]
            flux.append((W[4] + p) * vel[a] - sum(tau[m] * vel[m] for m in range(3)) - kap * gT[a])
            for m in range(5):
                R[m] = R[m] - op("cd10_1", flux[m], a)
        for m in range(5):
            Q[m] = dt * R[m] + rk_a[sub] * Q[m]
            W[m] = smooth(W[m] + rk_b[sub] * Q[m], "cf90", 1)
        rho = W[0]
        u, v, q = W[1] / rho, W[2] / rho, W[3] / rho
        p = (gam - 1.0) * rho * (W[4] / rho - 0.5 * (u * u + v * v + q * q))
    e = p / (gam - 1.0) / rho
    # W as the step leaves it: the filtered conserved variables
    return [torch.stack([x.permute(2, 1, 0) for x in W]).permute(3, 2, 1, 0), p, e * (gam - 1.0)]


def _stagg_matrix(c, op, h):
    """A staggered z operator; even / odd ends as the mirror image of the data about the wall."""
    n = c["n3"]
    a, b, al, taps, e_in, e_out, order = {
        "ddz_E2C": (63 / 62, 17 / 186, 9 / 62, (-1, 0, 1, 2), 1, 0, 1),
        "ddz_C2E": (63 / 62, 17 / 186, 9 / 62, (-2, -1, 0, 1), 0, 1, 1),
        "I_E2C": (0.75, 0.05, 0.3, (-1, 0, 1, 2), 1, 0, 0),
        "I_C2E": (0.75, 0.05, 0.3, (-2, -1, 0, 1), 0, 1, 0),
        "d2_C2C": (12 / 11, 3 / 44, 2 / 11, (-2, -1, 0, 1, 2), 0, 0, 2),
        "d2_E2E": (12 / 11, 3 / 44, 2 / 11, (-2, -1, 0, 1, 2), 1, 1, 2)}[op]
    wt = {1: (-b, -a, a, b), 0: (b, a, a, b), 2: (b, a, -2 * (a + b), a, b)}[order]
    rows = n + (e_out if c["walls"] else 0)
    cols = n + (e_in if c["walls"] else 0)
    flip = -1 if order == 1 else 1       # a first derivative changes the parity

    def fold(j, edge, sg):
        if not c["walls"]:
            return j % n, 1
        if j < 0:
            return (-j if edge else -1 - j), sg * c["bot"]
        last = n if edge else n - 1
        return (j, 1) if j <= last else ((2 * n - j if edge else 2 * n - 1 - j), sg * c["top"])

    A, B = np.zeros((rows, rows)), np.zeros((rows, cols))
    for i in range(rows):
        for o, v in ((-1, al), (0, 1.0), (1, al)):
            j, sg = fold(i + o, e_out, flip)
            A[i, j] += sg * v
        for o, v in zip(taps, wt):
            j, sg = fold(i + o, e_in, 1)
            B[i, j] += sg * v
    return torch.from_numpy(np.linalg.solve(A, B / h ** order)).to(DEV)


def _stagg_exact(c, f):
    h = _spacing(c["n3"] + (1 if c["walls"] else 0), c["walls"])
    out = []
    for op, src, e_out in (("ddz_E2C", 1, 0), ("ddz_C2E", 0, 1), ("I_E2C", 1, 0), ("I_C2E", 0, 1),
                           ("d2_C2C", 0, 0), ("d2_E2E", 1, 1)):
        M = _stagg_matrix(c, op, h)
        t = f[src].permute(2, 1, 0)[: M.shape[1]].reshape(M.shape[1], -1)
        y = torch.complex(M @ t.real, M @ t.imag) if t.is_complex() else M @ t
        y = y.reshape(M.shape[0], c["n2"], c["n1"])
        if e_out and not c["walls"]:
            y = torch.cat([y, y[:1]])
        out.append(y.permute(2, 1, 0))
    return out


def exact(case, seed):
    c = case
    s, w, fam = _shape(c), _walls(c), c["family"]
    f = _inputs(c, seed)
    if fam == "staggered":
        return _stagg_exact(c, f)
    f = [x.double() for x in f]
    h = _advdiff_spacing(c) if fam == "advdiff" else [_spacing(n, q) for n, q in zip(s, w)]

    def op(kind, a, x):
        wall = a == 2 if fam == "advdiff" else w[a]
        return _along(_matrix(kind, s[a], h[a] if kind.startswith("cd") else 1.0, wall), x, a)

    if fam == "gradient":
        return [op(c["kind"] + "_1", a, f[0]) for a in range(3)]
    if fam == "second":
        return [op(k, a, f[0]) for k in ("cd10_2", "cf90") for a in range(3)]
    if fam == "filter3d":
        return op("cf90", 2, op("cf90", 0, op("cf90", 1, f[0])))
    if fam == "adjoint":
        r = sum(op("cd06_1", a, f[a]) for a in range(3))
        grads = [_along(_matrix("cd06_1", s[a], h[a], False).t().contiguous(), r, a) for a in range(3)]
        return [0.5 * (r * r).sum(), *grads]
    if fam == "advdiff":
        u = f[0].requires_grad_(True)
        fn = [[functools.partial(op, k, a) for a in range(3)] for k in ("cd06_1", "cd06_2", "cf90")]
        u1 = _rk3(u, fn[0], fn[1], fn[2], _advdiff_dt(c))
        (g,) = torch.autograd.grad(torch.linalg.vector_norm(u1), u)
        return [u1.detach(), g]
    if fam == "cgrid":
        return _cgrid_exact(c, f)
    return op("cd10_1", c["axis"] - 1, f[0])
