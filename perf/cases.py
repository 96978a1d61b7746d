"""Timed cases: the solves that a user of the framework runs, through its public entry points.

A case is one call pattern on one tree:

  build_solve   build_solver + solve for new coefficients (the direct solver's whole job)
  solve         a built solver, new boundary data (the down pass)
  source        a built no-source ItI solver, a new source (the up pass, then the down pass)
  gradient      a loss's value and its derivative with respect to a coefficient field
  adaptive      build_solver + solve on a locally refined quadtree

Solutions are known in closed form so that the results can be checked without another solver:
the elliptic problems take random polynomials of a degree that the Gauss points of a leaf side
represent exactly, the Helmholtz problems plane waves of a wavenumber that a leaf resolves to
rounding.  The coefficients are the smooth variable fields of the framework's own workloads
(sums of Gaussian bumps); source and boundary data follow from the solution.
"""

import functools
import math

import numpy as np
import torch

import jaxhps_amd as jh
from jaxhps_amd.adjoint import differentiable_solve

DEV = "cuda"


def listed():
    return [
        # the quickstart: 2D Poisson on 64 small leaves; launches and host work decide
        dict(name="poisson2d_p8_L3", call="build_solve", kind="dtn2d", p=8, L=3, nsrc=1, terms="laplace",
             precision="fp64"),
        # 2D variable-coefficient elliptic problem with first-order and zeroth-order terms, 16 right-hand sides
        dict(name="elliptic2d_p16_L6_rhs16", call="build_solve", kind="dtn2d", p=16, L=6, nsrc=16, terms="full",
             precision="fp64"),
        # odd orders: no dimension is a multiple of a tile
        dict(name="elliptic2d_p11_L5_rhs3", call="build_solve", kind="dtn2d", p=11, L=5, nsrc=3, terms="full",
             precision="fp64"),
        # Helmholtz scattering at full size (4.2 M unknowns): the default precision and the mixed one
        dict(name="helmholtz_p16_L7", call="build_solve", kind="iti2d", p=16, L=7, nsrc=1, terms="helmholtz",
             precision="fp64"),
        dict(name="helmholtz_p16_L7_mixed", call="build_solve", kind="iti2d", p=16, L=7, nsrc=1, terms="helmholtz",
             precision="mixed"),
        # a moderate Helmholtz problem of odd order with several sources
        dict(name="helmholtz_p13_L4_rhs2", call="build_solve", kind="iti2d", p=13, L=4, nsrc=2, terms="helmholtz",
             precision="fp64"),
        # 3D variable-coefficient Poisson: 12288 unknowns in the root merge
        dict(name="poisson3d_p10_L3_rhs4", call="build_solve", kind="dtn3d", p=10, L=3, nsrc=4, terms="full",
             precision="fp64"),
        # a small 3D problem in mixed precision
        dict(name="poisson3d_p8_L2_mixed", call="build_solve", kind="dtn3d", p=8, L=2, nsrc=1, terms="full",
             precision="mixed"),
        # one factorisation, many incident waves: only the solve is repeated
        dict(name="resolve_p16_L6", call="solve", kind="iti2d", p=16, L=6, nsrc=1, terms="helmholtz",
             precision="fp64"),
        # one factorisation, many sources
        dict(name="newsource_p16_L6", call="source", kind="iti2d", p=16, L=6, nsrc=1, terms="helmholtz",
             precision="fp64"),
        # one step of an inverse-scattering loop: misfit and gradient in the contrast field
        dict(name="gradient_p16_L6", call="gradient", kind="iti2d", p=16, L=6, nsrc=1, terms="helmholtz",
             precision="fp64"),
        # a tree refined around a circular front: many small merges of mixed signatures
        dict(name="adaptive2d_p12_d6", call="adaptive", kind="dtn2d", p=12, L=6, nsrc=1, terms="laplace",
             precision="fp64"),
    ]


def draw(rng):
    call = rng.choice(["build_solve"] * 6 + ["solve", "source", "gradient", "adaptive"])
    kind = {"build_solve": rng.choice(["dtn2d", "iti2d", "dtn3d"]), "solve": rng.choice(["dtn2d", "iti2d"]),
            "source": "iti2d", "gradient": "iti2d", "adaptive": "dtn2d"}[call]
    precision, terms, nsrc = "fp64", "full", 1
    if kind == "dtn3d":
        p, L = rng.randint(6, 10), rng.randint(1, 3)
    else:
        p = rng.randint(8, 16)
        L = rng.randint(1, 7 if call == "build_solve" and kind == "iti2d" else 6)
        if call == "adaptive":
            L = rng.randint(3, 6)
        if kind == "iti2d":
            terms = "helmholtz"
    if call in ("build_solve", "solve"):
        nsrc = int(round(math.exp(rng.uniform(0.0, math.log(16 if kind == "dtn2d" else 4)))))
    if call == "build_solve":
        precision = rng.choice(["fp64", "fp64", "mixed"])
    if call == "adaptive" or (kind == "dtn2d" and rng.random() < 0.3):
        terms = "laplace"
    return dict(call=call, kind=kind, p=p, L=L, nsrc=nsrc, terms=terms, precision=precision)


# -- geometry, orders of points ---------------------------------------------------------------
def _front(case):
    """Cells (x0, x1, y0, y1) of the quadtree refined around the circle of radius 0.6, depth first."""
    def split(x0, x1, y0, y1, depth):
        s = x1 - x0
        near = abs(math.hypot((x0 + x1) / 2, (y0 + y1) / 2) - 0.6) < 2.0 * s
        if depth >= 2 and (depth >= case["L"] or not near):
            return (x0, x1, y0, y1, depth)
        xm, ym = (x0 + x1) / 2, (y0 + y1) / 2
        return [split(x0, xm, y0, ym, depth + 1), split(xm, x1, y0, ym, depth + 1),
                split(xm, x1, ym, y1, depth + 1), split(x0, xm, ym, y1, depth + 1)]
    return split(-1.0, 1.0, -1.0, 1.0, 0)


def _flat(tree):
    return [tree[:4]] if isinstance(tree, tuple) else [c for t in tree for c in _flat(t)]


def _boxes(case):
    """(n_leaves, 2 d) leaf bounds in the framework's leaf order."""
    if case["call"] == "adaptive":
        return np.array(_flat(_front(case)))
    d = 3 if case["kind"] == "dtn3d" else 2
    lo, s = np.full((1, d), -1.0), 2.0
    corners = [(0, 0), (1, 0), (1, 1), (0, 1)]
    if d == 3:  # the four upper octants first
        corners = [c + (1,) for c in corners] + [c + (0,) for c in corners]
    for _ in range(case["L"]):
        s /= 2
        lo = (lo[:, None, :] + s * np.array(corners, dtype=float)[None]).reshape(-1, d)
    return np.stack([lo, lo + s], -1).reshape(-1, 2 * d)


def _grid_order(p, d):
    """Index triples (pairs) of a leaf's Chebyshev points in the framework's order: the boundary first."""
    if d == 2:
        e = p - 1
        b = [(i, 0) for i in range(p)] + [(e, j) for j in range(1, p)]
        b += [(i, e) for i in range(p - 2, -1, -1)] + [(0, j) for j in range(p - 2, 0, -1)]
        return np.array(b + [(i, j) for i in range(1, e) for j in range(p - 2, 0, -1)])
    g = np.stack(np.meshgrid(*[np.arange(p)] * 3, indexing="ij"), -1).reshape(-1, 3)
    key = np.full(len(g), 6)
    for axis in (2, 1, 0):  # a point on several faces belongs to the first one in x, y, z order
        key[g[:, axis] == p - 1] = 2 * axis + 1
        key[g[:, axis] == 0] = 2 * axis
    return g[np.argsort(key, kind="stable")]


def _points(case):
    """(n_leaves, p^d, d) Chebyshev points of every leaf."""
    box, p = _boxes(case), case["p"]
    d = box.shape[1] // 2
    c = -np.cos(np.pi * np.arange(p) / (p - 1))
    idx = _grid_order(p, d)
    ax = [0.5 * (box[:, 2 * a + 1] - box[:, 2 * a])[:, None] * c + 0.5 * (box[:, 2 * a + 1] + box[:, 2 * a])[:, None]
          for a in range(d)]
    return np.stack([ax[a][:, idx[:, a]] for a in range(d)], -1)


@functools.lru_cache(maxsize=3)
def _domain(call, kind, p, L):
    """A program keeps one Domain for all its problems on that tree."""
    if kind == "dtn3d":
        return jh.Domain(p=p, q=p - 2, root=jh.DiscretizationNode3D(-1.0, 1.0, -1.0, 1.0, -1.0, 1.0), L=L)
    if call != "adaptive":
        return jh.Domain(p=p, q=p - 2, root=jh.DiscretizationNode2D(-1.0, 1.0, -1.0, 1.0), L=L)

    def node(tree, x0, x1, y0, y1, depth):
        if isinstance(tree, tuple):
            return jh.DiscretizationNode2D(x0, x1, y0, y1, depth=depth)
        xm, ym = (x0 + x1) / 2, (y0 + y1) / 2
        quads = [(x0, xm, y0, ym), (xm, x1, y0, ym), (xm, x1, ym, y1), (x0, xm, ym, y1)]
        kids = tuple(node(t, *b, depth + 1) for t, b in zip(tree, quads))
        return jh.DiscretizationNode2D(x0, x1, y0, y1, depth=depth, children=kids)
    return jh.Domain(p=p, q=p - 2, root=node(_front(dict(L=L)), -1.0, 1.0, -1.0, 1.0, 0))


# -- solutions and coefficients, the same on numpy arrays and torch tensors ---------------------
def _rng(seed, what):
    return np.random.default_rng([seed, what])


def _wavenumber(case):
    """The largest wavenumber that the Gauss points of a leaf side resolve to rounding."""
    q = case["p"] - 2
    half = 2.0 ** -case["L"]
    return (1e-15 * 2.0 ** (q - 1) * math.factorial(q)) ** (1.0 / q) / half


def _waves(case, seed):
    """Directions of the incident plane waves, one for each source."""
    a = _rng(seed, 1).uniform(0.0, 2 * math.pi, case["nsrc"])
    return np.stack([np.cos(a), np.sin(a)])


def _wave(case, seed, x):
    d = torch.as_tensor(_waves(case, seed)).to(x.device)
    return torch.exp(1j * _wavenumber(case) * (x @ d))


def _poly(case, seed, x):
    """Random polynomials (one for each source) and their first and second derivatives:
    values u, [du/dx_a], [d2u/dx_a2]."""
    d = x.shape[-1]
    deg = min(case["p"] - 3, 5)
    exps = [e for e in np.ndindex(*[deg + 1] * d) if sum(e) <= deg]
    co = torch.as_tensor(_rng(seed, 2).uniform(-1.0, 1.0, (len(exps), case["nsrc"]))).to(x.device)
    pw = [[torch.ones_like(x[..., 0])] for _ in range(d)]
    for a in range(d):
        for _ in range(deg):
            pw[a].append(pw[a][-1] * x[..., a])

    def term(e, der):
        t = 1.0
        for a in range(d):
            t = t * math.perm(e[a], der[a]) * pw[a][e[a] - der[a]]
        return t

    def total(der):
        out = torch.zeros(x.shape[:-1] + (case["nsrc"],), dtype=x.dtype, device=x.device)
        for i, e in enumerate(exps):
            if all(e[a] >= der[a] for a in range(d)):
                out += term(e, der)[..., None] * co[i]
        return out

    unit = np.eye(d, dtype=int).tolist()
    return (total([0] * d), [total(unit[a]) for a in range(d)],
            [total([2 * v for v in unit[a]]) for a in range(d)])


def _bumps(x, n, widths, amps, rng):
    """A sum of n Gaussian bumps and its gradient."""
    d = x.shape[-1]
    val, grad = torch.zeros_like(x[..., 0]), torch.zeros_like(x)
    for _ in range(n):
        c = torch.as_tensor(rng.uniform(-0.8, 0.8, d)).to(x.device)
        w, a = rng.uniform(*widths), rng.uniform(*amps)
        e = a * torch.exp(-((x - c) ** 2).sum(-1) / w**2)
        val += e
        grad += (-2.0 / w**2) * e[..., None] * (x - c)
    return val, grad


def _problem(case, seed):
    """Domain, PDEProblem keywords and boundary data, all in HBM."""
    dom = _domain(case["call"], case["kind"], case["p"], case["L"])
    x = torch.as_tensor(dom.interior_points).to(DEV)
    b = torch.as_tensor(dom.boundary_points).to(DEV)
    rng = _rng(seed, 3)
    d = x.shape[-1]
    one = case["nsrc"] == 1
    cut = (lambda t: t[..., 0].contiguous()) if one else (lambda t: t.contiguous())
    ones = torch.ones_like(x[..., 0])
    if case["kind"] == "iti2d":
        k = _wavenumber(case)
        h = 2.0 ** (1 - case["L"])
        con, _ = _bumps(x, 20, (max(0.02, 2 * h), max(0.05, 4 * h)), (0.5, 1.5), rng)
        src = -(k**2) * con[..., None] * _wave(case, seed, x)
        dirs = torch.as_tensor(_waves(case, seed)).to(DEV)
        n4 = b.shape[0] // 4
        nrm = torch.tensor([[0.0, -1.0], [1.0, 0.0], [0.0, 1.0], [-1.0, 0.0]], dtype=torch.float64, device=DEV)
        dn = nrm.repeat_interleave(n4, 0) @ dirs
        g = 1j * k * (dn + 1.0) * _wave(case, seed, b)
        return dom, dict(D_xx_coefficients=ones, D_yy_coefficients=ones, I_coefficients=k**2 * (1.0 - con),
                         source=cut(src), use_ItI=True, eta=k), cut(g)
    u, du, d2u = _poly(case, seed, x)
    names = ["D_xx", "D_yy", "D_zz"][:d]
    if case["terms"] == "laplace":
        kw = {f"{nm}_coefficients": -ones for nm in names}
        f = -sum(d2u)
    else:
        wid = (0.05, 0.2) if d == 2 else (0.1, 0.3)
        a, ga = _bumps(x, 8 if d == 2 else 6, wid, (0.5, 0.5), rng)
        a = a + 1.0
        kw = {f"{nm}_coefficients": -a for nm in names}
        for i, nm in enumerate(["D_x", "D_y", "D_z"][:d]):
            kw[f"{nm}_coefficients"] = -ga[..., i].contiguous()
        f = -(a[..., None] * sum(d2u)) - sum(ga[..., i, None] * du[i] for i in range(d))
        if d == 2:
            c, _ = _bumps(x, 4, (0.2, 0.6), (0.25, 0.25), rng)
            kw["I_coefficients"] = c
            f = f + c[..., None] * u
    g = _poly(case, seed, b)[0]
    return dom, dict(kw, source=cut(f)), cut(g)


# -- the cases ----------------------------------------------------------------------------------
def prepare(case, seed):
    dom, kw, g = _problem(case, seed)
    src = kw["source"]
    if case["call"] == "source":
        kw["source"] = None
    field = kw.get("I_coefficients")
    pde = jh.PDEProblem(dom, **kw)
    state = dict(call=case["call"], precision=case["precision"], pde=pde, g=g, source=src)
    if case["call"] in ("solve", "source"):
        jh.build_solver(pde, precision=case["precision"])
    if case["call"] == "gradient":
        state["field"] = field
        state["seen"] = 0.9 * _wave(case, seed, torch.as_tensor(dom.interior_points).to(DEV))[..., 0]
    return state


def run(state):
    pde, g, call = state["pde"], state["g"], state["call"]
    if call in ("build_solve", "adaptive"):
        jh.build_solver(pde, precision=state["precision"])
        return jh.solve(pde, g)
    if call == "solve":
        return jh.solve(pde, g)
    if call == "source":
        return jh.solve(pde, g, source=state["source"])
    field = state["field"].clone().requires_grad_(True)
    u = differentiable_solve(pde, g, I=field)
    loss = ((u - state["seen"]).abs() ** 2).sum()
    (grad,) = torch.autograd.grad(loss, field)
    return [u.detach(), grad]


def _merges(case):
    """[(merges, child side or face unknowns)] from the leaves' parents to the root."""
    q, L = case["p"] - 2, case["L"]
    if case["kind"] == "dtn3d":
        return [(8 ** (L - 1 - i), q * q * 4**i) for i in range(L)]
    return [(4 ** (L - 1 - i), q * 2**i) for i in range(L)]


def work(case):
    """Arithmetic of the elimination with its block zeros left out (real operations, complex ones
    four times), bytes of the inputs, of the solution and, where a built solver is applied, of its
    stored matrices."""
    p, s, cplx = case["p"], case["nsrc"], case["kind"] == "iti2d"
    q, d = p - 2, 3 if case["kind"] == "dtn3d" else 2
    n, ni = p**d, (p - 2) ** d
    nb, nq = n - ni, (4 * q if d == 2 else 6 * q * q)
    nl = len(_boxes(case))
    e = 16 if cplx else 8
    nco = {"laplace": d, "full": 6 if d == 3 else 5, "helmholtz": 3}[case["terms"]]
    merges = _merges(case) if case["call"] != "adaptive" else [(nl // 3, q)]
    leaf = 2 / 3 * ni**3 + 2 * ni**2 * (nb + s) + 2 * nq * ni * nb
    if cplx:
        # the interior block of a Helmholtz leaf is real; the impedance rows' complement is complex
        leaf += 2 * nb * ni * nb + 4 * (2 / 3 * nb**3 + 2 * nb**2 * nq + 2 * nq * nb * nq) + 4 * ni * nb * nq
        tree = sum(c * 4 * 874.7 * m**3 for c, m in merges)
    else:
        leaf += 2 * ni * nb * nq + 2 * nq * nb * nq
        # 2D: interfaces 5, 7 (and 3D: the x faces, then the y faces) do not couple to one another
        tree = sum(c * (470.0 if d == 2 else 7152.0) * m**3 for c, m in merges)
        if case["call"] != "adaptive":  # the root's own map is not formed
            tree -= (256.0 if d == 2 else 3456.0) * merges[-1][1] ** 3
    if cplx:
        tree -= 4 * 256.0 * merges[-1][1] ** 3
    vec = e * s * nl * n
    once = 8 * nco * nl * n + 2 * vec
    S = sum(c * m * m * ((8 * 8 if cplx else 4 * 8) if d == 2 else 12 * 24) for c, m in merges)
    down = e * (nl * n * nq + S) * (1 if case["precision"] == "fp64" else 0.5)
    if case["call"] == "solve":
        return {"bytes": down + 2 * vec, "flops": down / e * 2 * s * (4 if cplx else 1)}
    if case["call"] == "source":
        # besides the down pass: the leaves' factors, the interface factors, D12 and D21's nonzero halves, B's quarter
        up = 8 * nl * ni * (ni + nb) + e * sum(c * m * m * (16 + 8 + 8 + 16) for c, m in merges)
        return {"bytes": down + up + 3 * vec, "flops": (down + up) / e * 8 * s}
    if case["call"] == "gradient":
        return {"bytes": once + 3 * vec, "flops": nl * leaf + tree}
    return {"bytes": once, "flops": nl * leaf + tree}


def tolerance(case):
    """About four times the distance to exact(), which is the condition number's share: 3e-12 on
    the largest uniform trees, 8e-9 where the refined tree's interpolations are ill-conditioned
    (p = 16), and in mixed precision the refinement's own stopping tolerance of 1e-11."""
    if case["call"] == "adaptive":
        return {"rel": 4e-8 if case["p"] > 12 else 4e-10}
    return {"rel": 1e-10 if case["precision"] == "mixed" else 2e-11}


def exact(case, seed):
    """The solutions in closed form; the gradient has none."""
    x = torch.as_tensor(_points(case))
    u = _wave(case, seed, x) if case["kind"] == "iti2d" else _poly(case, seed, x)[0]
    u = u[..., 0] if case["nsrc"] == 1 else u
    return [u, None] if case["call"] == "gradient" else u
