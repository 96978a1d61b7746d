"""The unpivoted panel kernel and the conjugate-transposed GEMV at the edges
of their tiles, against float64 / complex128 numpy."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float64, torch.float32, torch.complex128, torch.complex64]
EPS = {torch.float64: 2.0**-53, torch.float32: 2.0**-24, torch.complex128: 2.0**-53, torch.complex64: 2.0**-24}


def _children(m, nm, dtype, gpu, seed):
    ne = 4 * m
    rng = np.random.default_rng(seed)
    T = 2.0 * np.eye(ne) + 0.3 * rng.standard_normal((4 * nm, ne, ne)) / np.sqrt(ne)
    if dtype.is_complex:
        T = T + 0.3j * rng.standard_normal(T.shape) / np.sqrt(ne)
    return torch.as_tensor(T, device=gpu).to(dtype).contiguous()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,nm", [(2, 1), (8, 3), (9, 2), (25, 16), (49, 1)])
def test_unpivoted_panel_factors(gpu, dtype, m, nm):
    """Interface matrices of 8 .. 196 unknowns (whole and partial 32-column
    panels, partial row and U12 tiles): L U is the gathered matrix.  The error of
    an LU without exchanges is n eps |L| |U| entrywise."""
    from jaxhps_amd._stages import merge_level
    from jaxhps_amd._tables import quad_merge_tables

    print(f"unpivoted panel {dtype} m={m} nm={nm}", flush=True)
    T = _children(m, nm, dtype, gpu, m)
    tb = quad_merge_tables(m, "dtn")
    out = merge_level(T, None, tb, pivot=False)
    assert (out.info == 0).all()
    n = 4 * m
    Th = T.cpu().numpy().reshape(nm, 4, n, n)
    D = np.zeros((nm, n, n), dtype=complex)
    for i, re in enumerate(tb.int_rows):
        for j, ce in enumerate(tb.int_cols):
            for a in (0, 2):
                for b in (0, 2):
                    if re[a] == ce[b]:
                        D[:, i, j] += Th[:, re[a], re[a + 1], ce[b + 1]]
    F = out.F_lu.cpu().numpy().astype(complex)
    Lo, Up = np.tril(F, -1) + np.eye(n), np.triu(F)
    bound = 4 * (n + 8) * EPS[dtype] * (np.abs(Lo) @ np.abs(Up))  # 4: complex products
    assert (np.abs(Lo @ Up - D) <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float64, torch.complex64])
@pytest.mark.parametrize("row", [0, 31, 32, 99])
def test_unpivoted_panel_rejects(gpu, dtype, row):
    """A zero row of the interface matrix (first, last of a panel, last of the
    matrix), or a NaN, marks its matrix alone with info = -1."""
    from jaxhps_amd._stages import merge_level
    from jaxhps_amd._tables import quad_merge_tables

    print(f"unpivoted panel rejects {dtype} row {row}", flush=True)
    m, nm = 25, 4
    tb = quad_merge_tables(m, "dtn")
    c0, l0, c1, l1 = (int(v) for v in tb.int_rows[row])
    for value in (0.0, float("nan")):
        T = _children(m, nm, dtype, gpu, row)
        T[4 * 2 + c0, l0, :] = value
        T[4 * 2 + c1, l1, :] = value
        info = merge_level(T, None, tb, pivot=False).info.cpu().numpy()
        assert info[2] == -1 and (np.delete(info, 2) == 0).all(), info


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nm", [4, 128])
def test_last_pivot_is_checked(gpu, dtype, nm):
    """The last pivot has no multipliers below it: not finite, subnormal or so
    large that its reciprocal is subnormal, it marks its matrix alone, in the
    panels for few matrices and in those for many."""
    from jaxhps_amd._stages import merge_level
    from jaxhps_amd._tables import quad_merge_tables

    tb = quad_merge_tables(25, "dtn")
    c0, l0, c1, l1 = (int(v) for v in tb.int_rows[-1])
    fi = torch.finfo(dtype)
    base = _children(25, nm, dtype, gpu, 1)
    for value in (float("nan"), float("inf"), fi.tiny / 4, fi.max / 8):
        print(f"last pivot {dtype} nm={nm} {value}", flush=True)
        T = base.clone()
        for c, l in ((c0, l0), (c1, l1)):
            T[4 * 2 + c, l, :] = 0.0
            T[4 * 2 + c, l, l] = value
        info = merge_level(T, None, tb, pivot=False).info.cpu().numpy()
        assert info[2] == -1 and (np.delete(info, 2) == 0).all(), (value, info)


def _natural_lu(A):
    """L and U of A without row exchanges (numpy)."""
    A = A.copy()
    for k in range(len(A) - 1):
        A[k + 1:, k] /= A[k, k]
        A[k + 1:, k + 1:] -= np.outer(A[k + 1:, k], A[k, k + 1:])
    return np.tril(A, -1), np.triu(A)


def _entries(tb, i, j):
    """The children's entries (child, row, column) that make D[i, j]."""
    r, c = tb.int_rows[i], tb.int_cols[j]
    return [(int(r[a]), int(r[a + 1]), int(c[b + 1])) for a in (0, 2) for b in (0, 2) if r[a] == c[b]]


# D[row, col] gets the large multiplier, outside every diagonal block
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.complex128])
@pytest.mark.parametrize("kind,m,nm,row,col", [
    ("quad", 40, 3, 150, 3),      # dense, 32 + 128 unknowns: the panel copied back
    ("quad", 25, 1024, 99, 2),    # many matrices, 36 + 64: in place, panel_check_kernel
    ("quad", 50, 3, 101, 60),     # dissected, one 50-wide block a group: later rows of group 1, in place
    ("quad", 70, 3, 279, 75),     # 70-wide blocks: later rows of group 1, copied back
    ("quad", 150, 2, 299, 155),   # 22 + 128 a group: rows of group 1 itself
    ("oct", 50, 2, 520, 160),     # group 3 of the x-interfaces, rows of a z-interface
    ("oct", 70, 1, 459, 430),     # the second slab's y-interfaces (12 + 128)
])
def test_multipliers_outside_the_diagonal_blocks_are_checked(gpu, dtype, kind, m, nm, row, col):
    """A multiplier above 64 in L21 alone marks its matrix, and no other, with
    info = -1: every diagonal block of the bad matrix factors well."""
    from jaxhps_amd._stages import merge_level
    from jaxhps_amd._tables import oct_merge_tables, quad_merge_tables

    print(f"multipliers outside {kind} m={m} nm={nm} D[{row}, {col}] {dtype}", flush=True)
    tb = oct_merge_tables(m) if kind == "oct" else quad_merge_tables(m, "dtn")
    g = torch.Generator(device=gpu).manual_seed(m)
    T = torch.randn(tb.nc * nm, tb.nec, tb.nec, generator=g, device=gpu, dtype=torch.float64).to(dtype)
    T = 0.1 * T / tb.nec**0.5 + 2.0 * torch.eye(tb.nec, device=gpu, dtype=dtype)
    bad = nm - 1
    assert (merge_level(T, None, tb, pivot=False).info == 0).all()
    # row `col` of D keeps its diagonal entry alone, so that eliminating it spreads nothing
    for j in range(tb.ni):
        for c, lr, lc in _entries(tb, col, j):
            if j != col:
                T[tb.nc * bad + c, lr, lc] = 0.0
    c, lr, lc = _entries(tb, row, col)[0]
    T[tb.nc * bad + c, lr, lc] = 1000.0
    # the oracle: of all multipliers that one alone passes the bound
    Tb = T[tb.nc * bad:].cpu().numpy().astype(complex)
    D = np.zeros((tb.ni, tb.ni), dtype=complex)
    for i in range(tb.ni):
        for a in (0, 2):
            for b in (0, 2):
                hit = tb.int_cols[:, b] == tb.int_rows[i, a]
                D[i, hit] += Tb[tb.int_rows[i, a], tb.int_rows[i, a + 1], tb.int_cols[hit, b + 1]]
    L, _ = _natural_lu(D)
    assert [tuple(x) for x in np.argwhere(np.abs(L) > 32)] == [(row, col)]
    info = merge_level(T, None, tb, pivot=False).info.cpu().numpy()
    assert info[bad] == -1 and (np.delete(info, bad) == 0).all(), info


@pytest.mark.parametrize("kind,m,nm,dtype", [
    ("quad", 47, 2, torch.float64), ("quad", 48, 3, torch.float32), ("quad", 65, 2, torch.complex128),
    ("quad", 129, 1, torch.float64), ("quad", 20, 40, torch.complex64), ("oct", 47, 1, torch.float64),
    ("oct", 49, 2, torch.float64), ("oct", 64, 1, torch.float32), ("iti", 65, 3, torch.complex128),
    ("iti", 20, 30, torch.complex64), ("quad", 17, 1024, torch.float64), ("quad", 36, 1024, torch.float32),
    ("iti", 21, 1024, torch.complex64)])
def test_block_elimination_matches_pivoted(gpu, kind, m, nm, dtype):
    """Natural-order block elimination (dense below 48 unknowns an interface,
    dissected from there; partial blocks, many and few matrices, first blocks of
    1, 2, 20, 68 and 80 unknowns) against the pivoted merge.  The matrices' condition is below 10, so both are within
    10 n eps of the exact result in the maximum norm."""
    from jaxhps_amd._stages import merge_level, up_level
    from jaxhps_amd._tables import oct_merge_tables, quad_merge_tables

    print(f"block elimination {kind} m={m} nm={nm} {dtype}", flush=True)
    tb = oct_merge_tables(m) if kind == "oct" else quad_merge_tables(m, "iti" if kind == "iti" else "dtn")
    g = torch.Generator(device=gpu).manual_seed(m)
    real = torch.float64

    def rand(*shape):
        x = torch.randn(shape, generator=g, device=gpu, dtype=real)
        return torch.complex(x, torch.randn(shape, generator=g, device=gpu, dtype=real)) if dtype.is_complex else x

    T = 0.1 * rand(tb.nc * nm, tb.nec, tb.nec) / tb.nec**0.5
    T = (T + (0.0 if kind == "iti" else 2.0) * torch.eye(tb.nec, device=gpu, dtype=T.dtype)).to(dtype).contiguous()
    h = rand(tb.nc * nm, tb.nec, 3).to(dtype).contiguous()
    nat = merge_level(T, h, tb, keep_factors=True, pivot=False)
    piv = merge_level(T, h, tb, keep_factors=True, pivot=True)
    assert (nat.info == 0).all()
    bound = 2 * 10 * tb.ni * EPS[dtype]
    for name in ("S", "T", "h", "gt"):
        a, b = getattr(nat, name), getattr(piv, name)
        assert float((a - b).abs().max() / b.abs().max()) < bound, name
    # the stored factors serve the up pass: the same data give the same result
    gt, ho = up_level(h, nat)
    assert float((gt - piv.gt).abs().max() / piv.gt.abs().max()) < bound
    assert float((ho - piv.h).abs().max() / piv.h.abs().max()) < bound


@pytest.mark.parametrize("pivot", [True, False])
def test_merge_without_row_map(gpu, pivot):
    """DtN merges whose internal order is the final one (adaptive trees): the
    rows of S and g_tilde come in internal order, T and h are the mapped
    merge's, and the solution goes straight to the output."""
    import copy

    from jaxhps_amd import profiling
    from jaxhps_amd._stages import merge_level
    from jaxhps_amd._tables import quad_merge_tables

    print(f"merge without row map pivot={pivot}", flush=True)
    tb = quad_merge_tables(37, "dtn")
    plain = copy.copy(tb)
    plain.cols_final, plain.upd = tb.int_cols, np.zeros((0, 4), dtype=np.int32)
    plain.reordered, plain.dissect, plain._dev = False, 0, {}
    T = _children(37, 3, torch.float64, gpu, 5)
    h = torch.randn(12, tb.nec, 2, device=gpu, dtype=torch.float64)
    mapped = merge_level(T, h, tb, pivot=pivot)
    out, kernels, _ = profiling.instrumented(lambda: merge_level(T, h, plain, pivot=pivot))
    names = [r["name"] for r in kernels]
    assert 0 < len(names) < 12  # the list holds at most 12
    assert not any("row_scatter" in nm for nm in names), names
    fin = torch.as_tensor(tb.final_of_internal, device=gpu).long()
    bound = 4 * tb.ni * EPS[torch.float64]
    for nm in ("S", "gt", "T", "h"):
        a, b = getattr(out, nm), getattr(mapped, nm)
        b = b[:, fin] if nm in ("S", "gt") else b
        assert float((a - b).abs().max() / b.abs().max()) < bound, nm


def test_merge_beyond_32_bit_indices(gpu):
    """A 3D merge whose S has more than 2^31 elements (32784 x 65568).  Columns
    of S put back into the children: the outgoing data of the two sides of
    every interface cancel, to n eps of the terms' sum."""
    from jaxhps_amd._stages import merge_level
    from jaxhps_amd._tables import oct_merge_tables

    if torch.cuda.mem_get_info(gpu)[0] < 64 << 30:
        pytest.skip("needs 64 GB of device memory")
    print("merge beyond 32-bit indices", flush=True)
    tb = oct_merge_tables(2732)
    assert tb.ni * tb.ne > 2**31
    g = torch.Generator(device=gpu).manual_seed(1)
    T = torch.randn(8, tb.nec, tb.nec, generator=g, device=gpu, dtype=torch.float32).mul_(0.1 / tb.nec**0.5)
    T.diagonal(dim1=1, dim2=2).add_(2.0)
    out = merge_level(T, None, tb, want_T=False, pivot=False)
    assert int(out.info[0]) == 0
    cols = torch.tensor([0, tb.ne // 2, tb.ne - 1], device=gpu)
    S = out.S[0][:, cols].double()
    del out
    src = torch.as_tensor(tb.child_src, device=gpu).long().reshape(-1)
    data = torch.where((src >= 0)[:, None], (src[:, None] == cols[None]).double(), S[(-src - 1).clamp(min=0)])
    data = data.reshape(8, tb.nec, -1)
    flux = torch.stack([T[c].double() @ data[c] for c in range(8)])
    size = torch.stack([T[c].double().abs() @ data[c].abs() for c in range(8)])
    c0, l0, c1, l1 = torch.as_tensor(tb.int_rows, device=gpu).long().T
    res = (flux[c0, l0] + flux[c1, l1]).abs() / (size[c0, l0] + size[c1, l1])
    assert float(res.max()) < tb.ni * EPS[torch.float32]


def test_merges_from_several_threads(gpu):
    """Merges with different eliminations (dissected 2D and 3D, dense ItI,
    pivoted) from four threads on one stream: each thread's factorisation
    switches are its own, so every result is the one it has alone."""
    import threading

    from jaxhps_amd._stages import merge_level
    from jaxhps_amd._tables import oct_merge_tables, quad_merge_tables

    print("merges from several threads", flush=True)
    jobs = []
    for tb, nm, pivot in ((quad_merge_tables(60, "dtn"), 3, False), (oct_merge_tables(49), 1, False),
                          (quad_merge_tables(20, "iti"), 8, False), (quad_merge_tables(60, "dtn"), 3, True)):
        g = torch.Generator(device=gpu).manual_seed(tb.nec)
        T = 0.1 * torch.randn(tb.nc * nm, tb.nec, tb.nec, generator=g, device=gpu, dtype=torch.float64) / tb.nec**0.5
        if tb.kind == "iti":
            T = T.to(torch.complex128)
        else:
            T = T + 2.0 * torch.eye(tb.nec, device=gpu, dtype=T.dtype)
        jobs.append((T.contiguous(), tb, pivot))
    alone = [merge_level(T, None, tb, pivot=pivot) for T, tb, pivot in jobs]
    torch.cuda.synchronize()
    wrong, start = [], threading.Barrier(len(jobs), timeout=60)

    def work(i):
        T, tb, pivot = jobs[i]
        start.wait()
        try:
            for _ in range(20):
                r = merge_level(T, None, tb, pivot=pivot)
                if not (torch.equal(r.S, alone[i].S) and torch.equal(r.T, alone[i].T)):
                    wrong.append(i)
        except Exception as e:  # reported by the assertion below
            wrong.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong


@pytest.mark.parametrize("p,L,k", [(12, 3, 20.0), (16, 3, 20.0), (8, 3, 12.0), (16, 2, 12.0)])
def test_indefinite_dtn_problems_keep_their_precision(gpu, monkeypatch, p, L, k):
    """DtN Helmholtz problems past the leaves' first eigenvalues, whose natural
    order elimination grows: the solution's distance to the exact discrete one
    is that of pivoting everywhere (5: the largest ratio that multipliers up to
    the bound showed is 3.3; 60 and 100 without it in the first two cases)."""
    import config_oracle as co
    import jaxhps_amd as jh
    from jaxhps_amd import _build_solver, _lib
    from jaxhps_amd.merge import _levels

    print(f"indefinite DtN p={p} L={L} k={k}", flush=True)
    dom = jh.Domain(p=p, q=p - 2, root=jh.DiscretizationNode2D(-1.0, 1.0, -1.0, 1.0), L=L)
    x = dom.interior_points
    rng = np.random.default_rng(3)
    con = 0.2 * np.exp(-((x - np.array([0.2, -0.1])) ** 2).sum(-1) / 0.09)
    one = np.ones(x.shape[:2])
    kw = dict(D_xx_coefficients=one, D_yy_coefficients=one, I_coefficients=k * k * (1 - con),
              source=rng.standard_normal(x.shape[:2]))
    g = rng.standard_normal(dom.boundary_points.shape[0])
    exact = co.exact_solution(dom, kw, g)

    def error():
        pde = jh.PDEProblem(dom, **kw)
        jh.build_solver(pde)
        return co.rel2(jh.solve(pde, g).cpu().numpy(), exact)

    natural = error()
    lib = _lib.load_library()

    class Pivoting:
        """The library with the leaves' switch left at partial pivoting."""

        def __getattr__(self, name):
            return (lambda h, v: 0) if name == "hps_set_leaf_pivoting" else getattr(lib, name)

    monkeypatch.setattr(_lib, "_lib", Pivoting())
    monkeypatch.setattr(_build_solver, "_levels", lambda *a, **kwargs: _levels(*a, **dict(kwargs, pivot=True)))
    assert natural <= 5 * error()


def _iti_leaves(gpu, p, L, k2, imag=0.0, extra=None):
    """An ItI problem with smooth coefficients on 4^L leaves (extra(x): a further
    zeroth-order term), and its leaf matrices B = [G; A_int] (complex128, numpy)
    for chosen leaves."""
    import jaxhps_amd as jh

    dom = jh.Domain(p=p, q=p - 2, root=jh.DiscretizationNode2D(-1.0, 1.0, -1.0, 1.0), L=L)
    x = dom.interior_points
    cf = {"D_xx": 1.0 + 0.2 * np.sin(x[..., 0]), "D_yy": 1.0 + 0.1 * x[..., 1], "D_x": 0.3 * x[..., 1],
          "I": k2 * (1.0 + 0.3 * np.cos(x[..., 0] + x[..., 1])) + 1j * imag}
    if extra is not None:
        cf["I"] = cf["I"] + extra(x)
    if imag == 0.0:
        cf["I"] = cf["I"].real
    pde = jh.PDEProblem(dom, use_ItI=True, eta=3.0, **{f"{n}_coefficients": a for n, a in cf.items()})
    nb = np.asarray(pde.P).shape[0]

    def matrix(leaf):
        A = sum(cf[nm][leaf][:, None]
                * (np.eye(p * p) if nm == "I" else np.asarray(getattr(pde, nm))) for nm, _ in pde.coefficient_list())
        return np.concatenate([np.asarray(pde.G), A[nb:]]).astype(complex)

    return pde, nb, matrix


@pytest.mark.parametrize("p,L,nsrc,dtype", [
    (5, 1, 0, torch.complex128), (8, 2, 1, torch.complex128), (16, 1, 3, torch.complex128), (9, 2, 2, torch.complex64),
    (10, 5, 1, torch.complex64), (11, 5, 3, torch.complex128), (14, 5, 1, torch.complex128)])
def test_condensed_leaves(gpu, p, L, nsrc, dtype):
    """Y, T, v, h and the kept factors' B^{-1} and B^{-H} of condensed leaves
    (one and several blocks, few and many leaves) against numpy solves with B.
    An eliminated system's error is within n eps cond, the impedance rows
    brought to the others' size first (a power of ten below B's condition)."""
    from jaxhps_amd._stages import HPS_KIND_ITI, leaf_apply_inverse, leaf_solve
    from jaxhps_amd.adjoint import _condensed_inverse_conjt

    print(f"condensed leaves p={p} L={L} nsrc={nsrc} {dtype}", flush=True)
    pde, nb, matrix = _iti_leaves(gpu, p, L, 4.0)
    nl, n = 4**L, p * p
    g = torch.Generator(device=gpu).manual_seed(p)
    f = torch.randn(nl, n, max(nsrc, 1), generator=g, device=gpu, dtype=dtype)
    res = leaf_solve(pde, HPS_KIND_ITI, dtype, gpu, source=f if nsrc else None, nsrc_zero=nsrc == 0)
    assert res.condensed is not None
    inv, invh = leaf_apply_inverse(res, f), _condensed_inverse_conjt(res, f)
    P, QH = np.asarray(pde.P), np.asarray(pde.QH)
    for leaf in {0, nl // 2 + 1, nl - 1}:
        B = matrix(leaf)
        scale = np.ones(n)
        scale[:nb] = np.abs(B[nb:]).max() / np.abs(B[:nb]).max()
        bound = n * EPS[dtype] * np.linalg.cond(scale[:, None] * B)
        fl = f[leaf].cpu().numpy().astype(complex)
        fi = fl.copy()
        fi[:nb] = 0.0
        rhs = np.zeros((n, P.shape[1]), dtype=complex)
        rhs[:nb] = P
        ref = {"Y": np.linalg.solve(B, rhs), "inv": np.linalg.solve(B, fl),
               "invh": np.linalg.solve(B.conj().T, fl)}
        ref["T"] = QH @ ref["Y"]
        got = {"Y": res.Y, "T": res.T, "inv": inv, "invh": invh}
        if nsrc:
            ref["v"] = np.linalg.solve(B, fi)
            ref["h"] = QH @ ref["v"]
            got.update(v=res.v, h=res.h)
        for nm, r in ref.items():
            # T and h: the error of Y and v through QH
            size = {"T": np.abs(QH).sum(1).max() * np.abs(ref["Y"]).max(),
                    "h": np.abs(QH).sum(1).max() * np.abs(ref.get("v", 0.0)).max()}.get(nm, np.abs(r).max())
            err = np.abs(got[nm][leaf].cpu().numpy() - r).max() / size
            assert err <= bound, (nm, leaf, err, bound)


@pytest.mark.parametrize("found_by", ["estimate", "checks"])
@pytest.mark.parametrize("kh", [2.0, 4.2, 4.5, 5.0, 8.0])
def test_condensed_leaves_lose_no_precision(gpu, monkeypatch, kh, found_by):
    """T of 16 leaves below and past the first Dirichlet eigenvalue (k h = 4.44)
    is as close to long double as through the factorisation of B (complex
    coefficients), leaf by leaf and whichever way the leaves are chosen.  Without
    the choice the ratio is 15 at k h = 4.5.  2: the two differ by rounding."""
    import jaxhps_amd as jh
    from jaxhps_amd import _stages
    from jaxhps_amd._stages import HPS_KIND_ITI, leaf_solve

    print(f"condensed leaves' precision k h = {kh} {found_by}", flush=True)
    monkeypatch.setattr(_stages, "LEAF_REDO_MIN", 0)
    monkeypatch.setattr(_stages, "LEAF_REDO_SHARE", 1.0)
    if found_by == "checks":
        monkeypatch.setattr(_stages, "LEAF_DEFINITE", float("inf"))
    p, L, k = 11, 2, 2.0 * kh
    dom = jh.Domain(p=p, q=p - 2, root=jh.DiscretizationNode2D(-1.0, 1.0, -1.0, 1.0), L=L)
    x = dom.interior_points
    one = np.ones(x.shape[:2])
    field = k * k * (1.0 - 0.1 * np.exp(-(x**2).sum(-1)))
    T = []
    for I in (field, field.astype(complex)):
        pde = jh.PDEProblem(dom, D_xx_coefficients=one, D_yy_coefficients=one, I_coefficients=I, use_ItI=True, eta=k)
        res = leaf_solve(pde, HPS_KIND_ITI, torch.complex128, gpu, nsrc_zero=True)
        T.append(res.T.cpu().numpy())
        if len(T) == 1:
            assert kh > 4.0 or (res.condensed is not None and res.condensed.redone is None)
    G, QH, P = (np.asarray(a).astype(np.clongdouble) for a in (pde.G, pde.QH, pde.P))
    nb, err = P.shape[0], np.zeros(2)

    def solve(A, B):  # no exchanges: 11 more bits than the results carry
        A, B = A.copy(), B.copy()
        for j in range(len(A)):
            l = A[j + 1:, j] / A[j, j]
            A[j + 1:, j + 1:] -= np.outer(l, A[j, j + 1:])
            B[j + 1:] -= np.outer(l, B[j])
        for j in range(len(A) - 1, -1, -1):
            B[j] /= A[j, j]
            B[:j] -= np.outer(A[:j, j], B[j])
        return B

    for leaf in range(16):
        A = np.asarray(pde.D_xx) + np.asarray(pde.D_yy) + np.diag(field[leaf])
        A = A[nb:].astype(np.longdouble)
        X = solve(A[:, nb:], A[:, :nb])
        Yb = solve(G[:, :nb] - G[:, nb:] @ X, P)
        ref = QH[:, :nb] @ Yb - QH[:, nb:] @ (X @ Yb)
        err += [float((np.abs(t[leaf] - ref) ** 2).sum() / (np.abs(ref) ** 2).sum()) for t in T]
    assert err[0] <= 2.0**2 * err[1], np.sqrt(err / 16)


def test_definiteness_is_read_before_or_after_alike(gpu, monkeypatch):
    """The coefficients' estimate gives one result whether it is read before the
    condensed stage (eta as large as the wavenumber) or after it."""
    from jaxhps_amd import _stages
    from jaxhps_amd._stages import HPS_KIND_ITI, leaf_solve

    print("definiteness read before or after", flush=True)
    for k2_extra in (False, True):
        res = []
        for first in (0.0, float("inf")):
            monkeypatch.setattr(_stages, "LEAF_LOOK_FIRST", first)
            pde = (_resonant_leaf if k2_extra else lambda *a: _iti_leaves(*a, 2000.0))(gpu, 8, 4)[0]
            res.append(leaf_solve(pde, HPS_KIND_ITI, torch.complex128, gpu, nsrc_zero=True))
        assert (res[0].condensed is None) == (res[1].condensed is None) == (not k2_extra)
        assert torch.equal(res[0].Y, res[1].Y) and torch.equal(res[0].T, res[1].T)


def test_condensed_build_leaves_the_complex_operators_alone(gpu):
    """A build whose leaves are condensed uploads the real differentiation
    operators, not a complex set beside them (a problem object per coefficient
    field pays for each)."""
    import jaxhps_amd as jh

    print("condensed build's operators", flush=True)
    pde, _, _ = _iti_leaves(gpu, 8, 2, 4.0)
    jh.build_solver(pde)
    assert pde._factors["leaf"].condensed is not None
    assert not {"diffops", "G"} & set(pde.device_ops(gpu, torch.complex128))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,nl", [(9, 1), (256, 300), (400, 70000)])
def test_mark_indefinite(gpu, dtype, n, nl):
    """Leaves with a point above the limit, or a NaN, are marked, whichever
    point it is; other entries of info stay, with one second-order field or two."""
    from jaxhps_amd import _lib

    print(f"mark indefinite {dtype} n={n} nl={nl}", flush=True)
    lib, h = _lib.load_library(), _lib.handle()
    g = torch.Generator(device=gpu).manual_seed(n)
    z = 3.9 * torch.rand(nl, n, generator=g, device=gpu, dtype=dtype)
    xx, yy = torch.full_like(z, 0.5), torch.full_like(z, 1.5)
    want = torch.zeros(nl, dtype=torch.int32, device=gpu)
    for leaf, point, value in ((0, n - 1, 4.5), (nl // 2, 0, float("nan")), (nl - 1, n // 2, float("inf"))):
        z[leaf, point] = value
        want[leaf] = -1
    want[nl // 3] = 7 if want[nl // 3] == 0 else -1
    for fields, limit in (((xx, yy), 2.0), ((2 * xx, None), 4.0)):
        info = torch.zeros_like(want)
        info[nl // 3] = 7
        rc = lib.hps_mark_indefinite(h, _lib.dtype_code(dtype), nl, n, _lib.ptr(z), _lib.ptr(fields[0]),
                                     _lib.ptr(fields[1]), limit, _lib.ptr(info))
        _lib.check(rc, h, "hps_mark_indefinite")
        assert torch.equal(info, want)


def test_condensed_leaves_give_way(gpu):
    """Complex coefficients, and a leaf at an eigenvalue of its Dirichlet
    problem, take the factorisation of B; the results stay right."""
    from jaxhps_amd._stages import HPS_KIND_ITI, leaf_solve

    print("condensed leaves give way", flush=True)
    for imag, k2 in ((0.5, 4.0), (0.0, None)):
        if k2 is None:  # the constant part nearest an eigenvalue of leaf 0
            pde, nb, matrix = _iti_leaves(gpu, 8, 1, 0.0)
            x = pde.domain.interior_points[0, nb:]
            A, W = matrix(0)[nb:, nb:].real, 1.0 + 0.3 * np.cos(x[:, 0] + x[:, 1])
            w = np.linalg.eigvals(-A / W[:, None])
            k2 = float(w[np.abs(w.imag) < 1e-9].real.min())
        pde, nb, matrix = _iti_leaves(gpu, 8, 1, k2, imag)
        res = leaf_solve(pde, HPS_KIND_ITI, torch.complex128, gpu, nsrc_zero=True)
        assert res.condensed is None
        B = matrix(0)
        rhs = np.zeros((64, pde.P.shape[1]), dtype=complex)
        rhs[:nb] = np.asarray(pde.P)
        ref = np.linalg.solve(B, rhs)
        err = np.abs(res.Y[0].cpu().numpy() - ref).max() / np.abs(ref).max()
        assert err <= 64 * 2.0**-53 * np.linalg.cond(B), err


def _resonant_leaf(gpu, p, L):
    """_iti_leaves with a bump in the zeroth-order coefficient for which the
    interior problem of leaf 0, at its centre, is singular."""
    h = 2.0 ** (1 - L)

    def bump(x):
        return np.exp(-((x - (h / 2 - 1.0)) ** 2).sum(-1) / h**2)

    pde, nb, matrix = _iti_leaves(gpu, p, L, 4.0)
    w = np.linalg.eigvals(-matrix(0)[nb:, nb:].real / bump(pde.domain.interior_points[0, nb:])[:, None])
    top = float(w[np.abs(w.imag) < 1e-9].real.min())
    return _iti_leaves(gpu, p, L, 4.0, extra=lambda x: top * bump(x))


@pytest.mark.parametrize("found_by", ["estimate", "checks"])
@pytest.mark.parametrize("nsrc,dtype", [(0, torch.complex128), (2, torch.complex128), (1, torch.complex64)])
def test_indefinite_leaves_alone_are_redone(gpu, monkeypatch, nsrc, dtype, found_by):
    """Among 256 leaves the few whose interior problem is not definite, found
    from the coefficients or by the kernels' checks, are factored directly and
    the others stay condensed; Y, T, v, h, B^{-1} and B^{-H} of both kinds against
    numpy solves with B, to the bound of test_condensed_leaves."""
    from jaxhps_amd import _stages
    from jaxhps_amd._stages import HPS_KIND_ITI, leaf_apply_inverse, leaf_solve
    from jaxhps_amd.adjoint import _leaf_inverse_conjt

    print(f"indefinite leaves redone nsrc={nsrc} {dtype} {found_by}", flush=True)
    if found_by == "checks":
        monkeypatch.setattr(_stages, "LEAF_DEFINITE", float("inf"))
    pde, nb, matrix = _resonant_leaf(gpu, 8, 4)
    nl, n = 256, 64
    g = torch.Generator(device=gpu).manual_seed(3)
    f = torch.randn(nl, n, max(nsrc, 1), generator=g, device=gpu, dtype=dtype)
    res = leaf_solve(pde, HPS_KIND_ITI, dtype, gpu, source=f if nsrc else None, nsrc_zero=nsrc == 0)
    assert res.condensed is not None and res.condensed.redone is not None
    redone = res.condensed.redone[0].cpu().tolist()
    assert 0 in redone and len(redone) <= nl // 4 and (res.info == 0).all()
    inv, invh = leaf_apply_inverse(res, f), _leaf_inverse_conjt(res, f)
    assert bool(torch.isfinite(inv.abs()).all()) and bool(torch.isfinite(invh.abs()).all())
    P, QH = np.asarray(pde.P), np.asarray(pde.QH)
    kept = [leaf for leaf in range(nl) if leaf not in redone]
    for leaf in {0, redone[-1], kept[0], kept[-1]}:
        B = matrix(leaf)
        scale = np.ones(n)
        scale[:nb] = np.abs(B[nb:]).max() / np.abs(B[:nb]).max()
        bound = n * EPS[dtype] * np.linalg.cond(scale[:, None] * B)
        fl = f[leaf].cpu().numpy().astype(complex)
        fi = fl.copy()
        fi[:nb] = 0.0
        rhs = np.zeros((n, P.shape[1]), dtype=complex)
        rhs[:nb] = P
        ref = {"Y": np.linalg.solve(B, rhs), "inv": np.linalg.solve(B, fl), "invh": np.linalg.solve(B.conj().T, fl)}
        got = {"Y": res.Y, "inv": inv, "invh": invh}
        size = {nm: np.abs(r).max() for nm, r in ref.items()}
        pairs = [("T", "Y", res.T)]
        if nsrc:
            ref["v"], got["v"] = np.linalg.solve(B, fi), res.v
            size["v"] = np.abs(ref["v"]).max()
            pairs.append(("h", "v", res.h))
        for nm, of, t in pairs:  # the error of Y and v through QH
            ref[nm], got[nm], size[nm] = QH @ ref[of], t, np.abs(QH).sum(1).max() * size[of]
        for nm, r in ref.items():
            err = np.abs(got[nm][leaf].cpu().numpy() - r).max() / size[nm]
            assert err <= bound, (nm, leaf, err, bound)


def test_solves_with_indefinite_leaves(gpu):
    """Build + solve, a new source and a gradient where some leaves are not
    condensed, against the same problem with its coefficients given as complex
    numbers (every leaf factored directly).  Both solve one system whose
    condition is below 1e6."""
    import jaxhps_amd as jh
    from jaxhps_amd.adjoint import differentiable_solve

    print("solves with indefinite leaves", flush=True)
    pde, _, _ = _resonant_leaf(gpu, 8, 4)
    dom = pde.domain
    cf = {f"{nm}_coefficients": torch.as_tensor(a, device=gpu) for nm, a in pde.coefficient_list()}
    g = torch.Generator(device=gpu).manual_seed(4)
    src, src2 = (torch.randn(256, 64, generator=g, device=gpu, dtype=torch.complex128) for _ in range(2))
    bd = torch.randn(dom.boundary_points.shape[0], generator=g, device=gpu, dtype=torch.complex128)
    got = []
    for cast in (lambda t: t, lambda t: t.to(torch.complex128)):
        p1 = jh.PDEProblem(dom, source=src, use_ItI=True, eta=3.0, **{k: cast(a) for k, a in cf.items()})
        jh.build_solver(p1)
        c = p1._factors["leaf"].condensed
        assert (c is not None and c.redone is not None) == (len(got) == 0)
        out = [jh.solve(p1, bd)]
        p2 = jh.PDEProblem(dom, use_ItI=True, eta=3.0, **{k: cast(a) for k, a in cf.items()})
        jh.build_solver(p2)
        out.append(jh.solve(p2, bd, source=src2))
        if not got:
            field = cf["I_coefficients"].clone().requires_grad_(True)
            u = differentiable_solve(p1, bd, I=field)
            (grad,) = torch.autograd.grad((u.abs() ** 2).sum(), field)
        else:
            from jaxhps_amd.adjoint import adjoint_lambda, coefficient_gradients

            lam = adjoint_lambda(p1, 2.0 * out[0])
            grad = coefficient_gradients(p1, out[0], lam)["I"]
        got.append(out + [grad])
    for nm, a, b in zip(("solve", "source", "gradient"), *got):
        assert float((a - b).abs().max() / b.abs().max()) < 1e6 * 64 * 2.0**-53, nm


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batch,M,N,K", [(1, 1, 1, 1), (3, 17, 2, 63), (2, 64, 1, 64), (2, 65, 2, 257), (1, 300, 1, 5),
                                         (5, 33, 1, 1000)])
def test_conjt_gemv(gpu, dtype, batch, M, N, K):
    """A^H B + C for one and two columns: remainders of the column tiles and of
    the rows each slice walks; K eps |A|^T |B| bounds the sum's rounding."""
    from jaxhps_amd.adjoint import _gemm_conjt

    print(f"conjt gemv {dtype} {(batch, M, N, K)}", flush=True)
    rng = np.random.default_rng(M + K)

    def rand(*s):
        x = rng.standard_normal(s) + (1j * rng.standard_normal(s) if dtype.is_complex else 0)
        return torch.as_tensor(x).to(dtype)

    A, B, C = rand(batch, K, M), rand(batch, K, N), rand(batch, M, N)
    out = _gemm_conjt(A.to(gpu), M, K * M, M, K, B.to(gpu), N, K * N, N, batch, C=C.to(gpu), beta=1.0)
    a, b, c = (t.numpy().astype(complex) for t in (A, B, C))
    ref = a.conj().transpose(0, 2, 1) @ b + c
    bound = 4 * (K + 2) * EPS[dtype] * (np.abs(a).transpose(0, 2, 1) @ np.abs(b) + np.abs(c))
    assert (np.abs(out.cpu().numpy() - ref) <= bound).all()


@pytest.mark.parametrize("conjt", [False, True])
def test_gemm_wide_rows(gpu, conjt):
    """Rows so far apart that a tile's byte offsets pass 4 GiB (8.3 M float64
    elements) take the 64-bit offsets; against the packed product."""
    from jaxhps_amd import _lib

    print(f"gemm wide rows conjt={conjt}", flush=True)
    lib, h = _lib.load_library(), _lib.handle()
    M, N, K, ld = 70, 20, 40, 8_300_000
    rows, cols = (K, M) if conjt else (M, K)
    g = torch.Generator(device=gpu).manual_seed(3)
    A = torch.empty(rows * ld, dtype=torch.float64, device=gpu).as_strided((rows, cols), (ld, 1))
    A.normal_(generator=g)
    B = torch.randn(K, N, generator=g, dtype=torch.float64, device=gpu)
    out = torch.empty(M, N, dtype=torch.float64, device=gpu)
    fn = lib.hps_gemm_batched_conjt if conjt else lib.hps_gemm_batched
    rc = fn(h, _lib.dtype_code(A.dtype), M, N, K, 1.0, A.data_ptr(), ld, 0, _lib.ptr(B), N, 0, 0.0, None, N, 0,
            _lib.ptr(out), N, 0, 1)
    _lib.check(rc, h, "gemm")
    a = A.cpu().numpy()
    ref = (a.T if conjt else a) @ B.cpu().numpy()
    bound = 2 * K * 2.0**-53 * (np.abs(a.T if conjt else a) @ np.abs(B.cpu().numpy()))
    assert (np.abs(out.cpu().numpy() - ref) <= bound).all()
