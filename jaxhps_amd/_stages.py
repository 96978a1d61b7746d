"""Device-side stage drivers: one C-ABI call per leaf stage / tree level.

These are the only functions that talk to libhps_mi355x; the public stage
functions (named like the reference's) and build_solver/solve sit on top.
All arrays are torch tensors resident in HBM.
"""

from __future__ import annotations

import ctypes
from dataclasses import dataclass
from typing import List, Optional, Tuple

import numpy as np
import torch

from . import _lib
from ._lib import HPS_DISSECT_NONE, HPS_KIND_DTN, HPS_KIND_ITI, check, dtype_code, load_library, ptr, workspace
from ._tables import MergeTables


def default_device():
    _lib._require_gpu()
    return torch.device("cuda", torch.cuda.current_device())


def to_device(x, device, dtype):
    if x is None:
        return None
    if isinstance(x, torch.Tensor):
        t = x
    else:
        t = torch.as_tensor(np.asarray(x))
    if not t.is_complex() and dtype.is_complex:
        t = t.to(torch.float64)
    t = t.to(device=device, dtype=dtype).contiguous()
    # the kernels read the memory: a view that is conjugated or negated on read is written out
    return t.resolve_conj().resolve_neg() if t.is_conj() or t.is_neg() else t


def is_complex_input(*arrs) -> bool:
    for a in arrs:
        if a is None:
            continue
        if isinstance(a, torch.Tensor):
            if a.is_complex():
                return True
        elif np.iscomplexobj(a):
            return True
    return False


def real_dtype(dt):
    return {torch.complex128: torch.float64, torch.complex64: torch.float32}.get(dt, dt)


def complex_dtype(dt):
    return {torch.float64: torch.complex128, torch.float32: torch.complex64}.get(dt, dt)


@dataclass
class LeafResult:
    Y: Optional[torch.Tensor]
    T: Optional[torch.Tensor]
    v: Optional[torch.Tensor]
    h: Optional[torch.Tensor]
    lu: torch.Tensor
    perm: torch.Tensor
    dinv: torch.Tensor
    info: torch.Tensor
    kind: int
    # ItI: the factored matrix is diag(s I_nb, I) B -- the incoming-impedance
    # rows scaled by the power of two s (a 0-dim device tensor), see
    # iti_row_scale; 1 for DtN.
    row_scale: Optional[torch.Tensor] = None
    nb: int = 0
    condensed: Optional[Condensed] = None


@dataclass
class Condensed:
    """Interior factors of condensed ItI leaves (hps_leaf_condensed); the
    leaf's lu, perm and dinv then factor the boundary system."""
    alu: torch.Tensor   # (nl, ni, n) real: [A_ib | LU(A_ii)]
    perm: torch.Tensor
    dinv: torch.Tensor
    X: torch.Tensor     # (nl, ni, nb + 2 nsrc) real: A_ii^{-1} [A_ib | f_i]
    Gi: torch.Tensor    # (nb, ni) real: interior columns of G
    # leaves that rejected the condensation, and their factorisation of B
    redone: Optional[Tuple[torch.Tensor, LeafResult]] = None


def iti_row_scale(pde, coeffs, clist, device):
    """Power-of-two factor s for the impedance rows G of the ItI leaf matrix
    B = [G; A_int], as a 0-dim float64 device tensor.

    G's entries are O(p^2/h) while the collocation rows carry O((p^2/h)^2)
    differentiation entries, so B is badly row-scaled: at p = 16 its
    condition number is ~3e5, and ~6e3 once the G rows are brought to the
    size of the A rows.  Factoring diag(s, 1) B instead of B (with the same
    scaling of the right-hand side's G rows) leaves every solution unchanged
    and cuts the factorisation's rounding error about tenfold.  s estimates
    max|A_int| / max|G| from the coefficient maxima and the operators'
    maxima; a power of two keeps the scaling exact."""
    key = ("iti_row_scale_ops", tuple(nm for nm, _ in clist))
    opmax = pde._dev_cache.get(key)
    if opmax is None:
        opmax = [1.0 if nm == "I" else float(np.abs(np.asarray(getattr(pde, nm))).max()) for nm, _ in clist]
        gmax = float(np.abs(np.asarray(pde.G)).max())
        opmax = pde._dev_cache[key] = (torch.tensor(opmax, dtype=torch.float64, device=device), gmax)
    om, gmax = opmax
    cmax = torch.amax(coeffs.abs().reshape(coeffs.shape[0], -1), dim=1).to(torch.float64)
    est = torch.amax(cmax * om.to(cmax.device)) / gmax
    return torch.exp2(torch.round(torch.log2(torch.clamp(est, min=1e-300))))


def scale_rhs_rows(leaf, rhs):
    """rhs (n_leaves, n, nsrc) with its first nb rows (the impedance rows)
    multiplied by the ItI leaf's row scale, as a new contiguous tensor."""
    out = rhs.contiguous().clone()
    if leaf.kind == HPS_KIND_ITI and leaf.row_scale is not None:
        out[:, : leaf.nb, :] *= leaf.row_scale.to(out.real.dtype if out.is_complex() else out.dtype)
    return out


def scale_batched(X, scale):
    """X[b] *= scale[b] in place (X contiguous, scale a float64 device vector)."""
    lib = load_library()
    h = _lib.handle()
    b = X.shape[0]
    n = X[0].numel()
    rc = lib.hps_scale_batched(h, dtype_code(X.dtype), b, n, n, ptr(scale), ptr(X))
    check(rc, h, "hps_scale_batched")


def leaf_solve(pde, kind: int, dtype, device, source=None, nsrc_zero=False, leaf_half_sides=None) -> LeafResult:
    """Run hps_leaf_solve over all leaves of `pde`.

    source: (n_leaves, n, nsrc) tensor in `dtype`, or None for a zero source
    (nsrc_zero=True gives the no-source leaf stage, nsrc = 0).
    leaf_half_sides (n_leaves,) float64 numpy array: leaves of different
    sizes with operators built for half side 1 -- each coefficient of a
    k-th order term is scaled by half^-k and T, h by 1/half (the operators
    are homogeneous in the half side)."""
    ops = pde.device_ops(device, dtype)
    names = pde.operator_names()
    clist = pde.coefficient_list()
    if not clist:
        raise ValueError("PDEProblem has no coefficients")
    coef_ops = np.array([-1 if nm == "I" else names.index(nm) for nm, _ in clist], dtype=np.int32)
    if nsrc_zero:
        nsrc = 0
        src = None
    else:
        if source is None:
            nsrc = 1
            src = None
        else:
            nsrc = source.shape[-1]
            src = source
    if kind == HPS_KIND_ITI and not is_complex_input(*[a for _, a in clist]):
        res = _leaf_condensed(pde, ops, dtype, device, clist, coef_ops, src, nsrc)
        if res is not None:
            return res
    coeffs = torch.stack([to_device(a, device, dtype) for _, a in clist]).contiguous()
    if leaf_half_sides is not None:
        hs = np.asarray(leaf_half_sides, dtype=np.float64)
        inv = torch.as_tensor(1.0 / hs).to(device)
        inv2 = torch.as_tensor(1.0 / (hs * hs)).to(device)
        for k, (nm, _) in enumerate(clist):
            order = 0 if nm == "I" else len(nm) - 2
            if order:
                scale_batched(coeffs[k], inv if order == 1 else inv2)
    res = _leaf_direct(pde, ops, kind, dtype, device, clist, coef_ops, coeffs, src, nsrc)
    if leaf_half_sides is not None:
        scale_batched(res.T, inv)
        if res.h is not None:
            scale_batched(res.h, inv)
    return res


def _leaf_direct(pde, ops, kind, dtype, device, clist, coef_ops, coeffs, src, nsrc) -> LeafResult:
    """Leaf stage by the factorisation of the whole leaf matrix, over the
    leaves of coeffs (ncoef, nl, n) and src (nl, n, nsrc)."""
    lib = load_library()
    h = _lib.handle()
    nl, n = coeffs.shape[1:]
    P, Q = ops["P"], ops["Q"]
    nb, nq = P.shape
    nrows = n - nb if kind == HPS_KIND_DTN else n
    Y = torch.empty((nl, n, nq), dtype=dtype, device=device)
    T = torch.empty((nl, nq, nq), dtype=dtype, device=device)
    v = torch.empty((nl, n, nsrc), dtype=dtype, device=device) if nsrc else None
    hv = torch.empty((nl, nq, nsrc), dtype=dtype, device=device) if nsrc else None
    lu = torch.empty((nl, nrows, n), dtype=dtype, device=device)
    perm = torch.empty((nl, nrows), dtype=torch.int32, device=device)
    dinv = torch.empty((nl, _lib.dinv_size(nrows)), dtype=dtype, device=device)
    info = torch.empty((nl,), dtype=torch.int32, device=device)
    ws = workspace(lib.hps_leaf_workspace(dtype_code(dtype), kind, nl, n, nb, nq, nsrc), device)
    cop = coef_ops.ctypes.data_as(ctypes.c_void_p)
    G = row_scale = None
    if kind == HPS_KIND_ITI:
        row_scale = iti_row_scale(pde, coeffs, clist, device)
        rs = row_scale.to(real_dtype(dtype))
        G = (ops["G"] * rs).contiguous()
        P = (P * rs).contiguous()

    def run():
        rc = lib.hps_leaf_solve(
            h, dtype_code(dtype), kind, nl, n, nb, nq, nsrc, len(clist), cop,
            ptr(coeffs), ptr(ops["diffops"]), ptr(P), ptr(Q), ptr(G), ptr(src),
            ptr(Y), ptr(T), ptr(v), ptr(hv), ptr(lu), ptr(perm), ptr(dinv), ptr(info), ptr(ws), ws.numel(),
        )
        check(rc, h, "hps_leaf_solve")

    # natural-order factorisation (the leaf matrices eliminate with multipliers
    # below 2), checked per leaf in the panel kernels: a rejected leaf
    # (info = -1) reruns the whole stage with partial pivoting
    lib.hps_set_leaf_pivoting(h, 0)
    try:
        run()
    finally:
        lib.hps_set_leaf_pivoting(h, 1)
    if bool((info < 0).any()):
        run()
    return LeafResult(Y, T, v, hv, lu, perm, dinv, info, kind, row_scale, nb)


# A leaf whose interior problem is not safely definite is factored directly: one
# whose I / (D_xx + D_yy) exceeds this part of the first Dirichlet eigenvalue
# (pi / h)^2 somewhere, or one that the condensed stage rejects.
LEAF_DEFINITE = 0.9
# With at least this many leaves, one a CU, and at most this share of such ones,
# they alone are factored directly: fewer leaves take as long as one, and one
# kind of factors is then half the launches of every later solve; and the
# condensed stage of all leaves plus a larger share costs more than factoring
# every leaf directly (p = 16, L = 7: 33 ms and 57 ms).
LEAF_REDO_MIN = 256
LEAF_REDO_SHARE = 0.4
# Which leaves are definite is read before the stage where eta h exceeds this: eta
# is usually the wavenumber, and the stage would likely be for nothing.  Below,
# it is read with the stage's own checks, which saves waiting for the GPU twice
# (p = 13, L = 4: 3.22 against 3.30 ms).  The order does not change the result.
LEAF_LOOK_FIRST = 3.0


def _too_many(count, nl):
    return count > 0 and (nl < LEAF_REDO_MIN or count > LEAF_REDO_SHARE * nl)


def _mark_indefinite(pde, coeffs, clist, info):
    """info = -1 for the leaves whose interior problem may not be definite,
    from the coefficients alone (LEAF_DEFINITE)."""
    nl, n = coeffs.shape[1:]
    field = {nm: at(coeffs, k * nl * n) for k, (nm, _) in enumerate(clist)}
    second = [field[nm] for nm in ("D_xx", "D_yy") if nm in field]
    if "I" not in field or not second:
        return  # the condensed stage's own checks decide
    hd = _lib.handle()
    limit = LEAF_DEFINITE * (np.pi / (2 * pde.half_side_len)) ** 2
    rc = load_library().hps_mark_indefinite(hd, dtype_code(coeffs.dtype), nl, n, field["I"], second[0],
                                            second[1] if len(second) == 2 else None, limit, ptr(info))
    check(rc, hd, "hps_mark_indefinite")


def _leaf_condensed(pde, full_ops, dtype, device, clist, coef_ops, src, nsrc) -> Optional[LeafResult]:
    """ItI leaf stage with real coefficients by static condensation, the leaves
    whose interior problem is not definite by the factorisation of B.  None where
    all leaves are to be factored that way."""
    ops = pde.condensed_ops(device, dtype)
    if ops is None:
        return None
    lib = load_library()
    h = _lib.handle()
    nl = pde.domain.n_leaves
    nb, nq = ops["P"].shape
    n = pde.domain.p**2
    ni = n - nb
    rdt = real_dtype(dtype)
    coeffs = torch.stack([to_device(a, device, rdt) for _, a in clist]).contiguous()
    def empty(*shape, dt=dtype):
        return torch.empty(shape, dtype=dt, device=device)

    info = empty(nl, dt=torch.int32)
    if pde.eta * 2 * pde.half_side_len > LEAF_LOOK_FIRST:
        _mark_indefinite(pde, coeffs, clist, info.zero_())
        if _too_many(int((info < 0).sum()), nl):
            return None
    Y, T = empty(nl, n, nq), empty(nl, nq, nq)
    v = empty(nl, n, nsrc) if nsrc else None
    hv = empty(nl, nq, nsrc) if nsrc else None
    alu, aperm = empty(nl, ni, n, dt=rdt), empty(nl, ni, dt=torch.int32)
    adinv, X = empty(nl, _lib.dinv_size(ni), dt=rdt), empty(nl, ni, nb + 2 * nsrc, dt=rdt)
    slu, sperm, sdinv = empty(nl, nb, nb), empty(nl, nb, dt=torch.int32), empty(nl, _lib.dinv_size(nb))
    ws = workspace(lib.hps_leaf_condensed_workspace(dtype_code(dtype), nl, n, nb, nq, nsrc), device)
    rc = lib.hps_leaf_condensed(
        h, dtype_code(dtype), nl, n, nb, nq, nsrc, len(clist), coef_ops.ctypes.data_as(ctypes.c_void_p), ptr(coeffs),
        ptr(ops["diffops"]), ptr(ops["GQ"]), ptr(ops["Gb"]), ptr(ops["Qb"]), ptr(ops["P"]), ptr(src), ptr(Y), ptr(T),
        ptr(v), ptr(hv), ptr(alu), ptr(aperm), ptr(adinv), ptr(X), ptr(slu), ptr(sperm), ptr(sdinv), ptr(info), ptr(ws),
        ws.numel(),
    )
    check(rc, h, "hps_leaf_condensed")
    res = LeafResult(Y, T, v, hv, slu, sperm, sdinv, info, HPS_KIND_ITI, None, nb,
                     Condensed(alu, aperm, adinv, X, ops["GQ"][:nb]))
    _mark_indefinite(pde, coeffs, clist, info)
    if bool((info < 0).any()):
        idx = (info < 0).nonzero().flatten()
        if _too_many(idx.numel(), nl):
            return None
        sub = _leaf_direct(pde, full_ops, HPS_KIND_ITI, dtype, device, clist, coef_ops, coeffs[:, idx].to(dtype).contiguous(),
                           None if src is None else src[idx], nsrc)
        for dst, part in ((Y, sub.Y), (T, sub.T), (v, sub.v), (hv, sub.h), (info, sub.info)):
            if dst is not None:
                dst[idx] = part
        sub.Y = sub.T = sub.v = sub.h = None
        res.condensed.redone = (idx, sub)
    return res


@dataclass
class MergeLevel:
    S: torch.Tensor
    T: Optional[torch.Tensor]
    h: Optional[torch.Tensor]
    gt: Optional[torch.Tensor]
    F_lu: torch.Tensor          # LU of D (DtN) or of W = I - D12 D21 (ItI)
    perm: torch.Tensor
    dinv: torch.Tensor
    info: torch.Tensor
    D12: Optional[torch.Tensor]
    D21: Optional[torch.Tensor]
    B: Optional[torch.Tensor]
    tables: MergeTables
    Finv: Optional[torch.Tensor] = None  # block inverses for few-column up-pass solves (hps_block_inverses)
    info_host: Optional[torch.Tensor] = None  # info on the host (set by merge._levels)


def merge_level(T_in, h_in, tables: MergeTables, keep_factors=False, want_T=True, pivot=True) -> MergeLevel:
    """One level of 4:1 / 8:1 merges.  T_in (nm*nc, nec, nec), h_in (nm*nc, nec, nsrc) or None.
    keep_factors also keeps B (and D12/D21 for ItI) for the up pass.
    pivot=False factors the interface matrices without row exchanges: a matrix
    that the panel kernels reject has info = -1 and needs pivot=True."""
    lib = load_library()
    hd = _lib.handle()
    dev = T_in.device
    dt = T_in.dtype
    nc, nec, ni, ne = tables.nc, tables.nec, tables.ni, tables.ne
    kind = HPS_KIND_ITI if tables.kind == "iti" else HPS_KIND_DTN
    nm = T_in.shape[0] // nc
    assert T_in.shape == (nm * nc, nec, nec), (T_in.shape, nm, nc, nec)
    nsrc = 0 if h_in is None else h_in.shape[-1]
    nf = ni // 2 if kind == HPS_KIND_ITI else ni
    rows, cols, ext, _, cols_final, final_of_internal = tables.device(dev)
    S = torch.empty((nm, ni, ne), dtype=dt, device=dev)
    T = torch.empty((nm, ne, ne), dtype=dt, device=dev) if want_T else None
    ho = torch.empty((nm, ne, nsrc), dtype=dt, device=dev) if (nsrc and want_T) else None
    gt = torch.empty((nm, ni, nsrc), dtype=dt, device=dev) if nsrc else None
    F_lu = torch.empty((nm, nf, nf), dtype=dt, device=dev)
    perm = torch.empty((nm, nf), dtype=torch.int32, device=dev)
    dinv = torch.empty((nm, _lib.dinv_size(nf)), dtype=dt, device=dev)
    info = torch.empty((nm,), dtype=torch.int32, device=dev)
    keep12 = keep_factors and kind == HPS_KIND_ITI
    D12 = torch.empty((nm, nf, nf), dtype=dt, device=dev) if keep12 else None
    D21 = torch.empty((nm, nf, nf), dtype=dt, device=dev) if keep12 else None
    B = torch.empty((nm, ne, ni), dtype=dt, device=dev) if keep_factors else None
    # the block inverses of low-precision levels for the refinement's up passes
    n_inv = lib.hps_block_inverses_elems(nf) if (dt in (torch.complex64, torch.float32) and nm < 128) else 0
    Finv = torch.empty((nm * n_inv,), dtype=dt, device=dev) if n_inv else None
    ws = workspace(lib.hps_merge_workspace(dtype_code(dt), kind, nm, ni, ne, nsrc), dev)
    upd = np.ascontiguousarray(tables.upd, dtype=np.int32)
    d12 = np.ascontiguousarray(tables.d12_blk, dtype=np.int32)
    d21 = np.ascontiguousarray(tables.d21_blk, dtype=np.int32)
    # the tables' elimination order serves natural-order factorisation only
    dissect = getattr(tables, "dissect", HPS_DISSECT_NONE)
    if kind == HPS_KIND_DTN and not getattr(tables, "reordered", False):
        final_of_internal = None  # the internal order is the final one
    try:
        if not pivot:
            check(lib.hps_set_merge_pivoting(hd, 0), hd, "hps_set_merge_pivoting")
            if dissect:
                by_child, pos = tables.by_child_device(dev)
                check(lib.hps_set_merge_dissection(hd, dissect, ptr(by_child), ptr(pos)), hd,
                      "hps_set_merge_dissection")
        rc = _merge_level_call(lib, hd, dt, kind, nm, nc, nec, ni, ne, nsrc, T_in, h_in, rows, cols, ext, cols_final,
                               final_of_internal, upd, d12, d21, S, T, ho, gt, F_lu, perm, dinv, info, D12, D21, B,
                               Finv, ws)
    finally:
        if not pivot:
            lib.hps_set_merge_pivoting(hd, 1)
            lib.hps_set_merge_dissection(hd, HPS_DISSECT_NONE, None, None)
    check(rc, hd, "hps_merge_level")
    return MergeLevel(S, T, ho, gt, F_lu, perm, dinv, info, D12, D21, B, tables, Finv)


def form_block_inverses(lvl: MergeLevel) -> None:
    """Store in lvl.Finv the inverses of the 256 x 256 diagonal blocks of the
    level's low-precision factors when its up-pass solves would otherwise take
    the blocked few-column path (fewer than 128 matrices of more than 256
    unknowns): the refinement's up passes then solve through them.
    merge_level keeps them already; this forms them for factors from
    elsewhere."""
    nm, n = lvl.F_lu.shape[0], lvl.F_lu.shape[-1]
    if lvl.F_lu.dtype not in (torch.complex64, torch.float32) or nm >= 128:
        return
    lib = load_library()
    elems = lib.hps_block_inverses_elems(n)
    if elems == 0:
        return
    hd = _lib.handle()
    dt = lvl.F_lu.dtype
    inv = torch.empty(nm * elems, dtype=dt, device=lvl.F_lu.device)
    ws = workspace(lib.hps_block_inverses_workspace(dtype_code(dt), n, nm), lvl.F_lu.device)
    rc = lib.hps_block_inverses(hd, dtype_code(dt), n, nm, ptr(lvl.F_lu), ptr(lvl.dinv), ptr(inv), ptr(ws), ws.numel())
    check(rc, hd, "hps_block_inverses")
    lvl.Finv = inv


def merge_factors_stable(F_lu, bound=64.0):
    """Device bool: the natural-order (unpivoted) LU factors of a merge level
    are usable -- every entry finite, no zero pivot, every multiplier at most
    `bound` in magnitude (partial pivoting would guarantee 1; the merge
    matrices of uniform trees give values below 4).  The stages themselves go
    by the kernels' own checks (info); this is for factors in hand, whoever
    formed them."""
    a = F_lu.abs()
    finite = torch.isfinite(a.amax(dim=(-2, -1)))
    mult = torch.tril(a, -1).amax(dim=(-2, -1))
    dmin = a.diagonal(dim1=-2, dim2=-1).amin(dim=-1)
    return (finite & (mult <= bound) & (dmin > 0)).all()


def _merge_level_call(lib, hd, dt, kind, nm, nc, nec, ni, ne, nsrc, T_in, h_in, rows, cols, ext, cols_final,
                      final_of_internal, upd, d12, d21, S, T, ho, gt, F_lu, perm, dinv, info, D12, D21, B, Finv, ws):
    return lib.hps_merge_level(
        hd, dtype_code(dt), kind, nm, nc, nec, ni, ne, nsrc,
        ptr(T_in), ptr(h_in), ptr(rows), ptr(cols), ptr(ext), ptr(cols_final), ptr(final_of_internal),
        upd.shape[0], upd.ctypes.data_as(ctypes.c_void_p),
        d12.shape[0], d12.ctypes.data_as(ctypes.c_void_p), d21.shape[0], d21.ctypes.data_as(ctypes.c_void_p),
        ptr(S), ptr(T), ptr(ho), ptr(gt), ptr(F_lu), ptr(perm), ptr(dinv), ptr(info),
        ptr(D12), ptr(D21), ptr(B), ptr(Finv), ptr(ws), ws.numel(),
    )


def down_level(S, gt, g_in, tables: MergeTables):
    """g_in (nm, ne, nsrc) -> children boundary data (nm*nc, nec, nsrc)."""
    lib = load_library()
    hd = _lib.handle()
    dev = S.device
    dt = S.dtype
    nc, nec, ni, ne = tables.nc, tables.nec, tables.ni, tables.ne
    nm = S.shape[0]
    nsrc = g_in.shape[-1]
    src = tables.device(dev)[3]
    g_out = torch.empty((nm * nc, nec, nsrc), dtype=dt, device=dev)
    ws = workspace(lib.hps_down_workspace(dtype_code(dt), nm, ni, nsrc), dev)
    rc = lib.hps_down_level(
        hd, dtype_code(dt), nm, nc, nec, ni, ne, nsrc, ptr(S), ptr(gt), ptr(g_in), ptr(src), ptr(g_out),
        ptr(ws), ws.numel(),
    )
    check(rc, hd, "hps_down_level")
    return g_out


def down_level_static(S, gt, g_in, tables: MergeTables):
    """down_level through hps_down_level_static: no workspace is allocated
    (the interface data live in the library's static per-GPU scratch).
    Calls that overlap on one GPU race on that scratch."""
    lib = load_library()
    hd = _lib.handle()
    dev = S.device
    dt = S.dtype
    nc, nec, ni, ne = tables.nc, tables.nec, tables.ni, tables.ne
    nm = S.shape[0]
    nsrc = g_in.shape[-1]
    src = tables.device(dev)[3]
    g_out = torch.empty((nm * nc, nec, nsrc), dtype=dt, device=dev)
    rc = lib.hps_down_level_static(hd, dtype_code(dt), nm, nc, nec, ni, ne, nsrc, ptr(S), ptr(gt), ptr(g_in),
                                   ptr(src), ptr(g_out))
    check(rc, hd, "hps_down_level_static")
    return g_out


def leaf_apply(Y, g, v):
    """u = Y g + v per leaf."""
    lib = load_library()
    hd = _lib.handle()
    nl, n, nq = Y.shape
    nsrc = g.shape[-1]
    u = torch.empty((nl, n, nsrc), dtype=Y.dtype, device=Y.device)
    rc = lib.hps_leaf_apply(hd, dtype_code(Y.dtype), nl, n, nq, nsrc, ptr(Y), ptr(g), ptr(v), ptr(u))
    check(rc, hd, "hps_leaf_apply")
    return u


def getrs_into(n, lu, lu_offset, lda, sA, perm, dinv, R, X):
    """X = A^{-1} R from factors stored in `lu` (element offset lu_offset,
    row stride lda, batch stride sA).  R, X: (batch, n, nrhs) contiguous."""
    lib = load_library()
    hd = _lib.handle()
    b = R.shape[0]
    nrhs = R.shape[2]
    es = lu.element_size()
    rc = lib.hps_getrs_batched(
        hd, dtype_code(lu.dtype), n, nrhs, ctypes.c_void_p(lu.data_ptr() + lu_offset * es), lda, sA, ptr(perm),
        ptr(dinv), ptr(R), nrhs, n * nrhs, ptr(X), nrhs, n * nrhs, b,
    )
    check(rc, hd, "hps_getrs_batched")
    return X


def leaf_apply_inverse(leaf: LeafResult, rhs):
    """v = (leaf operator)^{-1} rhs for a full collocation right-hand side
    rhs (n_leaves, n, nsrc): DtN solves the interior rows with A_ii (v is zero
    on the boundary); ItI solves with B = [G; A_int]."""
    if leaf.condensed is not None:
        return _apply_inverse_condensed(leaf, rhs)
    nl, nrows, n = leaf.lu.shape
    nsrc = rhs.shape[-1]
    if leaf.kind == HPS_KIND_DTN:
        nb = n - nrows
        R = rhs[:, nb:, :].contiguous()
        X = torch.empty_like(R)
        getrs_into(nrows, leaf.lu, nb, n, nrows * n, leaf.perm, leaf.dinv, R, X)
        v = torch.zeros((nl, n, nsrc), dtype=rhs.dtype, device=rhs.device)
        v[:, nb:, :] = X
        return v
    R = scale_rhs_rows(leaf, rhs)
    X = torch.empty_like(R)
    getrs_into(n, leaf.lu, 0, n, n * n, leaf.perm, leaf.dinv, R, X)
    return X


def at(t, offset=0):
    """Device address of a tensor's element `offset` (in its own elements)."""
    return ctypes.c_void_p(t.data_ptr() + offset * t.element_size())


def gemm_at(dtype, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, D, ldd, sD, batch, conjt=False):
    """hps_gemm_batched (conjt: op(A) = A^H, A stored K x M) on device addresses."""
    lib = load_library()
    hd = _lib.handle()
    fn = lib.hps_gemm_batched_conjt if conjt else lib.hps_gemm_batched
    check(fn(hd, dtype_code(dtype), M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, D, ldd, sD, batch), hd,
          "hps_gemm_batched")


def _apply_inverse_condensed(leaf: LeafResult, rhs):
    """B^{-1} rhs through the condensed factors: w = A_ii^{-1} r_i,
    u_b = S^{-1}(r_b - G_i w), u_i = w - X_b u_b.  The real factors take a
    complex right-hand side as twice as many real columns."""
    lib = load_library()
    hd = _lib.handle()
    c = leaf.condensed
    rhs = rhs.contiguous()
    nl, n, w = rhs.shape
    nb, ni = c.Gi.shape
    dt, rdt = rhs.dtype, c.alu.dtype
    w2, wr = 2 * w, c.X.shape[2]
    out = torch.empty_like(rhs)
    t = torch.empty((nl, nb, w), dtype=dt, device=rhs.device)
    rc = lib.hps_getrs_batched(hd, dtype_code(rdt), ni, w2, at(c.alu, nb), n, ni * n, ptr(c.perm), ptr(c.dinv),
                               at(rhs, nb * w), w2, n * w2, at(out, nb * w), w2, n * w2, nl)
    check(rc, hd, "hps_getrs_batched")
    gemm_at(rdt, nb, w2, ni, -1.0, ptr(c.Gi), ni, 0, at(out, nb * w), w2, n * w2, 1.0, at(rhs), w2, n * w2, at(t), w2,
            nb * w2, nl)
    rc = lib.hps_getrs_batched(hd, dtype_code(dt), nb, w, ptr(leaf.lu), nb, nb * nb, ptr(leaf.perm), ptr(leaf.dinv),
                               ptr(t), w, nb * w, at(out), w, n * w, nl)
    check(rc, hd, "hps_getrs_batched")
    gemm_at(rdt, ni, w2, nb, -1.0, ptr(c.X), wr, ni * wr, at(out), w2, n * w2, 1.0, at(out, nb * w), w2, n * w2,
            at(out, nb * w), w2, n * w2, nl)
    if c.redone is not None:
        idx, sub = c.redone
        out[idx] = leaf_apply_inverse(sub, rhs[idx])
    return out


def up_level(h_in, lvl: MergeLevel, inj=None, want_h=True):
    """New outgoing data through the factors kept by a merge level.
    h_in (nm*nc, nec, nsrc) -> (g_tilde (nm, ni, nsrc) final order, h_out (nm, ne, nsrc) or None)."""
    lib = load_library()
    hd = _lib.handle()
    tb = lvl.tables
    dev, dt = h_in.device, h_in.dtype
    kind = HPS_KIND_ITI if tb.kind == "iti" else HPS_KIND_DTN
    nm = lvl.F_lu.shape[0]
    nsrc = h_in.shape[-1]
    rows, _, ext, _, _, final_of_internal = tb.device(dev)
    if kind == HPS_KIND_DTN and not getattr(tb, "reordered", False):
        final_of_internal = None
    gt = torch.empty((nm, tb.ni, nsrc), dtype=dt, device=dev)
    ho = torch.empty((nm, tb.ne, nsrc), dtype=dt, device=dev) if want_h else None
    ws = workspace(lib.hps_up_workspace(dtype_code(dt), kind, nm, tb.ni, nsrc), dev)
    upd = np.ascontiguousarray(tb.upd, dtype=np.int32)
    rc = lib.hps_up_level(
        hd, dtype_code(dt), kind, nm, tb.nc, tb.nec, tb.ni, tb.ne, nsrc, ptr(h_in.contiguous()),
        ptr(inj.contiguous()) if inj is not None else None, ptr(rows), ptr(ext), ptr(final_of_internal),
        upd.shape[0], upd.ctypes.data_as(ctypes.c_void_p), ptr(lvl.F_lu), ptr(lvl.perm), ptr(lvl.dinv),
        ptr(lvl.Finv) if lvl.Finv is not None else None, ptr(lvl.D12), ptr(lvl.D21), ptr(lvl.B), ptr(gt), ptr(ho),
        ptr(ws), ws.numel(),
    )
    check(rc, hd, "hps_up_level")
    return gt, ho


def cast(t, dtype):
    """t converted to `dtype` on the device by hps_convert (t itself if it already has it)."""
    if t is None or t.dtype == dtype:
        return t
    lib = load_library()
    hd = _lib.handle()
    src = t.contiguous()
    out = torch.empty(src.shape, dtype=dtype, device=src.device)
    rc = lib.hps_convert(hd, dtype_code(src.dtype), dtype_code(dtype), src.numel(), ptr(src), ptr(out))
    check(rc, hd, "hps_convert")
    return out
