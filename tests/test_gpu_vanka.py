"""Vanka patch smoother on the GPU against the oracle.

FP64: the patch factors are formed with the oracle's operations (same pivots,
uncontracted updates) and the solves in the same order, so the smoother and the
V-cycle built on it agree bit for bit; GMRES / Newton iterates to 1e-12 with
iteration counts within one.  FP32 factors: within 1e-5 of FP64.
"""
import numpy as np
import pytest

import oracle_ctypes as O
from gascoignelib_amd import hip as H
from gascoignelib_amd.problem import Hierarchy, Level, block_operator, patches_from_cells
from gascoignelib_amd.structure import Mesh, assemble_hierarchy

pytestmark = pytest.mark.gpu

MGP = dict(mgtype="V", iterpre=2, iterpost=2, iterexact=4, omega=0.8, mgomega=1.0)


@pytest.fixture(scope="module")
def ctx():
    c = H.Context(0)
    yield c
    c.close()


def mesh_hierarchy(pre, B):
    """uniform cube hierarchy (levels 2^1 .. 2^pre cells per direction), scalar or
    the block operator of B components, and the Vanka patches of every level"""
    M = Mesh("cube.inp", 3, pre, 1)
    h = assemble_hierarchy(M)
    rng = np.random.default_rng(B)
    G = rng.uniform(-1, 1, (B, B))
    Cm, S = G @ G.T + B * np.eye(B), rng.uniform(-0.3, 0.3, (B, B))
    levels, patches = [], []
    for l, lev in enumerate(h.levels):
        val = lev.val if B == 1 else block_operator(lev, Cm, S)
        levels.append(Level(lev.n, B, lev.rowptr, lev.col, val, lev.transfer, lev.hn_kind,
                            dirichlet=lev.dirichlet,
                            dirichlet_comps=np.arange(B, dtype=np.int32), coords=lev.coords))
        patches.append(patches_from_cells(M.cells(l)))
    return Hierarchy(levels, 3, f"cube{pre}:B{B}"), patches


@pytest.mark.parametrize("B", [1, 4])
def test_vanka_solve_bitexact(ctx, B):
    h, patches = mesh_hierarchy(4 if B == 1 else 3, B)
    lev = h.fine
    A = H.CudaCSRMatrixInterface(ctx, lev.rowptr, lev.col, lev.val, B)
    x = np.random.default_rng(7).uniform(-1, 1, lev.n * B)
    X = H.CudaVectorInterface.from_global(ctx, x, B)
    H.VankaSmoother(ctx, A, patches[-1]).solve(X)
    xo = x.copy()
    O.Vanka(O.Matrix(lev.rowptr, lev.col, lev.val, B), patches[-1]).solve(xo)
    assert np.array_equal(X.copy_back(), xo)
    # FP32 factors and local solves
    X32 = H.CudaVectorInterface.from_global(ctx, x, B, "f32")
    H.VankaSmoother(ctx, A, patches[-1], "f32").solve(X32)
    assert np.abs(X32.copy_back() - xo).max() <= 1e-5 * np.abs(xo).max()


@pytest.mark.parametrize("B", [1, 4])
@pytest.mark.parametrize("order", [None, "lexicographic"])
def test_vcycle_with_vanka_vs_oracle(ctx, B, order):
    print(f"[vanka V-cycle B={B} order={order}]", flush=True)
    h, patches = mesh_hierarchy(4 if B == 1 else 3, B)
    f = np.random.default_rng(9).uniform(-1, 1, h.fine.n * B)
    for c in range(B):
        f[h.fine.dirichlet * B + c] = 0.0
    om = O.MG(h, ndirect=1, smoother="vanka", patches=patches, **MGP)
    xo = np.zeros_like(f)
    om.precondition(xo, f)
    mg = H.CudaMultiLevelSolver(ctx, h, ndirect=1, linear_smooth="vanka", patches=patches,
                                order=order, **MGP)
    X = mg.new_vector()
    mg.precondition(X, H.CudaVectorInterface.from_global(ctx, f, B))
    x = X.copy_back()
    if order is None:
        assert np.array_equal(x, xo)
    else:  # the same numbers, sums formed in the caller's order
        assert np.array_equal(x, xo)
    # Newton / GMRES with the Vanka V-cycle
    uo = np.zeros_like(f)
    _, orep = om.newton(uo, f, O.cginfo(1e-10, 1e-30, 100), O.nlinfo(1e-10, 1e-30, 30),
                        norm_kind=1)
    U = mg.new_vector()
    rep = mg.Solve(U, H.CudaVectorInterface.from_global(ctx, f, B), H.CGInfo(1e-10, 1e-30, 100),
                   H.NLInfo(1e-10, 1e-30, 30), norm_kind=1)
    u = U.copy_back()
    assert rep.newton_iterations == orep.newton_iterations
    assert abs(rep.gmres_iterations - orep.gmres_iterations) <= 1
    assert np.linalg.norm(u - uo) <= 1e-12 * np.linalg.norm(uo)


def test_vanka_mixed_precision_solve(ctx):
    h, patches = mesh_hierarchy(4, 4)
    f = np.random.default_rng(11).uniform(-1, 1, h.fine.n * 4)
    for c in range(4):
        f[h.fine.dirichlet * 4 + c] = 0.0
    om = O.MG(h, ndirect=1, smoother="vanka", patches=patches, **MGP)
    uo = np.zeros_like(f)
    om.newton(uo, f, O.cginfo(1e-12, 1e-30, 100), O.nlinfo(1e-12, 1e-30, 30), norm_kind=1)
    mg = H.CudaMultiLevelSolver(ctx, h, ndirect=1, linear_smooth="vanka", patches=patches,
                                prec="f32", krylov="fgmres", **MGP)
    U = mg.new_vector()
    rep = mg.Solve(U, H.CudaVectorInterface.from_global(ctx, f, 4), H.CGInfo(0.9e-10, 1e-30, 100),
                   H.NLInfo(1e-10, 1e-30, 30), norm_kind=1)
    assert H.N.NL_STATUS[rep.status] == "converged"
    assert np.linalg.norm(U.copy_back() - uo) <= 1e-8 * np.linalg.norm(uo)


def plane_problem(refine, B, seed, vary, children=4):
    """a 2D hierarchy's finest level with a B-component block operator, patches of
    9 nodes (4 cells) or 25 (16 cells); `vary`: a coefficient per cell, so that no two patches are equal"""
    M = Mesh("square.inp", 2, refine, 1)
    r = np.random.default_rng(seed)
    k = r.uniform(0.5, 2.0, len(M.cells(M.nlevels - 1))) if vary else None
    lev = assemble_hierarchy(M, k).fine
    C = np.eye(B) + 0.2 * r.uniform(-1, 1, (B, B))
    val = lev.val if B == 1 else block_operator(lev, C, 0.1 * r.uniform(-1, 1, (B, B)))
    return lev, np.asarray(val), patches_from_cells(M.cells(M.nlevels - 1), children), r


# local systems of 9 .. 125 unknowns (1 to 8 rows per lane, full and partial),
# patches that share factors and patches that do not (one wavefront each), up to
# 16,384 of them
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("B,refine,vary,children",
                         [(1, 2, True, 4), (1, 4, False, 4), (2, 4, True, 4), (4, 3, False, 4),
                          (5, 3, True, 4), (7, 3, True, 4), (8, 2, True, 4), (3, 4, True, 16),
                          (4, 4, False, 16), (5, 4, True, 16), (1, 8, True, 4)])
def test_vanka_solve_shapes(ctx, prec, B, refine, vary, children):
    print(f"[vanka B={B} refine={refine} vary={vary} {children} {prec}]", flush=True)
    lev, val, pat, r = plane_problem(refine, B, 100 * B + refine, vary, children)
    x = r.uniform(-1, 1, lev.n * B)
    A = H.CudaCSRMatrixInterface(ctx, lev.rowptr, lev.col, val, B)
    X = H.CudaVectorInterface.from_global(ctx, x, B, prec)
    H.VankaSmoother(ctx, A, pat, prec).solve(X)
    xo = x.copy()
    O.Vanka(O.Matrix(lev.rowptr, lev.col, val, B), pat).solve(xo)
    if prec == "f64":
        assert np.array_equal(X.copy_back(), xo)
    else:
        assert np.abs(X.copy_back() - xo).max() <= 1e-5 * np.abs(xo).max()


# factors and vectors outside the range in which the solves multiply by
# reciprocals: those patches are solved with plain divisions
@pytest.mark.parametrize("ascale,xscale", [(2.0 ** 500, 1.0), (2.0 ** -450, 2.0 ** -300),
                                           (1.0, 2.0 ** -800), (1.0, 2.0 ** 700)])
def test_vanka_solve_extreme_values(ctx, ascale, xscale):
    lev, val, pat, r = plane_problem(3, 2, 5, True)
    val = val * ascale
    x = r.uniform(-1, 1, lev.n * 2) * xscale
    x[::3] = 0.0
    X = H.CudaVectorInterface.from_global(ctx, x, 2)
    H.VankaSmoother(ctx, H.CudaCSRMatrixInterface(ctx, lev.rowptr, lev.col, val, 2), pat).solve(X)
    xo = x.copy()
    O.Vanka(O.Matrix(lev.rowptr, lev.col, val, 2), pat).solve(xo)
    assert np.array_equal(X.copy_back(), xo)


def class_problem(psize, B, npatches, nclasses, seed, band=None):
    """disjoint patches of `psize` nodes with `nclasses` different matrices in
    turn (full, or `band` nodes on each side of the diagonal), whose LU exchanges
    rows"""
    r = np.random.default_rng(seed)
    blk = r.uniform(-1, 1, (nclasses, psize, psize, B, B))
    i = np.arange(psize)
    keep = np.abs(i[:, None] - i[None]) <= (psize if band is None else band)
    rows, cols = np.nonzero(keep)
    n = npatches * psize
    rowptr = np.concatenate([[0], np.cumsum(np.tile(keep.sum(1), npatches))]).astype(np.int32)
    col = (np.arange(npatches)[:, None] * psize + cols[None]).reshape(-1).astype(np.int32)
    val = blk[np.arange(npatches) % nclasses][:, rows, cols].reshape(-1)
    return rowptr, col, val, np.arange(n, dtype=np.int32).reshape(npatches, psize), r


def check_vanka(ctx, rowptr, col, val, B, patches, x, prec, grouped):
    """the solve against the oracle: bit for bit in FP64; FP32 factors within what
    their rounding gives each patch, n_p 2^-24 times the condition of its matrix
    (times 4: factors, both triangles and the right-hand side)"""
    V = H.VankaSmoother(ctx, H.CudaCSRMatrixInterface(ctx, rowptr, col, val, B), patches, prec)
    assert (V.groups() > 0) == grouped
    X = H.CudaVectorInterface.from_global(ctx, x, B, prec)
    V.solve(X)
    xo = x.copy()
    O.Vanka(O.Matrix(rowptr, col, val, B), patches).solve(xo)
    if prec == "f64":
        assert np.array_equal(X.copy_back(), xo)
        return V
    P, m = len(patches), patches.shape[1] * B
    got, want = X.copy_back().reshape(P, m), xo.reshape(P, m)
    nc = min(P, 8)  # the classes come in turn
    A = np.zeros((nc, m, m))
    for p in range(nc):
        for a in range(patches.shape[1]):
            for q in range(rowptr[patches[p, a]], rowptr[patches[p, a] + 1]):
                b = col[q] - patches[p, 0]
                A[p, a * B:(a + 1) * B, b * B:(b + 1) * B] = val[q * B * B:(q + 1) * B * B].reshape(B, B)
    cond = np.array([np.linalg.cond(a) for a in A])
    for p in range(nc):
        bound = 4 * m * 2.0 ** -24 * cond[p] * np.linalg.norm(want[p])
        assert np.linalg.norm(got[p] - want[p]) <= bound
    return V


# local systems around the 16-row and 16-column batches and the second row of a
# lane (64, 65), each with a matrix of its own per patch (streamed) and with 8
# patches to a matrix (grouped)
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("psize,B", [(1, 1), (2, 1), (15, 1), (16, 1), (17, 1), (31, 1), (16, 2),
                                     (11, 3), (16, 3), (7, 7), (9, 7), (16, 4), (13, 5), (16, 5),
                                     (27, 3), (24, 4), (97, 1), (27, 4), (28, 4), (113, 1),
                                     (25, 5), (127, 1), (32, 4)])
def test_vanka_solve_both_kernels(ctx, prec, psize, B):
    print(f"[vanka both {psize}x{B} {prec}]", flush=True)
    for npatches, nclasses in ((41, 41), (40, 5)):
        rowptr, col, val, pat, r = class_problem(psize, B, npatches, nclasses, 10 * psize + B)
        x = r.uniform(-1, 1, npatches * psize * B)
        check_vanka(ctx, rowptr, col, val, B, pat, x, prec, nclasses < npatches)


# more workgroups than the chip holds at once: few patches to a matrix are
# streamed, enough are grouped; and more than 32 patches to a workgroup
@pytest.mark.parametrize("psize,B,npatches,nclasses,prec,grouped",
                         [(9, 1, 4096, 4096, "f64", False), (9, 1, 4096, 2048, "f64", True),
                          (27, 4, 1600, 800, "f64", False), (27, 4, 1600, 200, "f64", True),
                          (27, 4, 3200, 1600, "f32", False), (27, 4, 3200, 320, "f32", True),
                          (27, 4, 8200, 1, "f64", True)])
def test_vanka_solve_many_patches(ctx, psize, B, npatches, nclasses, prec, grouped):
    print(f"[vanka {npatches} patches, {nclasses} matrices, {psize}x{B} {prec}]", flush=True)
    rowptr, col, val, pat, r = class_problem(psize, B, npatches, nclasses, 3, band=1)
    x = r.uniform(-1, 1, npatches * psize * B)
    V = check_vanka(ctx, rowptr, col, val, B, pat, x, prec, grouped)
    if nclasses == 1:
        assert 32 * V.groups() < npatches


# the plain divisions of both kernels, with one and two rows per lane
@pytest.mark.parametrize("ascale,xscale", [(2.0 ** 500, 1.0), (2.0 ** -450, 2.0 ** -300),
                                           (1.0, 2.0 ** -800), (1.0, 2.0 ** 700)])
@pytest.mark.parametrize("psize,B", [(9, 2), (27, 4)])
def test_vanka_extreme_values_both_kernels(ctx, psize, B, ascale, xscale):
    for npatches, nclasses in ((17, 17), (24, 3)):
        rowptr, col, val, pat, r = class_problem(psize, B, npatches, nclasses, 8)
        x = r.uniform(-1, 1, npatches * psize * B) * xscale
        x[::3] = 0.0
        check_vanka(ctx, rowptr, col, val * ascale, B, pat, x, "f64", nclasses < npatches)
