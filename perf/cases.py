"""Performance cases of the multigrid solve path, from single operators to whole solves.

A case is one call (or one short chain of calls) that a program on top of
gascoignelib_amd.hip makes again and again, on meshes from the structure
producer.  The ranges:

  operators   the reference classes one by one in the caller's own numbering
  vanka       one application of the patch smoother, every patch different
  vcycle      one Vanka V-cycle of the Stokes-LPS channel (a preconditioner)
  stokes      a whole Stokes-LPS solve
  solve       Q1 Poisson / diffusion, 2D and 3D, Jacobi or ILU(0) smoothing,
              FP64 GMRES or a reduced-precision V-cycle in flexible GMRES
  q2          triquadratic Poisson, uniform or with adaptive levels
  gradient    forward and adjoint solve, dJ/dk per cell, DWR indicators
  assemble    a new coefficient: residual, re-assembled solver, one V-cycle

Boxes of a x b x c coarse cells, refined k times, give sizes that are not
powers of two.  Coefficients are 1 or vary from cell to cell (with the seed).
"""
import functools
import os
import tempfile

import numpy as np
import torch

from gascoignelib_amd import hip as H
from gascoignelib_amd import native as N
from gascoignelib_amd.problem import block_operator, patches_from_cells
from gascoignelib_amd.structure import (Mesh, assemble_hierarchy, colour_order, q2_hierarchy,
                                        stokes_hierarchy)


def listed():
    return [
        # a small 2D problem in FP64: every kernel is a launch, nothing fills the chip
        dict(name="solve_2d_32_f64", kind="solve", dim=2, macro="1x1", refine=5, coef="one",
             prec="f64", smoother="jacobi", order=False),
        # the reference algorithm in FP64 on a diffusion problem of ordinary size
        dict(name="solve_3d_96_var_f64", kind="solve", dim=3, macro="3x3x3", refine=5, coef="var",
             prec="f64", smoother="jacobi", order=True),
        # the largest: 2.1 M unknowns, f16-valued V-cycle in FP64 flexible GMRES
        dict(name="solve_3d_128_f16", kind="solve", dim=3, macro="1x1x1", refine=7, coef="one",
             prec="f16", smoother="jacobi", order=True),
        # the CPU path's default smoother
        dict(name="solve_3d_64_ilu_f64", kind="solve", dim=3, macro="1x1x1", refine=6, coef="one",
             prec="f64", smoother="ilu", order=True),
        # one step of a coefficient identification with goal-oriented indicators
        dict(name="gradient_48_f16", kind="gradient", dim=3, macro="3x3x3", refine=4, coef="var",
             prec="f16"),
        # 125-point rows, uniform mesh, mixed precision
        dict(name="q2_64_f16", kind="q2", refine=6, adaptive=0, prec="f16"),
        # 125-point rows, two adaptive refinements with hanging nodes, FP64
        dict(name="q2_16_adaptive_f64", kind="q2", refine=4, adaptive=2, prec="f64"),
        # saddle-point channel, FP32 Vanka V-cycle in FP64 flexible GMRES
        dict(name="stokes_32_f32", kind="stokes", macro="1x1x1", refine=5, visc=1.0, prec="f32"),
        # its preconditioner alone, in FP64
        dict(name="vcycle_stokes_32_f64", kind="vcycle", macro="1x1x1", refine=5, visc=1.0,
             prec="f64"),
        # the smoother alone on a linearised operator whose patches all differ
        dict(name="vanka_24_var_f32", kind="vanka", macro="3x3x3", refine=3, prec="f32"),
        # a program that calls the operators itself and keeps its own node numbers
        dict(name="operators_80x64x48_f64", kind="operators", dim=3, macro="5x4x3", refine=4,
             coef="var", prec="f64"),
        # a time step or Newton step: new coefficient, everything re-formed on the device
        dict(name="assemble_64_f16", kind="assemble", dim=3, macro="1x1x1", refine=6, coef="var",
             prec="f16"),
    ]


def draw(rng):
    kind = rng.choice(["solve", "solve", "gradient", "q2", "stokes", "vcycle", "vanka",
                       "operators", "assemble"])
    c = dict(kind=kind)

    def box(dim, most, least=300):
        """coarse cells and refinements of a box with about `least` .. `most` cells"""
        while True:
            macro = [rng.randint(1, 5) for _ in range(dim)]
            refine = rng.randint(2, 7)
            cells = float(np.prod([m << refine for m in macro]))
            if least <= cells <= most and rng.random() < 0.6:
                return "x".join(map(str, macro)), refine

    if kind == "solve":
        c["dim"] = rng.choice([2, 3, 3])
        c["smoother"] = rng.choice(["jacobi", "jacobi", "ilu"])
        most = 1.2e6 if c["smoother"] == "jacobi" else 3e5
        c["macro"], c["refine"] = box(c["dim"], most)
        c["coef"] = rng.choice(["one", "var"])
        c["prec"] = rng.choice(["f64", "f32", "f16"])
        c["order"] = rng.choice([True, True, False])
    elif kind == "gradient":
        c["dim"] = rng.choice([2, 3])
        c["macro"], c["refine"] = box(c["dim"], 2e5)
        c["coef"], c["prec"] = "var", rng.choice(["f64", "f32", "f16"])
    elif kind == "q2":
        c["adaptive"] = rng.choice([0, 1, 2])
        c["refine"] = rng.choice([4, 5, 6]) if c["adaptive"] == 0 else rng.choice([3, 4])
        c["prec"] = rng.choice(["f64", "f32", "f16"])
        c["x"], c["y"], c["z"] = (round(rng.uniform(0.3, 0.7), 3) for _ in range(3))
    elif kind in ("stokes", "vcycle"):
        # channels of 1 to 4 cubes in a row
        c["macro"], c["refine"] = rng.choice([("1x1x1", 3), ("1x1x1", 4), ("2x1x1", 3),
                                              ("2x1x1", 4), ("3x1x1", 3), ("3x1x1", 4),
                                              ("4x1x1", 4)])
        c["visc"] = round(10 ** rng.uniform(-1, 1), 3)
        c["prec"] = rng.choice(["f64", "f32"])
    elif kind == "vanka":
        c["macro"], c["refine"] = box(3, 3e4, 60)
        c["prec"] = rng.choice(["f64", "f32"])
    elif kind == "operators":
        c["dim"] = rng.choice([2, 3, 3])
        c["macro"], c["refine"] = box(c["dim"], 6e5, 60)
        c["coef"], c["prec"] = rng.choice(["one", "var"]), rng.choice(["f64", "f32", "f16"])
    else:
        c["dim"] = rng.choice([2, 3, 3])
        c["macro"], c["refine"] = box(c["dim"], 4e5)
        c["coef"], c["prec"] = "var", rng.choice(["f64", "f16"])
    return c


# ------------------------------------------------------------------- meshes
def _box_inp(macro, channel=False):
    """A coarse mesh of unit squares or cubes (scaled to a longest edge of 1; a
    channel keeps the unit cross-section), boundary colour 1, or inflow 1,
    walls 2 and outflow 3, written as .inp text to a temporary file."""
    dim = len(macro)
    nx, ny, nz = (list(macro) + [0])[:3]
    scale = 1.0 if channel else 1.0 / max(macro)
    at = lambda i, j, k=0: (k * (ny + 1) + j) * (nx + 1) + i  # noqa: E731
    verts = [(i * scale, j * scale, k * scale) for k in range(nz + 1) for j in range(ny + 1)
             for i in range(nx + 1)]
    cells, faces = [], []
    if dim == 2:
        cells = [("quad", (at(i, j), at(i + 1, j), at(i + 1, j + 1), at(i, j + 1)))
                 for j in range(ny) for i in range(nx)]
        faces += [(1, "line", (at(i, 0), at(i + 1, 0))) for i in range(nx)]
        faces += [(1, "line", (at(nx, j), at(nx, j + 1))) for j in range(ny)]
        faces += [(1, "line", (at(i + 1, ny), at(i, ny))) for i in range(nx)]
        faces += [(1, "line", (at(0, j + 1), at(0, j))) for j in range(ny)]
    else:
        for k in range(nz):
            for j in range(ny):
                for i in range(nx):
                    v = [at(i + a, j + b, k + c) for c in (0, 1)
                         for a, b in ((0, 0), (1, 0), (1, 1), (0, 1))]
                    cells.append(("hex", v))
                    wall, inflow, outflow = (2, 1, 3) if channel else (1, 1, 1)
                    for on, colour, q in ((k == 0, wall, (0, 1, 2, 3)),
                                          (k == nz - 1, wall, (5, 4, 7, 6)),
                                          (i == nx - 1, outflow, (1, 5, 6, 2)),
                                          (j == ny - 1, wall, (3, 2, 6, 7)),
                                          (i == 0, inflow, (0, 3, 7, 4)),
                                          (j == 0, wall, (1, 0, 4, 5))):
                        if on:
                            faces.append((colour, "quad", [v[t] for t in q]))
    lines = [f"{len(verts)} {len(cells) + len(faces)} 0 0 0"]
    lines += ["%d %r %r %r" % ((n,) + v) for n, v in enumerate(verts)]
    lines += ["%d 0 %s %s" % (n, t, " ".join(map(str, v))) for n, (t, v) in enumerate(cells)]
    lines += ["%d %d %s %s" % (n, col, t, " ".join(map(str, v)))
              for n, (col, t, v) in enumerate(faces)]
    fd, path = tempfile.mkstemp(suffix=".inp")
    with os.fdopen(fd, "w") as fh:
        fh.write("\n".join(lines) + "\n")
    return path


def _macro(case):
    return tuple(int(m) for m in case["macro"].split("x"))


@functools.lru_cache(maxsize=1)
def _mesh(macro, refine):
    path = _box_inp(macro)
    try:
        return Mesh(path, len(macro), refine, 1)
    finally:
        os.unlink(path)


@functools.lru_cache(maxsize=1)
def _stokes(macro, refine, visc):
    path = _box_inp(macro, channel=True)
    try:
        return stokes_hierarchy(refine, inp=path, visc=visc)
    finally:
        os.unlink(path)


@functools.lru_cache(maxsize=1)
def _q2(refine, adaptive, centre):
    return q2_hierarchy(refine, adaptive=adaptive, centre=centre)


@functools.lru_cache(maxsize=1)
def _ctx():
    return H.Context(0)


def _coefficient(points, seed):
    """exp of a seeded smooth random field, one value per point"""
    r = np.random.RandomState(seed % (1 << 31))
    g = np.zeros(len(points))
    for _ in range(6):
        w, b, a = r.normal(0, 6.0, points.shape[1]), r.uniform(0, 2 * np.pi), r.normal(0, 0.5)
        g += a * np.cos(points @ w + b)
    return np.exp(g)


def _hierarchy(case, seed):
    M = _mesh(_macro(case), case["refine"])
    k = None
    if case["coef"] == "var":
        l = M.nlevels - 1
        k = _coefficient(M.coords(l)[M.cells(l)].mean(axis=1), seed)
    return M, k, assemble_hierarchy(M, k)


def _rhs(lev, seed, salt=0):
    f = np.random.RandomState((seed * 7919 + salt) % (1 << 31)).uniform(-1, 1, lev.size)
    f.reshape(lev.n, lev.ncomp)[np.ix_(lev.dirichlet, lev.dirichlet_comps)] = 0.0
    for h in (lev.hn_edges, lev.hn_faces):
        if len(h):
            f[h[:, 0]] = 0.0
    return f


class _Memory:
    def __init__(self, v):
        self.owner = v  # the memory lives as long as a tensor refers to it
        kind = "<f8" if v.prec == "f64" else "<f4"
        self.__cuda_array_interface__ = {"shape": (v.n * v.n_comp,), "typestr": kind,
                                         "data": (N.hip().gh_vec_data(v.h), False), "version": 2}


def _view(v):
    """the vector's device memory as a tensor (no copy)"""
    return torch.as_tensor(_Memory(v), device="cuda")


def _vec(ctx, a, ncomp=1, prec="f64"):
    return H.CudaVectorInterface.from_global(ctx, a, ncomp, prec)


# ------------------------------------------------------------------ prepare
def _solver(ctx, hier, prec, sweeps=(2, 2), order="lexicographic", **kw):
    pre, post = sweeps
    args = dict(mgtype="V", iterpre=pre, iterpost=post, iterexact=10, omega=0.8, mgomega=1.0,
                ndirect=1000, prec=prec, krylov="gmres" if prec == "f64" else "fgmres",
                order=order)
    args.update(kw)
    return H.CudaMultiLevelSolver(ctx, hier, **args)


def prepare(case, seed):
    ctx = _ctx()
    return _PREPARE[case["kind"]](ctx, case, seed)


def _prepare_solve(ctx, case, seed):
    _, _, hier = _hierarchy(case, seed)
    order = "lexicographic" if case["order"] else None
    if case["smoother"] == "ilu":
        orders = [colour_order(l.rowptr, l.col)[0] for l in hier.levels]
        mg = _solver(ctx, hier, case["prec"], (1, 1), order, omega=1.0, linear_smooth="ilu",
                     ilu_orders=orders)
    else:
        pre = {"one": {"f64": (2, 2)}.get(case["prec"], (3, 2)),
               "var": {"f64": (3, 3)}.get(case["prec"], (2, 2))}[case["coef"]]
        mg = _solver(ctx, hier, case["prec"], pre, order)
    return _solve_state(ctx, case, mg, hier, seed)


def _solve_state(ctx, case, mg, hier, seed, rhs=None, nc=1):
    s = dict(kind=case["kind"], prec=case["prec"], mg=mg, U=mg.new_vector(),
             F=_vec(ctx, _rhs(hier.fine, seed) if rhs is None else rhs, nc))
    s["u"] = _view(s["U"])
    return s


def _prepare_q2(ctx, case, seed):
    hier = _q2(case["refine"], case["adaptive"],
               tuple(case.get(a, c) for a, c in zip("xyz", (0.671, 0.429, 0.431))))
    sweeps = ((3, 3) if case["adaptive"] else (3, 2)) if case["prec"] == "f64" else (2, 2)
    return _solve_state(ctx, case, _solver(ctx, hier, case["prec"], sweeps), hier, seed)


def _prepare_gradient(ctx, case, seed):
    M, k, hier = _hierarchy(case, seed)
    lev, l = hier.fine, M.nlevels - 1
    s = dict(kind="gradient", prec=case["prec"], fwd=_solver(ctx, hier, case["prec"]),
             adj=_solver(ctx, hier, case["prec"], adjoint=True))
    s["F"], s["G"] = _vec(ctx, _rhs(lev, seed)), _vec(ctx, _rhs(lev, seed, 1) / lev.n)
    s["cells"] = H.CoefficientCells(ctx, case["dim"], lev.coords, M.cells(l))
    s["patches"] = H.DwrPatches(ctx, case["dim"], lev.coords, M.patches(l))
    s["K"] = _vec(ctx, k)
    s["U"], s["Z"] = s["fwd"].new_vector(), s["adj"].new_vector()
    s["D"], s["E"] = (H.CudaVectorInterface(ctx, s["cells"].ncells) for _ in range(2))
    s["out"] = {n: _view(s[v]) for n, v in (("u", "U"), ("z", "Z"), ("dJdk", "D"), ("eta", "E"))}
    return s


def _stokes_rhs(hier, seed):
    """inflow of a seeded amplitude and a seeded smooth body force"""
    lev, r = hier.fine, np.random.RandomState(seed % (1 << 31))
    f = np.zeros((lev.n, 4))
    for c in (1, 2, 3):
        w, b = r.normal(0, 4.0, 3), r.uniform(0, 2 * np.pi)
        f[:, c] = hier.visc * np.cos(lev.coords @ w + b) / lev.n
    f[np.ix_(lev.dirichlet, lev.dirichlet_comps)] = 0.0
    return r.uniform(0.5, 1.5) * hier.rhs + f.reshape(-1)


def _prepare_stokes(ctx, case, seed):
    hier = _stokes(_macro(case), case["refine"], case["visc"])
    mg = _solver(ctx, hier, case["prec"], iterexact=4, ndirect=200, linear_smooth="vanka",
                 patches=hier.patches)
    s = _solve_state(ctx, case, mg, hier, seed, _stokes_rhs(hier, seed), 4)
    return s


def _vanka_problem(case, seed):
    M, k, hier = _hierarchy(dict(case, coef="var"), seed)
    r = np.random.RandomState(seed % (1 << 31))
    C = np.eye(4) + 0.2 * r.uniform(-1, 1, (4, 4))
    S = 0.05 * r.uniform(-1, 1, (4, 4))
    lev = hier.fine
    return lev, block_operator(lev, C, S), patches_from_cells(M.cells(M.nlevels - 1))


def _prepare_vanka(ctx, case, seed):
    lev, val, pat = _vanka_problem(case, seed)
    A = H.CudaCSRMatrixInterface(ctx, lev.rowptr, lev.col, val, 4)
    s = dict(kind="vanka", V=H.VankaSmoother(ctx, A, pat, case["prec"]))
    b = np.random.RandomState(seed % (1 << 31)).uniform(-1, 1, 4 * lev.n)
    s["B"], s["X"] = (_vec(ctx, b, 4, case["prec"]) for _ in range(2))
    s["x"] = _view(s["X"])
    return s


def _operator_inputs(lev, seed):
    r = np.random.RandomState(seed % (1 << 31))
    return r.uniform(-1, 1, lev.n), r.uniform(-1, 1, lev.n)


def _prepare_operators(ctx, case, seed):
    _, _, hier = _hierarchy(case, seed)
    lev, coarse = hier.fine, hier.level(hier.nlevels - 2)
    vp = "f64" if case["prec"] == "f64" else "f32"
    x, b = _operator_inputs(lev, seed)
    s = dict(kind="operators", A=H.CudaCSRMatrixInterface(ctx, lev.rowptr, lev.col, lev.val, 1,
                                                          case["prec"]),
             T=H.CudaMgInterpolatorNested(ctx, coarse.n, *lev.transfer),
             M=H.DirichletMask(ctx, lev.n, 1, lev.dirichlet),
             X=_vec(ctx, x, 1, vp), B=_vec(ctx, b, 1, vp))
    s.update((n, H.CudaVectorInterface(ctx, lev.n, 1, vp)) for n in ("Y", "R", "S", "W"))
    s["C"] = H.CudaVectorInterface(ctx, coarse.n, 1, vp)
    s["out"] = {n: _view(s[n]) for n in ("Y", "R", "S", "C")}
    return s


def _prepare_assemble(ctx, case, seed):
    M, _, hier = _hierarchy(dict(case, coef="one"), seed)
    nl = hier.nlevels
    mg = _solver(ctx, hier, case["prec"], (2, 2))
    r = np.random.RandomState(seed % (1 << 31))
    ks = [_coefficient(M.coords(l)[M.cells(l)].mean(axis=1), seed) for l in range(nl)]
    s = dict(kind="assemble", mg=mg, K=[_vec(ctx, k) for k in ks], ks=ks,
             cells=[H.CoefficientCells(ctx, case["dim"], M.coords(l), M.cells(l))
                    for l in range(nl)],
             U=_vec(ctx, r.uniform(-1, 1, hier.fine.n)), F=_vec(ctx, _rhs(hier.fine, seed)),
             R=mg.new_vector(), Z=mg.new_vector())
    s["out"] = {"r": _view(s["R"]), "z": _view(s["Z"])}
    return s


_PREPARE = dict(solve=_prepare_solve, q2=_prepare_q2, gradient=_prepare_gradient,
                stokes=_prepare_stokes, vcycle=_prepare_stokes, vanka=_prepare_vanka,
                operators=_prepare_operators, assemble=_prepare_assemble)


# ---------------------------------------------------------------------- run
def _solve(mg, U, F, prec):
    lin, vmax = (1e-10, 10) if prec == "f64" else (0.9e-10, 20)
    U.zero()
    rep = mg.Solve(U, F, H.CGInfo(lin, 1e-30, 100), H.NLInfo(1e-10, 1e-30, 50), vmax=vmax,
                   norm_kind=1)
    if N.NL_STATUS[rep.status] != "converged":
        raise RuntimeError("the solve did not converge: " + N.NL_STATUS[rep.status])


def run(s):
    kind = s["kind"]
    if kind in ("solve", "q2", "stokes"):
        _solve(s["mg"], s["U"], s["F"], s["prec"])
        return s["u"]
    if kind == "vcycle":
        s["mg"].precondition(s["U"], s["F"], x_is_zero=True)
        return s["u"]
    if kind == "vanka":
        s["X"].copy_from(s["B"])
        s["V"].solve(s["X"])
        return s["x"]
    if kind == "gradient":
        _solve(s["fwd"], s["U"], s["F"], s["prec"])
        _solve(s["adj"], s["Z"], s["G"], s["prec"])
        s["cells"].dJdk(s["Z"], s["U"], s["D"])
        s["patches"].estimate(s["U"], s["Z"], s["F"], s["K"], s["E"])
        return s["out"]
    if kind == "operators":
        s["A"].vmult(s["Y"], s["X"])
        s["A"].residual(s["R"], s["X"], s["B"])
        s["M"].zero(s["R"])
        s["T"].restrict_zero(s["C"], s["R"])
        s["S"].copy_from(s["X"])
        s["T"].prolongate_add(s["S"], s["C"])
        s["A"].smooth(s["S"], s["B"], s["W"], 2, 0.8)
        return s["out"]
    s["cells"][-1].form(s["R"], s["U"], s["F"], s["K"][-1], s["mg"].fine_mask)
    s["mg"].assemble_q1(s["cells"], s["K"])
    s["mg"].precondition(s["Z"], s["R"], x_is_zero=True)
    return s["out"]


# ----------------------------------------------------- what a pass must move
def _counts(case):
    """(nodes, operator entries, components) of the finest level"""
    kind = case["kind"]
    if kind == "q2":
        n = (1 << case["refine"]) ** 3 * (1 + 1.5 * case["adaptive"])
        return n, 62.0 * n, 1
    m = _macro(case)
    n = float(np.prod([(a << case["refine"]) + 1 for a in m]))
    if kind in ("stokes", "vcycle"):
        return n, 62.0 * n, 4
    return n, (27.0 if len(m) == 3 else 9.0) * n, 4 if kind == "vanka" else 1


def work(case):
    n, nnz, nc = _counts(case)
    v, m = 8.0 * n * nc, nnz * nc * nc
    size = {"f64": 8.0, "f32": 4.0, "f16": 2.0}[case["prec"]]
    kind = case["kind"]
    if kind in ("solve", "q2", "stokes"):  # the operator, the load and the solution
        return {"bytes": m * 8 + 2 * v, "flops": 2 * m}
    if kind == "vcycle":
        return {"bytes": m * size + 2 * v, "flops": 2 * m}
    if kind == "gradient":
        return {"bytes": m * 8 + 8 * v, "flops": 4 * m}
    if kind == "vanka":  # the patch factors (108 unknowns to 8 cells) and the vector
        return {"bytes": n / 8 * 108 * 108 * size + v / 8 * size * 2, "flops": n / 8 * 2 * 108 ** 2}
    if kind == "operators":
        sv = 8.0 if case["prec"] == "f64" else 4.0
        return {"bytes": m * size + 7 * n * sv, "flops": 8 * m}
    return {"bytes": m * size + 5 * v, "flops": 30 * m}


def tolerance(case):
    """four times what the outputs are off plain FP64 sums, and for solves what
    two iterations that both stop at 1e-10 are apart"""
    kind, prec = case["kind"], case["prec"]
    if kind in ("solve", "q2", "gradient"):
        return {"rel": 4e-10 if prec == "f64" else 1e-9}
    if kind == "stokes":
        return {"rel": 1e-8}
    if kind in ("assemble", "vcycle"):
        return {"rel": 1e-13 if prec == "f64" else 1e-5 if prec == "f16" else 2e-6}
    if kind == "vanka":
        return {"rel": 1e-13 if prec == "f64" else 2e-5}
    return {"rel": 2e-15 if prec == "f64" else 1e-6}


# -------------------------------------------------------------------- exact
def _dev(a, dtype=None):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype).cuda()


class _Csr:
    """A (block) CSR matrix on the GPU in FP64, as plain index sums."""

    def __init__(self, lev, val=None):
        nc = lev.ncomp
        self.n, self.nc = lev.n, nc
        self.row = _dev(np.repeat(np.arange(lev.n), np.diff(lev.rowptr)))
        self.col = _dev(lev.col.astype(np.int64))
        self.val = _dev(lev.val if val is None else val, torch.float64).reshape(-1, nc, nc)

    def __call__(self, x):
        t = torch.matmul(self.val, x.reshape(self.n, self.nc)[self.col].unsqueeze(-1)).squeeze(-1) \
            if self.nc > 1 else self.val[:, 0] * x[self.col].unsqueeze(-1)
        out = torch.zeros(self.n, self.nc, dtype=torch.float64, device="cuda")
        return out.index_add_(0, self.row, t).reshape(-1)

    def diagonal(self):
        d = torch.zeros(self.n, dtype=torch.float64, device="cuda")
        at = self.row == self.col
        return d.index_add_(0, self.row[at], self.val[at, 0, 0])


def _cg(A, b, tol=1e-14, most=4000):
    """conjugate gradients with the diagonal, on a symmetric operator"""
    x, r, d = torch.zeros_like(b), b.clone(), A.diagonal()
    z = r / d
    p, rz, stop = z.clone(), torch.dot(r, z), tol * float(torch.linalg.vector_norm(b))
    for it in range(most):
        q = A(p)
        a = rz / torch.dot(p, q)
        x += a * p
        r -= a * q
        if it % 20 == 19 and float(torch.linalg.vector_norm(r)) <= stop:
            break
        z = r / d
        new = torch.dot(r, z)
        p, rz = z + (new / rz) * p, new
    return x


def _patch_solve(A, lev, pat, x):
    """averages of the patch solves, patches in groups"""
    nc, nodes = lev.ncomp, _dev(pat.astype(np.int64))
    key = A.row * A.n + A.col  # ascending: rows ascend and so do their columns
    y = torch.zeros(lev.n, nc, dtype=torch.float64, device="cuda")
    count = torch.zeros(lev.n, dtype=torch.float64, device="cuda")
    xs, ps = x.reshape(lev.n, nc), pat.shape[1]
    for g in nodes.split(1024):
        want = (g[:, :, None] * A.n + g[:, None, :]).reshape(-1)
        at = torch.searchsorted(key, want).clamp(max=len(key) - 1)
        blk = A.val[at] * (key[at] == want).to(torch.float64)[:, None, None]
        m = blk.reshape(len(g), ps, ps, nc, nc).permute(0, 1, 3, 2, 4).reshape(len(g), ps * nc, -1)
        h = torch.linalg.solve(m.contiguous(), xs[g].reshape(len(g), ps * nc, 1))
        y.index_add_(0, g.reshape(-1), h.reshape(-1, nc))
        count.index_add_(0, g.reshape(-1), torch.ones(g.numel(), dtype=torch.float64, device="cuda"))
    return (y / count[:, None]).reshape(-1)


def _parents(lev):
    """(fine node, coarse node, weight) of the nodal interpolation"""
    c2f, z, v, a = (np.asarray(t, np.int64) for t in lev.transfer)
    f, c, w = [c2f], [np.arange(len(c2f))], [np.ones(len(c2f))]
    for t in (z, v, a):
        k = t.shape[1] - 1
        f.append(np.repeat(t[:, 0], k))
        c.append(t[:, 1:].reshape(-1))
        w.append(np.full(len(t) * k, 1.0 / k))
    return tuple(_dev(np.concatenate(q)) for q in (f, c, w))


def _restrict(par, uf, nc_nodes, nc=1):
    f, c, w = par
    out = torch.zeros(nc_nodes, nc, dtype=torch.float64, device="cuda")
    return out.index_add_(0, c, w[:, None] * uf.reshape(-1, nc)[f]).reshape(-1)


def _prolongate(par, uc, nf, nc=1):
    f, c, w = par
    out = torch.zeros(nf, nc, dtype=torch.float64, device="cuda")
    return out.index_add_(0, f, w[:, None] * uc.reshape(-1, nc)[c]).reshape(-1)


def _vcycle(levels, mats, smooth, sweeps, ndirect, l, b):
    """V-cycle from zero: smoothing, nodal transfers, Dirichlet rows zeroed"""
    lev, A = levels[l], mats[l]
    if lev.n < ndirect:
        m = torch.zeros(lev.n, lev.n, A.nc, A.nc, dtype=torch.float64, device="cuda")
        m[A.row, A.col] = A.val
        return torch.linalg.solve(m.permute(0, 2, 1, 3).reshape(lev.size, lev.size).contiguous(), b)

    def zero(v, at):
        v.reshape(at.n, at.ncomp)[_dev(at.dirichlet.astype(np.int64))[:, None],
                                  _dev(at.dirichlet_comps.astype(np.int64))[None]] = 0.0
        return v

    x = torch.zeros_like(b)
    for _ in range(sweeps[0]):
        x = x + 0.8 * smooth(l, b - A(x))
    par = _parents(lev)
    bc = zero(_restrict(par, b - A(x), levels[l - 1].n, A.nc), levels[l - 1])
    xc = _vcycle(levels, mats, smooth, sweeps, ndirect, l - 1, bc)
    x = x + zero(_prolongate(par, xc, lev.n, A.nc), lev)
    for _ in range(sweeps[1]):
        x = x + 0.8 * smooth(l, b - A(x))
    return x


def _element_matrices(dim, X):
    """unit-coefficient Q1 stiffness matrices of box cells with corners X
    (cells, corners, dim), from products of 1D stiffness and mass matrices"""
    h = (X.max(1) - X.min(1))
    bit = (X > X.min(1, keepdims=True) + 0.5 * h[:, None]).astype(np.int64)
    s = lambda d: np.where(bit[:, :, None, d] == bit[:, None, :, d], 1.0, -1.0) / h[:, d, None, None]  # noqa: E731
    m = lambda d: np.where(bit[:, :, None, d] == bit[:, None, :, d], 2.0, 1.0) * h[:, d, None, None] / 6  # noqa: E731
    if dim == 2:
        return s(0) * m(1) + m(0) * s(1)
    return s(0) * m(1) * m(2) + m(0) * s(1) * m(2) + m(0) * m(1) * s(2)


def exact(case, seed):
    kind = case["kind"]
    if kind == "stokes":  # indefinite and unsymmetric: no plain solver in seconds
        return None
    if kind == "q2":
        hier = _q2(case["refine"], case["adaptive"],
                   tuple(case.get(a, c) for a, c in zip("xyz", (0.671, 0.429, 0.431))))
        return _cg(_Csr(hier.fine), _dev(_rhs(hier.fine, seed)))
    if kind == "vcycle":
        hier = _stokes(_macro(case), case["refine"], case["visc"])
        mats = [_Csr(lev) for lev in hier.levels]
        b = _dev(_stokes_rhs(hier, seed))
        smooth = lambda l, r: _patch_solve(mats[l], hier.levels[l], hier.patches[l], r)  # noqa: E731
        return _vcycle(hier.levels, mats, smooth, (2, 2), 200, hier.nlevels - 1, b)
    if kind == "vanka":
        lev, val, pat = _vanka_problem(case, seed)
        lev.ncomp = 4
        b = np.random.RandomState(seed % (1 << 31)).uniform(-1, 1, 4 * lev.n)
        return _patch_solve(_Csr(lev, val), lev, pat, _dev(b))
    if kind == "assemble":
        return _exact_assemble(case, seed)
    M, k, hier = _hierarchy(case, seed)
    lev = hier.fine
    A = _Csr(lev)
    if kind == "solve":
        return _cg(A, _dev(_rhs(lev, seed)))
    if kind == "operators":
        x, b = (_dev(v) for v in _operator_inputs(lev, seed))
        y = A(x)
        r = b - y
        r[_dev(lev.dirichlet.astype(np.int64))] = 0.0
        par, d = _parents(lev), A.diagonal()
        c = _restrict(par, r, hier.level(hier.nlevels - 2).n)
        u = x + _prolongate(par, c, lev.n)
        for _ in range(2):
            u = u + 0.8 * (b - A(u)) / d
        return {"Y": y, "R": r, "S": u, "C": c}
    u, z = _cg(A, _dev(_rhs(lev, seed))), _cg(A, _dev(_rhs(lev, seed, 1) / lev.n))
    cells = M.cells(M.nlevels - 1)
    E = _dev(_element_matrices(case["dim"], lev.coords[cells]))
    t = _dev(cells.astype(np.int64))
    d = -(z[t].unsqueeze(1) @ E @ u[t].unsqueeze(2)).reshape(-1)
    return {"u": u, "z": z, "dJdk": d, "eta": None}


def _exact_assemble(case, seed):
    M = _mesh(_macro(case), case["refine"])
    r = np.random.RandomState(seed % (1 << 31))
    hier = assemble_hierarchy(M)
    levels, fine = hier.levels, hier.fine
    mats = []
    for l, lev in enumerate(levels):
        X, cells = M.coords(l), M.cells(l)
        k = _coefficient(X[cells].mean(axis=1), seed)
        E, t = _element_matrices(case["dim"], X[cells]), _dev(cells.astype(np.int64))
        A, npc = _Csr(lev), cells.shape[1]
        key = A.row * A.n + A.col
        A.val.zero_()
        for a in range(npc):
            for b in range(npc):
                at = torch.searchsorted(key, t[:, a] * A.n + t[:, b])
                A.val[:, 0, 0].index_add_(0, at, _dev(k * E[:, a, b]))
        if l == len(levels) - 1:
            u, f = _dev(r.uniform(-1, 1, fine.n)), _dev(_rhs(fine, seed))
            res = f - A(u)
            res[_dev(lev.dirichlet.astype(np.int64))] = 0.0
        isd = torch.zeros(A.n, dtype=torch.bool, device="cuda")
        isd[_dev(lev.dirichlet.astype(np.int64))] = True
        A.val[isd[A.row] | isd[A.col]] = 0.0
        A.val[isd[A.row] & (A.row == A.col)] = 1.0
        mats.append(A)
    diag = [A.diagonal() for A in mats]
    z = _vcycle(levels, mats, lambda l, v: v / diag[l], (2, 2), 1000, len(levels) - 1, res)
    return {"r": res, "z": z}
