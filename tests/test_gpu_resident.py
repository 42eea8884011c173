"""The resident CG (one launch, or one per stretch between hand-overs) against the separate kernels.

Sizes at the edges of its parts: one block (up to a few hundred rows), one row more than a
block's 512 threads, several rows per thread, rows whose entries lie in LDS (FP64, 27 entries,
more than 1,024 rows per block), lattices beyond that; every source of rows (K's columns, lattice planes, cell form),
9, 18 and 27 entries per row.  An explicit launch shape of the separate kernels (cg_elems)
selects those.  Both solve to a true residual of 1e-12, so their u differ by a few times
cond · 1e-12: 1e-8, the bar the other solver tests use."""
import ctypes

import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

import ferrite_amd as fa  # noqa: E402
from ferrite_amd.batch import BatchedPoisson, poisson_problem  # noqa: E402


def _move(g, nel, seed):
    """Interior nodes moved by up to a fifth of the cell size."""
    rng = np.random.default_rng(seed)
    inner = np.all((g.nodes > g.nodes.min(0) + 1e-12) & (g.nodes < g.nodes.max(0) - 1e-12), axis=1)
    h = (g.nodes.max(0) - g.nodes.min(0)) / np.array(nel)
    g.nodes[inner] += rng.uniform(-0.2, 0.2, (int(inner.sum()), g.sdim)) * h
    return g


def _poisson(nel, distort, **tune):
    ct = "Hexahedron" if len(nel) == 3 else "Quadrilateral"
    g = fa.generate_grid(ct, nel, (0.0,) * len(nel), (1.0,) * len(nel))
    if distort:
        _move(g, nel, 5)
    ip = fa.Lagrange(g.refshape, 1)
    dh = fa.DofHandler(g).add("u", ip).close()
    K = fa.allocate_matrix(fa.MI355XCSC, dh)
    f = fa.allocate_vector(K)
    fa.set_tuning(K, **tune)
    cv = fa.CellValues(fa.QuadratureRule(g.refshape, 2), ip)
    k = np.exp(np.random.default_rng(3).normal(0.0, 0.5, g.ncells))
    fa.assemble_global(fa.start_assemble(K, f), cv, fa.create_coloring(g), fa.PoissonElement(k=k, source=1.0))
    ch = fa.ConstraintHandler(dh)
    ch.add(fa.Dirichlet("u", g.facetsets["left"], lambda x, t: 1.0 + x[1])).close()
    fa.apply(K, f, ch)
    return K, f


def _check(K, f, mode, operator, kernels):
    A, b = K.to_scipy(), f.to_numpy()
    one = fa.solve(K, f, mode=mode, rtol=1e-12)
    two = fa.solve(K, f, mode=mode, rtol=1e-12)
    assert one.operator == operator and one.kernels == kernels and not one.gave_up
    assert np.array_equal(one.u, two.u) and one.iterations == two.iterations
    assert np.linalg.norm(b - A @ one.u) <= 2e-12 * np.linalg.norm(b)
    fa.set_tuning(K, cg_elems=8)
    sep = fa.solve(K, f, mode=mode, rtol=1e-12)
    assert sep.operator == operator and sep.kernels == "separate"
    assert np.linalg.norm(one.u - sep.u) <= 1e-8 * np.linalg.norm(sep.u)


@pytest.mark.parametrize("nel", [(3, 2), (15, 15), (22, 22), (30, 33), (71, 69), (5, 400), (7, 7, 7), (9, 8, 7),
                                 (2, 2, 200), (23, 19, 17), (63, 64, 65)])
def test_rows_of_K(nel):
    print("case resident rows of K", nel, flush=True)
    K, f = _poisson(nel, True, lattice=-1, cell_operator=-1)
    _check(K, f, "cg", "sell", "rows")
    if len(nel) == 2 or nel[0] < 60:
        fa.set_tuning(K, cg_elems=0)
        _check(K, f, "mixed", "sell", "rows")


@pytest.mark.parametrize("nel,kernels", [((71, 71, 71), "rows"), ((71, 71, 72), "separate"), ((72, 72, 72), "separate"),
                                         ((715, 715), "rows"), ((724, 724), "separate")])
def test_largest_rows_in_fp64(nel, kernels):
    """Meshes about as large as the rows of K may be in FP64, and larger ones."""
    print("case resident largest rows", nel, flush=True)
    K, f = _poisson(nel, False)
    A, b = K.to_scipy(), f.to_numpy()
    one = fa.solve(K, f, mode="cg", rtol=1e-8)
    assert one.kernels == kernels and one.operator == "sell"
    assert np.linalg.norm(b - A @ one.u) <= 1.01e-8 * np.linalg.norm(b)


@pytest.mark.parametrize("nel", [(15, 15), (24, 21), (71, 69), (7, 7, 7), (13, 12, 11), (40, 38, 36)])
@pytest.mark.parametrize("operator", ["lattice", "cells"])
def test_lattice_rows(nel, operator):
    print("case resident lattice rows", nel, operator, flush=True)
    forms = dict(lattice=1, cell_operator=-1) if operator == "lattice" else dict(lattice=0, cell_operator=1)
    K, f = _poisson(nel, operator == "lattice", **forms)
    for mode in ("mixed", "cg"):
        fa.set_tuning(K, cg_elems=0)
        _check(K, f, mode, operator, "rows")


def test_dofs_uploaded_after_the_pattern():
    """The context's dofs are no longer those of K's rows (more of them): positions of the rows are not to
    be had, and the separate kernels solve."""
    print("case resident dofs uploaded after the pattern", flush=True)
    K, _ = _poisson((12, 9), False, lattice=-1, cell_operator=-1)
    A, n = K.to_scipy(), K.n
    dofs = np.ascontiguousarray(2 * K.dh.cell_dofs, dtype=np.int64)
    K.ctx.call("fem_dofs_upload", 2 * n, 4, dofs.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)))
    b, u = np.ones(2 * n), np.zeros(2 * n)
    pd = ctypes.POINTER(ctypes.c_double)
    K.ctx.call("fem_matrix_upload", None, b.ctypes.data_as(pd))
    assert fa.solve(K, None, mode="cg", rtol=1e-12, download=False).kernels == "separate"
    K.ctx.call("fem_solution_download", u.ctypes.data_as(pd))
    assert np.linalg.norm(b[:n] - A @ u[:n]) <= 2e-12 * np.linalg.norm(b[:n])
    # fewer dofs than K has rows: f and u are too short
    few = np.minimum(K.dh.cell_dofs, n // 2)
    few = np.ascontiguousarray(few, dtype=np.int64)
    K.ctx.call("fem_dofs_upload", n // 2, 4, few.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)))
    with pytest.raises(fa.FemError, match="more rows than"):
        fa.solve(K, None, mode="cg", download=False)


@pytest.mark.parametrize("nel", [(90, 84, 80), (61, 140, 66), (200, 60, 50)])
def test_cell_bricks(nel):
    """More rows than the entries of which fit on chip: bricks of the cell form (uneven cuts,
    inhomogeneous prescribed rows on one side)."""
    print("case resident cell bricks", nel, flush=True)
    K, f = _poisson(nel, False)
    _check(K, f, "mixed", "cells", "bricks")


@pytest.mark.parametrize("nel", [(11, 11), (40, 23), (130, 64)])
def test_vector_field(nel):
    print("case resident vector field", nel, flush=True)
    g = _move(fa.generate_grid("Quadrilateral", nel, (0.0, 0.0), (2.0, 1.0)), nel, 6)
    ip = fa.Lagrange("RefQuadrilateral", 1) ** 2
    dh = fa.DofHandler(g).add("u", ip).close()
    K = fa.allocate_matrix(fa.MI355XCSC, dh)
    f = fa.allocate_vector(K)
    cv = fa.CellValues(fa.QuadratureRule("RefQuadrilateral", 2), ip)
    fa.assemble_global(fa.start_assemble(K, f), cv, fa.create_coloring(g), fa.ElasticityElement(nu=0.3))
    fa.add_point_load(K, f, [int(dh.cell_dofs[nel[1] // 2 * nel[0] + nel[0] // 2, 1])], [-1.0])   # an inner node
    ch = fa.ConstraintHandler(dh)
    ch.add(fa.Dirichlet("u", g.facetsets["left"] + g.facetsets["right"], lambda x, t: [0.0, 0.0])).close()
    fa.apply(K, f, ch)
    for mode in ("cg", "mixed"):
        fa.set_tuning(K, cg_elems=0)
        _check(K, f, mode, "sell", "rows")


@pytest.mark.parametrize("nel", [(40, 31), (14, 13, 12)])
@pytest.mark.parametrize("mode", ["cg", "mixed"])
def test_ends_without_convergence(nel, mode):
    """The step limit, and a tolerance below what FP64 reaches (the true residual stalls): the
    launch ends, and u is what it had reached."""
    print("case resident without convergence", nel, mode, flush=True)
    K, f = _poisson(nel, True)
    with pytest.raises(Exception, match="did not converge.* after 16 iterations"):
        fa.solve(K, f, mode=mode, rtol=1e-12, maxit=10)
    with pytest.raises(Exception, match="did not converge"):
        fa.solve(K, f, mode=mode, rtol=1e-19, maxit=20000)
    _check(K, f, mode, "sell" if mode == "cg" else "lattice", "rows")


@pytest.mark.parametrize("nel,forms,mode,kernels", [
    ((40, 31), dict(lattice=-1, cell_operator=-1), "cg", "rows"), ((14, 13, 12), {}, "mixed", "rows"),
    ((63, 64, 65), {}, "cg", "rows"), ((90, 84, 80), {}, "mixed", "bricks")])
def test_gives_up(nel, forms, mode, kernels):
    """A wait that runs out (no poll beyond the first allowed): every block leaves, the solve starts over on
    the separate kernels, which are used from then on until the tuning is set."""
    print("case resident gives up", nel, mode, flush=True)
    K, f = _poisson(nel, False, **forms)
    fa.set_wait_limit(K, 0)
    _gives_up(K, f, mode, kernels)


def _gives_up(K, f, mode, kernels):
    for _ in range(2):
        lost = fa.solve(K, f, mode=mode, rtol=1e-12)
        assert lost.kernels == "separate" and lost.gave_up
        fa.set_wait_limit(K)
    A, b = K.to_scipy(), f.to_numpy()
    assert np.linalg.norm(b - A @ lost.u) <= 2e-12 * np.linalg.norm(b)
    fa.set_tuning(K)
    back = fa.solve(K, f, mode=mode, rtol=1e-12)
    assert back.kernels == kernels and not back.gave_up and back.operator == lost.operator
    assert np.linalg.norm(back.u - lost.u) <= 1e-8 * np.linalg.norm(lost.u)


@pytest.mark.parametrize("nel,mode,kernels,limit", [
    ((40, 31), "cg", "rows", 0), ((14, 13, 12), "cg", "rows", 200_000), ((14, 13, 12), "mixed", "rows", 0),
    ((14, 13, 12), "mixed", "rows", 200_000), ((90, 84, 80), "mixed", "bricks", 2_000_000)])
def test_no_memory(nel, mode, kernels, limit):
    """Memory for the copy of the operator is not to be had (none, or its tables but not its values): the
    solve takes the separate kernels instead of failing, or bricks where those do fit."""
    print("case resident no memory", nel, mode, limit, flush=True)
    K, f = _poisson(nel, False)
    _no_memory(K, f, mode, kernels, limit)


def _no_memory(K, f, mode, kernels, limit):
    A, b = K.to_scipy(), f.to_numpy()
    small = "bricks" if mode == "mixed" and limit == 200_000 else "separate"
    for nbytes, ran in ((limit, small), (-1, kernels)):
        fa.set_copy_limit(K, nbytes)
        for _ in range(2):
            one = fa.solve(K, f, mode=mode, rtol=1e-12)
            assert one.kernels == ran and not one.gave_up
            assert np.linalg.norm(b - A @ one.u) <= 2e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("nel", [(40, 31), (14, 13, 12)])
@pytest.mark.parametrize("mode", ["cg", "mixed"])
@pytest.mark.parametrize("cg_elems", [0, 8])
@pytest.mark.parametrize("where,value", [("K", np.nan), ("K", np.inf), ("f", np.nan), ("f", np.inf)])
def test_no_numbers(nel, mode, cg_elems, where, value):
    """A NaN or an infinity in K or f: the solve ends and says that it did not converge."""
    print("case resident no numbers", nel, mode, cg_elems, where, value, flush=True)
    K, f = _poisson(nel, True, cg_elems=cg_elems)
    if where == "K":
        nz = K.nzval()
        nz[K.nnz // 2] = value
        K.set_nzval(nz)
    else:
        b = f.to_numpy()
        b[len(b) // 2] = value
        K.ctx.call("fem_matrix_upload", None, b.ctypes.data_as(ctypes.POINTER(ctypes.c_double)))
    with pytest.raises(fa.FemConvergenceError, match="did not converge"):
        fa.solve(K, f, mode=mode, rtol=1e-10, maxit=3200)


@pytest.mark.parametrize("nel", [(40, 31), (14, 13, 12)])
@pytest.mark.parametrize("delta", [0.5, 1e-3])
def test_hand_overs(nel, delta):
    """Many hand-overs (δ = 0.5) and few."""
    print("case resident hand-overs", nel, delta, flush=True)
    K, f = _poisson(nel, False)
    A, b = K.to_scipy(), f.to_numpy()
    one = fa.solve(K, f, mode="mixed", rtol=1e-12, inner_rtol=delta)
    assert one.kernels == "rows"
    assert one.outer_iterations >= (10 if delta == 0.5 else 3)
    assert np.linalg.norm(b - A @ one.u) <= 2e-12 * np.linalg.norm(b)
    assert abs(np.linalg.norm(b - A @ one.u) / np.linalg.norm(b) - one.relres) <= 1e-13


class _InPlace:
    """K.nzval for torch, through an address that is asked for once."""

    def __init__(self, K):
        p, n = ctypes.c_void_p(), ctypes.c_int64(0)
        K.ctx.call("fem_device_pointer", 0, ctypes.byref(p), ctypes.byref(n))
        self.__cuda_array_interface__ = dict(shape=(n.value,), typestr="<f8", data=(p.value, False), version=2)


_FORMS = [((40, 31), dict(lattice=-1, cell_operator=-1)), ((40, 31), dict(cell_operator=-1)), ((40, 31), {}),
          ((14, 13, 12), dict(lattice=-1, cell_operator=-1)), ((14, 13, 12), {})]


@pytest.mark.parametrize("nel,forms,mode,cg_elems",
                         [(*x, mode, e) for x in _FORMS for mode in ("mixed", "cg") for e in (0, 8)] +
                         [((90, 84, 80), {}, "mixed", 0)])
def test_K_written_in_place(nel, forms, mode, cg_elems):
    """A caller keeps K's address and writes K in place between solves: every solve is of the K
    that is there, on every form of the rows (the last case: bricks), resident or not."""
    print("case resident K in place", nel, forms, mode, cg_elems, flush=True)
    import torch
    K, f = _poisson(nel, False, cg_elems=cg_elems, **forms)
    nz = torch.as_tensor(_InPlace(K), device="cuda")
    one = fa.solve(K, f, mode=mode, rtol=1e-12)
    assert one.kernels == ("separate" if cg_elems else "bricks" if nel == (90, 84, 80) else "rows")
    u = one.u
    for scale in (2.0, 0.25):
        nz *= scale
        torch.cuda.synchronize()
        now = fa.solve(K, f, mode=mode, rtol=1e-12)
        u = u / scale
        A, b = K.to_scipy(), f.to_numpy()
        assert np.linalg.norm(b - A @ now.u) <= 2e-12 * np.linalg.norm(b)
        assert np.linalg.norm(now.u - u) <= 1e-8 * np.linalg.norm(u)


@pytest.mark.parametrize("nel", [(1, 1, 1), (2, 1, 1), (3, 3, 2), (5, 4, 4), (60, 1, 1), (2, 30, 3), (11, 12, 11),
                                 (13, 11, 11)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_q2_elements(nel, precision):
    """Parts of the Q2 element matrices: one cell, one block, blocks of up to six cells, one cell
    more than fits (13×11×11 > 6 · 256), FP64 and FP32 matrices in both solvers."""
    print("case resident q2 elements", nel, precision, flush=True)
    g = _move(fa.generate_grid("Hexahedron", nel, (0.0, 0.0, 0.0), (1.0, 0.8, 0.9)), nel, 7)
    ip = fa.Lagrange("RefHexahedron", 2) ** 3
    dh = fa.DofHandler(g).add("u", ip).close()
    K = fa.allocate_matrix(fa.MI355XCSC, dh)
    f = fa.allocate_vector(K)
    cv = fa.CellValues(fa.QuadratureRule("RefHexahedron", 3), ip)
    E = np.random.default_rng(4).uniform(0.5, 2.0, g.ncells)
    fa.assemble_global(fa.start_assemble(K, f), cv, fa.create_coloring(g), fa.ElasticityElement(E=E, nu=0.3),
                       precision=precision)
    fv = fa.FacetValues(fa.FacetQuadratureRule("RefHexahedron", 3), ip)
    fa.apply_traction(K, f, fv, g.facetsets["right"], (0.1, 0.0, -1.0))
    ch = fa.ConstraintHandler(dh)
    ch.add(fa.Dirichlet("u", g.facetsets["left"], lambda x, t: [0.0, 0.01, 0.0])).close()
    fa.apply(K, f, ch)
    # (60 slices 48 times as wide as thick: the FP32 recurrence does not get to 1e-12 with the
    # separate kernels either, 8e-12 and 5e-10)
    for mode in ("cg",) if nel == (60, 1, 1) else ("cg", "mixed"):
        fa.set_tuning(K, cg_elems=0)
        _check(K, f, mode, "elements", "separate" if nel == (13, 11, 11) else "elements")
        if nel == (5, 4, 4):
            fa.set_tuning(K, cg_elems=0)
            for limit in (0, 500_000):
                _no_memory(K, f, mode, "elements", limit)
            fa.set_wait_limit(K, 0)
            _gives_up(K, f, mode, "elements")


@pytest.mark.parametrize("grids", [
    [("Quadrilateral", (2, 2))], [("Hexahedron", (2, 1, 1))],
    [("Quadrilateral", (2, 2)), ("Quadrilateral", (71, 69)), ("Quadrilateral", (3, 300)), ("Quadrilateral", (16, 15))],
    [("Hexahedron", (9, 8, 7)), ("Quadrilateral", (40, 41)), ("Hexahedron", (30, 31, 32)), ("Hexahedron", (2, 2, 90)),
     ("Quadrilateral", (180, 170)), ("Hexahedron", (7, 7, 7)), ("Hexahedron", (2, 1, 1))]])
def test_batch(grids):
    """Systems sharing a launch: of one block and of many, 2D and 3D, one with f = 0 (all of
    its nodes prescribed).  First a
    tolerance out of reach (they stall, the separate kernels take over and end at the step
    limit), then one within reach, twice."""
    print("case resident batch", grids, flush=True)
    import scipy.sparse as sp
    b = BatchedPoisson(0)
    for i, (ct, nel) in enumerate(grids):
        k = np.exp(np.random.default_rng(i).normal(0.0, 0.5, int(np.prod(nel))))
        g, dh, colors, ch, k = poisson_problem(ct, nel, k)
        b.add(g, dh, colors, ch, k)
    b.finalize()
    if len(grids) > 1:      # (one unknown is solved exactly)
        with pytest.raises(fa.FemError, match="missed rtol"):
            b.run("mixed", rtol=1e-18, maxit=2000)
    us = []
    for _ in range(2):
        res = b.run("mixed", rtol=1e-11)
        assert res.converged == len(grids) and np.all(res.completion_ms > 0) and np.all(res.kernels == 1)
        us.append([b.download(i) for i in range(len(grids))])
    for i, p in enumerate(b.problems):
        nz, f, u = us[0][i]
        A = sp.csc_matrix((nz, p["rowval"] - 1, p["colptr"] - 1), shape=(p["ndofs"], p["ndofs"]))
        assert np.linalg.norm(f - A @ u) <= 1e-11 * np.linalg.norm(f) * 1.0001
        assert np.array_equal(u, us[1][i][2])
    b.close()


def test_batch_gives_up():
    """A launch that is not to be had: no memory for it, or a block of it gives up (the 2D problems
    are of one block each and wait for nobody).  The separate kernels solve its problems."""
    print("case resident batch gives up", flush=True)
    import scipy.sparse as sp
    grids = [("Quadrilateral", (9, 8)), ("Hexahedron", (30, 31, 32)), ("Quadrilateral", (7, 7)), ("Hexahedron", (9, 8, 7))]
    b = BatchedPoisson(0)
    for i, (ct, nel) in enumerate(grids):
        k = np.exp(np.random.default_rng(i).normal(0.0, 0.5, int(np.prod(nel))))
        b.add(*poisson_problem(ct, nel, k))
    b.finalize()
    # memory for the 2D rows but not for the 3D ones; then the wait limit
    for limit, polls, kernels in ((200_000, -1, [1, 0, 1, 0]), (0, -1, [0, 0, 0, 0]), (-1, -1, [1, 1, 1, 1]),
                                  (-1, 0, [1, 0, 1, 0]), (-1, -1, [0, 0, 0, 0])):
        b.set_copy_limit(limit)
        b.set_wait_limit(polls)
        res = b.run("mixed", rtol=1e-11)
        assert res.converged == len(grids) and list(res.kernels) == kernels
        for i, p in enumerate(b.problems):
            nz, f, u = b.download(i)
            A = sp.csc_matrix((nz, p["rowval"] - 1, p["colptr"] - 1), shape=(p["ndofs"], p["ndofs"]))
            assert np.linalg.norm(f - A @ u) <= 1e-11 * np.linalg.norm(f) * 1.0001
    b.close()


def test_contexts_on_threads():
    """Contexts on host threads of their own, whose one-launch solves want different amounts of LDS of
    the same kernels: each gets the u it gets alone, by the same kernels."""
    print("case resident contexts on threads", flush=True)
    from concurrent.futures import ThreadPoolExecutor
    systems = [(_poisson(nel, False), mode) for nel, mode in (
        ((24, 20, 17), "cg"), ((60, 58, 56), "cg"), ((47, 43, 41), "mixed"), ((14, 13, 12), "mixed"))]
    alone = [fa.solve(K, f, mode=mode, rtol=1e-11).u for (K, f), mode in systems]

    def repeat(i):
        (K, f), mode = systems[i]
        return [fa.solve(K, f, mode=mode, rtol=1e-11) for _ in range(20)]

    with ThreadPoolExecutor(len(systems)) as pool:
        for i, results in enumerate(pool.map(repeat, range(len(systems)))):
            for r in results:
                assert r.kernels == "rows" and not r.gave_up and np.array_equal(r.u, alone[i])


def _fan(m):
    """m quadrilaterals around one node, whose column has 2 m + 1 entries; u = 0 on two facets."""
    ang = np.arange(2 * m) * (np.pi / m)
    rad = np.where(np.arange(2 * m) % 2, 1.1, 1.0)
    nodes = np.vstack([[0.0, 0.0], np.stack([rad * np.cos(ang), rad * np.sin(ang)], axis=1)])
    cells = np.array([[1, 2 + 2 * i, 3 + 2 * i, 2 + (2 * i + 2) % (2 * m)] for i in range(m)])
    g = fa.Grid("Quadrilateral", cells, nodes, {"edge": [(1, 2), (m // 2, 3)]})
    dh = fa.DofHandler(g).add("u", fa.Lagrange(g.refshape, 1)).close()
    ch = fa.ConstraintHandler(dh)
    ch.add(fa.Dirichlet("u", g.facetsets["edge"], lambda x, t: 0.0)).close()
    return g, dh, fa.create_coloring(g), ch, 1.0 + np.arange(m) / m


def test_batch_of_which_some_do_not_fit():
    """One problem with a column of 29 entries and one of 895 k rows among problems that fit: only those
    two take the separate kernels.  One of 13 entries shares the launch of the 2D problems."""
    print("case resident batch of which some do not fit", flush=True)
    import scipy.sparse as sp
    b = BatchedPoisson(0)
    setups = [_fan(14)]
    for ct, nel in (("Quadrilateral", (950, 940)), ("Quadrilateral", (40, 41)), ("Hexahedron", (9, 8, 7))):
        setups.append(poisson_problem(ct, nel, np.exp(np.random.default_rng(1).normal(0.0, 0.3, int(np.prod(nel))))))
    setups.append(_fan(6))
    for s in setups:
        b.add(*s)
    b.finalize()
    res = b.run("fp64", rtol=1e-9)
    assert res.converged == 5 and list(res.kernels) == [0, 0, 1, 1, 1]
    for i, p in enumerate(b.problems):
        nz, f, u = b.download(i)
        A = sp.csc_matrix((nz, p["rowval"] - 1, p["colptr"] - 1), shape=(p["ndofs"], p["ndofs"]))
        assert np.linalg.norm(f) > 0 and np.linalg.norm(f - A @ u) <= 1e-9 * np.linalg.norm(f) * 1.0001
    b.close()
