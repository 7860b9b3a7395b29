"""The multifrontal factor (the default SHELLGPU_FACTOR) on matrices of known
solution: meshes of one front, fronts shorter and longer than a pivot block,
last blocks of every remainder, fronts longer than the staged vector pieces, the
stiffness of a shell of large fronts, batches of designs, several vectors per design, the captured solve, and
designs factored a few at a time where the memory left asks for it."""
import numpy as np
import pytest
import scipy.sparse as sp

import shellgpu as sg
from shellgpu.problems import BoxBeam, Cylinder

from helpers import random_mesh

pytestmark = pytest.mark.gpu

# diagonally dominant matrices with rows' off-diagonal sums at most 0.9 of
# the diagonal, equilibrated to about 1: condition number below 40, so the
# forward error of a backward stable solve is below ~ 40 eps times a modest
# factor (100 here) of the depth of the sums
TOL = 40 * 100 * 2.3e-16


def spd_values(rowp, cols, seed):
    """Symmetric diagonally dominant block values on a node pattern."""
    rng = np.random.default_rng(seed)
    n = len(rowp) - 1
    rows = np.repeat(np.arange(n), np.diff(rowp))
    v = rng.standard_normal((len(cols), 6, 6))
    t = np.lexsort((rows, cols))  # position of the transposed block
    up = rows < cols
    v[up] = v[t[up]].transpose(0, 2, 1)
    d = np.where(rows == cols)[0]
    v[d] = v[d] + v[d].transpose(0, 2, 1)
    off = np.zeros((n, 6))
    np.add.at(off, rows, np.abs(v).sum(2))
    i = np.arange(6)
    v[d[:, None], i, i] = 0.0
    off = np.zeros((n, 6))
    np.add.at(off, rows, np.abs(v).sum(2))
    v[d[:, None], i, i] = off / 0.9
    return v / off.mean()


def make(mesh, nb, bcs=True):
    ctx = sg.Context(0)
    ctx.set_mesh(mesh[0], mesh[1])
    ctx.set_material(70e9, 0.3)
    if bcs:
        ctx.set_bcs(np.arange(0, len(mesh[1]), 7), np.arange(0, len(mesh[1]), 7) % 63 + 1)
    ctx.set_designs(np.full((nb, len(mesh[0])), 0.002))
    return ctx


def bc_mask(nn):
    m = np.zeros((nn, 6), bool)
    nodes = np.arange(0, nn, 7)
    for k in range(6):
        m[nodes, k] = ((nodes % 63 + 1) >> k) & 1 == 1
    return m.ravel()


def system(ctx, nb, bcs, seed):
    """Values of nb designs, and right-hand sides b of known x."""
    rowp, cols = ctx.pattern()
    nn = len(rowp) - 1
    vals = np.stack([spd_values(rowp, cols, seed + d) for d in range(nb)])
    x = np.random.default_rng(seed + 99).standard_normal((nb, 6 * nn))
    b = np.empty_like(x)
    for d in range(nb):
        A = sp.bsr_matrix((vals[d], cols, rowp), shape=(6 * nn, 6 * nn))
        if bcs:
            m = bc_mask(nn)
            b[d] = np.where(m, x[d], A @ np.where(m, 0.0, x[d]))
        else:
            b[d] = A @ x[d]
    return vals, x, b


MESHES = {
    "1x3": lambda: (Cylinder(1, 3).conn, Cylinder(1, 3).Xpts),      # one front of 36 pivots
    "4x8": lambda: (Cylinder(4, 8).conn, Cylinder(4, 8).Xpts),      # two leaves
    "7x13": lambda: (Cylinder(7, 13).conn, Cylinder(7, 13).Xpts),
    "plate9x10": lambda: random_mesh(9, 10, 3),
    "33x65": lambda: (Cylinder(33, 65).conn, Cylinder(33, 65).Xpts),
    "box": lambda: (lambda b: (b.conn, b.Xpts))(BoxBeam(ns=40, nc=12, nh=5, nribs=4)),  # junctions
    "flat0": lambda: (Cylinder(12, 20).conn, 0.0 * Cylinder(12, 20).Xpts),  # coordinates say nothing
    "201x402": lambda: (Cylinder(201, 402).conn, Cylinder(201, 402).Xpts),  # fronts of 2,400 pivots
}


@pytest.mark.parametrize("mesh,nb,bcs", [("1x3", 1, False), ("4x8", 2, True), ("7x13", 3, True),
                                         ("plate9x10", 1, False), ("33x65", 2, True), ("box", 1, True),
                                         ("flat0", 1, False), ("201x402", 1, True)])
def test_known_solutions(mesh, nb, bcs):
    ctx = make(MESHES[mesh](), nb, bcs)
    vals, x, b = system(ctx, nb, bcs, 5)
    A = ctx.matrix()
    A.set_values(vals)
    if bcs:
        A.apply_bcs()
    F = ctx.factor()
    for _ in range(2):  # a second factor into the same buffers
        F.compute(A)
        y = ctx.vector()
        F.apply(ctx.vector(b), y)
        got = y.download().reshape(nb, -1)
        assert np.linalg.norm(got - x) <= TOL * np.linalg.norm(x)
    # in place
    y = ctx.vector(b)
    F.apply(y, y)
    assert np.array_equal(y.download().reshape(nb, -1), got)
    F.destroy()
    ctx.close()


def test_shell_stiffness_of_large_fronts():
    """K of a 201 x 402 cylinder, fronts of 2,400 pivots: one vector, and
    eleven through the factor of one design.  The solve multiplies by explicit
    inverses of the fronts' Cholesky factors, whose residuals grow with their
    condition, at most the root of K's (below 1e9); 1e3 covers the sums'
    lengths (up to 3,600 terms, 14 levels): 1e3 x 3.2e4 eps."""
    cyl = Cylinder(201, 402)
    thick = np.random.default_rng(51).uniform(0.0015, 0.0025, (1, cyl.nelems))
    ctx = sg.Context(0)
    ctx.set_mesh(cyl.conn, cyl.Xpts)
    ctx.set_material(70e9, 0.3)
    ctx.set_bcs(*cyl.bcs())
    ctx.set_designs(thick)
    K = ctx.matrix()
    ctx.assemble_mattype(sg.STIFFNESS, K)
    rowp, cols = ctx.pattern()
    n = 6 * cyl.nnodes
    A = sp.bsr_matrix((K.design_values(0), cols, rowp), shape=(n, n)).tocsr()
    F = ctx.factor()
    F.compute(K)
    norm = abs(A).sum(1).max()
    for vectors in (1, 11):
        ctx.set_designs(np.repeat(thick, vectors, 0))  # one factor, so many vectors
        b = np.random.default_rng(52).standard_normal((vectors, n))
        db = ctx.vector(b)
        ctx.vec_zero_bcs(db)
        b = db.download().reshape(vectors, n)
        y = ctx.vector()
        F.apply(db, y)
        for x, r in zip(y.download().reshape(vectors, n), b):
            eta = np.abs(A @ x - r).max() / (norm * np.abs(x).max() + np.abs(r).max())
            print(vectors, "vectors: backward error", eta)
            assert eta <= 1e3 * 3.2e4 * 2.3e-16
    F.destroy()
    ctx.close()


def test_indefinite_matrix_is_refused_and_named():
    mesh = MESHES["7x13"]()
    ctx = make(mesh, 3, False)
    vals, x, b = system(ctx, 3, False, 8)
    rowp, cols = ctx.pattern()
    diag = [rowp[i] + int(np.where(cols[rowp[i]:rowp[i + 1]] == i)[0][0]) for i in (40,)]
    bad = vals.copy()
    bad[1, diag[0], 2, 2] *= -1.0
    A = ctx.matrix()
    F = ctx.factor()
    A.set_values(bad)
    with pytest.raises(sg.ShellGPUError, match=r"in the Cholesky factorisation \(design 1\)"):
        F.compute(A)
    with pytest.raises(sg.ShellGPUError):
        F.apply(ctx.vector(b), ctx.vector())
    A.set_values(vals)
    F.compute(A)
    y = ctx.vector()
    F.apply(ctx.vector(b), y)
    assert np.linalg.norm(y.download() - x.ravel()) <= TOL * np.linalg.norm(x)
    ctx.close()


def test_captured_solve_matches_direct(monkeypatch):
    ctx = make(MESHES["7x13"](), 2)
    vals, x, b = system(ctx, 2, True, 11)
    A = ctx.matrix()
    A.set_values(vals)
    A.apply_bcs()
    F, G = ctx.factor(), ctx.factor()
    for f in (F, G):
        f.compute(A)
    y, z = ctx.vector(), ctx.vector()
    F.apply(ctx.vector(b), y)
    monkeypatch.setenv("SHELLGPU_GRAPH", "1")
    for rep in range(4):
        rhs = b * (rep + 1)
        G.apply(ctx.vector(rhs), z)
        F.apply(ctx.vector(rhs), y)  # eager work between the replays
        assert np.array_equal(y.download(), z.download())
    ctx.close()


@pytest.mark.parametrize("cases", [1, 2, 5, 8, 11, 16, 19])
def test_load_cases_share_one_factor(cases):
    """Identical designs: a factor of one design solves all vectors (16, or up
    to 8, at a time); every load case as if it were alone."""
    cyl = Cylinder(9, 16)
    rng = np.random.default_rng(3)
    f = rng.standard_normal((cases, 6 * cyl.nnodes))
    paths, lam = {}, {}
    for nb in (1, cases):
        ctx = sg.Context(0)
        ctx.set_mesh(cyl.conn, cyl.Xpts)
        ctx.set_material(70e9, 0.3)
        ctx.set_bcs(*cyl.bcs())
        ctx.set_designs(np.full((nb, cyl.nelems), 0.002))
        p, v = [], []
        for c in range(0, cases, nb):
            B = ctx.buckling(sigma=0.0, nev=2, max_lanczos=90, tol=1e-10)
            B.solve(force=f[c:c + nb])
            p.append(B.info()["path"])
            v.append(B.eigenvalues()[0])
            B.destroy()
        paths[nb], lam[nb] = np.concatenate(p), np.concatenate(v)
        ctx.close()
    # paths solved to 1e-12 by GMRES, condition ~ 1e6; loads to 1e-10
    assert np.linalg.norm(paths[cases] - paths[1]) <= 1e-8 * np.linalg.norm(paths[1])
    assert np.abs(lam[cases][:, 0] - lam[1][:, 0]).max() <= 1e-8 * np.abs(lam[1]).max()


def test_block_lanczos_solves_blocks(monkeypatch):
    cyl = Cylinder(10, 20)
    thick = np.random.default_rng(2).uniform(0.0015, 0.0025, (2, cyl.nelems))
    out = []
    for block in ("1", "4"):
        monkeypatch.setenv("SHELLGPU_LANCZOS_BLOCK", block)
        ctx = sg.Context(0)
        ctx.set_mesh(cyl.conn, cyl.Xpts)
        ctx.set_material(70e9, 0.3)
        ctx.set_bcs(*cyl.bcs())
        ctx.set_designs(thick)
        B = ctx.buckling(sigma=0.0, nev=3, max_lanczos=100, tol=1e-10)
        B.solve(force=cyl.edge_load(1.0))
        out.append(B.eigenvalues()[0])
        B.destroy()
        ctx.close()
    assert np.abs(out[0] - out[1]).max() <= 1e-8 * np.abs(out[0]).max()


@pytest.mark.parametrize("mesh,levels,largest", [("1x3", 1, 36), ("4x8", 2, 192)])
def test_info_describes_the_fronts(mesh, levels, largest):
    """4 x 8: 40 nodes, a separator of 8 between leaves of 8 and of 24; the
    largest front has 24 pivot and 8 boundary nodes."""
    with make(MESHES[mesh](), 2) as ctx:
        F = ctx.factor()
        assert F.info()[:2] == (levels, largest)
        F.destroy()


def test_order_follows_the_mesh_and_its_nodes():
    """The factors of a context share one order; new nodes or a new mesh get
    the order, and so the bits, that a context made with them has."""
    cyl = Cylinder(12, 20)
    nodes = [cyl.Xpts, cyl.Xpts * np.array([1.0, 9.0, 0.2]), cyl.Xpts]
    other = random_mesh(9, 10, 3)

    def solves(ctx, seed):
        vals, x, b = system(ctx, 1, False, seed)
        A = ctx.matrix()
        A.set_values(vals)
        out = []
        for _ in range(2):
            F, y = ctx.factor(), ctx.vector()
            F.compute(A)
            F.apply(ctx.vector(b), y)
            out.append(y.download())
            assert np.linalg.norm(out[-1] - x.ravel()) <= TOL * np.linalg.norm(x)
            F.destroy()
        A.destroy()
        assert np.array_equal(*out)
        return out[0]

    got = []
    with make((cyl.conn, nodes[0]), 1, False) as ctx:
        for X in nodes:
            ctx.set_nodes(X)
            got.append(solves(ctx, 41))
        ctx.set_mesh(*other)
        ctx.set_designs(np.full((1, len(other[0])), 0.002))
        got.append(solves(ctx, 42))
    for mesh, seed, g in [((cyl.conn, X), 41, h) for X, h in zip(nodes, got)] + [(other, 42, got[-1])]:
        with make(mesh, 1, False) as ctx:
            assert np.array_equal(solves(ctx, seed), g)


def test_every_part_of_a_mesh_needs_a_seed():
    """Two cylinders without a common node: refused until the ordering seed
    reaches both; then each is solved."""
    cyl = Cylinder(7, 13)
    nn = cyl.nnodes
    mesh = np.concatenate([cyl.conn, cyl.conn + nn]), np.concatenate([cyl.Xpts, cyl.Xpts + 3.0])
    with make(mesh, 1) as ctx:
        for seed in ([], [3]):
            ctx.set_ordering_seed(seed)
            with pytest.raises(sg.ShellGPUError, match="disconnected"):
                ctx.factor()
        ctx.set_ordering_seed([3, 2 * nn])
        with pytest.raises(sg.ShellGPUError, match="out of range"):
            ctx.factor()
        ctx.set_ordering_seed([3, nn + 5])
        vals, x, b = system(ctx, 1, True, 31)
        A = ctx.matrix()
        A.set_values(vals)
        A.apply_bcs()
        F = ctx.factor()
        F.compute(A)
        y = ctx.vector()
        F.apply(ctx.vector(b), y)
        assert np.linalg.norm(y.download() - x.ravel()) <= TOL * np.linalg.norm(x)
        F.destroy()


def test_designs_are_factored_in_the_memory_that_is_left():
    """Workspace for all designs at once does not fit beside the panels: the
    factor takes fewer at a time, with the same bits."""
    nb, gib = 12, 1 << 27  # gib: doubles
    cyl = Cylinder(100, 200)
    # per design 302 MiB of panels and 259 MiB of workspace (3.0 GiB for 12)
    panels, work = nb * 302 / 1024, nb * 259 / 1024
    ctx = make((cyl.conn, cyl.Xpts), nb)
    rowp, cols = ctx.pattern()
    base = spd_values(rowp, cols, 21)
    scale = 1.0 + 0.1 * np.arange(nb)
    x = np.random.default_rng(22).standard_normal((nb, 6 * cyl.nnodes))
    free = ~bc_mask(cyl.nnodes)
    x[:, ~free] = 0.0
    A = sp.bsr_matrix((base, cols, rowp), shape=(6 * cyl.nnodes,) * 2)
    b = np.stack([scale[d] * np.where(free, A @ x[d], 0.0) for d in range(nb)])
    K = ctx.matrix()
    K.set_values(base[None] * scale[:, None, None, None])
    K.apply_bcs()
    db, y = ctx.vector(b), ctx.vector()

    def solve():
        F = ctx.factor()
        assert abs(F.info()[2] - panels) <= 0.02 * panels
        F.compute(K)
        F.apply(db, y)
        F.destroy()
        return y.download().reshape(nb, -1)

    ref = solve()
    assert np.linalg.norm(ref - x) <= TOL * np.linalg.norm(x)
    # room for the panels and 0.7 of the workspace: for 6 designs, not for 12
    room = sg.DeviceArray(ctx, int((panels + 0.7 * work) * gib))
    held, size = [], 32 * gib
    while size >= gib // 8:
        try:
            held.append(sg.DeviceArray(ctx, size))
        except sg.ShellGPUError:
            size //= 4
    room.free()
    try:
        assert np.array_equal(solve(), ref)
    finally:
        for h in held:
            h.free()
    ctx.close()
