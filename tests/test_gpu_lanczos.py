"""The Lanczos kernels at their edges: a vector shorter than one workgroup's
rows (2,048), just below and above, more workgroups than the update adds up
itself (16), more basis vectors than one tile (64), and odd design counts;
loads against scipy on the assembled K and G; start vectors of no positive
norm are refused."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as sla

import shellgpu as sg
from shellgpu.problems import Cylinder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nc,nb,nev", [(4, 8, 1, 3), (9, 34, 1, 4), (9, 35, 3, 4), (14, 30, 2, 24), (40, 140, 1, 3)])
def test_loads_match_scipy(na, nc, nb, nev):
    cyl = Cylinder(na, nc)
    thick = np.random.default_rng(na).uniform(0.0015, 0.0025, (nb, cyl.nelems))
    ctx = sg.Context(0)
    ctx.set_mesh(cyl.conn, cyl.Xpts)
    ctx.set_material(70e9, 0.3)
    ctx.set_bcs(*cyl.bcs())
    ctx.set_designs(thick)
    B = ctx.buckling(sigma=0.0, nev=nev, max_lanczos=180, tol=1e-10)
    B.solve(force=cyl.edge_load(1.0))
    lam, err = B.eigenvalues()
    info = B.info()
    if nev > 20:
        assert info["steps"] > 64
    K, G = ctx.matrix(), ctx.matrix()
    ctx.assemble_mattype(sg.STIFFNESS, K)
    ctx.assemble_mattype(sg.GEOMETRIC, G, ctx.vector(info["path"]))
    rowp, cols = ctx.pattern()
    nodes, mask = cyl.bcs()
    free = np.ones((cyl.nnodes, 6), bool)
    for k in range(6):
        free[nodes[(mask >> k) & 1 == 1], k] = False
    free = np.where(free.ravel())[0]
    for d in range(nb):
        k, g = (sp.bsr_matrix((m.design_values(d), cols, rowp)).tocsc()[free][:, free] for m in (K, G))
        # the loads of smallest magnitude: largest |theta| of -G x = theta K x
        lu = sla.splu(k)
        op = sla.LinearOperator(k.shape, matvec=lu.solve, dtype=float)
        theta = sla.eigsh(-g, nev, M=k, Minv=op, which="LM", return_eigenvectors=False, ncv=4 * nev + 40)
        ref = np.sort(1.0 / theta[np.argsort(-np.abs(theta))])
        got = np.sort(lam[d])
        # converged to 1e-10; K has a condition number up to 1e9
        assert np.abs(got - ref).max() <= 1e-8 * np.abs(ref).max(), (got, ref)
        # the modes: K-normalised, residuals of the pencil
        for j in range(min(nev, 3)):
            phi = B.eigenvector(j)[d][free]
            assert abs(phi @ (k @ phi) - 1.0) <= 1e-8
    B.destroy()
    ctx.close()


def _context(nb, rho=2700.0, same=False, clamped=False):
    cyl = Cylinder(4, 8)
    ctx = sg.Context(0)
    ctx.set_mesh(cyl.conn, cyl.Xpts)
    ctx.set_material(70e9, 0.3, rho)
    if clamped:
        ctx.set_bcs(np.arange(cyl.nnodes, dtype=np.int32), np.full(cyl.nnodes, 63, np.int32))
    else:
        ctx.set_bcs(*cyl.bcs())
    ctx.set_designs(np.full((nb, cyl.nelems), 0.002) if same else
                    np.random.default_rng(1).uniform(0.0015, 0.0025, (nb, cyl.nelems)))
    return cyl, ctx


@pytest.mark.parametrize("nb", [1, 2])
@pytest.mark.parametrize("rho,clamped", [(0.0, False), (-2700.0, False), (2700.0, True)])
def test_frequencies_without_a_positive_mass_are_refused(rho, clamped, nb):
    """M zero or negative, or no free dof: the start vector's M norm is not
    positive, and no frequencies exist."""
    _, ctx = _context(nb, rho, clamped=clamped)
    fr = ctx.frequency(sigma=0.0, nev=2, max_lanczos=40, tol=1e-10)
    with pytest.raises(sg.ShellGPUError, match="error 6"):
        fr.solve()
    fr.destroy()
    ctx.close()


# sigma 0: buckling mode (identical designs) and shift estimate; 1e5: given shift
@pytest.mark.parametrize("sigma", [0.0, 1e5])
@pytest.mark.parametrize("nb,same", [(1, False), (2, False), (2, True)])
def test_buckling_without_a_free_dof_is_refused(sigma, nb, same):
    cyl, ctx = _context(nb, same=same, clamped=True)
    B = ctx.buckling(sigma=sigma, nev=2, max_lanczos=40, tol=1e-10)
    with pytest.raises(sg.ShellGPUError, match="error 6"):
        B.solve(force=cyl.edge_load(1.0))
    B.destroy()
    ctx.close()
