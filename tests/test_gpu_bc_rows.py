"""BC rows of assembled matrices: written by the element kernels up to 16,384
element copies, by a kernel of their own above.  Both against the same matrix
assembled without BCs, with the rows of the identity put in on the host, bit
for bit; a node listed twice carries both masks."""
import numpy as np
import pytest

import shellgpu as sg
from helpers import random_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nb", [(1, 1, 1), (5, 3, 2), (128, 1, 128), (128, 1, 129)])
def test_bc_rows_of_every_matrix(nx, ny, nb):
    conn, X = random_mesh(nx, ny, seed=nx + ny)
    nn, ne = X.shape[0], conn.shape[0]
    rng = np.random.default_rng(nb)
    thick = rng.uniform(0.002, 0.02, (nb, ne))
    u = 1e-3 * rng.standard_normal((nb, 6 * nn))
    nodes = np.array([0, nn - 1, 1, nn - 1], np.int32)
    mask = np.array([0x3F, 0x05, 0x38, 0x12], np.int32)
    rows = np.zeros((nn, 6), bool)
    for n, k in zip(nodes, mask):
        rows[n] |= (k >> np.arange(6)) & 1 == 1
    out = []
    for bcs in (True, False):
        with sg.Context(0) as ctx:
            ctx.set_mesh(conn, X)
            ctx.set_material(70e9, 0.3)
            if bcs:
                ctx.set_bcs(nodes, mask)
            ctx.set_designs(thick)
            du, A = ctx.vector(u), ctx.matrix()
            res = []
            for kind in (sg.STIFFNESS, sg.GEOMETRIC, sg.TANGENT_NONLINEAR, sg.GEOMETRIC_FD, sg.MASS):
                ctx.assemble_mattype(kind, A, du)
                res += [A.design_values(0), A.design_values(nb - 1)]
            R = ctx.vector()
            ctx.assemble_jacobian(A, R=R, u=du, model=sg.NONLINEAR, gamma=2.0)
            res += [A.design_values(0), A.design_values(nb - 1)]
            rowp, cols = ctx.pattern()
            out.append([np.array(r).reshape(-1, 6, 6) for r in res])
    brow = np.repeat(np.arange(nn), np.diff(rowp))
    eye = np.eye(6)
    for got, ref in zip(*out):
        ref = np.where(rows[brow][:, :, None], (brow == cols)[:, None, None] * eye, ref)
        assert np.array_equal(got, ref)
