"""Coordinate-derivative kernels at the edges of their launch: element counts
around the 32 of a workgroup, and more designs than one launch takes."""
import numpy as np
import pytest

import pyoracle as O
import shellgpu as sg
from helpers import random_mesh
from shellgpu.problems import Cylinder

pytestmark = pytest.mark.gpu


def mesh_ctx(conn, X, thick):
    ctx = sg.Context(0)
    ctx.set_mesh(conn, X)
    ctx.set_material(70e9, 0.3)
    ctx.set_designs(thick)
    return ctx


def five_point(f, t, h):
    return (f(t - 2 * h) - 8 * f(t - h) + 8 * f(t + h) - f(t + 2 * h)) / (12 * h)


@pytest.mark.parametrize("nx,ny", [(1, 1), (31, 1), (8, 4), (11, 3)])
def test_element_counts_around_a_workgroup(nx, ny):
    # elements of the size of a 3 x 3 mesh of the unit square, so that the
    # five-point differences (h = 3e-4, truncation ~ h^4) keep 1e-8
    conn, X = random_mesh(nx, ny, seed=7 * nx + ny)
    X = X * np.array([nx / 3, ny / 3, 1.0])
    nn, ne = X.shape[0], conn.shape[0]
    rng = np.random.default_rng(nx)
    thick = rng.uniform(0.002, 0.02, (2, ne))
    phi, psi = rng.standard_normal((2, 2, 6 * nn))
    u = 1e-3 * rng.standard_normal((2, 6 * nn))
    m = O.material()
    with mesh_ctx(conn, X, thick) as ctx:
        dphi, dpsi, du = ctx.vector(phi), ctx.vector(psi), ctx.vector(u)
        out = []
        for k in range(4):
            g = ctx.coord_vector()
            if k == 0:
                ctx.add_mat_xpt_sens_inner_product(g, sg.STIFFNESS, dphi)
            elif k == 1:
                ctx.add_mat_xpt_sens_inner_product(g, sg.GEOMETRIC, dphi, du)
            else:
                ctx.add_adj_res_xpt_product(g, dpsi, du, model=(sg.LINEAR, sg.NONLINEAR)[k - 2])
            out.append(g.download().reshape(2, -1))

    def scalar(k, d, e, Xe, idx):
        t = thick[d, e]
        if k == 0:
            return phi[d, idx] @ O.elem_stiffness(0, m, t, 0.0, Xe, np.zeros(24)) @ phi[d, idx]
        if k == 1:
            return phi[d, idx] @ O.elem_geometric_step(m, t, 0.0, Xe, u[d, idx], 1.0) @ phi[d, idx]
        return psi[d, idx] @ O.elem_residual(k - 2, m, t, 0.0, Xe, u[d, idx])

    for k in range(4):
        ref = np.zeros((2, 3 * nn))
        for d in range(2):
            for e in range(ne):
                idx = (6 * conn[e][:, None] + np.arange(6)).ravel()
                dof = (3 * conn[e][:, None] + np.arange(3)).ravel()
                Xe = X[conn[e]].ravel()
                for i in range(12):
                    def f(x, i=i):
                        Xp = Xe.copy()
                        Xp[i] = x
                        return scalar(k, d, e, Xp, idx)
                    ref[d, dof[i]] += five_point(f, Xe[i], 3e-4)
        err = np.abs(out[k] - ref).max() / np.abs(ref).max()
        print(k, err)
        assert err <= 1e-7, k


def test_more_designs_than_one_launch():
    # 32 elements: 8 Mi doubles of element gradients hold 21,845 designs
    cyl = Cylinder(4, 8)
    nb = 21846
    rng = np.random.default_rng(3)
    t, p = rng.uniform(0.0015, 0.0025, cyl.nelems), rng.standard_normal(6 * cyl.nnodes)
    with mesh_ctx(cyl.conn, cyl.Xpts, np.broadcast_to(t, (nb, cyl.nelems)).copy()) as ctx:
        phi = ctx.vector(np.broadcast_to(p, (nb, p.size)).copy())
        g = ctx.coord_vector()
        ctx.add_mat_xpt_sens_inner_product(g, sg.STIFFNESS, phi)
        g = g.download().reshape(nb, -1)
    assert np.abs(g[0]).max() > 0
    assert np.array_equal(g[0], g[-1]) and np.array_equal(g[0], g[nb // 2])


@pytest.mark.parametrize("nx,ny", [(1, 1), (31, 1), (8, 4), (11, 3)])
def test_thickness_and_path_products_around_a_workgroup(nx, ny):
    # the scalars are cubic in the thickness and s_G is affine in the path, so
    # five-point and two-point differences are exact: 1e-10 is their round-off
    conn, X = random_mesh(nx, ny, seed=5 * nx + ny)
    nn, ne = X.shape[0], conn.shape[0]
    rng = np.random.default_rng(nx + 1)
    thick = rng.uniform(0.002, 0.02, (2, ne))
    phi, psi, w = rng.standard_normal((3, 2, 6 * nn))
    u = 1e-3 * rng.standard_normal((2, 6 * nn))
    m = O.material()
    with mesh_ctx(conn, X, thick) as ctx:
        dphi, dpsi, du = ctx.vector(phi), ctx.vector(psi), ctx.vector(u)
        out = []
        for k in range(4):
            g = ctx.design_vector()
            if k == 0:
                ctx.add_mat_dv_sens_inner_product(g, sg.STIFFNESS, dphi)
            elif k == 1:
                ctx.add_mat_dv_sens_inner_product(g, sg.GEOMETRIC, dphi, du)
            else:
                ctx.add_adj_res_product(g, dpsi, du, model=(sg.LINEAR, sg.NONLINEAR)[k - 2])
            out.append(g.download().reshape(2, ne))
        gu = ctx.vector()
        ctx.eval_mat_sv_sens_inner_product(dphi, gu)
        gu = gu.download().reshape(2, -1)
    ref, sens, mag = np.zeros((4, 2, ne)), np.zeros(2), np.zeros(2)
    for d in range(2):
        for e in range(ne):
            idx = (6 * conn[e][:, None] + np.arange(6)).ravel()
            Xe, p, t = X[conn[e]].ravel(), phi[d, idx], thick[d, e]
            h = 0.05 * t
            ref[0, d, e] = five_point(
                lambda s: p @ O.elem_stiffness(0, m, s, 0.0, Xe, np.zeros(24)) @ p, t, h)
            ref[1, d, e] = five_point(
                lambda s: p @ O.elem_geometric_step(m, s, 0.0, Xe, u[d, idx], 1.0) @ p, t, h)
            for k in range(2):
                ref[2 + k, d, e] = O.elem_adj_res_dv(k, m, t, 0.0, psi[d, idx], Xe, u[d, idx])
            c = p @ O.elem_geometric_step(m, t, 0.0, Xe, w[d, idx], 1.0) @ p
            sens[d] += c
            mag[d] += abs(c)
    for k in range(4):
        err = np.abs(out[k] - ref[k]).max() / np.abs(ref[k]).max()
        print(k, err)
        assert err <= 1e-10, k
    err = np.abs((gu * w).sum(axis=1) - sens) / mag
    print("path", err)
    assert err.max() <= 1e-10
