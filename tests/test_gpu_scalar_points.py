"""The polynomial route's orders 0 and 1 for every number of lanes per element
(rules of 1 to 125 points, the last in two rounds of 64) and element counts
that do not fill a wavefront: the potential and its derivative against a
numpy sum over the same points."""
import numpy as np
import pytest

import getfem_amd as ga
from getfem_amd import core, meshes
from getfem_amd.workspace import GaWorkspace

pytestmark = pytest.mark.gpu

TET, HEX = "GT_PK(3,1)", "GT_QK(3,1)"
CASES = [(TET, "FEM_PK(3,%d)" % k, "IM_TETRAHEDRON(%d)" % r) for k, r in
         ((1, 1), (2, 1), (2, 2), (2, 3), (1, 5), (3, 5), (2, 6), (3, 8))]
CASES += [(HEX, "FEM_QK(3,%d)" % k, "IM_GAUSS_PARALLELEPIPED(3,%d)" % r) for k, r in
          ((1, 0), (1, 3), (2, 5), (2, 7), (2, 9))]


def reference(gt, fem, im, pts, cvx, dofs, P):
    """J = sum p^3 + p Grad_p.Grad_p and dJ/dp."""
    x, w = core.integration_rule(im)
    geo = "FEM_PK(3,1)" if gt == TET else "FEM_QK(3,1)"
    J, V = 0.0, np.zeros_like(P)
    for q in range(len(w)):
        phi, h = core.fem_eval(fem, x[q])
        _, hg = core.fem_eval(geo, x[q])
        K = np.einsum("evr,vc->erc", pts[cvx], hg)
        g = np.einsum("ecr,ic->eir", np.linalg.inv(K), h)
        wJ = np.abs(np.linalg.det(K)) * w[q]
        u = P[dofs]
        p, gp = u @ phi, np.einsum("ei,eir->er", u, g)
        s = (gp * gp).sum(axis=1)
        J += (wJ * (p ** 3 + p * s)).sum()
        v = (wJ * (3 * p * p + s))[:, None] * phi + np.einsum("e,er,eir->ei", 2 * wJ * p, gp, g)
        np.add.at(V, dofs, v)
    return J, V


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(c[1:]))
@pytest.mark.parametrize("n", [1, 2])
def test_potential_and_derivative(ctx, case, n):
    print("case: points per element", case, n, flush=True)
    gt, fem, im = case
    pts, cvx = meshes.regular_unit_mesh(n, gt)
    pts = meshes.jitter(pts, n) + 0.03 * np.sin(3.0 * pts[:, ::-1])
    cvx = cvx[:-1] if len(cvx) > 1 else cvx
    mesh = ga.Mesh(ctx, gt, pts, cvx)
    mf = ga.MeshFem(mesh, fem, 1)
    P = np.random.default_rng(n).uniform(0.5, 1.5, mf.nbdof())
    ws = GaWorkspace(ctx)
    ws.add_fem_variable("p", mf, P)
    ws.add_expression("p*p*p + p*(Grad_p.Grad_p)", ga.MeshIm(mesh, im), 1)
    ws.assembly(0)
    ws.assembly(1)
    J, V = reference(gt, fem, im, pts, cvx, mf.basic_dof_table(), P)
    assert abs(ws.assembled_potential() - J) <= 1e-12 * abs(J)
    assert np.linalg.norm(ws.assembled_vector() - V) <= 1e-12 * np.linalg.norm(V)
