"""Fields of one to three components in the order-0 and order-1 programs: a
linear field's integrals in closed form (its values and its gradient), and the
derivative with respect to a variable next to it."""
import numpy as np
import pytest

import getfem_amd as ga
from getfem_amd import meshes
from getfem_amd.workspace import GaWorkspace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q", [1, 2, 3])
@pytest.mark.parametrize("k", [1, 2])
def test_linear_field(ctx, q, k):
    print("case: scalar route components", q, k, flush=True)
    pts, cvx = meshes.regular_unit_mesh(2, "GT_PK(3,1)")
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", pts, cvx)
    mf = ga.MeshFem(mesh, "FEM_PK(3,%d)" % k, q)
    mfp = ga.MeshFem(mesh, "FEM_PK(3,1)", 1)
    rng = np.random.default_rng(q)
    A, b = rng.standard_normal((q, 3)), rng.standard_normal(q)
    d = (mf.basic_dof_nodes() @ A.T + b).ravel()
    M = np.full((3, 3), 0.25) + np.eye(3) / 12.0  # the second moments of the unit cube
    dd = b @ b + b @ A @ np.ones(3) + np.sum((A.T @ A) * M)
    for expr, ref in (("d.d" if q > 1 else "d*d", dd),
                      ("Grad_d:Grad_d" if q > 1 else "Grad_d.Grad_d", np.sum(A * A))):
        ws = GaWorkspace(ctx)
        ws.add_fem_variable("p", mfp, np.full(mfp.nbdof(), 2.0))
        ws.add_fem_constant("d", mf, d)
        ws.add_expression("p*(%s)" % expr, ga.MeshIm(mesh, "IM_TETRAHEDRON(5)"))
        ws.assembly(0)
        # sums of 48 elements and 15 points in FP64
        assert abs(ws.assembled_potential() - 2.0 * ref) <= 1e-12 * abs(ref)
        ws.assembly(1)
        assert abs(np.sum(ws.assembled_vector()) - ref) <= 1e-12 * abs(ref)
