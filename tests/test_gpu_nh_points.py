"""The point pass of the Neo-Hookean element computation (two elements per
wavefront, eight per workgroup) at element counts that leave the last
workgroup part empty: the residual alone and with the tangent against the
oracle, FP64 and FP32 tangents, and a change of pattern refused while the
pattern is pinned, twice in a row."""
import numpy as np
import pytest

import getfem_amd as ga
import oracle
from getfem_amd import meshes

pytestmark = pytest.mark.gpu

IM = "IM_GAUSS_PARALLELEPIPED(3,5)"


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("n", [1, 2, 3])
@pytest.mark.parametrize("prec,tol", [(ga.PREC_FP64, 1e-12), (ga.PREC_FP32, 1e-6)])
def test_residual_and_tangent(ctx, n, prec, tol):
    print("case: Neo-Hookean points", n, prec, flush=True)
    pts, cvx = meshes.regular_unit_mesh(n, "GT_QK(3,1)")
    pts = meshes.jitter(pts, n) + 0.01 * np.sin(7.0 * pts[:, ::-1])  # no axis-parallel face
    n_cv = cvx.shape[0]
    rng = np.random.default_rng(n)
    lam, mu = rng.uniform(5.0, 10.0, n_cv), rng.uniform(0.5, 1.0, n_cv)
    mesh = ga.Mesh(ctx, "GT_QK(3,1)", pts, cvx)
    mf = ga.MeshFem(mesh, "FEM_QK(3,2)", 3)
    plan = ga.Plan(mf, ga.MeshIm(mesh, IM), ga.TERM_NEOHOOKEAN, [lam, mu])
    plan.set_form(ga.FORM_PERQP, prec)
    U = 0.02 / n * rng.standard_normal(mf.nbdof())
    plan.set_state(U)
    plan.build_pattern()
    P = oracle.Problem(oracle.GT_QK31, pts, cvx, oracle.FEM_QK, 2, 3, mf.basic_dof_table(), mf.nbdof(), IM,
                       oracle.TERM_NEOHOOKEAN, coef_a=lam, coef_b=mu, U=U)
    V = P.assemble_vector()
    plan.assemble_residual()
    assert rel(plan.residual(), V) <= 1e-11
    alone = plan.residual()
    plan.assemble()
    assert np.array_equal(plan.residual(), alone)
    ip, ix, v = plan.csr()
    rip, rix, rv = oracle.csc_to_csr(*P.assemble_csc(), mf.nbdof())
    assert np.array_equal(ip, rip) and np.array_equal(ix, rix)
    assert rel(v, rv) <= tol


def test_refused_state_stays_refused(ctx):
    print("case: Neo-Hookean pinned pattern", flush=True)
    n = 2
    pts, cvx = meshes.regular_unit_mesh(n, "GT_QK(3,1)")  # unjittered: the zero state drops entries
    mesh = ga.Mesh(ctx, "GT_QK(3,1)", pts, cvx)
    mf = ga.MeshFem(mesh, "FEM_QK(3,2)", 3)
    plan = ga.Plan(mf, ga.MeshIm(mesh, IM), ga.TERM_NEOHOOKEAN, [10.0, 1.0])
    U = 0.01 * np.random.default_rng(3).standard_normal(mf.nbdof())
    zero = np.zeros_like(U)
    plan.set_state(U)
    nnz = plan.build_pattern()
    plan.assemble()
    v = plan.csr()[2]
    pid = plan.pattern_id()
    views = plan.torch_csr_view()
    for _ in range(2):  # the second time the stored keep bits are already those of the refused state
        plan.set_state(zero)
        with pytest.raises(ga.GfxError):
            plan.assemble()
    plan.set_state(U)
    plan.assemble()
    assert plan.pattern_id() == pid and np.array_equal(plan.csr()[2], v)
    del views
    plan.set_state(zero)
    plan.assemble()
    assert plan.pattern_id() != pid and plan.nnz is not None and plan.dims()[1] < nnz
