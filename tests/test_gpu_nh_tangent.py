"""The Neo-Hookean tangent's tiles and keep bits where elements drop entries: no
element, some of them and all of them, FP64 against the oracle (pattern and
values); a state that is not a number is never taken for one that keeps
everything."""
import numpy as np
import pytest

import getfem_amd as ga
import oracle
from getfem_amd import meshes

pytestmark = pytest.mark.gpu

IM = "IM_GAUSS_PARALLELEPIPED(3,5)"


def setup(ctx, n):
    pts, cvx = meshes.regular_unit_mesh(n, "GT_QK(3,1)")  # unjittered: an undeformed element drops entries
    mesh = ga.Mesh(ctx, "GT_QK(3,1)", pts, cvx)
    mf = ga.MeshFem(mesh, "FEM_QK(3,2)", 3)
    plan = ga.Plan(mf, ga.MeshIm(mesh, IM), ga.TERM_NEOHOOKEAN, [10.0, 1.0])
    return pts, cvx, mf, plan


def check(plan, mf, pts, cvx, U):
    P = oracle.Problem(oracle.GT_QK31, pts, cvx, oracle.FEM_QK, 2, 3, mf.basic_dof_table(), mf.nbdof(), IM,
                       oracle.TERM_NEOHOOKEAN, coef_a=np.full(cvx.shape[0], 10.0), coef_b=np.ones(cvx.shape[0]), U=U)
    ip, ix, v = plan.csr()
    rip, rix, rv = oracle.csc_to_csr(*P.assemble_csc(), mf.nbdof())
    assert np.array_equal(ip, rip) and np.array_equal(ix, rix)
    # sums of 27 points and up to 8 elements in FP64
    assert np.linalg.norm(v - rv) <= 1e-12 * np.linalg.norm(rv)


@pytest.mark.parametrize("n", [1, 3])
@pytest.mark.parametrize("moved", ["none", "some", "all"])
def test_keep_bits(ctx, n, moved):
    print("case: Neo-Hookean keep bits", n, moved, flush=True)
    pts, cvx, mf, plan = setup(ctx, n)
    U = 0.02 / n * np.random.default_rng(n).standard_normal(mf.nbdof())
    if moved == "none":
        U[:] = 0.0
    elif moved == "some":  # the nodes of the first element
        keep = np.zeros(mf.nbdof(), dtype=bool)
        for c in range(3):
            keep[mf.basic_dof_table()[0] + c] = True
        U[~keep] = 0.0
    plan.set_state(U)
    plan.build_pattern()  # the bits are written
    plan.assemble()
    check(plan, mf, pts, cvx, U)
    pid = plan.pattern_id()
    plan.set_state(1.001 * U)
    plan.assemble()  # and compared
    check(plan, mf, pts, cvx, 1.001 * U)
    assert plan.pattern_id() == pid
    plan.set_state(np.zeros_like(U))
    plan.assemble()  # elements that kept every entry no longer do
    check(plan, mf, pts, cvx, np.zeros_like(U))
    plan.set_state(U)
    plan.assemble()  # and do again
    check(plan, mf, pts, cvx, U)


def test_not_a_number_drops_entries(ctx):
    print("case: Neo-Hookean NaN state", flush=True)
    _, _, mf, plan = setup(ctx, 2)
    U = 0.01 * np.random.default_rng(1).standard_normal(mf.nbdof())
    plan.set_state(U)
    plan.build_pattern()
    plan.assemble()
    v = plan.csr()[2]
    views = plan.torch_csr_view()
    bad = U.copy()
    bad[5] = np.nan
    plan.set_state(bad)
    with pytest.raises(ga.GfxError):
        plan.assemble()
    plan.set_state(U)
    plan.assemble()
    assert np.array_equal(plan.csr()[2], v)
    del views
