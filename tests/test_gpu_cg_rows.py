"""The product of the device CG sums each row in the order of the plan's own
product, bit for bit: with b = K x from the latter, the residual b - K x that
CG starts from is zero exactly.  Vector fields by mean row length (up to 24: a
row per lane group; up to 64 and above: a wavefront per node), rows of one and
of several tiles, rows of full and of other nodes, and a scalar field."""
import numpy as np
import pytest

import getfem_amd as ga
import oracle
from tests import problems

pytestmark = pytest.mark.gpu

CASES = {  # n, degree, components, method, elements kept, range of the mean row length, longest row at least
    "scalar_p2": (3, 2, 1, "IM_TETRAHEDRON(5)", 1.0, (12, 64), 1),
    "one_cube_p1": (1, 1, 3, "IM_TETRAHEDRON(1)", 1.0, (1, 24), 1),
    "p1": (5, 1, 3, "IM_TETRAHEDRON(1)", 1.0, (24, 64), 1),
    "p1_ragged": (6, 1, 3, "IM_TETRAHEDRON(1)", 0.6, (24, 64), 1),
    "one_cube_p2": (1, 2, 3, "IM_TETRAHEDRON(5)", 1.0, (24, 64), 65),
    "p2": (4, 2, 3, "IM_TETRAHEDRON(5)", 1.0, (64, 1e9), 129),
    "p2_ragged": (4, 2, 3, "IM_TETRAHEDRON(5)", 0.8, (24, 64), 129),
    "p2_holes": (6, 2, 3, "IM_TETRAHEDRON(5)", 0.95, (64, 1e9), 129),
    "p3": (2, 3, 3, "IM_TETRAHEDRON(8)", 1.0, (64, 1e9), 257),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_start_residual_is_zero(ctx, name):
    import torch
    n, k, q, im, keep, (lo, hi), longest = CASES[name]
    rng = np.random.default_rng(31)
    lam = rng.lognormal(0.0, 1.0, 6 * n ** 3)
    case = problems.Case(n, k, q, im, oracle.TERM_ISO_ELAST if q == 3 else oracle.TERM_LAPLACE, lam=lam,
                         mu=lam[::-1].copy())
    kept = np.flatnonzero(rng.random(case.cvx.shape[0]) < keep)
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", case.pts, np.ascontiguousarray(case.cvx[kept]))
    mf = ga.MeshFem(mesh, case.fem, q)
    plan = ga.Plan(mf, ga.MeshIm(mesh, im), ga.TERM_ISO_ELAST if q == 3 else ga.TERM_LAPLACE,
                   [np.ascontiguousarray(c[kept]) for c in case.coefs()] if q == 3 else case.coefs())
    plan.build_pattern()
    plan.assemble()
    ip = plan.csr()[0]
    rows = np.diff(ip)
    assert lo < rows.mean() <= hi and rows.max() >= longest
    dx = torch.tensor(rng.standard_normal(rows.size), device="cuda")
    db = torch.empty_like(dx)
    x = dx.clone()
    torch.cuda.synchronize()
    print("case:", name, rows.size, rows.mean(), rows.max(), flush=True)
    plan.spmv(dx.data_ptr(), db.data_ptr())
    ctx.synchronize()
    assert db.abs().max() > 0
    assert plan.solve_cg(db.data_ptr(), dx.data_ptr(), rtol=1e-30, maxit=3) == (0, 0.0)
    assert torch.equal(dx, x)
