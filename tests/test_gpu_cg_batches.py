"""The device CG's iterations are launched in batches with the stopping test on
the device: the iterate after m iterations equals that of the same recurrence
on the host, for m around the batch edges, with rows of full and of other nodes
(3x3 block Jacobi) and with the diagonal (scalar field), and a solve to a
tolerance ends at the first iterate that meets it."""
import numpy as np
import pytest
import scipy.sparse as sp

import getfem_amd as ga
import oracle
from getfem_amd import _lib
from tests import problems

pytestmark = pytest.mark.gpu

CASES = {
    "p1_laplace_n6": (6, 1, 1, "IM_TETRAHEDRON(1)", oracle.TERM_LAPLACE),
    "p1_elast_n4": (4, 1, 3, "IM_TETRAHEDRON(1)", oracle.TERM_ISO_ELAST),
    "p2_elast_n3": (3, 2, 3, "IM_TETRAHEDRON(5)", oracle.TERM_ISO_ELAST),
    "p3_elast_n2": (2, 3, 3, "IM_TETRAHEDRON(8)", oracle.TERM_ISO_ELAST),
}


def host_cg(K, b, minv, m, rtol):
    x, r = np.zeros_like(b), b.copy()
    z = minv @ r
    p, rz, it = z.copy(), r @ z, 0
    while np.linalg.norm(r) / np.linalg.norm(b) > rtol and it < m:
        q = K @ p
        a = rz / (p @ q)
        x += a * p
        r -= a * q
        z = minv @ r
        rz, old = r @ z, rz
        p = z + rz / old * p
        it += 1
    return x, it, np.linalg.norm(r) / np.linalg.norm(b)


@pytest.mark.parametrize("name", sorted(CASES))
def test_iterates_and_counts(ctx, name):
    import torch
    n, k, q, im, term = CASES[name]
    lam = np.random.default_rng(5).lognormal(0.0, 0.5, 6 * n ** 3)
    case = problems.Case(n, k, q, im, term, lam=lam, mu=lam[::-1].copy())
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", case.pts, case.cvx)
    mf = ga.MeshFem(mesh, case.fem, q)
    plan = ga.Plan(mf, ga.MeshIm(mesh, im), ga.TERM_ISO_ELAST if q == 3 else ga.TERM_LAPLACE, case.coefs())
    plan.build_pattern()
    plan.assemble()
    face = np.flatnonzero(np.abs(mf.basic_dof_nodes()[:, 0]) < 1e-12)
    plan.dof_constraints((q * face[:, None] + np.arange(q)).ravel(), 0.0,
                         flags=_lib.BUILD_MATRIX | _lib.MODEL_SYMMETRIC)
    ip, ix, v = plan.csr()
    ndof = ip.size - 1
    K = sp.csr_matrix((v, ix, ip), shape=(ndof, ndof))
    blocks = [np.linalg.inv(K[q * u:q * u + q, q * u:q * u + q].toarray()) for u in range(ndof // q)]
    minv = sp.block_diag(blocks, format="csr")
    b = np.random.default_rng(6).standard_normal(ndof)
    db, dx = torch.tensor(b, device="cuda"), torch.empty(ndof, dtype=torch.float64, device="cuda")
    for m in (0, 1, 3, 4, 5, 8, 9, 17):
        print("case:", name, m, flush=True)
        dx.zero_()
        torch.cuda.synchronize()
        it, res = plan.solve_cg(db.data_ptr(), dx.data_ptr(), rtol=1e-30, maxit=m)
        x, hit, hres = host_cg(K, b, minv, m, 1e-30)
        assert it == hit == m
        # the recurrence amplifies rounding by far less than 1e4 over 17 iterations
        assert np.linalg.norm(dx.cpu().numpy() - x) <= 1e-12 * max(np.linalg.norm(x), 1e-300)
        assert abs(res - hres) <= 1e-12 * hres
    # the count at a tolerance: one iteration fewer does not meet it, and so
    # many asked for by number give the same iterate, bit for bit
    for rtol in (1e-1, 1e-3, 1e-6):
        dx.zero_()
        torch.cuda.synchronize()
        it, res = plan.solve_cg(db.data_ptr(), dx.data_ptr(), rtol=rtol, maxit=1000)
        x = dx.clone()
        assert res <= rtol
        for m in (it - 1, it):
            dx.zero_()
            torch.cuda.synchronize()
            got, r = plan.solve_cg(db.data_ptr(), dx.data_ptr(), rtol=1e-30, maxit=m)
            assert got == m and (r <= rtol) == (m == it)
        assert r == res and torch.equal(x, dx)
    dx.fill_(1.0)
    db.zero_()
    torch.cuda.synchronize()
    assert plan.solve_cg(db.data_ptr(), dx.data_ptr(), rtol=1e-8, maxit=5) == (0, 0.0)
    assert not dx.any()
