"""The check of the keep bits where an element's values are not finite: its
entries count as dropped, so a pinned pattern is refused, and the values that
it was built from bring it back bit for bit."""
import numpy as np
import pytest

import getfem_amd as ga
from getfem_amd import meshes

pytestmark = pytest.mark.gpu


# meshes where every element has an entry that no other element has
@pytest.mark.parametrize("k,q,n", [(1, 1, 1), (2, 1, 3), (2, 3, 3)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_not_finite(ctx, k, q, n, bad):
    print("case: keep bits of values that are not finite", k, q, n, bad, flush=True)
    pts, cvx = meshes.regular_unit_mesh(n, "GT_PK(3,1)")
    pts = meshes.jitter(pts, n)
    n_cv = cvx.shape[0]
    good = np.random.default_rng(k).uniform(0.5, 2.0, n_cv)
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", pts, cvx)
    plan = ga.Plan(ga.MeshFem(mesh, "FEM_PK(3,%d)" % k, q), ga.MeshIm(mesh, "IM_TETRAHEDRON(5)"),
                   ga.TERM_ISO_ELAST if q == 3 else ga.TERM_LAPLACE, [good, 1.5] if q == 3 else [good])
    plan.build_pattern()
    plan.assemble()
    v = plan.csr()[2]
    views = plan.torch_csr_view()
    for at in (0, n_cv - 1):  # the last element: the last group of 64 is part empty
        c = good.copy()
        c[at] = bad
        plan.set_coef(0, c)
        with pytest.raises(ga.GfxError):
            plan.assemble()
    plan.set_coef(0, good)
    plan.assemble()
    assert np.array_equal(plan.csr()[2], v)
    del views
