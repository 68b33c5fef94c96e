"""The keep signature (one bit per element, pair and component, 64 elements to
a word) behind the pattern build and its re-validation, at element counts that
do not fill the last group: after new coefficients the plan's CSR equals the
oracle's at those values, whether the bits stay (the pattern is kept) or
change (it is rebuilt), and a change refused because the pattern is pinned
stays refused until the values that the pattern was built from return."""
import numpy as np
import pytest

import getfem_amd as ga
import oracle
from tests import problems

pytestmark = pytest.mark.gpu

CASES = {
    "p1_laplace": (1, 1, oracle.TERM_LAPLACE), "p2_laplace": (2, 1, oracle.TERM_LAPLACE),
    "p3_laplace": (3, 1, oracle.TERM_LAPLACE), "p1_elast": (1, 3, oracle.TERM_ISO_ELAST),
    "p2_elast": (2, 3, oracle.TERM_ISO_ELAST), "p3_elast": (3, 3, oracle.TERM_ISO_ELAST),
}
IM = {1: "IM_TETRAHEDRON(1)", 2: "IM_TETRAHEDRON(5)", 3: "IM_TETRAHEDRON(8)"}


def coefs(n_cv, q, seed):
    rng = np.random.default_rng(seed)
    return [rng.lognormal(0.0, 0.5, n_cv) for _ in range(2 if q == 3 else 1)]


def at(case, c):
    if case.term == oracle.TERM_LAPLACE:
        case.a = c[0]
    else:
        case.lam, case.mu = c
    return case.oracle_csr()


def equal(plan, ref):
    ip, ix, v = plan.csr()
    assert np.array_equal(ip, ref[0]) and np.array_equal(ix, ref[1])
    assert np.linalg.norm(v - ref[2]) <= 1e-12 * np.linalg.norm(ref[2])


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("n", [1, 2, 3])
def test_new_coefficients(ctx, name, n):
    print("case: keep signature", name, n, flush=True)
    k, q, term = CASES[name]
    case = problems.Case(n, k, q, IM[k], term)
    n_cv = case.cvx.shape[0]
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", case.pts, case.cvx)
    mf = ga.MeshFem(mesh, case.fem, q)
    c0 = coefs(n_cv, q, 1)
    plan = ga.Plan(mf, ga.MeshIm(mesh, IM[k]), ga.TERM_ISO_ELAST if q == 3 else ga.TERM_LAPLACE, c0)
    plan.build_pattern()
    pid = plan.pattern_id()
    plan.assemble()
    equal(plan, at(case, c0))

    def assemble(c):
        for s, v in enumerate(c):
            plan.set_coef(s, v)
        plan.assemble()

    c1 = coefs(n_cv, q, 2)  # the same bits
    assemble(c1)
    equal(plan, at(case, c1))
    assert plan.pattern_id() == pid
    c2 = [v.copy() for v in c1]  # no entry of the first and last elements
    for v in c2:
        v[0] = v[-1] = 0.0
    refused = [v.copy() for v in c1]
    for v in refused:
        v[:] = 0.0
    assemble(c2)
    equal(plan, at(case, c2))
    pid = plan.pattern_id()
    views = plan.torch_csr_view()
    for _ in range(2):  # the second time the signature is already that of the refused values
        with pytest.raises(ga.GfxError):
            assemble(refused)
    assemble(c2)
    assert plan.pattern_id() == pid
    equal(plan, at(case, c2))
    del views
    assemble(c1)
    equal(plan, at(case, c1))


@pytest.mark.parametrize("name", ["p1_laplace", "p1_elast", "p2_elast", "p3_laplace"])
@pytest.mark.parametrize("n", [1, 2, 3])  # 6, 48 and 162 elements: groups of 64 that are and are not full
def test_void_elements_are_confirmed(ctx, name, n):
    """New coefficients with the same void elements (all of them 0): the check
    finds the stored bits again and nothing of the pattern is formed anew."""
    from tests.launches import kernels
    print("case: keep signature, void elements", name, n, flush=True)
    k, q, term = CASES[name]
    case = problems.Case(n, k, q, IM[k], term)
    n_cv = case.cvx.shape[0]
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", case.pts, case.cvx)
    c0, c1 = coefs(n_cv, q, 1), coefs(n_cv, q, 2)
    for v in c0 + c1:
        v[0] = v[-1] = 0.0
        v[64:128] = 0.0  # (at 162 elements) a whole group
    plan = ga.Plan(ga.MeshFem(mesh, case.fem, q), ga.MeshIm(mesh, IM[k]),
                   ga.TERM_ISO_ELAST if q == 3 else ga.TERM_LAPLACE, c0)
    plan.build_pattern()
    plan.assemble()

    def assemble():
        for s, v in enumerate(c1):
            plan.set_coef(s, v)
        plan.assemble()

    ran = kernels(assemble)
    equal(plan, at(case, c1))
    assert sum("k_keep<" in x for x in ran) == 1, ran
    assert not any("k_keep_words" in x or "k_mask" in x for x in ran), ran


@pytest.mark.parametrize("name", ["p1_laplace", "p2_elast"])
def test_a_body_without_material(ctx, name):
    """A plan built where every coefficient is 0 has no entries; coefficients
    given later bring them."""
    print("case: keep signature, no material", name, flush=True)
    k, q, term = CASES[name]
    case = problems.Case(2, k, q, IM[k], term)
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", case.pts, case.cvx)
    c = coefs(case.cvx.shape[0], q, 1)
    plan = ga.Plan(ga.MeshFem(mesh, case.fem, q), ga.MeshIm(mesh, IM[k]),
                   ga.TERM_ISO_ELAST if q == 3 else ga.TERM_LAPLACE, [0.0 * v for v in c])
    plan.build_pattern()
    plan.assemble()
    assert plan.csr()[1].size == 0
    for _ in range(2):
        for s, v in enumerate(c):
            plan.set_coef(s, v)
        plan.assemble()
        equal(plan, at(case, c))
