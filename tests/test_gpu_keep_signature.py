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


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("shape", ["flat", "needle"])
@pytest.mark.parametrize("ratio", [1e2, 1e4, 1e5])
def test_stretched_elements(ctx, name, shape, ratio):
    """Elements of a large aspect ratio, whose entries spread over its square:
    the stored pattern is the oracle's (per-point sums), from the build and
    after new coefficients that the check confirms or has formed anew."""
    print("case: keep signature, stretched", name, shape, ratio, flush=True)
    k, q, term = CASES[name]
    case = problems.Case(2, k, q, IM[k], term)
    case.pts = np.ascontiguousarray(case.pts * ([ratio, ratio, 1.0] if shape == "flat" else [ratio, 1.0, 1.0]))
    case.dofs, case.ndof = oracle.enumerate_dof(oracle.GT_PK31, case.pts, case.cvx, oracle.FEM_PK, k, q)
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", case.pts, case.cvx)
    n_cv = case.cvx.shape[0]
    plan = ga.Plan(ga.MeshFem(mesh, case.fem, q), ga.MeshIm(mesh, IM[k]),
                   ga.TERM_ISO_ELAST if q == 3 else ga.TERM_LAPLACE, coefs(n_cv, q, 1))
    plan.build_pattern()
    for seed in (1, 2):
        c = coefs(n_cv, q, seed)
        for s, v in enumerate(c):
            plan.set_coef(s, v)
        plan.assemble()
        ip, ix, v = plan.csr()
        ref = at(case, c)
        assert np.array_equal(ip, ref[0]) and np.array_equal(ix, ref[1])


def stretched(ratio, flat, seed):
    """A P3 elasticity body of aspect ratio `ratio` with its coefficients and
    the keys row * ndof + column of the oracle's stored entries."""
    case = problems.Case(2, 3, 3, IM[3], oracle.TERM_ISO_ELAST)
    case.pts = np.ascontiguousarray(case.pts * ([ratio, ratio, 1.0] if flat else [ratio, 1.0, 1.0]))
    case.dofs, case.ndof = oracle.enumerate_dof(oracle.GT_PK31, case.pts, case.cvx, oracle.FEM_PK, 3, 3)
    c = coefs(case.cvx.shape[0], 3, seed)
    ip, ix, _ = at(case, c)
    return case, c, np.repeat(np.arange(case.ndof, dtype=np.int64), np.diff(ip)) * case.ndof + ix


def kept_by_point_sums(case, c):
    """The same keys from the element matrices' sums over the points in float64."""
    P, W = ga.core.integration_rule(IM[3])
    X = case.pts[case.cvx]
    K = (X[:, 1:] - X[:, :1]).transpose(0, 2, 1)
    r, s = [1, 2, 0], [2, 0, 1]
    cof = K[:, r][:, :, r] * K[:, s][:, :, s] - K[:, r][:, :, s] * K[:, s][:, :, r]
    J = (K[:, 0] * cof[:, 0]).sum(axis=1)
    B, J = cof / J[:, None, None], np.abs(J)
    E = np.zeros((X.shape[0], 20, 3, 20, 3))
    for x, w in zip(P, W):
        g = np.einsum("erc,ic->eir", B, ga.core.fem_eval("FEM_PK(3,3)", x)[1])
        M = (J * c[0])[:, None, None, None, None] * np.einsum("eia,ejb->eiajb", g, g)
        M += (J * c[1])[:, None, None, None, None] * np.einsum("eib,eja->eiajb", g, g)
        M += ((J * c[1])[:, None, None] * np.einsum("eic,ejc->eij", g, g))[:, :, None, :, None] * np.eye(3)[:, None, :]
        E += w * M
    E = np.abs(E.reshape(X.shape[0], 60, 60))
    dofs = (case.dofs[:, :, None] + np.arange(3)).reshape(-1, 60).astype(np.int64)
    return np.unique((dofs[:, :, None] * case.ndof + dofs[:, None, :])[E > 1e-14 * E.max(axis=(1, 2), keepdims=True)])


def test_entries_at_the_threshold(ctx):
    """Where the entries of stretched elements spread across the threshold, the
    last bits of their sums decide.  No more stored entries differ from the
    oracle's than with sums over the points in float64 (and three standard
    deviations of so small a count)."""
    print("case: keep signature, entries at the threshold", flush=True)
    mine = theirs = 0
    for ratio in (1e6, 2e6, 3e6):
        for flat in (False, True):
            for seed in range(1, 9):
                case, c, ref = stretched(ratio, flat, seed)
                mesh = ga.Mesh(ctx, "GT_PK(3,1)", case.pts, case.cvx)
                plan = ga.Plan(ga.MeshFem(mesh, case.fem, 3), ga.MeshIm(mesh, IM[3]), ga.TERM_ISO_ELAST, c)
                plan.build_pattern()
                plan.assemble()
                ip, ix, _ = plan.csr()
                keys = np.repeat(np.arange(case.ndof, dtype=np.int64), np.diff(ip)) * case.ndof + ix
                mine += np.setxor1d(keys, ref).size
                theirs += np.setxor1d(kept_by_point_sums(case, c), ref).size
    print("entries that differ: %d, by sums over the points %d" % (mine, theirs), flush=True)
    assert mine <= theirs + 3 * theirs ** 0.5


@pytest.mark.parametrize("name", sorted(CASES))
def test_regular_meshes_are_confirmed(ctx, name):
    """The roundings left of entries that are 0 (right angles) stay clear of
    the threshold: new coefficients are confirmed by the check alone."""
    from tests.launches import kernels
    print("case: keep signature, regular mesh", name, flush=True)
    k, q, term = CASES[name]
    case = problems.Case(3, k, q, IM[k], term, jitter=False)
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", case.pts, case.cvx)
    c0, c1 = (coefs(case.cvx.shape[0], q, seed) for seed in (1, 2))
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
    assert not any("k_keep_words" in x or "k_keep_points" in x or "k_mask" in x for x in ran), ran


@pytest.mark.parametrize("ratio", [1e6, 3e6])
def test_entries_at_the_threshold_follow_the_values(ctx, ratio):
    """New coefficients and back, where entries lie at the threshold: the
    pattern is that of a plan made at those coefficients."""
    print("case: keep signature, entries at the threshold, new values", ratio, flush=True)
    case, c, _ = stretched(ratio, True, 1)
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", case.pts, case.cvx)
    mf, mim = ga.MeshFem(mesh, case.fem, 3), ga.MeshIm(mesh, IM[3])
    plan = ga.Plan(mf, mim, ga.TERM_ISO_ELAST, c)
    plan.build_pattern()
    seen = set()
    for values in (coefs(c[0].size, 3, 2), c, [c[0], 0.25 * c[1]], [2.0 * v for v in c], c):
        for s, v in enumerate(values):
            plan.set_coef(s, v)
        plan.assemble()
        new = ga.Plan(mf, mim, ga.TERM_ISO_ELAST, values)
        new.build_pattern()
        new.assemble()
        for a, b in zip(plan.csr(), new.csr()):
            assert np.array_equal(a, b)
        seen.add(plan.csr()[1].size)
    assert len(seen) > 2
