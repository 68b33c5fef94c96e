"""The polynomial route's element matrices through the reference tensor (affine
elements, a program without fem fields) against the same program with a data
field that is 1 everywhere, which goes through the points: the same pattern and
values for every pair of slots (value, gradient), numbers of components and
degrees, at element counts that leave the last workgroup and its last pass part
empty."""
import numpy as np
import pytest

import getfem_amd as ga
from getfem_amd import meshes
from getfem_amd.workspace import GaWorkspace

pytestmark = pytest.mark.gpu

# (components and degree of u, of p, expression in k)
CASES = {
    "v2_s1": (3, 2, 1, 1, "k*Sym(Grad_u):Grad_Test_u - p*Div_Test_u - Test_p*Div_u - k*p*Test_p"),
    "v1_s2": (3, 1, 1, 2, "k*Grad_u:Grad_Test_u + k*u.Grad_Test_p + Grad_p.Grad_Test_p"),
    "v3_s1": (3, 3, 1, 1, "k*u.Test_u + Grad_u:Grad_Test_u - k*p*Div_Test_u + k*p*Test_p"),
    "s3_s2": (1, 3, 1, 2, "k*Grad_u.Grad_Test_u + u*Test_u + k*p*Test_u + Grad_p.Grad_Test_u + p*Test_p"),
    "w2_v1": (2, 2, 3, 1, "k*u.Test_u + k*Grad_p:Grad_Test_p + p.Test_p"),
    "v1_w1": (3, 1, 2, 1, "k*Div_u*Div_Test_u + k*p.Test_p"),
    "w1_s1": (2, 1, 1, 2, "u.Test_u + k*p*Test_p + k*Grad_p.Grad_Test_p"),
}


def matrix(ctx, mfu, mfp, mim, expr, scale, data):
    ws = GaWorkspace(ctx)
    ws.add_fem_variable("u", mfu, np.zeros(mfu.nbdof()), first=0)
    ws.add_fem_variable("p", mfp, np.zeros(mfp.nbdof()), first=mfu.nbdof())
    if data is not None:
        ws.add_fem_constant("one", data, np.ones(data.nbdof()))
        expr = expr.replace("k*", "k*one*") if "k*" in expr else expr
        # terms without k: multiplied as well
        expr = " + ".join("one*(%s)" % t if "one" not in t else t for t in expr.replace(" - ", " + (-1)*").split(" + "))
    ws.add_expression(expr.replace("k*", "%r*" % scale), mim)
    ws.assembly(2)
    return ws.assembled_matrix_csr()


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("n", [1, 2, 9])
def test_reference_and_points(ctx, name, n):
    qu, ku, qp, kp, expr = CASES[name]
    if n == 9 and ku == 3 and qu == 3:
        n = 6
    print("case: polynomial reference tensor", name, n, flush=True)
    pts, cvx = meshes.regular_unit_mesh(n, "GT_PK(3,1)")
    pts = meshes.jitter(pts, n) + 0.01 * np.sin(7.0 * pts[:, ::-1])
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", pts, cvx)
    mfu = ga.MeshFem(mesh, "FEM_PK(3,%d)" % ku, qu)
    mfp = ga.MeshFem(mesh, "FEM_PK(3,%d)" % kp, qp)
    one = ga.MeshFem(mesh, "FEM_PK_DISCONTINUOUS(3,0)", 1)
    mim = ga.MeshIm(mesh, "IM_TETRAHEDRON(%d)" % (8 if ku == 3 else 5))
    a = matrix(ctx, mfu, mfp, mim, expr, 1.5, None)
    b = matrix(ctx, mfu, mfp, mim, expr, 1.5, one)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    # rounding of at most 15 (43 for degree 8) points and 16 slot pairs a value
    assert np.linalg.norm(a[2] - b[2]) <= 1e-13 * np.linalg.norm(b[2])


def sorted_matrix(ctx, mfu, mfp, mim, expr, scale):
    """The matrix of constant programs with the kept entries sorted."""
    ws = GaWorkspace(ctx)
    ws.add_fem_variable("u", mfu, first=0)
    ws.add_fem_variable("p", mfp, first=mfu.nbdof())
    ws.add_expression(expr.replace("k*", "%r*" % scale), mim)
    ws.set_structure_limit(0)
    ws.assembly(2)
    return ws.assembled_matrix_csr()


@pytest.mark.parametrize("limit", [None, 0])
@pytest.mark.parametrize("shape", ["flat", "needle"])
@pytest.mark.parametrize("ku", [2, 3])
def test_entries_at_the_threshold(ctx, shape, ku, limit):
    """Stretched elements, whose entries spread across the threshold: the stored
    entries are those of the sums over the points, one for one, whether the
    structure is kept or not."""
    print("case: polynomial reference tensor, entries at the threshold", shape, ku, limit, flush=True)
    pts, cvx = meshes.regular_unit_mesh(2, "GT_PK(3,1)")
    pts = meshes.jitter(pts, 2)
    expr = "k*Div_u*Div_Test_u + k*Sym(Grad_u):Grad_Test_u + p*Test_p"
    near = 0
    for ratio in (1e6, 2e6, 3e6, 4e6, 5e6, 6e6, 7e6, 8e6):
        mesh = ga.Mesh(ctx, "GT_PK(3,1)", pts * ([ratio, 1.3 * ratio, 1.0] if shape == "flat" else [ratio, 1.0, 1.0]), cvx)
        mfu, mfp = ga.MeshFem(mesh, "FEM_PK(3,%d)" % ku, 3), ga.MeshFem(mesh, "FEM_PK(3,1)", 1)
        one = ga.MeshFem(mesh, "FEM_PK_DISCONTINUOUS(3,0)", 1)
        mim = ga.MeshIm(mesh, "IM_TETRAHEDRON(%d)" % (8 if ku == 3 else 5))
        a = matrix(ctx, mfu, mfp, mim, expr, 1.5, None) if limit is None else sorted_matrix(ctx, mfu, mfp, mim, expr, 1.5)
        b = matrix(ctx, mfu, mfp, mim, expr, 1.5, one)
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
        assert np.linalg.norm(a[2] - b[2]) <= 1e-13 * np.linalg.norm(b[2])
        near += np.array_equal(a[2], b[2])
    assert near  # (some of the bodies have entries near the threshold: the same sums)


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("jittered", [False, True])
def test_ordinary_meshes_stay_with_the_reference_tensor(ctx, name, jittered):
    """The roundings left of entries that are 0 stay clear of the threshold."""
    from tests.launches import kernels
    qu, ku, qp, kp, expr = CASES[name]
    print("case: polynomial reference tensor, ordinary mesh", name, jittered, flush=True)
    pts, cvx = meshes.regular_unit_mesh(3, "GT_PK(3,1)")
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", meshes.jitter(pts, 3) if jittered else pts, cvx)
    mfu = ga.MeshFem(mesh, "FEM_PK(3,%d)" % ku, qu)
    mfp = ga.MeshFem(mesh, "FEM_PK(3,%d)" % kp, qp)
    ran = kernels(lambda: matrix(ctx, mfu, mfp, ga.MeshIm(mesh, "IM_TETRAHEDRON(%d)" % (8 if ku == 3 else 5)), expr,
                                 1.5, None))
    assert any("k_poly_ref" in x for x in ran) and not any("k_poly_mat" in x for x in ran), ran
