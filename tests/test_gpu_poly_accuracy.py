"""How far the polynomial route's matrices and vectors are from the exact ones, in long
double: no further than the sum over the rule's points in plain float64, the
order that the reference assembles in, but for a tenth (two ways of rounding
one sum).  Exact: where the integrand is a polynomial that the rule integrates
(constant coefficients on tetrahedra), its integral; otherwise the sum over the
points of the same tables."""
import numpy as np
import pytest

import getfem_amd as ga
from getfem_amd import core, meshes
from getfem_amd.workspace import GaWorkspace

pytestmark = pytest.mark.gpu

CASES = {  # geometry, element of u, rule, whether the integrand reads a field
    "p2_const": ("GT_PK(3,1)", "FEM_PK(3,2)", "IM_TETRAHEDRON(5)", False),
    "p3_const": ("GT_PK(3,1)", "FEM_PK(3,3)", "IM_TETRAHEDRON(8)", False),
    "p2_field": ("GT_PK(3,1)", "FEM_PK(3,2)", "IM_TETRAHEDRON(5)", True),
    "p3_field": ("GT_PK(3,1)", "FEM_PK(3,3)", "IM_TETRAHEDRON(8)", True),
    "q1_const": ("GT_QK(3,1)", "FEM_QK(3,1)", "IM_GAUSS_PARALLELEPIPED(3,4)", False),
    "q1_field": ("GT_QK(3,1)", "FEM_QK(3,1)", "IM_GAUSS_PARALLELEPIPED(3,4)", True),
}
MU = 0.8


def lagrange(k, x):
    """Values and gradients of the Pk base at the points x in long double, in
    the library's node order."""
    L = np.longdouble
    lam = np.concatenate([1 - x.sum(axis=1, keepdims=True), x], axis=1)
    dlam = np.array([[-1, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]], dtype=L)
    out = {}
    for a in np.ndindex(*[k + 1] * 4):
        if sum(a) != k:
            continue
        v, g = np.ones(x.shape[0], dtype=L), np.zeros((x.shape[0], 3), dtype=L)
        for b in range(4):
            for j in range(a[b]):  # a factor (k lambda_b - j) / (j + 1)
                f, df = (k * lam[:, b] - j) / (j + 1), dlam[b] * k / L(j + 1)
                g = g * f[:, None] + v[:, None] * df
                v = v * f
        node = int(np.argmax(core.fem_eval("FEM_PK(3,%d)" % k, np.array(a[1:]) / k)[0]))
        out[node] = (v, g)
    return np.stack([out[i][0] for i in sorted(out)], axis=1), np.stack([out[i][1] for i in sorted(out)], axis=1)


def fine_rule(m):
    """Collapsed Gauss rule of the tetrahedron in long double, exact up to degree 2 m - 3."""
    t = np.polynomial.legendre.leggauss(m)[0].astype(np.longdouble)
    for _ in range(3):  # Newton on the Legendre polynomial
        p0, p1 = np.ones_like(t), t
        for j in range(2, m + 1):
            p0, p1 = p1, ((2 * j - 1) * t * p1 - (j - 1) * p0) / j
        dp = m * (p0 - t * p1) / (1 - t * t)
        t = t - p1 / dp
    w, t = 1 / ((1 - t * t) * dp * dp), (t + 1) / 2
    a, b, c = (v.ravel() for v in np.meshgrid(t, t, t, indexing="ij"))
    wa, wb, wc = (v.ravel() for v in np.meshgrid(w, w, w, indexing="ij"))
    return np.stack([a, b * (1 - a), c * (1 - a) * (1 - b)], axis=1), wa * wb * wc * (1 - a) ** 2 * (1 - b)


def point_sum(T, x, g1, W, phi, gref, psi, P):
    """sum_q w |J| c (2 mu Sym(Grad_u):Grad_Test_u + mu u.Test_u), c = 1 + p^2, in
    the type T; x: the elements' vertices, P: the field's nodal values or None."""
    x, nd = x.astype(T), phi.shape[1]
    E = np.zeros((x.shape[0], nd, 3, nd, 3), dtype=T)
    eye, mu = np.eye(3, dtype=T), T(MU)
    for q in range(len(W)):
        K = np.einsum("evr,vc->erc", x, g1[q].astype(T))
        r, s = [1, 2, 0], [2, 0, 1]
        cof = K[:, r][:, :, r] * K[:, s][:, :, s] - K[:, r][:, :, s] * K[:, s][:, :, r]
        J = (K[:, 0] * cof[:, 0]).sum(axis=1)
        h = np.einsum("erc,ic->eir", cof / J[:, None, None], gref[q].astype(T))
        c = mu * (1 + (P.astype(T) @ psi[q].astype(T)) ** 2) if P is not None else mu + 0 * J
        f = phi[q].astype(T)
        dot = np.einsum("eic,ejc->eij", h, h) + np.outer(f, f)
        M = np.einsum("eib,eja->eiajb", h, h) + dot[:, :, None, :, None] * eye[None, None, :, None, :]
        E += (T(W[q]) * np.abs(J))[:, None, None, None, None] * (c[:, None, None, None, None] * M)
    return E.reshape(x.shape[0], 3 * nd, 3 * nd)


@pytest.mark.parametrize("seed", [1, 2])
@pytest.mark.parametrize("name", sorted(CASES))
def test_matrix(ctx, name, seed):
    print("case: accuracy of the polynomial route", name, seed, flush=True)
    gt, fem, im, field = CASES[name]
    n = 3 if fem == "FEM_QK(3,1)" else 2
    pts, cvx = meshes.regular_unit_mesh(n, gt)
    pts = meshes.jitter(pts, n, seed=seed)
    mesh = ga.Mesh(ctx, gt, pts, cvx)
    mf, mfp = ga.MeshFem(mesh, fem, 3), ga.MeshFem(mesh, fem, 1)
    p = np.random.default_rng(seed).uniform(0.5, 1.5, mfp.nbdof())
    ws = GaWorkspace(ctx)
    ws.add_fem_variable("u", mf)
    ws.add_fem_constant("p", mfp, p)
    ws.add_fixed_size_constant("mu", MU)
    ws.add_expression(("(1+p*p)*" if field else "") + "(mu*(Grad_u + Grad_u'):Grad_Test_u + mu*u.Test_u)",
                      ga.MeshIm(mesh, im))
    ws.assembly(2)
    ip, ix, v = ws.assembled_matrix_csr()
    P, W = core.integration_rule(im)
    phi, gref = (np.stack(a) for a in zip(*(core.fem_eval(fem, x) for x in P)))
    corner = np.array([[-1.0, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    g1 = [core.fem_eval("FEM_QK(3,1)", x)[1] if gt == "GT_QK(3,1)" else corner for x in P]
    args = (pts[cvx], g1, W, phi, gref, phi, p[mfp.basic_dof_table()] if field else None)
    dofs = mf.basic_dof_table().reshape(cvx.shape[0], -1)
    dofs = (dofs[:, :: dofs.shape[1] // phi.shape[1]][:, :, None] + np.arange(3)).reshape(cvx.shape[0], -1)
    N = mf.nbdof()
    key, inv = np.unique(dofs[:, :, None].astype(np.int64) * N + dofs[:, None, :], return_inverse=True)
    mat = np.repeat(np.arange(N), np.diff(ip)).astype(np.int64) * N + ix
    at = np.searchsorted(key, mat)
    assert np.array_equal(key[at], mat)

    def assembled(T, args):
        m = np.zeros(key.size, dtype=T)
        np.add.at(m, inv.ravel(), point_sum(T, *args).ravel())
        return m[at]

    fine = args
    if gt == "GT_PK(3,1)" and not field:
        x, w = fine_rule(5)
        fine = (pts[cvx], [corner] * len(w), w) + lagrange(int(fem[9]), x) + (None, None)
    exact = assembled(np.longdouble, fine)
    norm = np.sqrt((exact * exact).sum())
    far = [float(np.sqrt(((a - exact) ** 2).sum()) / norm) for a in (v, assembled(np.float64, args))]
    print("error %.3e, of the sum over the points in float64 %.3e" % tuple(far), flush=True)
    assert far[0] <= 1.1 * far[1]


def point_vector(T, x, g1, W, phi, gref, psi, P, U):
    """The same integrand's vector at the nodal values U, a point after another."""
    x, U = x.astype(T), U.astype(T)
    V = np.zeros(U.shape, dtype=T)
    mu = T(MU)
    for q in range(len(W)):
        K = np.einsum("evr,vc->erc", x, g1[q].astype(T))
        r, s = [1, 2, 0], [2, 0, 1]
        cof = K[:, r][:, :, r] * K[:, s][:, :, s] - K[:, r][:, :, s] * K[:, s][:, :, r]
        J = (K[:, 0] * cof[:, 0]).sum(axis=1)
        h = np.einsum("erc,ic->eir", cof / J[:, None, None], gref[q].astype(T))
        c = mu * (1 + (P.astype(T) @ psi[q].astype(T)) ** 2) if P is not None else mu + 0 * J
        H = np.einsum("eia,eic->eac", U, h)
        u = np.einsum("eia,i->ea", U, phi[q].astype(T))
        S = c[:, None, None] * (H + H.transpose(0, 2, 1))
        v = np.einsum("eac,eic->eia", S, h) + (c[:, None] * u)[:, None, :] * phi[q].astype(T)[None, :, None]
        V += (T(W[q]) * np.abs(J))[:, None, None] * v
    return V


@pytest.mark.parametrize("seed", [1, 2, 3])
@pytest.mark.parametrize("name", ["p2_const", "p3_const", "p3_field", "q1_const", "q1_field"])
def test_vector(ctx, name, seed):
    """(The element vectors' sums over the points are compensated: no tenth.)"""
    print("case: accuracy of the polynomial route's vector", name, seed, flush=True)
    gt, fem, im, field = CASES[name]
    n = 4 if fem == "FEM_QK(3,1)" else 3
    pts, cvx = meshes.regular_unit_mesh(n, gt)
    pts = meshes.jitter(pts, n, seed=seed)
    mesh = ga.Mesh(ctx, gt, pts, cvx)
    mf, mfp = ga.MeshFem(mesh, fem, 3), ga.MeshFem(mesh, fem, 1)
    rng = np.random.default_rng(seed)
    p, u = rng.uniform(0.5, 1.5, mfp.nbdof()), rng.standard_normal(mf.nbdof())
    ws = GaWorkspace(ctx)
    ws.add_fem_variable("u", mf, u)
    ws.add_fem_constant("p", mfp, p)
    ws.add_fixed_size_constant("mu", MU)
    ws.add_expression(("(1+p*p)*" if field else "") + "(mu*(Grad_u + Grad_u'):Grad_Test_u + mu*u.Test_u)",
                      ga.MeshIm(mesh, im))
    ws.assembly(1)
    V = ws.assembled_vector()
    P, W = core.integration_rule(im)
    phi, gref = (np.stack(a) for a in zip(*(core.fem_eval(fem, x) for x in P)))
    corner = np.array([[-1.0, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    g1 = [core.fem_eval("FEM_QK(3,1)", x)[1] if gt == "GT_QK(3,1)" else corner for x in P]
    dofs = mf.basic_dof_table().reshape(cvx.shape[0], -1)
    dofs = dofs[:, :: dofs.shape[1] // phi.shape[1]][:, :, None] + np.arange(3)
    args = (pts[cvx], g1, W, phi, gref, phi, p[mfp.basic_dof_table()] if field else None, u[dofs])

    def assembled(T):
        v = np.zeros(V.size, dtype=T)
        np.add.at(v, dofs.ravel(), point_vector(T, *args).ravel())
        return v

    exact = assembled(np.longdouble)
    far = [float(np.sqrt(((a - exact) ** 2).sum() / (exact ** 2).sum())) for a in (V, assembled(np.float64))]
    print("error %.3e, of the sum over the points in float64 %.3e" % tuple(far), flush=True)
    assert far[0] <= far[1]
