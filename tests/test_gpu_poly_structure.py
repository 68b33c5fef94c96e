"""The polynomial route's matrix from its candidate structure: after values
that make entries vanish, return and change sign, the CSR equals (bit for bit)
that of a workspace made at those values, for blocks of every tile shape
(test fields of 1 and 3 components, degrees 1 to 3), on constant and on
field-dependent programs and on hexahedra."""
import numpy as np
import pytest

import getfem_amd as ga
from getfem_amd import meshes
from getfem_amd.workspace import GaWorkspace

pytestmark = pytest.mark.gpu

IM = {"GT_PK(3,1)": "IM_TETRAHEDRON(5)", "GT_QK(3,1)": "IM_GAUSS_PARALLELEPIPED(3,4)"}
CASES = {
    "p2v_p1_const": ("GT_PK(3,1)", "FEM_PK(3,2)", "FEM_PK(3,1)", "rho*Sym(Grad_u):Grad_Test_u - rho*p*Div_Test_u"
                     " - rho*Test_p*Div_u - p*Test_p"),
    "p1v_p2_const": ("GT_PK(3,1)", "FEM_PK(3,1)", "FEM_PK(3,2)", "rho*Grad_u:Grad_Test_u + u.Grad_Test_p"
                     " + rho*Grad_p.Grad_Test_p"),
    "p3v_p1_const": ("GT_PK(3,1)", "FEM_PK(3,3)", "FEM_PK(3,1)", "rho*u.Test_u - rho*p*Div_Test_u + p*Test_p"),
    "p2v_p1_field": ("GT_PK(3,1)", "FEM_PK(3,2)", "FEM_PK(3,1)", "rho*(1+p*p)*Grad_u:Grad_Test_u"
                     " + rho*p*p*p*Test_p + Grad_p.Grad_Test_p"),
    "q2_q1_hex": ("GT_QK(3,1)", "FEM_QK(3,2)", "FEM_QK(3,1)", "rho*Grad_u.Grad_Test_u + rho*p*Test_u + Grad_p.Grad_Test_p"),
}


def workspace(ctx, mfs, mim, vals, expr):
    mfu, mfp, mfr = mfs
    ws = GaWorkspace(ctx)
    ws.add_fem_variable("u", mfu, vals["u"], first=0)
    ws.add_fem_variable("p", mfp, vals["p"], first=mfu.nbdof())
    ws.add_fem_constant("rho", mfr, vals["rho"])
    ws.add_expression(expr, mim)
    return ws


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("n", [1, 2])
def test_pattern_follows_values(ctx, name, n):
    print("case: candidate structure", name, n, flush=True)
    gt, femu, femp, expr = CASES[name]
    pts, cvx = meshes.regular_unit_mesh(n, gt)
    pts = meshes.jitter(pts, n)
    mesh = ga.Mesh(ctx, gt, pts, cvx)
    mfu = ga.MeshFem(mesh, femu, 1 if name == "q2_q1_hex" else 3)
    mfp = ga.MeshFem(mesh, femp, 1)
    mfr = ga.MeshFem(mesh, "FEM_PK_DISCONTINUOUS(3,0)" if gt == "GT_PK(3,1)" else femp, 1)
    mim = ga.MeshIm(mesh, IM[gt])
    rng = np.random.default_rng(n)
    vals = {"u": rng.standard_normal(mfu.nbdof()), "p": rng.uniform(0.5, 1.5, mfp.nbdof()),
            "rho": rng.uniform(0.5, 2.0, mfr.nbdof())}
    ws = workspace(ctx, (mfu, mfp, mfr), mim, vals, expr)
    r0 = vals["rho"]
    some = r0.copy()
    some[:: 2] = 0.0
    sizes = []
    for rho in (r0, some, 0.0 * r0, r0, -some):
        vals["rho"] = rho
        ws.set_values("rho", rho)
        ws.assembly(2)
        got = ws.assembled_matrix_csr()
        ref = workspace(ctx, (mfu, mfp, mfr), mim, vals, expr)
        ref.assembly(2)
        for a, b in zip(got, ref.assembled_matrix_csr()):
            assert np.array_equal(a, b)
        sizes.append(got[2].size)
    assert sizes[2] < sizes[0] == sizes[3]


@pytest.mark.parametrize("name", sorted(CASES))
def test_same_matrix_without_the_structure(ctx, name):
    """A limit below the number of candidates has the kept entries sorted at
    every assembly: the same CSR bit for bit, also where values vanish and
    return, where everything vanishes, and after the limit is lifted again."""
    print("case: matrix without the structure", name, flush=True)
    gt, femu, femp, expr = CASES[name]
    pts, cvx = meshes.regular_unit_mesh(2, gt)
    pts = meshes.jitter(pts, 2)
    mesh = ga.Mesh(ctx, gt, pts, cvx)
    mfs = (ga.MeshFem(mesh, femu, 1 if name == "q2_q1_hex" else 3), ga.MeshFem(mesh, femp, 1),
           ga.MeshFem(mesh, "FEM_PK_DISCONTINUOUS(3,0)" if gt == "GT_PK(3,1)" else femp, 1))
    mim = ga.MeshIm(mesh, IM[gt])
    rng = np.random.default_rng(7)
    vals = {"u": rng.standard_normal(mfs[0].nbdof()), "p": rng.uniform(0.5, 1.5, mfs[1].nbdof()),
            "rho": rng.uniform(0.5, 2.0, mfs[2].nbdof())}
    ws, ref = workspace(ctx, mfs, mim, vals, expr), workspace(ctx, mfs, mim, vals, expr)
    ws.set_structure_limit(1000)
    some = vals["rho"].copy()
    some[:: 2] = 0.0

    def same(rho):
        for w in (ws, ref):
            w.set_values("rho", rho)
            w.assembly(2)
        got, want = ws.assembled_matrix_csr(), ref.assembled_matrix_csr()
        for a, b in zip(got, want):
            assert np.array_equal(a, b)
        return want[2].size

    sizes = [same(rho) for rho in (vals["rho"], some, 0.0 * some, -vals["rho"])]
    assert sizes[2] < sizes[1] <= sizes[0] == sizes[3]
    ws.set_structure_limit(2**31 - 1)
    same(some)
    with pytest.raises(ga.GfxError):
        ws.set_structure_limit(-1)


def test_matrix_without_blocks(ctx):
    """An expression whose second derivative vanishes: an empty matrix, whose
    arrays are there all the same."""
    import ctypes

    from getfem_amd import _lib
    print("case: matrix without blocks", flush=True)
    pts, cvx = meshes.regular_unit_mesh(1)
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", pts, cvx)
    mf = ga.MeshFem(mesh, "FEM_PK(3,2)", 1)
    ws = GaWorkspace(ctx)
    ws.add_fem_variable("u", mf)
    ws.add_expression("3*u", ga.MeshIm(mesh, "IM_TETRAHEDRON(5)"))
    ws.assembly(2)
    ip, ix, v = ws.assembled_matrix_csr()
    assert ip.size == mf.nbdof() + 1 and not ip.any() and ix.size == v.size == 0
    p = [ctypes.c_void_p() for _ in range(3)]
    n, nnz = ctypes.c_int64(), ctypes.c_int64()
    _lib.check(_lib.lib().gfx_ws_device_csr(ws.h, ctypes.byref(n), ctypes.byref(nnz), *[ctypes.byref(x) for x in p]),
               ctx.h)
    assert nnz.value == 0 and all(x.value for x in p)
    assert ws.assembled_matrix().nnz == 0
