"""Assemblies on the polynomial route that fail: the results of the last good
one are not handed out under the failed one's name, the next good assembly
gives what a new workspace gives, and nothing is left running."""
import numpy as np
import pytest

import getfem_amd as ga
from getfem_amd import meshes
from getfem_amd.workspace import GaWorkspace

pytestmark = pytest.mark.gpu

MESH = {"tets": ("GT_PK(3,1)", "FEM_PK(3,2)", "FEM_PK(3,1)", "IM_TETRAHEDRON(5)"),
        "hexes": ("GT_QK(3,1)", "FEM_QK(3,1)", "FEM_QK(3,1)", "IM_GAUSS_PARALLELEPIPED(3,3)")}
EXPR = {"constant": "2*mu*Sym(Grad_u):Grad_Test_u - p*Div_Test_u - Test_p*Div_u - p*Test_p",
        "field": "(1+p*p)*Grad_u:Grad_Test_u + mu*p*p*p*Test_p"}


def model(ctx, kind, expr):
    gt, fu, fp, im = MESH[kind]
    pts, cvx = meshes.regular_unit_mesh(2, gt)
    pts = meshes.jitter(pts, 2)
    mesh = ga.Mesh(ctx, gt, pts, cvx)
    mfu, mfp = ga.MeshFem(mesh, fu, 3), ga.MeshFem(mesh, fp, 1)
    rng = np.random.default_rng(1)
    ws = GaWorkspace(ctx)
    ws.add_fem_variable("u", mfu, rng.standard_normal(mfu.nbdof()), first=0)
    ws.add_fem_variable("p", mfp, rng.uniform(0.5, 1.5, mfp.nbdof()), first=mfu.nbdof())
    ws.add_fixed_size_constant("mu", 0.8)
    ws.add_expression(EXPR[expr], ga.MeshIm(mesh, im))
    return ws, mesh, pts, cvx


@pytest.mark.parametrize("kind", sorted(MESH))
@pytest.mark.parametrize("expr", sorted(EXPR))
def test_degenerate_element(ctx, kind, expr):
    print("case: failed assembly", kind, expr, flush=True)
    ws, mesh, pts, cvx = model(ctx, kind, expr)
    ws.assembly(2)
    ws.assembly(1)
    good = ws.assembled_matrix_csr() + (ws.assembled_vector(),)
    flat = pts.copy()
    flat[cvx[3]] = flat[cvx[3][0]]
    mesh.set_points(flat)
    for _ in range(2):
        for order in (2, 1):
            with pytest.raises(ga.GfxError, match="degenerate"):
                ws.assembly(order)
        with pytest.raises(ga.GfxError, match="no matrix assembled"):
            ws.assembled_matrix_csr()
        with pytest.raises(ga.GfxError, match="no order-1 assembly"):
            ws.assembled_vector()
    mesh.set_points(pts)
    ws.assembly(2)
    ws.assembly(1)
    for a, b in zip(ws.assembled_matrix_csr() + (ws.assembled_vector(),), good):
        assert np.array_equal(a, b)


def test_vector_of_an_earlier_setup(ctx):
    """A vector whose buffer was given back with the setup that it came from
    is not handed out any more."""
    print("case: vector of an earlier setup", flush=True)
    ws, mesh, _, _ = model(ctx, "tets", "constant")
    ws.assembly(1)
    ws.assembled_vector()
    ws.add_expression("p*Test_p", ga.MeshIm(mesh, "IM_TETRAHEDRON(5)"))
    with pytest.raises(ga.GfxError):  # (two mesh_ims: refused after the setup was dropped)
        ws.assembly(1)
    with pytest.raises(ga.GfxError, match="no order-1 assembly"):
        ws.assembled_vector()


def test_refusal_waits_for_its_uploads():
    """An assembly that is refused after the variables' values went on their
    way (here: more than 2^31 dofs) returns when the stream has ended."""
    import torch
    print("case: refusal behind a busy stream", flush=True)
    c = ga.Context(0)
    side = torch.cuda.Stream()
    c.set_stream(side.cuda_stream)
    pts, cvx = meshes.regular_unit_mesh(2)
    mesh = ga.Mesh(c, "GT_PK(3,1)", pts, cvx)
    mfu, mfp = ga.MeshFem(mesh, "FEM_PK(3,2)", 3), ga.MeshFem(mesh, "FEM_PK(3,1)", 1)
    ws = GaWorkspace(c)
    ws.add_fem_variable("u", mfu, np.ones(mfu.nbdof()), first=0)
    ws.add_fem_variable("p", mfp, np.ones(mfp.nbdof()), first=2**31)
    ws.add_expression("u.Test_u + p*Test_p", ga.MeshIm(mesh, "IM_TETRAHEDRON(5)"))
    with pytest.raises(ga.GfxError, match="dofs"):  # (the setup's own waits are over)
        ws.assembly(2)
    x = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(200):
            x = torch.clamp(x @ x, -1, 1)
    busy = not side.query()
    with pytest.raises(ga.GfxError, match="dofs"):
        ws.assembly(2)
    assert busy and side.query()
