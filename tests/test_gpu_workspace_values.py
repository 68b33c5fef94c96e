"""What the polynomial route reads between assemblies: values given on the host
and on the device in turn, constants that change and stay, each against a
workspace made at those values (bit for bit, matrix and vector)."""
import numpy as np
import pytest

import getfem_amd as ga
from getfem_amd import meshes
from getfem_amd.workspace import GaWorkspace

pytestmark = pytest.mark.gpu

EXPR = "k*(1+c*p*p)*Grad_u:Grad_Test_u - p*Div_Test_u - Test_p*Div_u - c*p*p*p*Test_p"


def workspace(ctx, mfu, mfp, mim, u, p, k, c):
    ws = GaWorkspace(ctx)
    ws.add_fem_variable("u", mfu, u, first=0)
    ws.add_fem_variable("p", mfp, p, first=mfu.nbdof())
    ws.add_fixed_size_constant("k", k)
    ws.add_fixed_size_constant("c", c)
    ws.add_expression(EXPR, mim)
    return ws


def answers(ws):
    ws.assembly(2)
    m = ws.assembled_matrix_csr()
    ws.assembly(1)
    return tuple(m) + (ws.assembled_vector(),)


@pytest.mark.parametrize("n", [1, 3])
def test_values_in_turn(ctx, n):
    import torch
    print("case: values of the polynomial route", n, flush=True)
    pts, cvx = meshes.regular_unit_mesh(n, "GT_PK(3,1)")
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", meshes.jitter(pts, n), cvx)
    mfu, mfp = ga.MeshFem(mesh, "FEM_PK(3,2)", 3), ga.MeshFem(mesh, "FEM_PK(3,1)", 1)
    mim = ga.MeshIm(mesh, "IM_TETRAHEDRON(5)")
    rng = np.random.default_rng(n)
    u = [rng.standard_normal(mfu.nbdof()) for _ in range(3)]
    p = [rng.uniform(0.5, 1.5, mfp.nbdof()) for _ in range(3)]
    ws = workspace(ctx, mfu, mfp, mim, u[0], p[0], 2.0, 0.5)
    now = [u[0], p[0], 2.0, 0.5]

    def check():
        for a, b in zip(answers(ws), answers(workspace(ctx, mfu, mfp, mim, *now))):
            assert np.array_equal(a, b)

    check()
    d = torch.from_numpy(p[1]).cuda()
    torch.cuda.synchronize()
    ws.set_values_device("p", d.data_ptr())  # p on the device, u on the host
    now[1] = p[1]
    check()
    d.zero_()  # the caller's array is read when it is given
    torch.cuda.synchronize()
    check()
    ws.set_values("k", 3.0)  # one constant changes
    now[2] = 3.0
    check()
    ws.set_values("p", p[2])  # back to the host
    now[1] = p[2]
    check()
    ws.set_values("u", u[2])
    ws.set_values("k", 2.0)
    now[0], now[2] = u[2], 2.0
    check()
