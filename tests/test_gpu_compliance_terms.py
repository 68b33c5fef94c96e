"""The compliance kernels' exponent forms (whole exponents by products, others
by pow), element counts around the workgroup's 256, vertex gathers of few and
many incidences, and every choice of outputs, against torch autograd of the
same sum in float64."""
import numpy as np
import pytest

import getfem_amd as ga
from getfem_amd import meshes

pytestmark = pytest.mark.gpu

LAM, MU, EMIN = 1.2, 0.8, 1e-3


def reference(cvx, dofs, rho, X, u, penal):
    import torch
    x = X[cvx]
    K = (x[:, 1:] - x[:, :1]).transpose(1, 2)
    B = torch.linalg.inv(K).transpose(1, 2)
    h = torch.tensor([[-1.0, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]], dtype=torch.float64, device=X.device)
    g = torch.matmul(h, B.transpose(1, 2))
    H = torch.matmul(u.reshape(-1, 3)[dofs].transpose(1, 2), g)
    eps = (H + H.transpose(1, 2)) / 2
    W = LAM * H.diagonal(dim1=1, dim2=2).sum(-1) ** 2 + 2 * MU * (eps ** 2).sum(dim=(1, 2))
    return ((EMIN + rho ** penal * (1 - EMIN)) * torch.linalg.det(K).abs() / 6 * W).sum()


@pytest.mark.parametrize("n", [1, 3, 7])
@pytest.mark.parametrize("penal", [1.0, 2.5, 3.0, 8.0, 9.0])
def test_against_autograd(ctx, n, penal):
    import torch

    from getfem_amd.torch_ops import Compliance, compliance
    print("case: compliance", n, penal, flush=True)
    pts, cvx = meshes.regular_unit_mesh(n)
    pts = meshes.jitter(pts, n)
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", pts, cvx)
    mf = ga.MeshFem(mesh, "FEM_PK(3,1)", 3)
    op = Compliance(mf, ga.MeshIm(mesh, "IM_TETRAHEDRON(1)"), LAM, MU, EMIN, penal)
    dev = "cuda"
    args = [torch.tensor(a, device=dev, requires_grad=True) for a in
            (meshes.simp_density(cvx.shape[0]), pts, meshes.random_state(mf.nbdof()))]
    J = compliance(*args, op)
    got = torch.autograd.grad(J, args)
    dofs = torch.tensor(mf.basic_dof_table() // 3, device=dev).long()
    Jr = reference(torch.tensor(cvx, device=dev).long(), dofs, *args, penal)
    ref = torch.autograd.grad(Jr, args)
    assert abs(float(J.detach() - Jr.detach())) <= 1e-13 * abs(float(Jr.detach()))
    for a, b in zip(got, ref):
        assert float((a - b).norm()) <= 1e-13 * float(b.norm())
    # outputs one at a time, on another stream than torch's default one
    rho, X, u = (a.detach() for a in args)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        J1 = torch.empty((), dtype=torch.float64, device=dev)
        for k, like in enumerate((rho, X, u)):
            out = [J1, None, None, None]
            out[1 + k] = torch.empty_like(like)
            op.eval(rho, X, u, out=tuple(out))
            op.check()
            side.synchronize()
            assert torch.equal(out[1 + k], got[k]) and torch.equal(J1, J.detach())


@pytest.mark.parametrize("penal", [2.0, 3.0, 5.0, 8.0])
def test_whole_exponents_are_correctly_rounded(ctx, penal):
    """dJ/drho of unit tetrahedra under a unit strain is p rho^(p-1) w: the
    power (within half an ulp, 2^-53 relative, and terms of its square) and one
    product with w may round, p = 2, 3, 5 and 8 by a third."""
    from fractions import Fraction

    import torch

    from getfem_amd.torch_ops import Compliance
    print("case: compliance exponent", penal, flush=True)
    n = 1500
    unit = np.array([[0.0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    pts = (unit[None] + 2.0 * np.arange(n)[:, None, None]).reshape(-1, 3)
    mesh = ga.Mesh(ctx, "GT_PK(3,1)", pts, np.arange(4 * n, dtype=np.int32).reshape(n, 4))
    mf = ga.MeshFem(mesh, "FEM_PK(3,1)", 3)
    mim = ga.MeshIm(mesh, "IM_TETRAHEDRON(1)")
    op = Compliance(mf, mim, 0.0, 0.5, 0.0, penal)  # 2 mu = 1: W = 1
    u = np.zeros(mf.nbdof())
    u[0::3] = mf.basic_dof_nodes()[:, 0] % 2.0  # the first coordinate in the element
    rho = np.random.default_rng(int(penal)).uniform(0.05, 1.0, n)
    out = [torch.empty((), dtype=torch.float64, device="cuda"), torch.empty(n, dtype=torch.float64, device="cuda"),
           None, None]
    dev = [torch.tensor(a, device="cuda") for a in (rho, pts, u)]
    torch.cuda.synchronize()
    op.eval(*dev, out=tuple(out))
    op.check()
    w = Fraction(float(mim.points()[1].sum()))
    p = int(penal)
    worst = max(abs(Fraction(float(g)) / (p * Fraction(float(r)) ** (p - 1) * w) - 1)
                for g, r in zip(out[1].cpu().numpy(), rho))
    assert float(worst) <= 3.1 * 2.0 ** -53
