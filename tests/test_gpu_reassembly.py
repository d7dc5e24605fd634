"""GPU: Assemble called again on a form whose coefficient or geometry changed.

Bars: bitwise against a form created afterwards: the same kernels on the same
operator data.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _form(M, fes, k, mass=False):
    a = M.BilinearForm(fes)
    a.SetAssemblyLevel(M.AssemblyLevel.PARTIAL)
    c = M.PWConstCoefficient(k)
    a.AddDomainIntegrator(M.DiffusionIntegrator(c))
    if mass:
        a.AddDomainIntegrator(M.MassIntegrator(c))
    a.Assemble()
    return a


def _space(M, p, n):
    mesh = M.Mesh.MakeCartesian3D(n, n, n)
    mesh.Perturb(0.2, p)
    return mesh, M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))


def _low(torch, a, x, prec):
    y = torch.full_like(x, float("nan"))
    a.MultLowPrecision(x, y, prec)
    return y


@pytest.mark.parametrize("prec", ["PREC_FP32", "PREC_BF16_PA"])
@pytest.mark.parametrize("p,mass", [(1, False), (3, True), (6, False)])
def test_reduced_precision_follows_the_operator(h1pa, torch_cuda, prec, p, mass):
    """The reduced-precision copy of the operator data is made again after a
    re-assembly, for a coefficient changed in place and for moved nodes."""
    M, torch = h1pa, torch_cuda
    prec = getattr(M, prec)
    mesh, fes = _space(M, p, 4)
    rng = np.random.default_rng(p)
    k = torch.from_numpy(rng.uniform(0.5, 2.0, fes.GetNE())).cuda()
    x = torch.from_numpy(rng.uniform(-1, 1, fes.GetNDofs())).cuda().float()
    a = _form(M, fes, k, mass)
    old = _low(torch, a, x, prec)
    k.mul_(3.0).add_(torch.linspace(0, 1, fes.GetNE(), dtype=k.dtype, device=k.device))
    a.Assemble()
    got = _low(torch, a, x, prec)
    assert not torch.equal(got, old)
    assert torch.equal(got, _low(torch, _form(M, fes, k, mass), x, prec))
    mesh.Perturb(0.1, 77)
    a.Assemble()
    moved = _low(torch, a, x, prec)
    assert not torch.equal(moved, got)
    assert torch.equal(moved, _low(torch, _form(M, fes, k, mass), x, prec))


def test_bf16_cycle_follows_the_operator(h1pa, torch_cuda):
    """A multigrid cycle in BF16, set up after a re-assembly."""
    M, torch = h1pa, torch_cuda
    mesh, fes = _space(M, 4, 4)
    rng = np.random.default_rng(1)
    k = torch.from_numpy(rng.uniform(0.5, 2.0, fes.GetNE())).cuda()
    x = torch.from_numpy(rng.uniform(-1, 1, fes.GetNDofs())).cuda()
    a = _form(M, fes, k)

    def cycle(form):
        mg = M.PMultigrid(form, [1, 2, 4], cycle_precision=M.PREC_BF16_PA)
        y = torch.full_like(x, float("nan"))
        mg.Mult(x, y)
        torch.cuda.synchronize()
        return y

    old = cycle(a)
    k.copy_(k.flip(0) * 2.0)
    a.Assemble()
    got = cycle(a)
    assert not torch.equal(got, old)
    assert torch.equal(got, cycle(_form(M, fes, k)))


def _queue(M, torch, what, fes, a, x, n):
    """n results of one kind queued on the current stream, which read the operator
    data; and the vector that each writes."""
    ess = fes.GetBoundaryTrueDofs()
    if what == "low":
        x = x.float()
    ys = [torch.full_like(x, float("nan")) for _ in range(n)]
    if what == "mult":
        f = [lambda y: a.Mult(x, y)]
    elif what == "low":
        f = [lambda y: a.MultLowPrecision(x, y, M.PREC_BF16_PA)]
    elif what == "diagonal":
        f = [a.AssembleDiagonal]
    else:
        A = M.ConstrainedOperator(a, ess)
        S = M.OperatorChebyshevSmoother(A, None, ess, 2) if what == "smoother" else A
        f = [lambda y: S.Mult(x, y)]
    return ys, f[0]


@pytest.mark.parametrize("what", ["mult", "low", "diagonal", "constrained", "smoother"])
def test_products_queued_on_another_stream(h1pa, torch_cuda, what):
    """Products queued on one stream when another re-assembles apply the operator
    they were queued with: bitwise the product before.  On the same stream they
    need no wait, and with a second stream in between they do again."""
    M, torch = h1pa, torch_cuda
    mesh, fes = _space(M, 4, 24)
    k = torch.full((fes.GetNE(),), 2.0, dtype=torch.float64, device="cuda")
    x = torch.rand(fes.GetNDofs(), dtype=torch.float64, device="cuda")
    a = _form(M, fes, k)
    st = [torch.cuda.Stream() for _ in range(3)]
    for queue, assemble in ((0, 1), (1, 1), (2, 0), (0, 0), (1, 0)):
        want, f = _queue(M, torch, what, fes, a, x, 1)
        f(want[0])
        ys, f = _queue(M, torch, what, fes, a, x, 30)
        f(ys[0])
        torch.cuda.synchronize()
        with torch.cuda.stream(st[queue]):
            for y in ys:
                f(y)
        with torch.cuda.stream(st[assemble]):
            k.add_(1.0)
            a.Assemble()
        torch.cuda.synchronize()
        assert all(torch.equal(y, want[0]) for y in ys), (queue, assemble)
