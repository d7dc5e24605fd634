"""GPU: solves that end on (A d, d) = 0 or on an (A d, d) that is not finite, in
the first iteration: nothing may be written after it, on either side of the
size from which CG sums its products in kernels of their own, and in a batch with
and without a slot too large for folded sums.

The right-hand sides make (B r, r) an ordinary number and (A d, d) not: with
b = s D v and d = D^-1 b = s v, (B r, r) = s^2 (v, D v) and (A d, d) = s^2 (v, A v).
For a smooth v every product of the second is below half the smallest double,
2.5e-324, where the largest of the first is 3e-323; for the highest eigenvector the
second is c > 1 times the first, which is chosen as the largest double over sqrt(c).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BIG = np.finfo(np.float64).max


def _system(M, torch, p, n):
    mesh = M.Mesh.MakeCartesian3D(n, n, n)
    fes = M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))
    a = M.BilinearForm(fes)
    a.SetAssemblyLevel(M.AssemblyLevel.PARTIAL)
    a.AddDomainIntegrator(M.DiffusionIntegrator(M.ConstantCoefficient(100.0)))
    a.Assemble()
    ess = fes.GetBoundaryTrueDofs()
    zero = torch.zeros(fes.GetNDofs(), dtype=torch.float64, device="cuda")
    A, _, _ = a.FormLinearSystem(ess, zero, zero)
    D = torch.empty_like(zero)
    a.AssembleDiagonal(D)
    return dict(mesh=mesh, fes=fes, a=a, A=A, D=D, ess=ess, free=_free(torch, fes, ess))


def _free(torch, fes, ess):
    f = torch.ones(fes.GetNDofs(), dtype=torch.float64, device="cuda")
    f[ess.long()] = 0.0
    return f


def _apply(torch, s, v):
    out = torch.empty_like(v)
    s["A"].Mult(v, out)
    return out


def _ends_at_zero(torch, s):
    """b with (B r, r) > 0 and every product of (A d, d) zero: v from inverse-like
    smoothing, (1 - D^-1 A / 3) applied often (its smooth part stays)."""
    v = s["free"].clone()
    for _ in range(60):
        v = v - _apply(torch, s, v) * s["free"] / s["D"] / 3.0
    top = float((s["D"] * v * v).max())
    low = float((v * _apply(torch, s, v)).abs().max())
    assert low < 0.07 * top
    return s["D"] * v * s["free"] * np.sqrt(3e-323 / 1e-300 / top) * 1e-150


def _ends_at_infinity(torch, s):
    g = torch.Generator(device="cuda").manual_seed(1)
    v = torch.rand(s["D"].numel(), dtype=torch.float64, device="cuda", generator=g) - 0.5
    for _ in range(40):
        v = _apply(torch, s, v) * s["free"] / s["D"]
        v = v / v.abs().max()
    nom = float((s["D"] * v * v).sum())
    c = float((v * _apply(torch, s, v)).sum()) / nom
    assert c > 1.2
    return s["D"] * v * np.sqrt(BIG / np.sqrt(c) / nom), v, c


# 4,913, 117,649 and 226,981 DOFs fold the scalar steps, 300,763 do not
@pytest.mark.parametrize("p,n", [(2, 8), (2, 24), (3, 20), (2, 33)])
def test_cg_ends_before_an_update(h1pa, torch_cuda, p, n):
    M, torch = h1pa, torch_cuda
    s = _system(M, torch, p, n)
    cg = M.CGSolver()
    cg.SetRelTol(1e-10)
    cg.SetMaxIter(50)
    cg.SetOperator(s["A"])
    cg.SetPreconditioner(M.OperatorJacobiSmoother(s["a"], s["ess"]))
    zero, inf = _ends_at_zero(torch, s), _ends_at_infinity(torch, s)[0]
    for every in (1, 8):
        cg.check_every = every
        for _ in range(5):
            x = torch.full_like(zero, float("nan"))
            cg.Mult(zero, x)
            assert not cg.GetConverged() and cg.GetNumIterations() == 0
            assert not bool(x.any())  # NaN counts as nonzero
            x.fill_(float("nan"))
            with pytest.raises(M.H1paError):
                cg.Mult(inf, x)
            assert not bool(x.any())
    # an ordinary solve afterwards
    cg.SetMaxIter(2000)
    b = s["D"] * s["free"]
    cg.Mult(b, x)
    r = b - _apply(torch, s, x)
    assert cg.GetConverged() and float(r.norm() / b.norm()) < 1e-8


@pytest.mark.parametrize("K", [1, 2, 3, 8])
@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("prec", ["PREC_FP64", "PREC_FP32", "PREC_BF16_PA"])
def test_batch_ends_before_an_update(h1pa, torch_cuda, prec, large, K):
    """As above; mixed slots run FP32 inner iterations, in which (A d, d) is zero
    because b = 1e-60 rounds to zero, and not finite because A d overflows FP32.
    They share the batch with ordinary solves, and (large) with a slot of 1.1M
    DOFs, which no folded sum takes."""
    M, torch = h1pa, torch_cuda
    mode = getattr(M, prec)
    s = _system(M, torch, 2, 8)
    if mode == M.PREC_FP64:
        zero, inf = _ends_at_zero(torch, s), _ends_at_infinity(torch, s)[0]
    else:
        zero = s["D"] * s["free"] * 1e-60
        v = _ends_at_infinity(torch, s)[1]
        inf = s["D"] * v
        inf = inf * (3.3e38 / inf.abs().max())
    b = s["D"] * s["free"]
    rhs = [zero, b, inf, b * 2.0]
    xs = [torch.full_like(b, float("nan")) for _ in rhs]
    bs = M.BatchSolver(precision=mode, iters_per_replay=K)
    tags = [bs.Add(s["A"], q, x, rel_tol=1e-10, max_iter=400) for q, x in zip(rhs, xs)]
    if large:
        t = _system(M, torch, 3, 35)
        bl = t["D"] * t["free"]
        xl = torch.empty_like(bl)
        tags.append(bs.Add(t["A"], bl, xl, rel_tol=1e-2, max_iter=400))
    bs.Run()
    res = dict(bs.Poll())
    assert not res[tags[0]]["converged"] and not bool(xs[0].any())
    assert res[tags[2]]["status"] == M.H1PA_ENONFINITE and not bool(xs[2].any())
    for k, f in ((1, 1.0), (3, 2.0)):
        assert res[tags[k]]["converged"]
        r = b * f - _apply(torch, s, xs[k])
        assert float(r.norm() / b.norm()) < 1e-7
