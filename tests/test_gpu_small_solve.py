"""GPU: CG on systems small enough for the folded scalar steps.

The stopping iteration, the result and the failure states must not depend on
how often the host looks (the state is read one look late), and must match the
oracle's iteration count (+-1) on both sides of the size rule (262,144 DOFs).
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(M, torch, p, n, seed=1):
    mesh = M.Mesh.MakeCartesian3D(n, n, n)
    mesh.Perturb(0.2, seed)
    fes = M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))
    a = M.BilinearForm(fes)
    a.SetAssemblyLevel(M.AssemblyLevel.PARTIAL)
    a.AddDomainIntegrator(M.DiffusionIntegrator(M.SinCosCoefficient()))
    a.Assemble()
    b = torch.from_numpy(np.random.default_rng(seed).uniform(-1, 1, fes.GetNDofs())).cuda()
    ess = fes.GetBoundaryTrueDofs()
    A, X, B = a.FormLinearSystem(ess, torch.zeros_like(b), b)
    cg = M.CGSolver()
    cg.SetRelTol(1e-10)
    cg.SetMaxIter(5000)
    cg.SetOperator(A)
    cg.SetPreconditioner(M.OperatorJacobiSmoother(a, ess))
    return dict(mesh=mesh, fes=fes, a=a, A=A, X=X, B=B, cg=cg, b=b)


@pytest.mark.parametrize("p,n", [(1, 1), (1, 2), (2, 3), (3, 5), (4, 4), (6, 3), (8, 2), (1, 62),
                                 (1, 63), (1, 64)])
def test_looks_do_not_matter(orc, h1pa, torch_cuda, p, n):
    M, torch = h1pa, torch_cuda
    s = _system(M, torch, p, n)
    ref = None
    for every in (1, 2, 3, 8, 50):
        s["cg"].check_every = every
        x = torch.full_like(s["X"], float("nan"))
        s["cg"].Mult(s["B"], x)
        got = (x, s["cg"].GetNumIterations(), s["cg"].GetConverged(), s["cg"].GetFinalNorm())
        if ref is None:
            ref = got
            P = orc.Problem(n, p, perturb=0.2, seed=1, coeff="sincos")
            X, B = P.form_linear_system(np.zeros(P.ndofs), s["b"].cpu().numpy())
            its = P.pcg(B, rel_tol=1e-10, max_iter=5000)[1]["iterations"]
            assert got[2] and abs(got[1] - its) <= 1
        assert torch.equal(got[0], ref[0]) and got[1:] == ref[1:], every


@pytest.mark.parametrize("limit", [1, 2, 7, 8, 9, 17])
def test_iteration_limit(h1pa, torch_cuda, limit):
    M, torch = h1pa, torch_cuda
    s = _system(M, torch, 3, 6)
    s["cg"].SetMaxIter(limit)
    ref = None
    for every in (1, 4, 8):
        s["cg"].check_every = every
        x = torch.empty_like(s["X"])
        s["cg"].Mult(s["B"], x)
        assert not s["cg"].GetConverged() and s["cg"].GetNumIterations() == limit
        assert ref is None or torch.equal(x, ref)
        ref = x


def test_zero_and_nan_right_hand_sides(h1pa, torch_cuda):
    M, torch = h1pa, torch_cuda
    s = _system(M, torch, 2, 6)
    x = torch.full_like(s["X"], float("nan"))
    s["cg"].Mult(torch.zeros_like(s["B"]), x)
    assert s["cg"].GetConverged() and not bool(x.any())
    with pytest.raises(M.H1paError):
        s["cg"].Mult(s["B"] * float("nan"), x)
    s["cg"].Mult(s["B"], x)  # the next solve is not disturbed
    assert s["cg"].GetConverged()


def test_threads_and_streams(h1pa, torch_cuda):
    """Solves side by side on their own streams share the pool of state blocks."""
    M, torch = h1pa, torch_cuda
    systems = [_system(M, torch, p, n, seed=p) for p, n in ((1, 9), (2, 6), (3, 5), (4, 4))]
    refs = []
    for s in systems:
        x = torch.empty_like(s["X"])
        s["cg"].Mult(s["B"], x)
        refs.append((x, s["cg"].GetNumIterations()))
    torch.cuda.synchronize()
    bad = []

    def work(k):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for _ in range(6):
                x = torch.empty_like(systems[k]["X"])
                systems[k]["cg"].Mult(systems[k]["B"], x)
                st.synchronize()
                if not torch.equal(x, refs[k][0]) or \
                        systems[k]["cg"].GetNumIterations() != refs[k][1]:
                    bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(systems))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("pre,post,cycle", [(1, 1, "V"), (2, 2, "V"), (0, 1, "V"), (1, 0, "V"),
                                            (1, 1, "W")])
def test_cycle_is_its_public_pieces(h1pa, torch_cuda, order, pre, post, cycle):
    """The fused two-level cycle against the same cycle composed of the public
    operators, smoothers and transfers (rounding: 1e-12 on quantities that a
    cycle amplifies by less than 100)."""
    M, torch = h1pa, torch_cuda
    s = _system(M, torch, 4, 3)
    mesh, fes = s["mesh"], s["fes"]
    mg = M.PMultigrid(s["a"], [1, 4], smoother_order=order, pre_smoothing=pre,
                      post_smoothing=post, cycle=cycle, coarse_rel_tol=1e-12, coarse_max_iter=500)
    lo = M.FiniteElementSpace(mesh, M.H1_FECollection(1, 3))
    al = M.BilinearForm(lo)
    al.SetAssemblyLevel(M.AssemblyLevel.PARTIAL)
    al.AddDomainIntegrator(M.DiffusionIntegrator(M.SinCosCoefficient()))
    al.Assemble()
    essl, essh = lo.GetBoundaryTrueDofs(), fes.GetBoundaryTrueDofs()
    Al = M.ConstrainedOperator(al, essl)
    T = M.TransferOperator(lo, fes)
    S = M.OperatorChebyshevSmoother(s["A"], None, essh, order)
    cg = M.CGSolver()
    cg.SetRelTol(1e-13)
    cg.SetMaxIter(2000)
    cg.SetOperator(Al)
    cg.SetPreconditioner(M.OperatorJacobiSmoother(al, essl))

    def apply(op, v, n):
        out = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
        (op.MultTranspose if op is T else op.Mult)(v, out)
        return out

    N, n = fes.GetNDofs(), lo.GetNDofs()
    x = s["b"]
    y = torch.zeros_like(x)
    for _ in range(pre):
        y = y + apply(S, x - apply(s["A"], y, N), N)
    r = apply(T, x - apply(s["A"], y, N), n)
    c = torch.empty_like(r)
    cg.Mult(r, c)
    up = torch.empty_like(x)
    T.Mult(c, up)
    y = y + up
    for _ in range(post):
        y = y + apply(S, x - apply(s["A"], y, N), N)
    got = torch.full_like(x, float("nan"))
    mg.Mult(x, got)
    # the coarse solves stop at 1e-12 and 1e-13 of their right-hand side
    assert float((got - y).norm() / y.norm()) < 1e-9
