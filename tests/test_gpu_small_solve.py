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


# What two cycles that stop their coarse solves at t and t' may differ by: CG stops
# on |r| <= t |b| in the norm of D^-1, so its error is at most t sqrt(k) of the
# solution in the energy norm, k the condition number of D^-1 A; below 10 on the
# coarse systems here (8 and 27 free DOFs, coefficient 0.5 to 1.5), and as much again
# from the energy norm to the 2-norm: 10 (t + t') = 1.1e-11 a coarse solve.  A
# correction is at most a few times the cycle's result, and a W cycle of three
# levels adds two: 1e-10.  Rounding is far below (1e-15 amplified by less than 100).
CYCLE_BAR = 1e-10


def _level(M, mesh, p):
    fes = M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))
    a = M.BilinearForm(fes)
    a.SetAssemblyLevel(M.AssemblyLevel.PARTIAL)
    a.AddDomainIntegrator(M.DiffusionIntegrator(M.SinCosCoefficient()))
    a.Assemble()
    ess = fes.GetBoundaryTrueDofs()
    return dict(fes=fes, a=a, ess=ess, n=fes.GetNDofs(), A=M.ConstrainedOperator(a, ess))


class _Cycle:
    """MultigridBase::Cycle from the public operators, smoothers and transfers."""

    def __init__(self, M, torch, mesh, orders, order, pre, post, w):
        self.torch, self.pre, self.post, self.w = torch, pre, post, w
        self.lv = [_level(M, mesh, p) for p in orders]
        for L in self.lv[1:]:
            L["S"] = M.OperatorChebyshevSmoother(L["A"], None, L["ess"], order)
        self.T = [M.TransferOperator(a["fes"], b["fes"]) for a, b in zip(self.lv, self.lv[1:])]
        cg = self.cg = M.CGSolver()
        cg.SetRelTol(1e-13)
        cg.SetMaxIter(2000)
        cg.SetOperator(self.lv[0]["A"])
        cg.SetPreconditioner(M.OperatorJacobiSmoother(self.lv[0]["a"], self.lv[0]["ess"]))

    def _to(self, f, v, n):
        out = self.torch.full((n,), float("nan"), dtype=self.torch.float64, device="cuda")
        f(v, out)
        return out

    def __call__(self, l, x, y):
        L = self.lv[l]
        if l == 0:
            return self._to(self.cg.Mult, x, L["n"])
        A, S, n = L["A"], L.get("S"), L["n"]
        for _ in range(self.pre):
            y = y + self._to(S.Mult, x - self._to(A.Mult, y, n), n)
        T, nc = self.T[l - 1], self.lv[l - 1]["n"]
        r = self._to(T.MultTranspose, x - self._to(A.Mult, y, n), nc)
        c = self(l - 1, r, self.torch.zeros_like(r))
        if self.w:
            c = self(l - 1, r, c)
        y = y + self._to(T.Mult, c, n)
        for _ in range(self.post):
            y = y + self._to(S.Mult, x - self._to(A.Mult, y, n), n)
        return y


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("pre,post,cycle", [(1, 1, "V"), (2, 2, "V"), (0, 1, "V"), (1, 0, "V"),
                                            (1, 1, "W"), (0, 2, "W")])
@pytest.mark.parametrize("orders,n", [([1, 4], 3), ([1, 2, 4], 3), ([1, 3, 7], 4)])
def test_cycle_is_its_public_pieces(h1pa, torch_cuda, order, pre, post, cycle, orders, n):
    """The fused cycle against the same one composed of the public operators,
    smoothers and transfers; with a level between, whose iterate starts from zero
    without being filled where the first smoothing writes it whole."""
    M, torch = h1pa, torch_cuda
    s = _system(M, torch, orders[-1], n)
    mg = M.PMultigrid(s["a"], orders, smoother_order=order, pre_smoothing=pre,
                      post_smoothing=post, cycle=cycle, coarse_rel_tol=1e-12, coarse_max_iter=500)
    ref = _Cycle(M, torch, s["mesh"], orders, order, pre, post, cycle == "W")
    x = s["b"]
    y = ref(len(orders) - 1, x, torch.zeros_like(x))
    for _ in range(2):  # the second one finds the levels' vectors as the first left them
        got = torch.full_like(x, float("nan"))
        mg.Mult(x, got)
        err = float((got - y).norm() / y.norm())
        print(f"[case] {orders} order={order} {pre},{post},{cycle}: {err:.1e}", flush=True)
        assert err < CYCLE_BAR
