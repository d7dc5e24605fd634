"""GPU: the E -> L row table of the fused operators.

On structured meshes Mult (native E-vector, row table) must equal the
composition R^T A_E R of the public pieces (lexicographic E-vector, CSR table)
bit for bit: the same element arithmetic, the same order of every row's sum.
Sizes cross the rules on rows per thread.  Star meshes (S hexahedra around an
edge) have rows wider than the table's for S >= 5, which the CSR table serves:
every consumer of the rows against the oracle.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-13


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def _form(M, fes, coeff=None):
    a = M.BilinearForm(fes)
    a.SetAssemblyLevel(M.AssemblyLevel.PARTIAL)
    a.AddDomainIntegrator(M.DiffusionIntegrator(coeff or M.SinCosCoefficient()))
    a.Assemble()
    return a


@pytest.mark.parametrize("p,dims", [(1, (1, 1, 1)), (1, (9, 7, 5)), (2, (1, 1, 1)), (2, (5, 4, 3)),
                                    (3, (16, 15, 14)), (4, (9, 8, 7)), (4, (20, 19, 18)),
                                    (5, (3, 2, 2)), (6, (5, 5, 4)), (7, (4, 3, 3)), (8, (3, 3, 2)),
                                    (2, (62, 62, 62)), (2, (96, 96, 96))])
def test_mult_is_the_composition_bitwise(h1pa, torch_cuda, p, dims):
    M, torch = h1pa, torch_cuda
    mesh = M.Mesh.MakeCartesian3D(*dims)
    mesh.Perturb(0.2, p)
    fes = M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))
    a = _form(M, fes)
    R = fes.GetElementRestriction()
    g = torch.Generator(device="cuda").manual_seed(p)
    x = torch.rand(fes.GetNDofs(), dtype=torch.float64, device="cuda", generator=g) * 2 - 1
    y = torch.full_like(x, float("nan"))
    a.Mult(x, y)
    xe = torch.empty(fes.ne * fes.dof, dtype=torch.float64, device="cuda")
    ye = torch.zeros_like(xe)
    R.Mult(x, xe)
    a.AddMultPA_E(xe, ye)
    z = torch.empty_like(x)
    R.MultTranspose(ye, z)
    assert torch.equal(y, z)


def _star(S, layers):
    """S prisms of one quadrilateral each around a central edge, extruded."""
    t = np.linspace(0, 2 * np.pi, 2 * S, endpoint=False)
    ring = np.stack([np.cos(t), np.sin(t)], 1) * np.where(np.arange(2 * S) % 2, 1.3, 1.0)[:, None]
    flat = np.concatenate([[[0.0, 0.0]], ring])
    nf = len(flat)
    xyz = np.concatenate([np.column_stack([flat, np.full(nf, z)]) for z in range(layers + 1)])
    quads = [(0, 1 + 2 * s, 2 + 2 * s, 1 + (2 * s + 2) % (2 * S)) for s in range(S)]
    ev, bq = [], []
    for l in range(layers):
        for q in quads:
            ev.append([v + l * nf for v in q] + [v + (l + 1) * nf for v in q])
        for k in range(2 * S):
            i, j = 1 + k, 1 + (k + 1) % (2 * S)
            bq.append([i + l * nf, j + l * nf, j + (l + 1) * nf, i + (l + 1) * nf])
    for q in quads:
        bq.append([v for v in q[::-1]])
        bq.append([v + layers * nf for v in q])
    return np.array(ev, np.int32), np.array(bq, np.int32), xyz


@pytest.mark.parametrize("S", [3, 5, 7])
@pytest.mark.parametrize("p", [1, 2, 4, 7])
def test_wide_rows(orc, h1pa, torch_cuda, S, p):
    M, torch = h1pa, torch_cuda
    ev, bq, xyz = _star(S, 3)
    mesh = M.Mesh.FromArrays(xyz, ev, bq)
    fes = M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))
    P = orc.Problem(None, p, mesh_arrays=(ev, bq, xyz), coeff="sincos")
    assert np.array_equal(fes.GetElementRestriction().Offsets().cpu().numpy(), P.offsets)
    if S >= 5:
        assert np.diff(P.offsets).max() > 8
    a = _form(M, fes)
    n = P.ndofs
    x = np.random.default_rng(S + p).uniform(-1, 1, n)
    xd = torch.from_numpy(x).cuda()
    y = torch.full_like(xd, float("nan"))
    a.Mult(xd, y)
    assert _rel(y.cpu().numpy(), P.mult(x)) < RTOL
    a.AssembleDiagonal(y)
    assert _rel(y.cpu().numpy(), P.diagonal()) < RTOL
    lf = M.LinearForm(fes)
    lf.AddDomainIntegrator(M.DomainLFIntegrator(M.ConstantCoefficient(1.0)))
    assert _rel(lf.Assemble().cpu().numpy(), P.rhs(1.0)) < RTOL
    x32, y32 = xd.float(), torch.full((n,), float("nan"), dtype=torch.float32, device="cuda")
    a.MultLowPrecision(x32, y32, M.PREC_FP32)
    # FP32 data, vectors and sums of 6 contractions of (p + 2) terms
    assert _rel(y32.cpu().numpy().astype(float), P.mult(x32.cpu().numpy().astype(float))) < 2e-5
    # boundary DOFs (interior rows written directly), then a list that holds
    # interior DOFs too (they go through the E-vector)
    some = np.unique(np.concatenate([P.ess[::2], np.arange(n - 1, 0, -3)])).astype(np.int32)
    for ess in (P.ess, some):
        P.set_ess(ess)
        e = torch.from_numpy(np.ascontiguousarray(ess)).cuda()
        if ess is not some:
            e = fes.GetBoundaryTrueDofs()
        A, X, B = a.FormLinearSystem(e, torch.zeros_like(xd), xd)
        A.Mult(xd, y)
        assert _rel(y.cpu().numpy(), P.constrained_mult(x)) < RTOL
        cg = M.CGSolver()
        cg.SetRelTol(1e-12)
        cg.SetMaxIter(2000)
        cg.SetOperator(A)
        cg.SetPreconditioner(M.OperatorJacobiSmoother(a, e))
        cg.Mult(B, X)
        A.Mult(X, y)
        # CG stops on the preconditioned residual, 1e-12 of the first
        assert cg.GetConverged() and _rel(y.cpu().numpy(), B.cpu().numpy()) < 1e-9
        ir, X2 = M.IRSolver(M.PREC_BF16_PA), X.clone()
        ir.SetRelTol(1e-10)
        ir.SetOperator(A)
        ir.Mult(B, X2)
        bs = M.BatchSolver(precision=M.PREC_BF16_PA, use_graph=False)
        X3 = X.clone()
        bs.Add(A, B, X3, rel_tol=1e-10)
        bs.Run()
        bs.Poll()
        for Z in (X2, X3):
            assert _rel(Z.cpu().numpy(), X.cpu().numpy()) < 1e-7
    ch = M.OperatorChebyshevSmoother(A, None, e, 2)
    ch.Mult(xd, y)
    assert bool(torch.isfinite(y).all())
    assert _rel(y.cpu().numpy(), P.chebyshev_mult(ch.GetCoefficients(), x)) < 1e-11
