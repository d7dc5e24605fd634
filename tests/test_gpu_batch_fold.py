"""GPU: the batch's merged element launch and folded scalar steps.

Bars: bitwise.  A solve's iterates depend neither on the replay length (FP64
mode; odd lengths leave an iteration unfolded) nor on whether a slot too large
for folding, or a single order (no merged launch), shares the batch.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(M, torch, p, n, seed):
    mesh = M.Mesh.MakeCartesian3D(n, n, n)
    mesh.Perturb(0.15, seed)
    fes = M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))
    a = M.BilinearForm(fes)
    a.SetAssemblyLevel(M.AssemblyLevel.PARTIAL)
    a.AddDomainIntegrator(M.DiffusionIntegrator(M.SinCosCoefficient()))
    a.Assemble()
    N = fes.GetNDofs()
    b = torch.from_numpy(np.random.default_rng(seed).uniform(-1, 1, N)).cuda()
    A, X, B = a.FormLinearSystem(fes.GetBoundaryTrueDofs(), torch.zeros_like(b), b)
    return mesh, fes, a, A, X, B


def _solve(M, probs, precision, K, rel=1e-10, graph=True, max_iter=10000):
    bs = M.BatchSolver(precision=precision, iters_per_replay=K, use_graph=graph)
    out = [q[4].clone().fill_(float("nan")) for q in probs]
    tags = [bs.Add(q[3], q[5], o, rel_tol=rel, max_iter=max_iter) for q, o in zip(probs, out)]
    bs.Run()
    res = dict(bs.Poll())
    return out, [res[t]["iterations"] for t in tags]


SMALL = [(1, 9), (2, 5), (3, 4), (4, 3), (5, 3), (6, 2), (7, 2), (8, 2)]


@pytest.mark.parametrize("max_iter", [10000, 7])
def test_replay_length_fp64(h1pa, torch_cuda, max_iter):
    M, torch = h1pa, torch_cuda
    probs = [_problem(M, torch, p, n, p) for p, n in SMALL]
    ref, its = _solve(M, probs, M.PREC_FP64, 1, max_iter=max_iter)
    for K in (2, 3, 8, 9):
        for graph in (True, False):
            got, i2 = _solve(M, probs, M.PREC_FP64, K, graph=graph, max_iter=max_iter)
            assert i2 == its, K
            assert all(torch.equal(a, b) for a, b in zip(got, ref)), K


@pytest.mark.parametrize("prec", ["PREC_FP64", "PREC_FP32", "PREC_BF16_PA"])
@pytest.mark.parametrize("K", [3, 8])
def test_alone_in_mix_and_beside_a_large_slot(h1pa, torch_cuda, prec, K):
    M, torch = h1pa, torch_cuda
    precision = getattr(M, prec)
    probs = [_problem(M, torch, p, n, p) for p, n in SMALL]
    alone = [_solve(M, [q], precision, K) for q in probs]  # one order: no merged launch
    got, its = _solve(M, probs, precision, K)
    assert its == [a[1][0] for a in alone]
    assert all(torch.equal(g, a[0][0]) for g, a in zip(got, alone))
    # 1.1M DOFs: more chunks than a folded sum takes; loose tolerance, few iterations
    big = _problem(M, torch, 3, 35, 5)
    bs = M.BatchSolver(precision=precision, iters_per_replay=K)
    out = [q[4].clone().fill_(float("nan")) for q in probs]
    xb = big[4].clone()
    bs.Add(big[3], big[5], xb, rel_tol=1e-10, tag=99)
    for i, (q, o) in enumerate(zip(probs, out)):
        bs.Add(q[3], q[5], o, rel_tol=1e-10, tag=i)
    while bs.Launch():
        bs.Wait()
        for t, r in bs.Poll():
            if t < 99:
                assert r["iterations"] == its[t]
    assert all(torch.equal(g, o) for g, o in zip(got, out))
