"""GPU: the sum-factorized element geometry against the oracle's, at every
node order (1..8) and number of points (1..10), so at every kernel that is
chosen by them, with element counts that leave the last block partly filled.

Bar: 1e-13 relative (2-norm).  A Jacobian entry is three nested sums of at most
nine products with table entries of size at most ~50 (the derivative row of
order 8), each rounded to 2^-53 of its partial sums: below 27 * 2^-53 * 30 on
the entries of a mesh whose nodes move by a few percent of h, 9e-14 at worst
and far less in the mean that the 2-norm takes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-13


def _rel(a, b):
    return np.linalg.norm(np.ravel(a) - np.ravel(b)) / np.linalg.norm(b)


def _nodes(orc, M, torch, dims, g, seed):
    """A mesh with order-g nodes given by the caller, moved at random by 0.05 h."""
    mesh = M.Mesh.MakeCartesian3D(*dims)
    om = orc.CartesianMesh(*dims)
    X = om.nodes_curved(om.vertices(), g, 0.0).copy()
    X += np.random.default_rng(seed).uniform(-0.05, 0.05, X.size).reshape(X.shape) / (max(dims) * g * g)
    mesh.SetNodes(g, torch.from_numpy(np.ravel(X).copy()).cuda())
    return mesh, X


@pytest.mark.parametrize("g", range(1, 9))
@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 4, 3)])
def test_geometric_factors_every_order(orc, h1pa, torch_cuda, g, dims):
    mesh, X = _nodes(orc, h1pa, torch_cuda, dims, g, g)
    ne = int(np.prod(dims))
    for q in range(1, 11):
        J, P = orc.geom(ne, g, q, X)
        Xq, Jq, dJ = (t.cpu().numpy() for t in mesh.GetGeometricFactors(q))
        assert _rel(Xq, P) < RTOL and _rel(Jq, J) < RTOL, (g, q)
        Jr = np.asarray(J).reshape(ne, 3, 3, -1)
        assert _rel(dJ, np.linalg.det(Jr.transpose(0, 3, 2, 1))) < RTOL, (g, q)


@pytest.mark.parametrize("p", range(1, 9))
@pytest.mark.parametrize("g", range(1, 9))
def test_pa_data_every_order(orc, h1pa, torch_cuda, p, g):
    M, dims = h1pa, (5, 3, 3)
    mesh, X = _nodes(orc, M, torch_cuda, dims, g, 10 * p + g)
    ne = int(np.prod(dims))
    fes = M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))
    kv = np.random.default_rng(p).uniform(0.5, 2.0, ne)
    for q in (p + 1, p + 2):
        J, P = orc.geom(ne, g, q, X)
        W = orc.tensor_weights(q)
        for coeff, k in ((M.SinCosCoefficient(), orc.coeff_sincos(q, ne, P)),
                         (M.PWConstCoefficient(torch_cuda.from_numpy(kv).cuda()),
                          np.repeat(kv, q ** 3))):
            a = M.BilinearForm(fes)
            a.SetAssemblyLevel(M.AssemblyLevel.PARTIAL)
            a.AddDomainIntegrator(M.DiffusionIntegrator(coeff, q))
            a.AddDomainIntegrator(M.MassIntegrator(coeff, q))
            a.Assemble()
            a.Assemble()  # in place, into the same buffers
            dd, dm = a.PAData()
            assert _rel(dd.cpu().numpy(), orc.diffusion_setup(q, ne, W, J, k)) < RTOL
            assert _rel(dm.cpu().numpy(), orc.mass_setup(q, ne, W, J, k)) < RTOL


@pytest.mark.parametrize("p", range(1, 9))
@pytest.mark.parametrize("g", [1, 2, 3, 4, 5, 6, 7, 8])
def test_domain_rhs_every_order(orc, h1pa, torch_cuda, p, g):
    """b = sum over elements and points of w det J f B: sums of positive weights
    against basis values below 1 in size, so the same bar holds."""
    M, dims = h1pa, (5, 3, 3)
    mesh, X = _nodes(orc, M, torch_cuda, dims, g, 100 * p + g)
    ne = int(np.prod(dims))
    fes = M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))
    gmap = fes.GetElementRestriction().GatherMap().cpu().numpy()
    fq = np.random.default_rng(p).uniform(-1, 1, (p + 1) ** 3 * ne)
    for coeff, kw in ((M.ConstantCoefficient(1.5), dict(f=1.5)),
                      (M.QuadratureFunctionCoefficient(torch_cuda.from_numpy(fq).cuda()),
                       dict(fq=fq))):
        lf = M.LinearForm(fes)
        lf.AddDomainIntegrator(M.DomainLFIntegrator(coeff))
        ref = np.zeros(fes.GetNDofs())
        np.add.at(ref, gmap, np.ravel(orc.domain_lf(p, ne, g, X, **kw)))
        assert _rel(lf.Assemble().cpu().numpy(), ref) < RTOL


@pytest.mark.parametrize("p", range(1, 9))
@pytest.mark.parametrize("g", [1, 0])
def test_physical_derivatives_every_rule(orc, h1pa, torch_cuda, p, g):
    """Straight-sided (the Jacobian is formed with the field) and isoparametric
    meshes, at every rule and both layouts.  The gradient multiplies by J^-T, of
    condition number below 4 on these meshes: the bar of the factors times 4."""
    M, dims, g = h1pa, (5, 3, 3), g or p
    mesh, X = _nodes(orc, M, torch_cuda, dims, g, 1000 * p + g)
    ne = int(np.prod(dims))
    fes = M.FiniteElementSpace(mesh, M.H1_FECollection(p, 3))
    flags = M.QI_VALUES | M.QI_PHYSICAL_DERIVATIVES
    for q in range(p + 1, min(p + 3, 10) + 1):
        J, _ = orc.geom(ne, g, q, X)
        for vdim in (1, 3):
            xE = np.random.default_rng(q).uniform(-1, 1, (p + 1) ** 3 * vdim * ne)
            for layout in (0, 1):
                qi = fes.GetQuadratureInterpolator(q, vdim)
                qi.SetOutputLayout(layout)
                val = torch_cuda.full((q ** 3 * vdim * ne,), np.nan, dtype=torch_cuda.float64,
                                      device="cuda")
                der = torch_cuda.full((3 * val.numel(),), np.nan, dtype=torch_cuda.float64,
                                      device="cuda")
                qi.Mult(torch_cuda.from_numpy(xE).cuda(), flags, val, der, None)
                ref = orc.qinterp(p, q, vdim, ne, xE, flags, by_vdim=bool(layout), J=J)
                assert _rel(val.cpu().numpy(), np.ravel(ref[0])) < RTOL
                assert _rel(der.cpu().numpy(), np.ravel(ref[1])) < 4 * RTOL
