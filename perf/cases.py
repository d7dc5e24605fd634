"""The work that programs on this framework have it do, as cases to be timed.

Each case goes through the public entry points only: the applies of a
partially assembled operator, its set-up, the right-hand side, the
evaluation of fields at quadrature points, and the solvers.

`exact` recomputes a case in plain torch, 64 bits, with dense 1D contractions.
How the vectors are laid out -- which vertices an element has, which L-DOF an
element's node is, where the interior vertices of a perturbed mesh lie -- it
reads from the framework's tables and vertex list; every computed number is
its own.
"""
import math

import numpy as np
import torch

import mfem_amd as M

DEV = "cuda"

# The geometry factor of a curved mesh: x' = x + CURVE sin(2 pi y) sin(2 pi z) and cyclic.
CURVE = 0.05
# Vertex perturbation of the straight-sided meshes, in element widths.
PERTURB = 0.2


def listed():
    return [
        # The smallest problem that is solved in earnest (117,649 DOFs): every apply of a
        # Krylov or time loop on it is two short launches.
        dict(name="mult_p3_small", kind="mult", integ="diffusion", p=3, nx=16, ny=16, nz=16, q=0),
        # Low order on a ragged grid, where the quadrature data weigh most per DOF.
        dict(name="mult_p2_ragged", kind="mult", integ="diffusion", p=2, nx=61, ny=53, nz=47, q=0),
        # The benchmark's own apply: 31.9M DOFs at p = 4, the largest call.
        dict(name="mult_p4_large", kind="mult", integ="diffusion", p=4, nx=79, ny=79, nz=79, q=0),
        # High order, where the contractions cost as much as the data.
        dict(name="mult_p8_high", kind="mult", integ="diffusion", p=8, nx=31, ny=29, nz=27, q=0),
        # A mass operator (projection, explicit time stepping).
        dict(name="mass_p6", kind="mult", integ="mass", p=6, nx=27, ny=27, nz=27, q=0),
        # The reduced-precision apply of an inner solver: FP32 vectors, BF16 operator data.
        dict(name="mult_bf16_p6", kind="mult_lp", precision="bf16", p=6, nx=40, ny=40, nz=40),
        # New coefficient or new geometry on a curved mesh: operator data, Jacobi diagonal and
        # the first residual (what a nonlinear or moving-mesh program does each outer step).
        dict(name="assemble_p4_curved", kind="assemble", geom=4, p=4, nx=32, ny=32, nz=32),
        # The right-hand side of a source given at the quadrature points.
        dict(name="rhs_p5", kind="rhs", geom=1, p=5, nx=23, ny=23, nz=23),
        # A field's values and physical gradient at the quadrature points (post-processing,
        # nonlinear coefficients).
        dict(name="interpolate_p3", kind="interpolate", geom=1, p=3, nx=40, ny=39, nz=38, q=5, vdim=1),
        # A small FP64 Jacobi-PCG solve to 1e-12, whole.
        dict(name="pcg_p3_small", kind="pcg", p=3, nx=16, ny=16, nz=16, rel=1e-12),
        # A solve with CG preconditioned by p-multigrid (BF16 cycle) on a curved mesh.
        dict(name="multigrid_p6", kind="multigrid", p=6, nx=17, ny=17, nz=17, rel=1e-10),
        # Many small mixed-precision solves advanced together, as a server has them.
        dict(name="batch_small", kind="batch", count=24, nlo=4, nhi=10, plo=2, phi=6, rel=1e-10),
    ]


# Largest work of a drawn case: that of the largest listed one.
MOST_BYTES = 5.9e9
MOST_ELEMENTS = 500000


def _dofs(c):
    p = c["p"]
    return (c["nx"] * p + 1) * (c["ny"] * p + 1) * (c["nz"] * p + 1)


def _elements(c):
    return c["nx"] * c["ny"] * c["nz"]


def _grid(rng, p, lo, hi):
    """A ragged grid of about log-uniform DOF count in [lo, hi] at order p."""
    target = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    n = max(1.0, (target ** (1.0 / 3.0) - 1.0) / p)
    dims = [max(2, round(n * rng.uniform(0.85, 1.15))) for _ in range(3)]
    while dims[0] * dims[1] * dims[2] > MOST_ELEMENTS:
        dims = [max(2, d - 1) for d in dims]
    return dims


def draw(rng):
    kind = rng.choice(["mult", "mult", "mult", "mult", "mult_lp", "assemble", "rhs",
                       "interpolate", "pcg", "multigrid", "batch"])
    if kind == "batch":
        nlo = rng.randint(3, 6)
        plo = rng.randint(1, 4)
        return dict(kind=kind, count=rng.randint(4, 24), nlo=nlo, nhi=nlo + rng.randint(0, 4),
                    plo=plo, phi=min(6, plo + rng.randint(0, 4)), rel=1e-10)
    p = rng.randint(1, 8)
    c = dict(kind=kind, p=p)
    if kind == "mult":
        c["integ"] = rng.choice(["diffusion", "diffusion", "mass", "both"])
        c["q"] = rng.choice([0, 0, 0, p + 1])
        dims = _grid(rng, p, 1e3, 3.0e7)
    elif kind == "mult_lp":
        c["precision"] = rng.choice(["bf16", "fp32"])
        dims = _grid(rng, p, 1e4, 1.4e7)
    elif kind == "assemble":
        c["geom"] = rng.choice([1, p, 2])
        dims = _grid(rng, p, 1e4, 4e6)
    elif kind == "rhs":
        c["geom"] = rng.choice([1, p])
        dims = _grid(rng, p, 1e4, 2e6)
    elif kind == "interpolate":
        c["geom"] = rng.choice([1, p])
        c["q"] = rng.choice([q for q in (p + 1, p + 2, p + 3) if q <= 10])
        c["vdim"] = rng.choice([1, 3])
        dims = _grid(rng, p, 1e4, 2e6)
    elif kind == "pcg":
        c["rel"] = rng.choice([1e-8, 1e-10, 1e-12])
        dims = _grid(rng, p, 1e4, 4e5)
    else:
        c["p"] = p = rng.randint(2, 8)
        c["rel"] = rng.choice([1e-8, 1e-10])
        dims = _grid(rng, p, 5e4, 1.1e6)
    c["nx"], c["ny"], c["nz"] = dims
    while work(c)["bytes"] > MOST_BYTES:
        c["nx"], c["ny"], c["nz"] = (max(2, n - 1) for n in (c["nx"], c["ny"], c["nz"]))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(1000003 * (seed % 1000003) + salt)


def _uniform(n, g, lo=-1.0, hi=1.0):
    return torch.rand(n, dtype=torch.float64, device=DEV, generator=g) * (hi - lo) + lo


def _mesh(c, seed):
    mesh = M.Mesh.MakeCartesian3D(c["nx"], c["ny"], c["nz"])
    if c["kind"] == "multigrid":
        mesh.SetCurvature(c["p"], CURVE)
    elif c.get("geom", 1) > 1:
        mesh.SetCurvature(c["geom"], CURVE)
    else:
        mesh.Perturb(PERTURB, seed)
    return mesh


def _space(c, seed):
    mesh = _mesh(c, seed)
    return mesh, M.FiniteElementSpace(mesh, M.H1_FECollection(c["p"], 3))


def _log_uniform(ne, seed):
    """A coefficient of one value per element, log-uniform over four decades."""
    return torch.exp(_uniform(ne, _gen(seed, 7), math.log(1e-2), math.log(1e2)))


def _form(fes, integrators):
    a = M.BilinearForm(fes)
    a.SetAssemblyLevel(M.AssemblyLevel.PARTIAL)
    for i in integrators:
        a.AddDomainIntegrator(i)
    a.Assemble()
    return a


def _mult_integrators(c):
    k = M.SinCosCoefficient()
    q = c.get("q", 0)
    out = []
    if c.get("integ", "diffusion") in ("diffusion", "both"):
        out.append(M.DiffusionIntegrator(k, q))
    if c.get("integ") in ("mass", "both"):
        out.append(M.MassIntegrator(k, q))
    return out


def _batch_problems(c, seed):
    """Orders and sizes of the requests of a batch, the same for every seed."""
    rng = np.random.default_rng(c["count"])
    return [dict(kind="request", p=int(rng.integers(c["plo"], c["phi"] + 1)),
                 nx=int(n), ny=int(n), nz=int(n))
            for n in rng.integers(c["nlo"], c["nhi"] + 1, c["count"])]


def _orders(p):
    """Multigrid levels: the order halved (rounding up) down to 1."""
    o = [p]
    while o[-1] > 1:
        o.append((o[-1] + 1) // 2)
    return list(reversed(o))


def _system(a, fes, seed):
    """The constrained system of the boundary DOFs with a random right-hand side."""
    n = fes.GetNDofs()
    b = _uniform(n, _gen(seed, 11))
    ess = fes.GetBoundaryTrueDofs()
    A, X, B = a.FormLinearSystem(ess, torch.zeros(n, dtype=torch.float64, device=DEV), b)
    return A, X, B, ess


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "batch":
        problems = []
        for i, r in enumerate(_batch_problems(c, seed)):
            mesh, fes = _space(r, seed + i)
            a = _form(fes, [M.DiffusionIntegrator(M.SinCosCoefficient())])
            A, X, B, _ = _system(a, fes, seed + i)
            problems.append((mesh, fes, a, A, X, B))
        solver = M.BatchSolver(precision=M.PREC_BF16_PA)
        return dict(c=c, problems=problems, solver=solver)
    mesh, fes = _space(c, seed)
    n, ne = fes.GetNDofs(), fes.GetNE()
    s = dict(c=c, mesh=mesh, fes=fes)
    if kind in ("mult", "mult_lp"):
        s["a"] = _form(fes, _mult_integrators(c))
        s["x"] = _uniform(n, _gen(seed))
        if kind == "mult_lp":
            s["x"] = s["x"].float()
            s["prec"] = M.PREC_BF16_PA if c["precision"] == "bf16" else M.PREC_FP32
        s["y"] = torch.empty_like(s["x"])
        if kind == "mult_lp":  # the reduced-precision copy of the operator data is made once
            s["a"].MultLowPrecision(s["x"], s["y"], s["prec"])
    elif kind == "assemble":
        s["k"] = _log_uniform(ne, seed)
        s["a"] = _form(fes, [M.DiffusionIntegrator(M.PWConstCoefficient(s["k"]))])
        s["x"] = _uniform(n, _gen(seed))
        s["y"], s["diag"] = torch.empty_like(s["x"]), torch.empty_like(s["x"])
    elif kind == "rhs":
        f = _uniform((c["p"] + 1) ** 3 * ne, _gen(seed))
        s["lf"] = M.LinearForm(fes)
        s["lf"].AddDomainIntegrator(M.DomainLFIntegrator(M.QuadratureFunctionCoefficient(f)))
    elif kind == "interpolate":
        nq = c["q"] ** 3
        s["qi"] = fes.GetQuadratureInterpolator(c["q"], c["vdim"])
        s["xe"] = _uniform(fes.dof * c["vdim"] * ne, _gen(seed))
        s["val"] = torch.empty(nq * c["vdim"] * ne, dtype=torch.float64, device=DEV)
        s["der"] = torch.empty(nq * c["vdim"] * 3 * ne, dtype=torch.float64, device=DEV)
    else:
        if kind == "pcg":
            integ = [M.DiffusionIntegrator(M.SinCosCoefficient())]
        else:
            integ = [M.DiffusionIntegrator(M.PWConstCoefficient(_log_uniform(ne, seed)))]
            s["k"] = integ[0].coeff.data
        a = s["a"] = _form(fes, integ)
        A, X, B, ess = _system(a, fes, seed)
        s["X"], s["B"], s["cg"] = X, B, M.CGSolver()
        s["cg"].SetRelTol(c["rel"])
        s["cg"].SetMaxIter(5000)
        s["cg"].SetOperator(A)
        if kind == "pcg":
            s["cg"].SetPreconditioner(M.OperatorJacobiSmoother(a, ess))
        else:
            s["mg"] = M.PMultigrid(a, _orders(c["p"]), cycle_precision=M.PREC_BF16_PA,
                                   coarse_jacobi=True)
            s["cg"].SetPreconditioner(s["mg"])
    return s


def run(state):
    s, kind = state, state["c"]["kind"]
    if kind == "mult":
        s["a"].Mult(s["x"], s["y"])
        return s["y"]
    if kind == "mult_lp":
        s["a"].MultLowPrecision(s["x"], s["y"], s["prec"])
        return s["y"]
    if kind == "assemble":
        s["a"].Assemble()
        s["a"].AssembleDiagonal(s["diag"])
        s["a"].Mult(s["x"], s["y"])
        return s["diag"], s["y"]
    if kind == "rhs":
        return s["lf"].Assemble()
    if kind == "interpolate":
        qi = s["qi"]
        qi.Mult(s["xe"], qi.VALUES | qi.PHYSICAL_DERIVATIVES, s["val"], s["der"], None)
        return s["val"], s["der"]
    if kind == "batch":
        for mesh, fes, a, A, X, B in s["problems"]:
            s["solver"].Add(A, B, X, rel_tol=s["c"]["rel"])
        s["solver"].Run()
        s["solver"].Poll()
        return [q[4] for q in s["problems"]]
    s["cg"].Mult(s["B"], s["X"])
    return s["X"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _apply_flops(c, D, Q, diff, mass):
    """Multiply-adds (as 2) of the sum-factorized applies, there and back."""
    f = 0
    if diff:
        f += 10 * D ** 3 * Q + 12 * D ** 2 * Q ** 2 + 12 * D * Q ** 3 + 15 * Q ** 3
    if mass:
        f += 4 * (D ** 3 * Q + D ** 2 * Q ** 2 + D * Q ** 3) + Q ** 3
    return f * _elements(c)


def _apply_bytes(c, diff, mass, value=8, data=8, q=0):
    """Operator data and the element-to-DOF map once, both vectors once."""
    Q, D = q or c["p"] + 2, c["p"] + 1
    per = data * Q ** 3 * ((6 if diff else 0) + (1 if mass else 0)) + 4 * D ** 3
    return _elements(c) * per + 2 * value * _dofs(c)


def work(case):
    c, kind = case, case["kind"]
    if kind == "batch":
        # every request's system read once and its solution written: the iterations a method
        # takes are not work that the path cannot do without
        parts = [work(dict(r, kind="pcg")) for r in _batch_problems(c, 0)]
        return {k: sum(w[k] for w in parts) for k in ("bytes", "flops")}
    p, ne, n = c["p"], _elements(c), _dofs(c)
    D, Q = p + 1, c.get("q", 0) or p + 2
    if kind == "mult":
        diff, mass = c["integ"] != "mass", c["integ"] != "diffusion"
        return dict(bytes=_apply_bytes(c, diff, mass, q=Q), flops=_apply_flops(c, D, Q, diff, mass))
    if kind == "mult_lp":
        data = 2 if c["precision"] == "bf16" else 4
        return dict(bytes=_apply_bytes(c, True, False, 4, data), flops=_apply_flops(c, D, Q, True, False))
    if kind in ("pcg", "multigrid"):
        # one apply's data, the right-hand side and the solution
        return dict(bytes=_apply_bytes(c, True, False), flops=_apply_flops(c, D, Q, True, False))
    Dg = c.get("geom", 1) + 1
    nodes = 24 * Dg ** 3 * ne
    geometry = 2 * 9 * (Dg ** 3 * Q + Dg ** 2 * Q ** 2 + Dg * Q ** 3) * ne
    if kind == "assemble":
        # nodes in, operator data out and in again for the diagonal and the apply
        data = 48 * Q ** 3 * ne
        return dict(bytes=nodes + 8 * ne + 3 * data + 8 * D ** 3 * ne + 3 * 8 * n,
                    flops=geometry + 60 * Q ** 3 * ne + 2 * _apply_flops(c, D, Q, True, False))
    if kind == "rhs":
        Q = D
        return dict(bytes=nodes + 8 * Q ** 3 * ne + 4 * D ** 3 * ne + 8 * n,
                    flops=geometry + 2 * (Q ** 3 * D + Q ** 2 * D ** 2 + Q * D ** 3) * ne)
    return dict(bytes=nodes + 8 * c["vdim"] * ne * (D ** 3 + 4 * Q ** 3),
                flops=geometry + c["vdim"] * ne * 2 * (2 * D ** 3 * Q + 3 * D ** 2 * Q ** 2 + 4 * D * Q ** 3 + 10 * Q ** 3))


def tolerance(case):
    kind = case["kind"]
    # Each is about four times the largest distance seen between the framework and `exact`
    # over the listed and some drawn cases.
    if kind == "mult":
        return {"rel": 2e-14, "max": 4e-13}
    if kind == "mult_lp":  # FP32 sums; the stored BF16 data are the same on both sides
        return {"rel": 5e-7, "max": 1e-5}
    if kind in ("assemble", "rhs", "interpolate"):
        return {"rel": 1.5e-13, "max": 4e-12}
    # Whole solves stop at their own tolerance: an iteration more or less, as another order of
    # a sum gives, changes the result by about the distance to the solution.
    return {"rel": 100 * case["rel"]}


# ---------------------------------------------------------------------------
# the same in plain torch
# ---------------------------------------------------------------------------
def _gauss_legendre(n):
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (x + 1.0), 0.5 * w


def _gauss_lobatto(p):
    """The p + 1 Gauss-Lobatto points on [0, 1]: ends and roots of P_p'."""
    P = np.polynomial.legendre.Legendre.basis(p)
    d1, d2 = P.deriv(), P.deriv(2)
    r = np.sort(d1.roots().real) if p > 1 else np.zeros(0)
    for _ in range(3):
        r = r - d1(r) / d2(r) if p > 1 else r
    return 0.5 * (np.concatenate([[-1.0], r, [1.0]]) + 1.0)


def _lagrange(nodes, x):
    """B[q, d], G[q, d]: the Lagrange basis on `nodes` and its derivative at x (long double)."""
    t, x = nodes.astype(np.longdouble), np.asarray(x, np.longdouble)
    D = len(t)
    B, G = np.ones((len(x), D), np.longdouble), np.zeros((len(x), D), np.longdouble)
    for d in range(D):
        for k in range(D):
            if k != d:
                B[:, d] *= (x - t[k]) / (t[d] - t[k])
        for m in range(D):
            if m == d:
                continue
            g = np.full(len(x), 1 / (t[d] - t[m]), np.longdouble)
            for k in range(D):
                if k not in (d, m):
                    g *= (x - t[k]) / (t[d] - t[k])
            G[:, d] += g
    to = lambda a: torch.tensor(a.astype(np.float64), device=DEV)  # noqa: E731
    return to(B), to(G)


def _contract(u, z, y, x):
    """out[e, a, b, c] = sum z[a, k] y[b, j] x[c, i] u[e, k, j, i]"""
    u = torch.tensordot(u, x, ([3], [1]))            # e k j c
    u = torch.tensordot(u, y, ([2], [1]))            # e k c b
    u = torch.tensordot(u, z, ([1], [1]))            # e c b a
    return u.permute(0, 3, 2, 1)


class _Exact:
    """Geometry, operator data and maps of one case, element by element."""

    def __init__(self, c, seed, Q, k=None, mesh_fes=None):
        self.mesh, self.fes = mesh_fes or _space(c, seed)
        p, ne = c["p"], self.fes.GetNE()
        self.p, self.D, self.Q, self.ne, self.n = p, p + 1, Q, ne, self.fes.GetNDofs()
        self.gmap = self.fes.GetElementRestriction().GatherMap().long().view(ne, -1)
        v = torch.tensor(self.mesh.GetVertices(), device=DEV)
        ev = torch.tensor(self.mesh.Topology()["ev"].astype(np.int64), device=DEV)
        corners = v[ev[:, [0, 1, 3, 2, 4, 5, 7, 6]]].view(ne, 2, 2, 2, 3)  # e z y x comp
        g = c["p"] if c["kind"] == "multigrid" else c.get("geom", 1)
        if g > 1:
            s = _gauss_lobatto(g)
            N = torch.tensor(np.stack([1 - s, s], 1), device=DEV)
            P = [_contract(corners[..., i], N, N, N) for i in range(3)]
            tp = 2 * math.pi
            P = [P[i] + CURVE * torch.sin(tp * P[(i + 1) % 3]) * torch.sin(tp * P[(i + 2) % 3])
                 for i in range(3)]
            self.nodes = torch.stack(P, -1)
        else:
            self.nodes = corners
        xq, wq = _gauss_legendre(Q)
        self.B, self.G = _lagrange(_gauss_lobatto(p), xq)
        self.gB, self.gG = _lagrange(_gauss_lobatto(g), xq)
        w = torch.tensor(wq, device=DEV)
        self.W = w[:, None, None] * w[None, :, None] * w[None, None, :]
        self.k = k
        per = 40 * Q ** 3 * 8
        step = max(1, int(3e9 / per))
        self.chunks = [slice(i, min(ne, i + step)) for i in range(0, ne, step)]

    def jacobian(self, sl):
        X, B, G = self.nodes[sl], self.gB, self.gG
        J = [[_contract(X[..., r], *(G if d == c else B for d in (2, 1, 0))) for c in range(3)]
             for r in range(3)]
        det = (J[0][0] * (J[1][1] * J[2][2] - J[2][1] * J[1][2])
               - J[1][0] * (J[0][1] * J[2][2] - J[2][1] * J[0][2])
               + J[2][0] * (J[0][1] * J[1][2] - J[1][1] * J[0][2]))
        return J, det

    def adjugate(self, J):
        """adj[c][r] with J^-1 = adj / det."""
        m = lambda i, j, k, l: J[i][j] * J[k][l]  # noqa: E731
        return [[m(1, 1, 2, 2) - m(1, 2, 2, 1), m(0, 2, 2, 1) - m(0, 1, 2, 2), m(0, 1, 1, 2) - m(0, 2, 1, 1)],
                [m(1, 2, 2, 0) - m(1, 0, 2, 2), m(0, 0, 2, 2) - m(0, 2, 2, 0), m(0, 2, 1, 0) - m(0, 0, 1, 2)],
                [m(1, 0, 2, 1) - m(1, 1, 2, 0), m(0, 1, 2, 0) - m(0, 0, 2, 1), m(0, 0, 1, 1) - m(0, 1, 1, 0)]]

    def coefficient(self, sl):
        if self.k is not None:
            return self.k[sl].view(-1, 1, 1, 1)
        B = self.gB
        x, y, z = (_contract(self.nodes[sl][..., i], B, B, B) for i in range(3))
        tp = 2 * math.pi
        return 1 + 0.5 * torch.sin(tp * x) * torch.cos(tp * y) * torch.sin(tp * z)

    def data(self, sl, diff=True, mass=False):
        """Diffusion data (c, d) as the upper triangle, mass data."""
        J, det = self.jacobian(sl)
        wk = self.W * self.coefficient(sl)
        D = None
        if diff:
            A = self.adjugate(J)
            s = wk / det
            D = {(i, j): s * sum(A[i][r] * A[j][r] for r in range(3)) for i in range(3) for j in range(i, 3)}
        return D, (wk * det if mass else None)

    def element_mult(self, u, D, m):
        B, G = self.B, self.G
        y = 0
        if D is not None:
            g = [_contract(u, *(G if d == c else B for d in (2, 1, 0))) for c in range(3)]
            for i in range(3):
                h = sum(D[min(i, j), max(i, j)] * g[j] for j in range(3))
                y = y + _contract(h, *((G if d == i else B).t() for d in (2, 1, 0)))
        if m is not None:
            y = y + _contract(m * _contract(u, B, B, B), B.t(), B.t(), B.t())
        return y

    def mult(self, x, diff=True, mass=False, kept=None):
        y = torch.zeros(self.n, dtype=torch.float64, device=DEV)
        for i, sl in enumerate(self.chunks):
            D, m = kept[i] if kept else self.data(sl, diff, mass)
            u = x[self.gmap[sl]].view(-1, self.D, self.D, self.D)
            y.index_add_(0, self.gmap[sl].reshape(-1), self.element_mult(u, D, m).reshape(-1))
        return y

    def diagonal(self, kept=None):
        y = torch.zeros(self.n, dtype=torch.float64, device=DEV)
        B, G = self.B, self.G
        pair = {(0, 0): B * B, (1, 1): G * G, (0, 1): B * G}
        for n, sl in enumerate(self.chunks):
            D = (kept[n] if kept else self.data(sl))[0]
            e = 0
            for (i, j), v in D.items():
                t = []
                for d in (2, 1, 0):
                    t.append(pair[tuple(sorted((int(i == d), int(j == d))))].t())
                e = e + (1 if i == j else 2) * _contract(v, *t)
            y.index_add_(0, self.gmap[sl].reshape(-1), e.reshape(-1))
        return y

    def solve(self, b):
        """The system constrained on the boundary, by Jacobi-PCG as far as it goes."""
        free = torch.ones(self.n, dtype=torch.float64, device=DEV)
        free[self.fes.GetBoundaryTrueDofs().long()] = 0
        kept = [self.data(sl) for sl in self.chunks]
        dinv = free / self.diagonal(kept)
        x, r = torch.zeros_like(b), b * free
        z = dinv * r
        d, nom = z.clone(), torch.dot(r, z)
        first = nom.item()
        for it in range(20000):
            q = self.mult(d, kept=kept) * free
            alpha = nom / torch.dot(d, q)
            x += alpha * d
            r -= alpha * q
            z = dinv * r
            new = torch.dot(r, z)
            d = z + (new / nom) * d
            nom = new
            if it % 20 == 19 and nom.item() < 1e-30 * first:
                break
        return x


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "batch":
        out = []
        for i, r in enumerate(_batch_problems(c, seed)):
            E = _Exact(r, seed + i, r["p"] + 2)
            out.append(E.solve(_uniform(E.n, _gen(seed + i, 11))))
        return out
    Q = c.get("q", 0) or c["p"] + 2
    if kind == "rhs":
        E = _Exact(c, seed, c["p"] + 1)
        f = _uniform((c["p"] + 1) ** 3 * E.ne, _gen(seed)).view(E.ne, E.Q, E.Q, E.Q)
        b = torch.zeros(E.n, dtype=torch.float64, device=DEV)
        for sl in E.chunks:
            v = E.W * E.jacobian(sl)[1] * f[sl]
            b.index_add_(0, E.gmap[sl].reshape(-1), _contract(v, E.B.t(), E.B.t(), E.B.t()).reshape(-1))
        return b
    if kind == "interpolate":
        E = _Exact(c, seed, Q)
        D, vd, nq = E.D, c["vdim"], Q ** 3
        xe = _uniform(D ** 3 * vd * E.ne, _gen(seed)).view(E.ne, vd, D, D, D)
        val, der = [], []
        for sl in E.chunks:
            J, det = E.jacobian(sl)
            A = E.adjugate(J)
            for_val, for_der = [], [[None] * vd for _ in range(3)]
            for k in range(vd):
                for_val.append(_contract(xe[sl, k], E.B, E.B, E.B))
                g = [_contract(xe[sl, k], *(E.G if d == i else E.B for d in (2, 1, 0))) for i in range(3)]
                for r in range(3):
                    for_der[r][k] = sum(A[i][r] * g[i] for i in range(3)) / det
            val.append(torch.stack(for_val, 1).reshape(-1, vd * nq))
            der.append(torch.stack([torch.stack(x, 1) for x in for_der], 1).reshape(-1, 3 * vd * nq))
        return torch.cat(val).reshape(-1), torch.cat(der).reshape(-1)
    if kind == "mult":
        E = _Exact(c, seed, Q)
        return E.mult(_uniform(E.n, _gen(seed)), c["integ"] != "mass", c["integ"] != "diffusion")
    if kind == "mult_lp":
        # the operator that is stored: the data rounded once to what the precision keeps
        E = _Exact(c, seed, Q)
        x = _uniform(E.n, _gen(seed)).float().double()
        low = torch.bfloat16 if c["precision"] == "bf16" else torch.float32
        y = torch.zeros(E.n, dtype=torch.float64, device=DEV)
        for sl in E.chunks:
            D, _ = E.data(sl)
            D = {ij: v.float().to(low).double() for ij, v in D.items()}
            u = x[E.gmap[sl]].view(-1, E.D, E.D, E.D)
            y.index_add_(0, E.gmap[sl].reshape(-1), E.element_mult(u, D, None).reshape(-1))
        return y
    if kind == "assemble":
        E = _Exact(c, seed, Q, k=_log_uniform(_elements(c), seed))
        kept = [E.data(sl) for sl in E.chunks]
        return E.diagonal(kept), E.mult(_uniform(E.n, _gen(seed)), kept=kept)
    k = _log_uniform(_elements(c), seed) if kind == "multigrid" else None
    E = _Exact(c, seed, Q, k=k)
    return E.solve(_uniform(E.n, _gen(seed, 11)))
