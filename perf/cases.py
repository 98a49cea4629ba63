"""Performance cases of the spectral-element operator path.

Each case is one call, or one short sequence of calls, that a program built on
``geoflow_amd`` makes: explicit Burgers steps, Helmholtz solves, sphere
advection, an ensemble step, a gradient through the adjoint, and the operators
called one at a time by a program with a time stepper of its own.  Sizes are
those of the benchmark and of the tests, and ragged ones between them.

``exact`` restates the box cases in plain torch FP64 (nodes and weights from
numpy's Legendre routines, assembly on the box's node lattice); the linear
solves are done directly by fast diagonalisation, the adjoint by autograd.
Sphere and terrain cases have no such restatement.
"""
import functools
import math

import numpy as np
import torch

import geoflow_amd as ga
from geoflow_amd import workloads
from geoflow_amd.device import Context, Mesh
from geoflow_amd.ensemble import Ensemble, MemberSpec

NU = 0.02        # viscosity of the Burgers and ensemble workloads
W8 = 8           # bytes of an FP64 value


def listed():
    return [
        # The 2-D Burgers run of the parity tests: a small mesh stepped many
        # times, where the launches of a step count.
        dict(name="burgers2d_16x16_p4", kind="burgers", dim=2, p=4, nx=16, ny=16, nz=1,
             order=4, steps=10, Lx=1.0, Ly=1.0, Lz=1.0),
        # The benchmark's step: 16.8 M nodes, three components, RK4.
        dict(name="burgers3d_32_p7", kind="burgers", dim=3, p=7, nx=32, ny=32, nz=32,
             order=4, steps=4, Lx=1.0, Ly=1.0, Lz=1.0),
        # A box as a regional run has it: unequal extents and counts, another
        # order of element and of the scheme.
        dict(name="burgers3d_ragged_p5_rk3", kind="burgers", dim=3, p=5, nx=19, ny=14, nz=11,
             order=3, steps=5, Lx=2.0, Ly=1.5, Lz=1.0),
        # The benchmark's Helmholtz solve (Dirichlet box, Jacobi).
        dict(name="cg_box_32_p7", kind="cgbox", p=7, nx=32, ny=32, nz=32, periodic=False,
             coef=0.1, precond=1, precision=0),
        # The same operator with FP32 recurrences and FP64 updates, at an
        # order with an odd number of nodes.
        dict(name="cg_box_mixed_20_p6", kind="cgbox", p=6, nx=20, ny=20, nz=20, periodic=False,
             coef=0.1, precond=1, precision=1),
        # A small solve without a preconditioner (the reference's default):
        # an iteration is a few short kernels.
        dict(name="cg_box_small_5x4x3_p4", kind="cgbox", p=4, nx=5, ny=4, nz=3, periodic=False,
             coef=0.1, precond=0, precision=0),
        # A solve on a terrain-following mesh (metrics at every node).
        dict(name="cg_terrain_10x9x6_p6", kind="cgnode", mesh="terrain3d", p=6, nx=10, ny=9,
             nz=6, level=0, coef=0.1, precision=0),
        # Tracer advection on the sphere, bench's order and viscosity.
        dict(name="sphere_adv_l5_p5", kind="sphere", p=5, level=5, order=4, steps=10),
        # One implicit-viscous step of a batched ensemble of uneven members.
        dict(name="ensemble_8", kind="ensemble", members="4:12,6:8,8:8,4:16,6:12,8:12,4:8,6:8",
             precision=0),
        # A gradient through the checkpointed adjoint, the adjoint workload's
        # order and checkpoint ratio on a shorter window.
        dict(name="adjoint_12_p6", kind="adjoint", p=6, nx=12, ny=12, nz=12, order=4, steps=6,
             ckpt=3),
        # The right-hand side and its assembly, for a stepper of one's own.
        dict(name="rhs_24_p7", kind="rhs", p=7, nx=24, ny=24, nz=24, Lx=1.0, Ly=1.0, Lz=1.0),
        # The operators one by one on a ragged box: gradient, advection,
        # Helmholtz with a coefficient field and in FP32, assembly.
        dict(name="operators_21x17x13_p5", kind="operators", p=5, nx=21, ny=17, nz=13, Lx=1.4,
             Ly=1.0, Lz=0.9),
    ]


def draw(rng):
    def logint(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    def box(p, lo, hi, nodes):
        while True:
            n = [logint(lo, hi) for _ in range(3)]
            if n[0] * n[1] * n[2] * (p + 1) ** 3 <= nodes:
                return dict(p=p, nx=n[0], ny=n[1], nz=n[2])

    def lengths():
        return dict(Lx=round(rng.uniform(0.5, 2.0), 3), Ly=round(rng.uniform(0.5, 2.0), 3),
                    Lz=round(rng.uniform(0.5, 2.0), 3))

    kind = rng.choice(["burgers2d", "burgers3d", "cgbox", "cgnode", "sphere", "ensemble",
                       "adjoint", "rhs", "operators"])
    if kind == "burgers2d":
        return dict(kind="burgers", dim=2, p=rng.randint(2, 9), nx=logint(4, 96),
                    ny=logint(4, 96), nz=1, order=rng.randint(2, 4), steps=rng.randint(2, 12),
                    **lengths())
    if kind == "burgers3d":
        return dict(kind="burgers", dim=3, order=rng.randint(2, 4), steps=rng.randint(2, 5),
                    **box(rng.randint(3, 8), 3, 32, 8_000_000), **lengths())
    if kind == "cgbox":
        return dict(kind="cgbox", periodic=rng.random() < 0.3,
                    coef=round(10 ** rng.uniform(-3, -0.7), 5), precond=int(rng.random() < 0.8),
                    precision=int(rng.random() < 0.4), **box(rng.randint(3, 8), 3, 24, 4_000_000))
    if kind == "cgnode":
        if rng.random() < 0.5:
            return dict(kind="cgnode", mesh="sphere", p=rng.randint(3, 6), nx=0, ny=0, nz=0,
                        level=rng.randint(1, 3), coef=round(10 ** rng.uniform(-3, -1), 5),
                        precision=int(rng.random() < 0.4))
        return dict(kind="cgnode", mesh="terrain3d", level=0,
                    coef=round(10 ** rng.uniform(-3, -1), 5),
                    precision=int(rng.random() < 0.4), **box(rng.randint(3, 7), 3, 12, 250_000))
    if kind == "sphere":
        return dict(kind="sphere", p=rng.randint(3, 7), level=rng.randint(2, 4),
                    order=rng.randint(2, 4), steps=rng.randint(3, 10))
    if kind == "ensemble":
        mem = ",".join("%d:%d" % (rng.choice((4, 6, 8)), rng.choice((4, 6, 8, 12)))
                       for _ in range(rng.randint(3, 9)))
        return dict(kind="ensemble", members=mem, precision=int(rng.random() < 0.4))
    if kind == "adjoint":
        return dict(kind="adjoint", order=rng.randint(2, 4), steps=rng.randint(3, 7),
                    ckpt=rng.randint(2, 4), **box(rng.randint(3, 7), 3, 14, 400_000))
    if kind == "rhs":
        return dict(kind="rhs", **box(rng.randint(3, 8), 3, 28, 8_000_000), **lengths())
    return dict(kind="operators", **box(rng.randint(3, 8), 3, 28, 4_000_000), **lengths())


# ---------------------------------------------------------------------------
# Meshes.  The host grid does not depend on the fields, so a program (and this
# file) forms it once; the device mesh is made for every state.
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=2)
def _box_grid(dim, p, ne, L, periodic):
    b = ga.GF_BDY_PERIODIC if periodic else ga.GF_BDY_DIRICHLET
    return ga.BoxGrid(dim, p, list(ne), P1=L, bdy=[b] * (2 * dim), device_maps=dim == 3)


@functools.lru_cache(maxsize=2)
def _node_grid(mesh, p, ne, level):
    if mesh == "sphere":
        return ga.IcosGrid(p, level, radius=1.0)
    return ga.TerrainBoxGrid3D(p, list(ne), amp=0.1)


class Lattice:
    """The node lattice of a box of equal elements: FP64 tables in torch."""

    def __init__(self, dim, p, ne, L, periodic):
        self.dim, self.p, self.N, self.ne, self.per = dim, p, p + 1, list(ne[:dim]), periodic
        self.h = [L[d] / ne[d] for d in range(dim)]
        P = np.polynomial.legendre.Legendre.basis(p)
        x = np.concatenate([[-1.0], np.sort(P.deriv().roots().real), [1.0]])
        for _ in range(3):  # Newton steps on (1 - x^2) P'(x) at the inner nodes
            f, g = P.deriv()(x[1:-1]), P.deriv(2)(x[1:-1])
            x[1:-1] -= f / g
        x = 0.5 * (x - x[::-1])
        w = 2.0 / (p * (p + 1) * P(x) ** 2)
        pv = P(x)
        D = np.zeros((p + 1, p + 1))
        for i in range(p + 1):
            for j in range(p + 1):
                if i != j:
                    D[i, j] = pv[i] / (pv[j] * (x[i] - x[j]))
        D[0, 0], D[p, p] = -p * (p + 1) / 4.0, p * (p + 1) / 4.0
        self.x, self.w, self.Dn = x, w, D
        dev = dict(dtype=torch.float64, device="cuda")
        self.D = torch.tensor(D, **dev)
        n1 = [ne[d] * p if periodic else ne[d] * p + 1 for d in range(dim)]
        self.n1 = n1
        self.idx = []
        for d in range(dim):
            g = (torch.arange(ne[d])[:, None] * p + torch.arange(p + 1)[None, :]) % n1[d]
            shape = [1] * (2 * dim)
            shape[dim - 1 - d], shape[2 * dim - 1 - d] = ne[d], p + 1
            self.idx.append(g.reshape(shape).cuda())
        wt = torch.tensor(w, **dev)
        m = wt
        for _ in range(dim - 1):
            m = m[..., None] * wt  # every axis the same weights
        self.mass = m * math.prod(0.5 * h for h in self.h)
        self.dx = min(self.h) * 0.5 * float(x[1] - x[0])
        one = torch.ones(self.shape(), **dev)
        self.mult = self.total(one)
        am = self.smooth((one * self.mass))
        self.imass = 1.0 / am

    def shape(self):
        return tuple(reversed(self.ne)) + (self.N,) * self.dim

    def local(self, lat):
        """Lattice values at every element's nodes."""
        return lat[tuple(reversed(self.idx))]

    def coords(self):
        """Lattice coordinates as broadcastable axes (x, y[, z])."""
        out = []
        for d in range(self.dim):
            c = (np.arange(self.ne[d])[:, None] + 0.5 * (self.x[None, :-1] + 1)) * self.h[d]
            c = c.reshape(-1)
            if not self.per:
                c = np.append(c, self.ne[d] * self.h[d])
            s = [1] * self.dim
            s[self.dim - 1 - d] = -1
            out.append(torch.tensor(c, dtype=torch.float64, device="cuda").reshape(s))
        return out

    def fold(self, u):
        """Sums of the copies of every lattice node."""
        dim, p = self.dim, self.p
        for d in range(dim):  # direction d: element axis and node axis joined
            # the axes still unfolded are (el axes of dims dim-1..d), lattice
            # axes of the directions done, then node axes: bring (el, node) of
            # direction d to the end
            ea = dim - 1 - d
            u = u.movedim((ea, u.dim() - 1), (-2, -1))
            ne = self.ne[d]
            body, last = u[..., :p], u[..., p]
            if self.per:
                body = torch.cat([body[..., :1] + torch.roll(last, 1, -1)[..., None],
                                  body[..., 1:]], -1)
                lat = body.reshape(body.shape[:-2] + (ne * p,))
            else:
                first = torch.cat([body[..., 0, :1][..., None, :],
                                   body[..., 1:, :1] + last[..., :-1, None]], -2)
                body = torch.cat([first, body[..., 1:]], -1)
                lat = torch.cat([body.reshape(body.shape[:-2] + (ne * p,)), last[..., -1:]], -1)
            u = lat.movedim(-1, ea)
            # after direction d the lattice axis stands where its element
            # axis stood and the remaining node axes end with direction d+1
        return u

    def total(self, u):
        return self.local(self.fold(u))

    def smooth(self, u):
        return self.total(u) / self.mult

    def ref(self, u, d, trans=False):
        """D (or its transpose) along direction d of every element."""
        A = self.D.T if trans else self.D
        s = u.shape
        N = self.N
        v = u.reshape(-1, N, N ** d)
        if d == 0:
            return (u.reshape(-1, N) @ A.T).reshape(s)
        return torch.matmul(A, v).reshape(s)

    def deriv(self, u, d):
        return self.ref(u, d) * (2.0 / self.h[d])

    def lap(self, u, pf=None):
        """Weak (element-wise) Laplacian, with a coefficient field."""
        out = None
        for d in range(self.dim):
            g = self.ref(u, d) * (2.0 / self.h[d]) ** 2 * self.mass
            if pf is not None:
                g = g * pf
            t = self.ref(g, d, True)
            out = t if out is None else out + t
        return out

    def advect(self, q, us):
        s = 0.0
        for d, v in enumerate(us):
            s = s + v * self.deriv(q, d)
        return self.mass * s

    def rhs(self, us, nu):
        return [self.imass * (-nu * self.lap(u) - self.advect(u, us)) for u in us]

    def step(self, us, nu, dt, order):
        c = {1: [1.0], 2: [0.5, 0.5], 3: [0.25, 0.0, 0.75],
             4: [1 / 6, 1 / 3, 1 / 3, 1 / 6]}[order]
        b = {1: [0], 2: [0, 1.0], 3: [0, 1 / 3, 2 / 3], 4: [0, 0.5, 0.5, 1.0]}[order]
        acc, K = list(us), None
        for s in range(order):
            v = us if s == 0 else [u + b[s] * dt * k for u, k in zip(us, K)]
            if s == order - 1:
                v = [self.smooth(a) for a in v]
            K = [self.smooth(k) for k in self.rhs(v, nu)]
            acc = [a + c[s] * dt * k for a, k in zip(acc, K)]
        return [self.smooth(a) for a in acc]

    def solve(self, lat, p, q):
        """(p L + q M)^-1 of an assembled lattice vector, homogeneous Dirichlet
        or periodic, by the generalised eigenvectors of each direction."""
        T, lam = [], []
        for d in range(self.dim):
            n, h = self.n1[d], self.h[d]
            K, M = np.zeros((n, n)), np.zeros(n)
            Ke = self.Dn.T @ np.diag(self.w) @ self.Dn * (2.0 / h)
            for e in range(self.ne[d]):
                ix = (e * self.p + np.arange(self.N)) % n
                # an element that is its own neighbour has one index twice
                np.add.at(K, (ix[:, None], ix[None, :]), Ke)
                np.add.at(M, ix, self.w * h / 2)
            keep = np.arange(n) if self.per else np.arange(1, n - 1)
            s = 1.0 / np.sqrt(M[keep])
            ev, Z = np.linalg.eigh(K[np.ix_(keep, keep)] * s[:, None] * s[None, :])
            full = np.zeros((n, len(keep)))
            full[keep] = Z * s[:, None]
            T.append(torch.tensor(full, dtype=torch.float64, device="cuda"))
            lam.append(torch.tensor(ev, dtype=torch.float64, device="cuda"))
        u = lat
        for d in range(self.dim):
            ax = self.dim - 1 - d
            u = torch.movedim(torch.movedim(u, ax, -1) @ T[d], -1, ax)
        den = q
        for d in range(self.dim):
            s = [1] * self.dim
            s[self.dim - 1 - d] = -1
            den = den + p * lam[d].reshape(s)
        u = u / den
        for d in range(self.dim):
            ax = self.dim - 1 - d
            u = torch.movedim(torch.movedim(u, ax, -1) @ T[d].T, -1, ax)
        return u


def _geometry(case):
    dim = case.get("dim", 3)
    ne = (case["nx"], case["ny"], case["nz"])[:dim]
    L = (case.get("Lx", 1.0), case.get("Ly", 1.0), case.get("Lz", 1.0))
    return dim, case["p"], ne, L, case.get("periodic", True)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _waves(lat, g, ncomp, modes=10):
    """Random periodic fields of low wavenumber, continuous over elements."""
    xs = lat.coords()
    out = []
    for _ in range(ncomp):
        k = torch.randint(-3, 4, (modes, lat.dim), generator=g, device="cuda").tolist()
        a = torch.randn(modes, generator=g, device="cuda", dtype=torch.float64).tolist()
        f = torch.rand(modes, generator=g, device="cuda", dtype=torch.float64).tolist()
        u = 0.0
        for m in range(modes):
            arg = 2 * math.pi * f[m]
            for d in range(lat.dim):
                arg = arg + 2 * math.pi * k[m][d] / (lat.h[d] * lat.ne[d]) * xs[d]
            u = u + a[m] / (2.0 + sum(v * v for v in k[m])) * torch.cos(arg)
        out.append(lat.local(u.expand(tuple(reversed(lat.n1)))).contiguous().reshape(-1))
    return out


def _noise(lat, g):
    """N(0, 1) per distinct node, as the benchmark's right-hand side."""
    u = torch.randn(tuple(reversed(lat.n1)), generator=g, device="cuda", dtype=torch.float64)
    return lat.local(u).reshape(-1)


def _members(case):
    return [MemberSpec(*map(int, m.split(":"))) for m in case["members"].split(",")]


def _inputs(case, seed):
    """The fields of a case, from the seed: the box cases' lattice and fields."""
    g = _gen(seed)
    if case["kind"] == "ensemble":
        lats = [Lattice(3, m.p, [m.ne] * 3, (1.0, 1.0, 1.0), True) for m in _members(case)]
        return lats, [_waves(l, g, 3, 6) for l in lats]
    lat = Lattice(*_geometry(case))
    if case["kind"] == "cgbox":
        return lat, [_noise(lat, g)]
    if case["kind"] == "adjoint":
        return lat, _waves(lat, g, 6)
    if case["kind"] == "operators":
        return lat, _waves(lat, g, 5)
    return lat, _waves(lat, g, lat.dim)


def _dt(lat):
    return min(0.02 * lat.dx ** 2 / NU, 0.05 * lat.dx)


ENS_DT = 5e-5
TOL = 1e-11  # solves: the benchmark's 1e-10 and one digit more


def prepare(case, seed):
    kind = case["kind"]
    ctx = Context(0)
    st = dict(case=case)
    if kind in ("cgnode", "sphere"):
        g = _node_grid(case.get("mesh", "sphere"), case["p"],
                       (case.get("nx", 0), case.get("ny", 0), case.get("nz", 0)), case["level"])
        m = st["mesh"] = Mesh(ctx, g)
        if kind == "cgnode":
            f = torch.from_numpy(workloads.unique_normal(g, seed=seed)).cuda()
            st["b"] = m.mass_apply(f)
            st["xb"] = torch.zeros_like(f) if g.mask is not None else None
        else:
            lat0, lon0 = workloads.bell_centre(seed)
            h = workloads.cosine_bell(*g.xyz, lat0, lon0)
            v = workloads.williamson1_velocity(*g.xyz, 2 * np.pi, np.pi / 4)
            st["u"] = [torch.from_numpy(a).cuda() for a in [h] + v]
        return st
    lat, fields = _inputs(case, seed)
    if kind == "ensemble":
        st["ens"] = Ensemble(ctx, _members(case), device_maps=True)
        st["u"] = st["ens"].new_state(lambda i, g: fields[i])
        return st
    m = st["mesh"] = Mesh(ctx, _box_grid(*_geometry(case)))
    if kind == "cgbox":
        st["b"] = m.mass_apply(fields[0])
        st["xb"] = None if case["periodic"] else torch.zeros_like(fields[0])
        return st
    st["dt"] = _dt(lat)
    st["u"] = fields[:3]
    if kind == "adjoint":
        st["target"] = fields[3:]
        st["mass"] = m.mass_apply(torch.ones_like(fields[0]))
    if kind == "operators":
        st["q"] = fields[3]
        st["coef"] = 1.0 + 0.2 * torch.tanh(fields[4])
        st["q32"] = fields[3].float()
        st["out"] = [m.new(), m.new(), m.new(torch.float32)]
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    m = st.get("mesh")
    if kind == "burgers":
        return m.burgers_steps(st["u"], NU, st["dt"], case["steps"], order=case["order"])
    if kind == "sphere":
        return m.burgers_steps(st["u"], 5e-5, 1e-4, case["steps"], mode=1,
                               order=case["order"])[0]
    if kind in ("cgbox", "cgnode"):
        x, _ = m.cg_solve(st["b"], xb=st["xb"], p=case["coef"], q=1.0, maxit=20000, tol=TOL,
                          normtype=4, precond=case.get("precond", 1),
                          precision=case["precision"], raise_on_error=True)
        return x
    if kind == "ensemble":
        st["ens"].imex_step(st["u"], NU, ENS_DT, precision=case["precision"], tol=1e-12)
        return st["u"]
    if kind == "adjoint":
        u = [a.clone() for a in st["u"]]
        m.burgers_steps(u, NU, st["dt"], case["steps"], order=case["order"])
        lam = [st["mass"] * (a - t) for a, t in zip(u, st["target"])]
        return m.burgers_adjoint(st["u"], lam, NU, st["dt"], case["steps"], order=case["order"],
                                 ckpt=case["ckpt"])
    if kind == "rhs":
        return [m.dss(k, "smooth") for k in m.burgers_rhs(st["u"], NU)]
    o = st["out"]
    return dict(grad=m.grad(st["q"]), adv=m.advect(st["q"], st["u"], out=o[0]),
                helm=m.dss(m.helmholtz(st["q"], p=st["coef"], q=1.0, out=o[1]), "sum"),
                helm32=m.helmholtz_f32(st["q32"], p=0.1, q=1.0, out=o[2]))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("cgnode", "sphere"):
        return None
    lat, fields = _inputs(case, seed)
    if kind == "ensemble":
        res = {}
        for ms, la, fs in zip(_members(case), lat, fields):
            us = [f.reshape(la.shape()) for f in fs]
            new = []
            for u in us:
                b = la.mass * u - ENS_DT * la.advect(u, us)
                new.append(la.local(la.solve(la.fold(b), NU * ENS_DT, 1.0)).reshape(-1))
            res.setdefault(ms.p, []).append(new)
        return {p: [torch.cat([v[c] for v in res[p]]) for c in range(3)] for p in res}
    fs = [f.reshape(lat.shape()) for f in fields]
    flat = lambda v: v.reshape(-1)  # noqa: E731
    if kind == "cgbox":
        return flat(lat.local(lat.solve(lat.fold(lat.mass * fs[0]), case["coef"], 1.0)))
    dt = _dt(lat)
    if kind == "burgers":
        us = fs
        for _ in range(case["steps"]):
            us = lat.step(us, NU, dt, case["order"])
        return [flat(u) for u in us]
    if kind == "adjoint":
        u0 = [f.clone().requires_grad_(True) for f in fs[:3]]
        us = u0
        for _ in range(case["steps"]):
            us = lat.step(us, NU, dt, case["order"])
        lam = [(lat.mass * (a - t)).detach() for a, t in zip(us, fs[3:])]
        return [flat(g) for g in torch.autograd.grad(us, u0, lam)]
    if kind == "rhs":
        return [flat(lat.smooth(k)) for k in lat.rhs(fs, NU)]
    u, q, coef = fs[:3], fs[3], 1.0 + 0.2 * torch.tanh(fs[4])
    q32 = q.float().double()
    return dict(grad=[flat(lat.deriv(q, d)) for d in range(3)], adv=flat(lat.advect(q, u)),
                helm=flat(lat.total(lat.lap(q, coef) + lat.mass * q)),
                helm32=flat(0.1 * lat.lap(q32) + lat.mass * q32))


def _cg_iterations(case):
    """Rough count of CG iterations to the tolerance: the square root of the
    condition number of (q M + p L), in nodes per direction."""
    if case["kind"] == "cgnode" and case["mesh"] == "sphere":
        n1 = 4 * 2 ** case["level"] * case["p"]
    else:
        n1 = max(case["nx"], case["ny"], case["nz"]) * case["p"]
    return 10 + 19.0 * n1 * math.sqrt(case["coef"])


def work(case):
    """Values that have to move and operations that have to be done, by the
    mathematics: one read and one write of every evolved field in each stage
    (a stage needs its neighbours' previous one), of x, r and w in each
    iteration (an iteration has two global sums)."""
    kind, p = case["kind"], case.get("p", 0)
    N = p + 1
    if kind == "ensemble":
        n = flops = 0
        for m in _members(case):
            n += m.ndof
            flops += m.ndof * 3 * (6 * 12 * (m.p + 1) + 60)
        return dict(bytes=float(n * 3 * W8 * (2 + 6 * 6)), flops=float(flops))
    if kind == "sphere" or (kind == "cgnode" and case["mesh"] == "sphere"):
        n, dim = 60 * 4 ** case["level"] * N * N, 2
    else:
        dim, _, ne, _, _ = _geometry(case)
        n = math.prod(ne) * N ** dim
    lap = 4 * dim * N + 8
    if kind == "sphere":
        s = case["order"] * case["steps"]
        return dict(bytes=float(n * W8 * s * (2 + 5)), flops=float(n * s * (lap + 10)))
    if kind == "burgers":
        s = case["order"] * case["steps"]
        return dict(bytes=float(n * W8 * dim * s * 2), flops=float(n * s * dim * (lap + 10)))
    if kind in ("cgbox", "cgnode"):
        it = _cg_iterations(case)
        w = 4 if case["precision"] else 8
        metric = {"sphere": 4, "terrain3d": 7}.get(case.get("mesh"), 0)
        return dict(bytes=float(n * w * it * (6 + metric)), flops=float(n * it * (lap + 14)))
    if kind == "adjoint":
        # forward twice, stage states once more, each stage's transpose
        s = case["order"] * case["steps"]
        return dict(bytes=float(n * W8 * 3 * s * (2 + 2 + 2 + 3)),
                    flops=float(n * s * 3 * (5 * lap + 40)))
    if kind == "rhs":
        return dict(bytes=float(n * W8 * 6), flops=float(n * 3 * (lap + 10)))
    return dict(bytes=float(n * (W8 * (1 + 3 + 4 + 1 + 3) + 8)), flops=float(n * (4 * lap)))
