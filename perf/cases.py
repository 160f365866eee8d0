"""Performance cases of the Helmholtz/Poisson solve path.

Each case is a call that a time-stepping program makes through
nek5000_amd.solver on fields resident on the GPU:

  axhelm    Field.axhelm          one operator apply
  dssum     Field.dssum           one direct-stiffness sum
  helmholtz Field.hmholtz         a velocity component or a scalar, Jacobi PCG
  step      Batch.hmholtz         the viscous solves of one time step together
  pressure  Field.hmholtz('PRES') flexible CG or GMRES with the h1mg V-cycle

Meshes are boxes of nx x ny x nz elements of width 1/32, every node moved by
the sine map of the benchmark (0.1 element widths), Dirichlet walls except
where a case is periodic in x.  Right-hand sides are B f with f ~ U(-1, 1) per
unique node.  exact() restates geometry, operator and solves in plain torch.
"""
import math

import numpy as np
import torch

from nek5000_amd import solver
from nek5000_amd.mesh import BoxMesh

# The viscous coefficients of a BDF3 step: h1 = nu, h2 = bd(1)/dt with
# bd(1) = 11/6 and dt = 1e-3 (the benchmark's time-step solves).
NU, BD_DT = 1.0e-3, 11.0 / 6.0e-3
WIDTH = 1.0 / 32.0  # element width
RTOL = 1.0e-8  # relative residual of every solve
DEFORM = 0.1

# What a solve needs per local node and iteration, in 8-byte words (mixed
# solves keep their iteration in 4-byte ones): Jacobi PCG reads p, r, d, six
# factors and bm1 and writes p and w in the operator, reads and writes the
# shared part of w in the assembly, and reads p, w, x, r and two weights and
# writes x and r in the update; the multigrid-preconditioned iteration has the
# operator's 13, 2.4 of its assembly, 6 of the vector updates and dots, and
# about 15 in the V-cycle.  Nominal iteration counts for RTOL.
PCG_WORDS, PCG_ITERS = 22.0, {"uniform": 12, "field": 24}
PRES_WORDS, PRES_ITERS = 36.0, 16
PRES_FLOPS = 700.0  # per node and iteration: operator and local solves


def listed():
    return [
        # operator applies: a small mesh of low order, where the call itself
        # counts; varying viscosity (turbulence model) at the usual order on
        # a mesh larger than the caches; constant coefficients at high order
        dict(name="axhelm-small-n5", kind="axhelm", nx=6, ny=5, nz=7, lx1=6, coef="uniform"),
        dict(name="axhelm-visc-n7", kind="axhelm", nx=30, ny=29, nz=28, lx1=8, coef="field"),
        dict(name="axhelm-n11", kind="axhelm", nx=17, ny=18, nz=16, lx1=12, coef="uniform"),
        # averaging a field at element boundaries
        dict(name="dssum-n9", kind="dssum", nx=20, ny=22, nz=21, lx1=10),
        # one velocity component: a small case (or one rank of a
        # strong-scaled one) and a large one
        dict(name="velocity-small", kind="helmholtz", nx=6, ny=7, nz=8, lx1=8, coef="uniform",
             precision=0, periodic=False),
        dict(name="velocity-large", kind="helmholtz", nx=32, ny=32, nz=32, lx1=8,
             coef="uniform", precision=0, periodic=False),
        # a scalar with varying diffusivity in a channel (periodic in x)
        dict(name="scalar-field-n9", kind="helmholtz", nx=14, ny=13, nz=15, lx1=10,
             coef="field", precision=0, periodic=True),
        # the same solves with the iteration in single precision
        dict(name="velocity-mixed", kind="helmholtz", nx=26, ny=25, nz=27, lx1=8,
             coef="uniform", precision=2, periodic=False),
        # three velocity components and two scalars of one time step
        dict(name="step-batch", kind="step", nx=10, ny=11, nz=12, lx1=8, scalars=2,
             precision=0),
        # pressure: flexible CG on a large mesh, the single-precision variant
        # on a medium one, and the default GMRES on a small one
        dict(name="pressure-large", kind="pressure", nx=30, ny=31, nz=29, lx1=8,
             method="fcg", precision=0),
        dict(name="pressure-mixed", kind="pressure", nx=17, ny=16, nz=18, lx1=8,
             method="fcg", precision=2),
        dict(name="pressure-gmres-n5", kind="pressure", nx=12, ny=11, nz=13, lx1=6,
             method="gmres", precision=0),
    ]


def _dims(rng, lo, hi):
    """Three element counts around the cube root of a count spread over its
    logarithm."""
    e = math.exp(rng.uniform(math.log(lo), math.log(hi))) ** (1.0 / 3.0)
    cap = hi ** (1.0 / 3.0)
    return {k: max(3, int(min(e * rng.uniform(0.85, 1.15), cap))) for k in ("nx", "ny", "nz")}


def draw(rng):
    kind = rng.choice(["axhelm", "axhelm", "dssum", "helmholtz", "helmholtz", "step",
                       "pressure", "pressure"])
    if kind in ("axhelm", "dssum"):
        lx1 = rng.randint(4, 14)
        c = dict(kind=kind, lx1=lx1, **_dims(rng, 60, 1.1e7 / lx1 ** 3))
        if kind == "axhelm":
            c["coef"] = rng.choice(["uniform", "field"])
        return c
    if kind == "helmholtz":
        lx1 = rng.choice([6, 7, 8, 8, 9, 10])
        precision = rng.choice([0, 0, 2])
        return dict(kind=kind, lx1=lx1, precision=precision, periodic=rng.random() < 0.3,
                    coef="uniform" if precision else rng.choice(["uniform", "field"]),
                    **_dims(rng, 60, 1.2e7 / lx1 ** 3))
    if kind == "step":
        lx1 = rng.choice([6, 8, 8, 10])
        return dict(kind=kind, lx1=lx1, scalars=rng.randint(1, 3), precision=rng.choice([0, 2]),
                    **_dims(rng, 60, 1.5e6 / lx1 ** 3))
    lx1 = rng.choice([6, 8, 8, 10])
    method = rng.choice(["fcg", "fcg", "gmres"])
    return dict(kind=kind, lx1=lx1, method=method,
                precision=rng.choice([0, 2]) if method == "fcg" else 0,
                **_dims(rng, 120, 1.0e7 / lx1 ** 3))


# ---------------------------------------------------------------------------
# inputs: plain torch, shared by prepare() and exact()
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _lattice(c):
    """For every local node the number of its point of the global lattice
    (equal at all copies of a shared node), and the lattice's size."""
    n, d = c["lx1"] - 1, "cuda"
    per = bool(c.get("periodic", False))
    px, py, pz = (c["nx"] * n if per else c["nx"] * n + 1), c["ny"] * n + 1, c["nz"] * n + 1
    a = torch.arange(c["lx1"], device=d)

    def axis(cnt):
        return torch.arange(cnt, device=d)[:, None] * n + a

    ix, iy, iz = axis(c["nx"]) % px, axis(c["ny"]), axis(c["nz"])
    ids = (ix[None, None, :, None, None, :]
           + px * (iy[None, :, None, None, :, None] + py * iz[:, None, None, :, None, None]))
    return ids.reshape(-1), px * py * pz


def _shape(c):
    return (c["nx"] * c["ny"] * c["nz"], c["lx1"], c["lx1"], c["lx1"])


def _node_field(c, seed):
    """U(-1, 1) per unique node."""
    ids, cnt = _lattice(c)
    v = torch.rand(cnt, generator=_gen(seed), device="cuda", dtype=torch.float64)
    return (2.0 * v - 1.0)[ids].reshape(_shape(c)).contiguous()


def _coefs(c, seed, xyz):
    """h1, h2 of a case: constants, or smooth positive fields."""
    if c["kind"] == "pressure":
        one = torch.ones(_shape(c), dtype=torch.float64, device="cuda")
        return one, torch.zeros_like(one)
    h1 = torch.full(_shape(c), NU, dtype=torch.float64, device="cuda")
    h2 = torch.full(_shape(c), BD_DT, dtype=torch.float64, device="cuda")
    if c.get("coef", "uniform") == "field":
        x, y, z = xyz
        # whole periods over the box, so that a periodic x stays continuous
        kx = 2.0 * math.pi / (c["nx"] * WIDTH)
        s = 0.1 * (seed % 7)
        h1 = h1 * (1.5 + torch.sin(kx * x + s) * torch.cos(9.0 * y) * torch.cos(7.0 * z))
        h2 = h2 * (1.0 + 0.2 * torch.cos(kx * x + s) * torch.sin(5.0 * y))
    return h1.contiguous(), h2.contiguous()


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------
class _State:
    """Handles and arrays of one case; gives the library's handles back."""

    def __init__(self):
        self.fields, self.batch = [], None

    def __del__(self):
        try:
            if self.batch is not None:
                self.batch.destroy()
            for f in self.fields:
                f.destroy()
        except Exception:  # at interpreter exit the library may be gone
            pass


def _box(c):
    return BoxMesh(c["nx"], c["ny"], c["nz"], c["lx1"],
                   lengths=(c["nx"] * WIDTH, c["ny"] * WIDTH, c["nz"] * WIDTH),
                   deform=DEFORM, periodic_x=bool(c.get("periodic", False)))


def _step_boxes(c):
    """The velocity mesh and the (smaller) scalar meshes of a time step."""
    out = [dict(c, kind="helmholtz", coef="uniform", periodic=False)]
    for k in range(c["scalars"]):
        out.append(dict(out[0], nx=max(2, c["nx"] * 2 // 3 - k), ny=max(2, c["ny"] * 2 // 3),
                        periodic=k % 2 == 1))
    return out


def _step_solves(c):
    """(box, seed offset) of every solve: three components, then the scalars."""
    boxes = _step_boxes(c)
    return [(0, 0), (0, 1), (0, 2)] + [(k, 2 + k) for k in range(1, len(boxes))]


def prepare(case, seed):
    c, st = case, _State()
    st.kind = c["kind"]
    if st.kind == "step":
        boxes = _step_boxes(c)
        st.fields = [solver.box_field(_box(b)) for b in boxes]
        solves = _step_solves(c)
        st.batch = solver.Batch([st.fields[k] for k, _ in solves])
        mass = [f.mass()[0] for f in st.fields]
        coefs = [_coefs(b, seed, None) for b in boxes]
        st.rhs0 = [(mass[k] * _node_field(boxes[k], 97 * seed + o)).contiguous()
                   for k, o in solves]
        st.solves = [dict(u=st.fields[k].zeros(), rhs=torch.empty_like(r), h1=coefs[k][0],
                          h2=coefs[k][1], mask=st.fields[k].mask, mult=st.fields[k].mult,
                          tli=-RTOL) for (k, _), r in zip(solves, st.rhs0)]
        st.params = solver.default_params(istep=20, precision=c["precision"])
        return st
    box = _box(c)
    f = solver.box_field(box, multigrid=st.kind == "pressure")
    st.fields = [f]
    v = _node_field(c, seed)
    if st.kind == "dssum":
        # contributions of each element to its copies of a node
        st.u0, st.u = f.mass()[0] * v, torch.empty_like(v)
        return st
    xyz = None
    if c.get("coef") == "field":
        xyz = [torch.as_tensor(a, device="cuda") for a in box.xyz()]
    st.h1, st.h2 = _coefs(c, seed, xyz)
    if st.kind == "axhelm":
        st.u, st.au = v, f.zeros()
        return st
    st.rhs0 = f.mass()[0] * v
    st.rhs, st.u = torch.empty_like(v), f.zeros()
    if st.kind == "helmholtz":
        st.name, st.maxit = "VELX", 900
        st.params = solver.default_params(istep=20, precision=c["precision"])
    else:
        st.name, st.maxit = "PRES", 200
        st.params = solver.default_params(istep=20, param21=-RTOL, precision=c["precision"],
                                          param42=2 if c["method"] == "fcg" else 0)
    return st


def run(st):
    f = st.fields[0]
    if st.kind == "axhelm":
        f.axhelm(st.au, st.u, st.h1, st.h2)
        return st.au
    if st.kind == "dssum":
        st.u.copy_(st.u0)
        f.dssum(st.u)
        return st.u
    if st.kind == "step":
        for q, r in zip(st.solves, st.rhs0):
            q["rhs"].copy_(r)
        st.batch.hmholtz(st.solves, 900, params=st.params)
        return [[q["u"], q["rhs"]] for q in st.solves]
    # the solve assembles and masks its right-hand side in place
    st.rhs.copy_(st.rhs0)
    f.hmholtz(st.name, st.u, st.rhs, st.h1, st.h2, f.mask, f.mult, -RTOL, st.maxit,
              params=st.params)
    return [st.u, st.rhs]


def work(case):
    c = case
    n = float(np.prod(_shape(c)))
    lx1 = c["lx1"]
    apply_flops = 12.0 * lx1 + 21.0
    if c["kind"] == "axhelm":
        # u, six factors, bm1, h1 and h2 in, au out
        return dict(bytes=8.0 * 11 * n, flops=apply_flops * n)
    if c["kind"] == "dssum":
        # the copy of the input, then the shared nodes read and written
        shared = 1.0 - ((lx1 - 2.0) / lx1) ** 3
        return dict(bytes=8.0 * n * (2 + 2 * shared) + 4.0 * n * shared, flops=n * shared)
    word = 4.0 if c.get("precision") == 2 else 8.0
    if c["kind"] == "pressure":
        return dict(bytes=word * PRES_WORDS * PRES_ITERS * n, flops=PRES_FLOPS * PRES_ITERS * n)
    if c["kind"] == "step":
        boxes = _step_boxes(c)
        n = float(sum(np.prod(_shape(boxes[k])) for k, _ in _step_solves(c)))
    field = c.get("coef") == "field"  # then h1 and h2 are read as well
    iters = PCG_ITERS["field" if field else "uniform"]
    return dict(bytes=word * (PCG_WORDS + 2.0 * field) * iters * n,
                flops=(apply_flops + 14.0) * iters * n)


def tolerance(case):
    k = case["kind"]
    if k in ("axhelm", "dssum"):
        # 64-bit sums; measured 1e-14 to 5e-13 from exact(), most of it the
        # rounding of coordinates that the geometric factors amplify
        return dict(rel=2e-12)
    # solves to a relative residual of 1e-8: measured 2e-9 to 3.2e-8 from
    # exact(), the error that the last iterate keeps
    return dict(rel=1.3e-7)


# ---------------------------------------------------------------------------
# plain torch, 64 bits
# ---------------------------------------------------------------------------
def _gll(n):
    """Gauss-Lobatto-Legendre points, weights and derivative matrix."""
    N = n - 1
    P = np.polynomial.legendre.Legendre.basis(N)
    z = np.concatenate([[-1.0], np.sort(P.deriv().roots().real), [1.0]])
    for _ in range(3):  # Newton on P' at the interior points
        z[1:-1] -= P.deriv()(z[1:-1]) / P.deriv(2)(z[1:-1])
    p = P(z)
    w = 2.0 / (N * n * p ** 2)
    D = np.zeros((n, n))
    for i in range(n):
        for j in range(n):
            if i != j:
                D[i, j] = p[i] / (p[j] * (z[i] - z[j]))
    D[0, 0], D[-1, -1] = -N * n / 4.0, N * n / 4.0
    return z, w, D


class _Plain:
    """The operator, assembly and mask of a case's mesh in plain torch."""

    def __init__(self, c):
        n = c["lx1"]
        z, w, D = _gll(n)
        t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device="cuda")  # noqa: E731
        self.D, self.shape = t(D), _shape(c)
        q = t((z + 1.0) / 2.0 * WIDTH)

        def axis(cnt):
            return torch.arange(cnt, device="cuda")[:, None] * WIDTH + q

        full = (c["nz"], c["ny"], c["nx"], n, n, n)
        x = axis(c["nx"])[None, None, :, None, None, :].expand(full)
        y = axis(c["ny"])[None, :, None, None, :, None].expand(full)
        zz = axis(c["nz"])[:, None, None, :, None, None].expand(full)
        tau = 2.0 * math.pi
        s = DEFORM * WIDTH * torch.sin(tau * x) * torch.sin(tau * y) * torch.sin(tau * zz)
        self.xyz = [(a + s).reshape(self.shape) for a in (x, y, zz)]
        g = [self.grad(a) for a in self.xyz]  # g[a][b] = d x_a / d r_b
        cof = [[None] * 3 for _ in range(3)]  # J d r_b / d x_a
        for a in range(3):
            for b in range(3):
                a1, a2, b1, b2 = (a + 1) % 3, (a + 2) % 3, (b + 1) % 3, (b + 2) % 3
                cof[a][b] = g[a1][b1] * g[a2][b2] - g[a1][b2] * g[a2][b1]
        jac = sum(g[0][b] * cof[0][b] for b in range(3))
        w = t(w)
        w3 = w[:, None, None] * w[:, None] * w
        self.G = {(b, d): sum(cof[a][b] * cof[a][d] for a in range(3)) * w3 / jac
                  for b in range(3) for d in range(b, 3)}
        self.mass = jac * w3
        self.ids, self.cnt = _lattice(c)
        m = torch.ones(full, dtype=torch.float64, device="cuda")
        if not c.get("periodic", False):
            m[:, :, 0, :, :, 0] = 0.0
            m[:, :, -1, :, :, -1] = 0.0
        m[:, 0, :, :, 0, :] = 0.0
        m[:, -1, :, :, -1, :] = 0.0
        m[0, :, :, 0, :, :] = 0.0
        m[-1, :, :, -1, :, :] = 0.0
        self.mask = torch.ones(self.cnt, dtype=torch.float64, device="cuda")
        self.mask[self.ids[m.reshape(-1) == 0.0]] = 0.0

    def grad(self, u):
        return (torch.matmul(u, self.D.t()), torch.matmul(self.D, u),
                torch.einsum("kl,elji->ekji", self.D, u))

    def apply(self, u, h1, h2):
        u = u.reshape(self.shape)
        d = self.grad(u)
        f = [h1 * sum(self.G[min(b, q), max(b, q)] * d[q] for q in range(3)) for b in range(3)]
        return (torch.matmul(f[0], self.D) + torch.matmul(self.D.t(), f[1])
                + torch.einsum("lk,elji->ekji", self.D, f[2]) + h2 * self.mass * u)

    def gather(self, v):
        return torch.zeros(self.cnt, dtype=torch.float64, device="cuda").index_add_(
            0, self.ids, v.reshape(-1))

    def solve(self, f, h1, h2, rtol=1e-13, most=4000):
        """The assembled, masked problem by conjugate gradients, one value
        per unique node; the local values of its solution and of its
        right-hand side."""
        D2 = self.D ** 2
        diag = h1 * (torch.matmul(self.G[0, 0], D2) + torch.matmul(D2.t(), self.G[1, 1])
                     + torch.einsum("lk,elji->ekji", D2, self.G[2, 2])) + h2 * self.mass
        m = self.mask / self.gather(diag)
        r = self.gather(self.mass * f) * self.mask
        x, z, b = torch.zeros_like(r), m * r, r.clone()
        p, rz, end = z.clone(), float(torch.dot(r, z)), rtol * float(r.norm())
        for it in range(most):
            w = self.gather(self.apply(p[self.ids], h1, h2)) * self.mask
            a = rz / float(torch.dot(p, w))
            x += a * p
            r -= a * w
            if it % 10 == 9 and float(r.norm()) <= end:
                break
            z = m * r
            rz, old = float(torch.dot(r, z)), rz
            p = z + (rz / old) * p
        return [v[self.ids].reshape(self.shape) for v in (x, b)]


def exact(case, seed):
    c = case
    n = float(np.prod(_shape(c)))
    if c["kind"] == "pressure" and n > 6.0e6:
        return None  # thousands of plain iterations on a large mesh
    if c["kind"] == "step":
        boxes, out, last = _step_boxes(c), [], None
        for k, o in _step_solves(c):
            if last is None or last[0] != k:
                last = (k, _Plain(boxes[k]))
            h1, h2 = _coefs(boxes[k], seed, None)
            out.append(last[1].solve(_node_field(boxes[k], 97 * seed + o), h1, h2))
        return out
    P = _Plain(c)
    v = _node_field(c, seed)
    if c["kind"] == "dssum":
        return P.gather(P.mass * v)[P.ids].reshape(P.shape)
    h1, h2 = _coefs(c, seed, P.xyz)
    if c["kind"] == "axhelm":
        return P.apply(v, h1, h2)
    return P.solve(v, h1, h2)
