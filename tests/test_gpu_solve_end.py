"""A solve returns only when nothing of it is left to run: the next one, on
another stream and without a synchronization by the caller, uses the same work
space and state at once, and the solution can be read there.  Each result
equals, bit for bit, that of the solve alone."""
import numpy as np
import pytest

from problems import Problem, box

pytestmark = pytest.mark.gpu

REPEATS = 12


def _alternate(jobs, solve):
    """solve(job) -> (solution, iterations), alone and then on two streams in
    turn, each solution copied on the other stream right after its solve."""
    import torch

    alone = []
    for job in jobs:
        u, its = solve(job)
        torch.cuda.synchronize()
        alone.append((u.cpu().numpy(), its))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for k in range(REPEATS * len(jobs)):
        with torch.cuda.stream(streams[k % 2]):
            u, its = solve(jobs[k % len(jobs)])
        with torch.cuda.stream(streams[(k + 1) % 2]):
            got.append((u, u.clone(), its))
    torch.cuda.synchronize()
    for k, (u, copy, its) in enumerate(got):
        ref, ref_its = alone[k % len(jobs)]
        assert its == ref_its
        assert np.array_equal(u.cpu().numpy(), ref), k
        assert np.array_equal(copy.cpu().numpy(), ref), k


@pytest.mark.parametrize("fused", [True, False])
def test_cggo(gpu, fused):
    # weights that do not sum to 1 per node take the general path
    P = Problem(box((4, 3, 3), 6, deform=0.1))
    F = gpu.box_field(P.box)
    h1, h2, mult = F.zeros() + 1.0, F.zeros() + 3.0, F.mult * (1.0 if fused else 0.5)
    prm = gpu.default_params(istep=20, param22=0.0, restol=0.0)
    jobs = []
    for k, tol in enumerate((-1e-9, -1e-3, -1e-6)):
        f = P.field.dssum(P.bm1 * P.uniform_field(70 + k)) * P.mask
        jobs.append((F.to_dev(f), tol))

    def solve(job):
        u = F.zeros()
        out = F.cggo(u, job[0], h1, h2, F.mask, mult, job[1], 200, params=prm)
        return u, out["niter"]

    _alternate(jobs, solve)
    F.destroy()


@pytest.mark.parametrize("fused", [True, False])
def test_flexible_cg(gpu, fused):
    # a pressure mask that is not the hierarchy's fine mask takes the general
    # path: here the hierarchy has Neumann faces on top, the mask Dirichlet ones
    b = box((4, 3, 3), 6, deform=0.1)
    P = Problem(b)
    F = gpu.box_field(b)
    fbc = b.fast_bc()
    top = (np.arange(b.nel) // (b.nelx * b.nely)) == b.nelz - 1
    fbc[top, 5] = 2  # Neumann
    F.h1mg_setup(b.fast_bc() if fused else fbc, b.vertex, *b.xyz())
    h1, h2 = F.zeros() + 1.0, F.zeros()
    jobs = [(F.to_dev(P.field.dssum(P.bm1 * P.uniform_field(80 + k)) * P.mask), tol)
            for k, tol in enumerate((-1e-9, -1e-2, -1e-5))]

    def solve(job):
        u = job[0].clone()
        out = F.hmh_flex_cg(u, h1, h2, F.mult, 60,
                            params=gpu.default_params(istep=20, param21=job[1], param42=2))
        return u, out["niter"]

    _alternate(jobs, solve)
    F.destroy()


@pytest.mark.parametrize("kind", ["hmholtz", "mixed", "noalloc", "batch"])
def test_zero_right_hand_side(gpu, kind):
    # the solution 0 is there when the call returns, read on another stream
    import torch

    F = gpu.box_field(box((10, 10, 10), 8))
    h1, h2, zero = F.zeros() + 1.0, F.zeros() + 3.0, F.zeros()
    prm = gpu.default_params(istep=20, precision=2 if kind == "mixed" else 0)
    us = [F.zeros() + 1.0 for _ in range(20)]
    rhs = zero.clone()
    B = gpu.Batch([F, F]) if kind == "batch" else None
    q = [dict(u=None, rhs=rhs, h1=h1, h2=h2, mask=F.mask, mult=F.mult, tli=-1e-8),
         dict(u=F.zeros(), rhs=F.mass()[0] * F.mask, h1=h1, h2=h2, mask=F.mask, mult=F.mult,
              tli=-1e-8)]
    streams, copies = [torch.cuda.Stream(), torch.cuda.Stream()], []
    torch.cuda.synchronize()
    for u in us:
        with torch.cuda.stream(streams[0]):
            if kind == "batch":
                q[0]["u"] = u
                niter = B.hmholtz(q, 900, params=prm)[0][0]["niter"]
            elif kind == "noalloc":
                niter = F.cggo(u, rhs, h1, h2, F.mask, F.mult, -1e-8, 900, params=prm,
                               noalloc=True)["niter"]
            else:
                niter = F.hmholtz("VELX", u, rhs, h1, h2, F.mask, F.mult, -1e-8, 900,
                                  params=prm)["niter"]
        assert niter == 0
        with torch.cuda.stream(streams[1]):
            copies.append(u.clone())
    torch.cuda.synchronize()
    assert all(bool((c == 0.0).all()) for c in copies)
    if B is not None:
        B.destroy()
    F.destroy()
