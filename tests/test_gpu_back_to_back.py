"""Solves of one mesh, one after the other on alternating streams with no
synchronization by the caller: a solve returns only when nothing of it is
left to run in the mesh's work space, although its last kernels run after the
report that ends it.  Every result equals, bit for bit, that of the solve
alone; maxit 1 ends on the iteration limit, a loose tolerance on the first
exit test."""
import numpy as np
import pytest

from problems import Problem, box

pytestmark = pytest.mark.gpu

LIMITS = [(200, -1e-9), (1, -1e-9), (200, 1e3)]  # maxit, tolerance


@pytest.mark.parametrize("kind", ["jacobi", "mixed", "batch", "gmres", "flex-mixed"])
def test_alternating_streams(gpu, kind):
    import torch

    b = box((4, 3, 3), 6, deform=0.1)
    P = Problem(b)
    F = gpu.box_field(b)
    F.h1mg_setup(b.fast_bc(), b.vertex, *b.xyz())
    h1, h2 = F.zeros() + 1.0, F.zeros() + 3.0
    name = "PRES" if kind in ("gmres", "flex-mixed") else "VELX"
    B = gpu.Batch([F, F]) if kind == "batch" else None

    def solve(rhs, maxit, tol):
        if B is not None:
            qs = [dict(u=F.zeros(), rhs=rhs.clone(), h1=h1, h2=h2 * (k + 1), mask=F.mask,
                       mult=F.mult, tli=tol) for k in range(2)]
            outs, _ = B.hmholtz(qs, maxit, params=gpu.default_params(
                istep=20, param22=0.0, restol=0.0))
            return [q["u"] for q in qs], [o["niter"] for o in outs]
        prm = gpu.default_params(istep=20, param22=0.0, restol=0.0,
                                 param42=2 if kind == "flex-mixed" else 0,
                                 param21=tol, precision=2 if "mixed" in kind else 0)
        u = F.zeros()
        out = F.hmholtz(name, u, rhs.clone(), h1, h2, F.mask, F.mult, tol, maxit, params=prm)
        return [u], [out["niter"]]

    rhs = [F.to_dev(P.bm1 * P.uniform_field(50 + k)) for k in range(3)]
    jobs = [(r, *lim) for r in rhs for lim in LIMITS]
    alone = []
    for job in jobs:
        us, its = solve(*job)
        torch.cuda.synchronize()
        alone.append(([u.cpu().numpy() for u in us], its))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for k, job in enumerate(jobs):
        with torch.cuda.stream(streams[k % 2]):
            got.append(solve(*job))
    torch.cuda.synchronize()
    for k, ((us, its), (ref, ref_its)) in enumerate(zip(got, alone)):
        print(kind, k, its, ref_its, flush=True)
        assert its == ref_its
        for u, e in zip(us, ref):
            assert np.array_equal(u.cpu().numpy(), e)
    if B is not None:
        B.destroy()
    F.destroy()
