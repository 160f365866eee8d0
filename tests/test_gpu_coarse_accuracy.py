"""The direct coarse solver where its problem is ill-conditioned: refined on
stretched elements, and not used at all where the problem is singular to
rounding (the AMG-preconditioned CG takes it, as for problems that are too
large)."""
import numpy as np
import pytest

from problems import box
from test_gpu_hsmg import build, host, l2rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel,lengths", [
    ((13, 15, 14), (1.0, 1.0, 0.01)),  # 1:100, parts and a separator
    ((12, 11, 13), (1e-3, 1.0, 1e-3)),  # rods of 1:1000, one inverse, refined
    ((13, 15, 14), (1.0, 1.0, 1e-3)),  # plates of 1:1000, parts, refined
])
def test_stretched_neumann(gpu, nel, lengths):
    # against the oracle's factor: either carries eps times the condition number
    # of its problem, 1e6 to 1e9 here
    P, mg, F = build(gpu, dict(nel=nel, lx1=4, lengths=lengths, deform=0.05, neumann_all=True))
    rng = np.random.default_rng(5)
    r = P.field.dssum(P.bm1 * rng.standard_normal(P.shape))
    r -= r.sum() / r.size  # what a pressure solve hands the V-cycle
    zo = mg.solve(r.copy())
    zd = F.zeros()
    F.h1mg_solve(zd, F.to_dev(r))
    e = l2rel(host(zd), zo)
    print(f"[coarse accuracy] {nel} {lengths} rel L2 = {e:.3e}", flush=True)
    assert F.h1mg_info()["crs_avg_iters"] == 0.0
    assert e < 1e-7
    F.destroy()


@pytest.mark.parametrize("nel", [(12, 12, 12), (10, 12, 13), (16, 12, 13)])
def test_second_region_without_dirichlet_face(gpu, nel):
    """A box cut in two, the right half with Neumann faces only: the coarse
    matrix is singular, its last pivot rounding of either sign."""
    b = box(nel, 4)
    F = gpu.box_field(b)
    ix = np.arange(b.nel) % b.nelx
    right = ix >= b.nelx // 2
    vertex, fbc = b.vertex.reshape(b.nel, 8).copy(), b.fast_bc()
    vertex[right] += vertex.max() + 1
    fbc[right] = np.where(fbc[right] == 1, 2, fbc[right])
    fbc[ix == b.nelx // 2, 0] = 2
    fbc[ix == b.nelx // 2 - 1, 1] = 2
    try:
        F.h1mg_setup(fbc, vertex, *b.xyz())
    except gpu.NekAmdError as e:  # the AMG set-up refuses what it finds indefinite
        print(f"[coarse accuracy] cut {nel} {e}", flush=True)
        assert "not SPD" in str(e)
    else:
        F.h1mg_solve(F.zeros(), F.mass()[0] * F.mask)
        info = F.h1mg_info()
        print(f"[coarse accuracy] cut {nel} {info}", flush=True)
        assert info["crs_avg_iters"] > 0.0
    F.destroy()
