"""The V-cycle on one stream (up to 2e6 local nodes) and on three: pressure
solves on both sides of the line, their solutions checked by the true residual
formed with axhelm and dssum (the solvers stop at 1e-9 of the first residual in
a norm whose weights differ by less than 100 on these meshes)."""
import numpy as np
import pytest

from problems import box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("param42", [0, 2])
@pytest.mark.parametrize("nel", [(6, 5, 4), (20, 20, 10)])
def test_pressure_residual(gpu, nel, param42):
    b = box(nel, 8, deform=0.05)
    F = gpu.box_field(b, multigrid=True)
    rng = np.random.default_rng(9)
    f = F.to_dev(rng.uniform(-1, 1, F.shape))
    h1, h2 = F.zeros() + 1.0, F.zeros()
    rhs = f.clone()
    u = F.zeros()
    out = F.hmholtz("PRES", u, rhs, h1, h2, F.mask, F.mult, -1e-9, 100,
                    params=gpu.default_params(param42=param42, param21=-1e-9))
    au = F.zeros()
    F.axhelm(au, u, h1, h2)
    F.dssum(au)
    F.dssum(f)
    r = f * F.mask - au * F.mask
    e = float((r * r * F.mult).sum().sqrt() / (f * f * F.mask * F.mult).sum().sqrt())
    print(nel, param42, out["niter"], e, flush=True)
    assert out["converged"] and 0 < out["niter"] < 60
    assert e < 1e-7
    F.destroy()
