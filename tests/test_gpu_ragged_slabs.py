"""setprec, axhelm and a Jacobi solve where the last block of the element
kernels is not full (several elements share a block below lx1 8), at every kind
of default kernel (element-staged, matrix cores by element and by planes) and
for constant and varying h1 and h2, against the oracle.  Bounds: the operator
sums 3 lx1 products per node twice, 1e-13 of the largest value; the solves stop
at 1e-10, their iteration counts within 1 of the oracle's, give or take how far
those move when the right-hand side moves by one rounding (0, but 283 to 286 of
284 iterations at lx1 16 with varying h1 and h2)."""
import numpy as np
import pytest

from problems import Problem, box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kinds", ["cc", "ff", "cf"])
@pytest.mark.parametrize("lx1", [2, 3, 5, 7, 8, 10, 11, 12, 13, 16])
def test_ragged(gpu, lx1, kinds):
    b = box((3, 1, 1) if lx1 > 8 else (5, 3, 1), lx1, deform=0.05)
    P = Problem(b)
    F = gpu.box_field(b)
    h = [np.full(P.shape, v) if k == "c" else v * (1.5 + 0.5 * P.uniform_field(60 + q))
         for q, (k, v) in enumerate(zip(kinds, (0.8, 2.5)))]
    hd = [F.to_dev(a) for a in h]
    print(lx1, kinds, flush=True)
    d = F.zeros()
    F.setprec(d, *hd)
    ref = P.field.setprec(*h)
    assert np.abs(d.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max()
    u = P.uniform_field(71)
    au = F.zeros()
    F.axhelm(au, F.to_dev(u), *hd)
    ref = P.field.axhelm(u, *h)
    assert np.abs(au.cpu().numpy() - ref).max() <= 1e-13 * lx1 * np.abs(ref).max()
    if lx1 == 2:  # no free node in this box
        F.destroy()
        return
    from oracle import oracle as O

    rhs = P.bm1 * P.uniform_field(72)
    uo, _, ito, _, _ = P.field.hmholtz(rhs, *h, -1e-10, 400, O.Params(20, 0.0, 0.0, 0.0))
    x = F.zeros()
    out = F.hmholtz("VELX", x, F.to_dev(rhs), *hd, F.mask, F.mult, -1e-10, 400,
                    params=gpu.default_params(istep=20, param22=0.0, restol=0.0))
    rng, its = np.random.default_rng(lx1), [ito]
    for _ in range(4):
        r = rhs * (1.0 + np.finfo(float).eps * rng.choice([-1.0, 1.0], rhs.shape))
        its.append(P.field.hmholtz(r, *h, -1e-10, 400, O.Params(20, 0.0, 0.0, 0.0))[2])
    slack = 1 + max(its) - min(its)
    print(out["niter"], its, flush=True)
    assert min(its) - slack <= out["niter"] <= max(its) + slack
    assert np.linalg.norm(x.cpu().numpy() - uo) <= 1e-8 * np.linalg.norm(uo)
    F.destroy()
