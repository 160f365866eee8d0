"""Jacobi PCG where one group of shared nodes is larger than a wavefront: the
step length then comes from a kernel of its own after the assembly, not from
the packet kernel.  All corners of all elements are one degree of freedom (64
elements: its multiplicity, a power of 2, inverts exactly).
The solution's residual, formed with axhelm and dssum, meets the tolerance: the
solve stops at 1e-11 of the first residual in a norm weighted by 1/mass, whose
weights here differ by less than 1e3."""
import numpy as np
import pytest

from problems import box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 2])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("nel,lx1", [((4, 4, 4), 3), ((8, 4, 2), 4)])
def test_group_beyond_a_wavefront(gpu, nel, lx1, masked, precision):
    b = box(nel, lx1, deform=0.05)
    F = gpu.Field(lx1, b.nel)
    F.geom_from_xyz(*b.xyz())
    glo, _ = b.glo_num()
    glo = np.array(glo, dtype=np.int64).reshape(b.nel, lx1, lx1, lx1)
    corners = np.unique(glo[:, ::lx1 - 1, ::lx1 - 1, ::lx1 - 1])
    glo[np.isin(glo, corners)] = corners[0]
    F.gs_setup(glo.reshape(-1))
    mask = F.to_dev(b.face_mask()) if masked else F.zeros() + 1.0
    F.dsop(mask, "*")
    mult = F.zeros() + 1.0
    F.dssum(mult)
    mult = 1.0 / mult
    h1, h2 = F.zeros() + 1.0, F.zeros() + 2.0
    rng = np.random.default_rng(3)
    rhs = F.to_dev(rng.uniform(-1, 1, F.shape))
    rhs = rhs * mult
    u = F.zeros()
    out = F.hmholtz("VELX", u, rhs, h1, h2, mask, mult, -1e-11, 400,
                    params=gpu.default_params(istep=20, param22=0.0, restol=0.0,
                                              precision=precision))
    au = F.zeros()
    F.axhelm(au, u, h1, h2)
    F.dssum(au)
    r = (rhs - au * mask).cpu().numpy()  # rhs is assembled and masked by the solve
    e = float(np.linalg.norm(r) / np.linalg.norm(rhs.cpu().numpy()))
    print(nel, lx1, masked, precision, out["niter"], e, flush=True)
    assert out["converged"] and 0 < out["niter"] < 400
    assert e < 1e-8
    F.destroy()
