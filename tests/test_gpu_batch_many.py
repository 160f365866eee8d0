"""The largest batch (64 solves, the host taking them in turn): every solve's
iteration count and solution equal, bit for bit, those of nkd_hmholtz."""
import numpy as np
import pytest

from problems import box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 2])
def test_sixty_four_solves(gpu, precision):
    import torch

    meshes = [gpu.box_field(box((3, 2, 2), 6, deform=0.1)), gpu.box_field(box(2, 5))]
    prm = gpu.default_params(istep=20, param22=0.0, restol=0.0, precision=precision)
    fields, solves, ref = [], [], []
    for k in range(64):
        F = meshes[k % 2]
        g = torch.Generator(device="cuda")
        g.manual_seed(k)
        v = torch.rand(F.shape, generator=g, dtype=torch.float64, device="cuda")
        q = dict(rhs=F.mass()[0] * v, h1=F.zeros() + 1.0, h2=F.zeros() + 0.5 * k, mask=F.mask,
                 mult=F.mult, tli=-1e-9 if k % 3 else -1e-3)
        u = F.zeros()
        out = F.hmholtz("VELX", u, q["rhs"].clone(), q["h1"], q["h2"], F.mask, F.mult, q["tli"],
                        900, params=prm)
        fields.append(F)
        solves.append(dict(q, u=F.zeros()))
        ref.append((u.cpu().numpy(), out["niter"]))
    B = gpu.Batch(fields)
    outs, slowest = B.hmholtz(solves, 900, params=prm)
    torch.cuda.synchronize()
    print(f"[batch many] precision {precision}: {sorted({o['niter'] for o in outs})} iterations, "
          f"{slowest} enqueued", flush=True)
    for q, out, (u, niter) in zip(solves, outs, ref):
        assert out["niter"] == niter
        assert np.array_equal(q["u"].cpu().numpy(), u)
    B.destroy()
    for F in meshes:
        F.destroy()
