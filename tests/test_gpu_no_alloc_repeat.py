"""nkd_cggo_noalloc called again and again takes no memory: neither device
memory nor host memory that the GPU can reach (each allocation of that kind
is a mapping of its own in /proc/self/maps)."""
import pytest

from problems import box

pytestmark = pytest.mark.gpu


def _mappings():
    with open("/proc/self/maps") as f:
        return sum(1 for _ in f)


def test_noalloc_takes_no_memory(gpu):
    import torch

    F = gpu.box_field(box(2, 4))
    f = F.mass()[0] * F.mask
    h1, h2, x = F.zeros() + 1.0, F.zeros() + 10.0, F.zeros()

    def solves(count):
        for _ in range(count):
            F.cggo(x, f, h1, h2, F.mask, F.mult, -1e-8, 20, noalloc=True)

    solves(20)
    maps, free = _mappings(), torch.cuda.mem_get_info()[0]
    solves(200)
    grown = _mappings() - maps
    print(f"[noalloc] mappings {maps} -> +{grown}, device bytes "
          f"{free - torch.cuda.mem_get_info()[0]}", flush=True)
    assert grown < 20  # (one per call where a call allocates)
    assert torch.cuda.mem_get_info()[0] >= free
    F.destroy()
