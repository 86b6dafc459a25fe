"""Device memory of a handle per particle of its capacity: the particle arrays
and their scratch (337 bytes), and for the shape function two record planes and
the block boxes (65)."""
import pytest
import torch

from piclas_amd import mesh as M
from piclas_amd import stage

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,kw,want", [(3, dict(deposition=stage.DEPO_NONE), 337),
                                       (2, dict(deposition=stage.DEPO_SF, sf_radius=0.3), 337 + 65),
                                       (3, dict(deposition=stage.DEPO_SF, sf_radius=0.3), 337 + 65)])
def test_bytes_per_particle(N, kw, want):
    cap = 16_000_000
    print("case handle memory", N, kw, flush=True)
    mesh = M.cartesian_box((4, 4, 4))
    with stage.PICStage(mesh, N, max_particles=1, **kw):     # (code and queues of the device)
        pass
    free = torch.cuda.mem_get_info()[0]
    with stage.PICStage(mesh, N, max_particles=cap, **kw):
        taken = free - torch.cuda.mem_get_info()[0]
    # some hundred arrays, each rounded up to 64 KB at least and to 2 MB where it is larger
    assert taken <= want * cap + 48 * 2 ** 21 + 100 * 2 ** 16, taken / cap
