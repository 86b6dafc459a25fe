"""pic_set_particles and pic_get_particles order the particles on the device:
counts around the sort's tiles of 4096 keys, meshes of one to three digits of
element ids, particles outside, elements given, missing or half given,
refused calls.  Everything is compared exactly."""
import numpy as np
import pytest

from piclas_amd import mesh as M
from piclas_amd import stage

pytestmark = pytest.mark.gpu


def _particles(n, hi, seed, spread):
    rng = np.random.Generator(np.random.PCG64(seed))
    pos = rng.uniform(0.0, 1.0, (n, 3)) ** 3 * hi * spread     # crowded towards one corner, some outside
    return np.hstack([pos, rng.normal(size=(n, 3)) * 1e5]), rng.integers(1, 4, n).astype(np.int32)


@pytest.mark.parametrize("shape,n", [((3, 3, 3), 0), ((3, 3, 3), 1), ((1, 1, 1), 5000), ((5, 7, 4), 4095),
                                     ((5, 7, 4), 4096), ((16, 16, 1), 4097), ((17, 16, 1), 12289), ((9, 31, 10), 70001),
                                     ((42, 41, 43), 30011)])
@pytest.mark.parametrize("given", ["all", "none", "half"])
def test_round_trip(shape, n, given):
    print("case hand-over", shape, n, given, flush=True)
    hi = np.array(shape) / 8.0
    mesh = M.cartesian_box(shape, hi=tuple(hi), periodic=(False, False, False))
    part, species = _particles(n, hi, 3, 1.0 if given == "all" else 1.2)
    isnew = (np.arange(n) % 3 == 0).astype(np.uint8)
    owner = np.where((part[:, :3] < hi).all(1), mesh.element_of(part[:, :3]), 0).astype(np.int32)
    elem = {"all": owner, "none": None, "half": np.where(np.arange(n) % 2 == 0, owner, 0).astype(np.int32)}[given]
    with stage.PICStage(mesh, 1, max_particles=max(n, 1), charge=(1.0, -1.0, 0.0), mass=(1e-26, 1e-27, 1e-26),
                        mpf=(1.0, 1.0, 1.0)) as s:
        s.set_particles(part, elem=elem, species=species, is_new=isnew)
        got, el, inside = s.particles()
        assert np.array_equal(got, part) and np.array_equal(el, owner) and np.array_equal(inside, owner > 0)
        pd, pi = s.particle_data()
        order = np.argsort(np.where(owner > 0, owner, shape[0] * shape[1] * shape[2] + 1), kind="stable")
        order = order[:int((owner > 0).sum())]
        assert np.array_equal(pd, np.hstack([part, species[:, None].astype(float)])[order])
        assert np.array_equal(pi[:, 1] - pi[:, 0], np.bincount(owner, minlength=mesh.nElems + 1)[1:])
        if n == 0:
            return
        # a refused call leaves the particles as they are
        for bad in (dict(elem=np.where(np.arange(n) == n - 1, mesh.nElems + 1, owner).astype(np.int32), species=species),
                    dict(elem=np.where(np.arange(n) == 0, -1, owner).astype(np.int32), species=species),
                    dict(elem=owner, species=np.where(np.arange(n) == n // 2, 4, species).astype(np.int32)),
                    dict(elem=owner, species=np.where(np.arange(n) == n // 2, 0, species).astype(np.int32))):
            with pytest.raises(stage.StageError, match="out of range"):
                s.set_particles(part[::-1].copy(), is_new=isnew, **bad)
            again = s.particles()
            assert np.array_equal(again[0], part) and np.array_equal(again[1], owner)
