"""Hand-over of particles that fill few elements of a mesh: the segment offsets
of long runs of empty elements before, between and after them.  Exact."""
import numpy as np
import pytest

from piclas_amd import mesh as M
from piclas_amd import stage

pytestmark = pytest.mark.gpu

SHAPE = (67, 64, 32)      # 137,216 elements: three digits of the sort


@pytest.fixture(scope="module")
def mesh():
    return M.cartesian_box(SHAPE)


@pytest.mark.parametrize("n", [0, 1, 255, 5000])
@pytest.mark.parametrize("where", ["first", "middle", "last", "ends", "none"])
def test_clustered(mesh, where, n):
    print("case clustered hand-over", where, n, flush=True)
    ne = mesh.nElems
    rng = np.random.Generator(np.random.PCG64(2))
    cells = {"first": [0], "middle": [ne // 2 + 3], "last": [ne - 1], "ends": [0, ne - 1], "none": [0]}[where]
    cell = rng.choice(cells, n)
    ijk = np.stack([cell % SHAPE[0], cell // SHAPE[0] % SHAPE[1], cell // (SHAPE[0] * SHAPE[1])], 1)
    part = np.hstack([(ijk + rng.uniform(0.1, 0.9, (n, 3))) / np.array(SHAPE), rng.normal(size=(n, 3))])
    elem = (cell + 1).astype(np.int32)
    if where == "none":   # outside, so in no element
        part[:, 0] += 2.0
        elem[:] = 0
    with stage.PICStage(mesh, 1, max_particles=max(n, 1), deposition=stage.DEPO_NONE) as s:
        s.set_particles(part, elem=elem)
        got, el, inside = s.particles()
        _, pi = s.particle_data()
    assert np.array_equal(got, part) and np.array_equal(el, elem) and np.array_equal(inside, elem > 0)
    count = np.bincount(elem, minlength=ne + 1)[1:]
    assert np.array_equal(pi[:, 1], np.cumsum(count)) and np.array_equal(pi[:, 0], np.cumsum(count) - count)
