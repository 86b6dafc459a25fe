"""Start guess 2 where two Gauss points are equally near to some ulp: a particle
gets the same start, and so the same bits of xi, whether its wave holds one
element (scalar loads, one minimum of keys) or several.

The particles move in their z-plane near the columns of Gauss points of the lowest
layer of elements, a few ulp about the middle of two points of a column.  They are stepped
128 to an element, so that every wave of 64 holds one, and 4 to an element, so
that every wave holds sixteen."""
import numpy as np
import pytest

from piclas_amd import stage
from piclas_amd import workloads as W

pytestmark = pytest.mark.gpu


def _step(w, E, state, elem):
    with stage.PICStage(w.mesh, w.N, max_particles=len(state), **W.stage_kwargs(w)) as s:
        s.set_field(E)
        s.set_particles(state, elem=elem, species=np.ones(len(state), np.int32))
        s.time_step(w.dt, 1)
        ps, el, _ = s.particles()
        assert np.array_equal(el, elem)
        return np.hstack([ps, s.part_pos_ref()])


@pytest.mark.parametrize("N", [3, 4, 7])
def test_uniform_and_mixed_waves(N):
    w = W.annulus_plasma(shape=(2, 8, 2), n_total=100, dt=2e-9)
    w.N = N
    print("case start ties N=%d" % N, flush=True)
    n1 = N + 1
    xg = W.curved_dof_positions(w.mesh, N).reshape(w.mesh.nElems, n1, n1, n1, 3)      # k, j, i
    low = np.flatnonzero(xg[..., 2].max((1, 2, 3)) < 0.5)
    assert len(low) == 16
    rng = np.random.Generator(np.random.PCG64(17))
    per = 128
    state, elem = np.zeros((len(low), per, 6)), np.zeros((len(low), per), np.int32)
    for a, e in enumerate(low):
        i, j, k = rng.integers(0, n1, per), rng.integers(0, n1, per), rng.integers(0, n1 - 1, per)
        A, B = xg[e, k, j, i], xg[e, k + 1, j, i]
        p = 0.5 * (A + B)
        p[:, :2] += 0.002 * rng.uniform(-1.0, 1.0, (per, 2))
        p[:, 2] += np.arange(per) % 33 * np.spacing(p[:, 2]) - 16 * np.spacing(p[:, 2])
        state[a, :, :3], elem[a] = p, e + 1
        state[a, :, 3:5] = 5e4 * rng.uniform(-1.0, 1.0, (per, 2))     # some 1e-4 of a step of 2e-9
    E = np.zeros((w.mesh.nElems, n1 ** 3, 3))
    uniform = _step(w, E, state.reshape(-1, 6), elem.ravel()).reshape(len(low), per, 9)
    for q in range(0, per, 4):
        mixed = _step(w, E, state[:, q:q + 4].reshape(-1, 6), elem[:, q:q + 4].ravel()).reshape(len(low), 4, 9)
        assert np.array_equal(mixed, uniform[:, q:q + 4]), q
