"""Steps of few particles: the push takes its movers through the face walk
itself, and k_dest scans the element counts.  Fast particles that cross several
elements in a step, out of two open walls and around the other directions, at
element counts on both sides of the scan's limit and particle counts that do
not fill the last wave, eager and as a graph.  Bit for bit what the staged calls
give, which keep the movers' list and run the walk in its own kernel; owners and
removals are the oracle's (the field times dt^2 makes round-off grow about
fivefold a step, so positions are not held to the bars of one step).
"""
import numpy as np
import pytest

from piclas_amd import mesh as M, stage, workloads as W
from test_gpu_parity import deformed_box, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("shape,N,n", [((3, 3, 3), 3, 1), ((3, 4, 5), 1, 1000), ((8, 8, 16), 3, 20011),
                                       ((5, 5, 41), 2, 20011)])
def test_walk_and_scan(oracle_mod, shape, N, n, graph):
    m = M.cartesian_box(shape, periodic=(False, True, True))
    rng = np.random.default_rng(20261206)
    x = rng.uniform(0.0, 1.0, (n, 3))
    v = rng.normal(0.0, 1e6, (n, 3))
    xg = W.dof_positions(m, N)
    E = W.fourier_field(xg.reshape(-1, 3), (1.0, 1.0, 1.0), 4, 1e3, rng).reshape(xg.shape)
    w = W.Workload("small", m, N, np.hstack([x, v]), m.element_of(x), np.ones(n, np.int32), E,
                   (0, 0, 0, 0, 0, 0.01), stage.DEPO_CVWM, 0.0, 2, 1e-7, 4, (-W.ELEMENTARY_CHARGE,),
                   (W.ELECTRON_MASS,), (1e3,))
    s, o = run_pair(oracle_mod, w, 0)
    s.set_tuning(use_graph=graph)
    s.time_step(w.dt, 4)
    o.time_step(w.dt, 4)
    s.deposition()
    t, _ = run_pair(oracle_mod, w, 4, staged=True)
    ps, el, ins = s.particles()
    _, oel, oins = o.particles()
    assert np.array_equal(ins, oins) and np.array_equal(el[ins], oel[ins])
    for a, b in zip((ps, el, ins), t.particles()):
        assert np.array_equal(a, b)
    assert np.array_equal(s.part_source(), t.part_source())
    s.close()
    t.close()


@pytest.mark.parametrize("nx", [3, 5, 21])
def test_arrivals_in_caller_order(oracle_mod, nx):
    """Many arrivals per element on general elements, where a wave (up to 8,192 elements) or 8 lanes order them:
    the same bits in every run, though the atomics hand out the places in any order."""
    n = max(40000, 8 * nx ** 3)
    w = deformed_box(W.thermal_cube(nx=nx, ppc=-(-n // nx ** 3), steps=2))
    out = []
    for _ in range(3):
        with stage.PICStage(w.mesh, w.N, max_particles=len(w.PartState), **W.stage_kwargs(w)) as s:
            s.set_field(0.0 * w.E)
            s.set_particles(w.PartState, elem=w.elem, species=w.species)
            before = s.particles()[1]
            s.time_step(3000 * w.dt, 2)   # a thermal step of 0.2
            s.deposition()
            out.append(s.particles() + (s.part_source(),))
    assert (out[0][1] != before).sum() > len(before) // 4
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a, b)
