"""Tensor-grid gather with one wave per target element: meshes of so many
elements, or so few particles, that no waves share a target, with fixed and with
persistent waves (sf_persistent takes the targets from counters), exponents
compiled in (2, 3) and at run time (4).  Against the oracle, and the persistent
waves bit for bit against the fixed ones, eager and as a graph."""
import numpy as np
import pytest

from piclas_amd import mesh as M
from piclas_amd import stage
from piclas_amd import workloads as W

pytestmark = pytest.mark.gpu


def _box(shape, n):
    rng = np.random.Generator(np.random.PCG64(5))
    hi = np.array(shape) / 8.0
    mesh = M.cartesian_box(shape, hi=tuple(hi))
    pos = rng.uniform(0.0, 1.0, (n, 3)) ** 2 * hi     # crowded towards one corner
    return mesh, np.hstack([pos, W.maxwellian(rng, n, 2.0, stage.ELECTRON_MASS)]), mesh.element_of(pos)


# below and above 64 particles per element, and just above 16,384 elements
@pytest.mark.parametrize("alpha", [2, 3, 4])
@pytest.mark.parametrize("shape,n", [((17, 13, 19), 5000), ((17, 13, 19), 64 * 17 * 13 * 19 - 1), ((26, 26, 25), 40000)])
def test_one_wave_per_target(oracle_mod, shape, n, alpha):
    print("case one wave per target", shape, n, alpha, flush=True)
    mesh, part, elem = _box(shape, n)
    kw = dict(deposition=stage.DEPO_SF, sf_radius=0.19, sf_alpha=alpha)
    with stage.PICStage(mesh, 3, max_particles=n, **kw) as s:
        s.set_particles(part, elem=elem)
        s.deposition()
        PS = s.part_source()
        s.set_tuning(sf_persistent=True)
        for _ in range(2):      # (the counters start at zero each time)
            s.deposition()
            assert np.array_equal(s.part_source(), PS)
    o = oracle_mod.Oracle(mesh, 3, **kw)
    o.set_particles(part, elem=elem)
    o.deposition()
    ref = o.part_source()
    for c in (slice(0, 3), slice(3, 4)):
        assert np.abs(PS[..., c] - ref[..., c]).max() <= 1e-12 * np.abs(ref[..., c]).max()


@pytest.mark.parametrize("alpha", [2, 3, 4])
@pytest.mark.parametrize("graph", [False, True])
def test_persistent_steps(graph, alpha):
    mesh, part, elem = _box((17, 17, 17), 20000)
    print("case persistent steps graph=%s alpha=%d" % (graph, alpha), flush=True)
    out = []
    for persistent in (False, True):
        with stage.PICStage(mesh, 3, max_particles=len(part), deposition=stage.DEPO_SF, sf_radius=0.19,
                            sf_alpha=alpha) as s:
            s.set_tuning(use_graph=graph and persistent, sf_persistent=persistent)
            s.set_field(np.full((mesh.nElems, 64, 3), 10.0))
            s.set_particles(part, elem=elem)
            for _ in range(3):
                s.time_step(1e-8, 4)
                s.deposition()
                out.append(s.particles() + (s.part_source(),))
    for a, b in zip(out[:3], out[3:]):
        for u, v in zip(a, b):
            assert np.array_equal(u, v)
