"""RefMapping boundary tracking of long lists: up to 65,536 particles go to the
resident waves, more to all workgroups in full waves, more than 262,144 in
several passes; and steps of 2^20 particles and more.

Every particle starts within a tenth of an element of a wall or a z side and
crosses it in the step, so that the list holds all of them: half are wrapped by
the periodic z sides, half leave through the open walls.  Bars as in the other
boundary tests: inside flags and owners exact, positions 1e-12."""
import numpy as np
import pytest

from piclas_amd import mesh as M
from piclas_amd import stage
from piclas_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65536, 65537, 270001])
def test_long_lists(oracle_mod, n):
    print("case boundary list", n, flush=True)
    m = M.annulus((3, 12, 3))
    rng = np.random.Generator(np.random.PCG64(21))
    th, z = 2 * np.pi * rng.uniform(0.0, 1.0, n), rng.uniform(0.05, 0.95, n)
    r = rng.uniform(0.6, 0.9, n)
    part = np.zeros((n, 6))
    kind = np.arange(n) % 4
    z[kind == 0], part[kind == 0, 5] = 0.99, 1.0
    z[kind == 1], part[kind == 1, 5] = 0.01, -1.0
    r[kind == 2], r[kind == 3] = 0.98, 0.52
    out = np.where(kind == 2, 1.0, np.where(kind == 3, -1.0, 0.0))
    part[:, 0], part[:, 1], part[:, 2] = r * np.cos(th), r * np.sin(th), z
    part[:, 3], part[:, 4] = out * np.cos(th), out * np.sin(th)
    kw = dict(tracking=stage.TRACK_REFMAPPING, refmapping_guess=2, charge=(0.0,), mass=(1.0,), mpf=(1.0,))
    o = oracle_mod.Oracle(m, 1, **kw)
    o.set_field(np.zeros((m.nElems, 8, 3)))
    o.set_particles(part, elem=np.zeros(n, np.int32))
    assert o.locate() == 0
    o.time_step(0.05, 1)
    ops, oel, oins = o.particles()
    with stage.PICStage(m, 1, max_particles=n, **kw) as s:
        s.set_field(np.zeros((m.nElems, 8, 3)))
        s.set_particles(part, elem=None, species=np.ones(n, np.int32))
        s.time_step(0.05, 1)
        ps, el, ins = s.particles()
    assert np.array_equal(ins, kind < 2) and np.array_equal(ins, oins)
    assert np.array_equal(el[ins], oel[ins])
    assert np.abs(ps[:, :3] - ops[:, :3]).max() <= 1e-12


def test_a_million_particles():
    """2^20 + 77 particles against the same particles in two halves: a particle's step does not depend on the others."""
    w = W.annulus_plasma(shape=(8, 32, 8), n_total=2 ** 20 + 77, dt=2e-9)
    n = len(w.PartState)
    print("case RefMapping", n, flush=True)
    kw = W.stage_kwargs(w)
    kw["deposition"] = stage.DEPO_NONE

    def steps(sel):
        with stage.PICStage(w.mesh, w.N, max_particles=n, **kw) as s:
            s.set_field(w.E)
            s.set_particles(w.PartState[sel], species=w.species[sel])
            s.time_step(w.dt, 2)
            return s.particles() + (s.part_pos_ref(),)

    ps, el, ins, ref = steps(slice(None))
    assert (~ins).sum() > 100
    for sel in (slice(0, None, 2), slice(1, None, 2)):
        hps, hel, hins, href = steps(sel)
        assert np.array_equal(hins, ins[sel]) and np.array_equal(hel, el[sel])
        assert np.abs(hps[:, :3] - ps[sel, :3]).max() <= 1e-12
        assert np.abs(hps[:, 3:] - ps[sel, 3:]).max() <= 1e-12 * np.abs(ps[:, 3:]).max()
        assert np.abs(href[hins] - ref[sel][hins]).max() <= 1e-12
