"""Most particles leave their element: the mover lists of the push, their walk by
64 workgroups and more, and the re-sort of that many arrivals, on elements with
bilinear faces.  One force-free step, so positions and owners are held to the
bars of the other parity tests."""
import dataclasses

import numpy as np
import pytest

from piclas_amd import stage
from piclas_amd import workloads as W
from test_gpu_parity import compare, deformed_box, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("staged", [False, True])
@pytest.mark.parametrize("ppc", [1, 131, 140, 400])      # 125, 16,375, 17,500 and 50,000 particles
def test_most_particles_move_on(oracle_mod, ppc, staged):
    w = deformed_box(W.thermal_cube(nx=5, ppc=ppc, steps=1))
    w = dataclasses.replace(w, E=0.0 * w.E, external_field=(0.0,) * 6, dt=0.4 / 6e5)      # a thermal step of two elements
    s, o = run_pair(oracle_mod, w, 1, staged=staged, sf_radius=w.sf_radius)
    assert compare(s, o, 1.0) == 0
    s.close()


def test_more_than_a_row_of_workgroups():
    """150,120 particles (ten workgroups per list): the fused step against the staged calls, bit for bit."""
    w = deformed_box(W.thermal_cube(nx=6, ppc=695, steps=1))
    print("case movers n=%d" % len(w.PartState), flush=True)
    out = []
    for staged in (False, True):
        with stage.PICStage(w.mesh, w.N, max_particles=len(w.PartState), **W.stage_kwargs(w)) as s:
            s.set_field(0.0 * w.E)
            s.set_particles(w.PartState, elem=w.elem, species=w.species)
            if staged:
                s.interpolate_field_to_particle()
                s.push_boris_leapfrog(0.3 / 6e5)
                s.perform_tracking()
            else:
                s.time_step(0.3 / 6e5, 1)
            s.deposition()
            out.append(s.particles() + (s.part_source(),))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
