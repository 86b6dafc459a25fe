"""Start guess 2 in waves of one element: the nearest Gauss point is found from
one minimum of keys (squared distance with the point's place in its last bits).
Degrees at the edges of the scalar chunks, at the smallest and at the largest
number of points; half of the particles start at rest at the elements' middles, so
that the ions meet points that are almost equally near.  The bars are those of the
other RefMapping tests.
"""
import dataclasses

import numpy as np
import pytest

from piclas_amd import workloads as W
from test_gpu_parity import run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2, 4, 7])
def test_dense_refmapping_degrees(oracle_mod, N):
    w = W.annulus_plasma(shape=(2, 8, 2), n_total=12000, dt=2e-9)
    xg = W.curved_dof_positions(w.mesh, N)
    E = 1e3 * np.cos(2.0 * xg[..., [1, 2, 0]])
    mid = W.curved_dof_positions(w.mesh, 2)[:, 13]          # the middle of the 27 points of degree 2
    ps = w.PartState.copy()
    ps[::2, :3] = mid[np.arange(len(ps[::2])) % len(mid)]
    ps[::2, 3:] = 0.0
    w = dataclasses.replace(w, N=N, E=E, PartState=ps)
    s, o = run_pair(oracle_mod, w, 3)
    ps, el, ins = s.particles()
    ops, oel, oins = o.particles()
    assert np.array_equal(ins, oins)
    assert np.array_equal(el[ins], oel[ins])
    assert np.abs(ps[ins, :3] - ops[ins, :3]).max() <= 1e-12
    vmax = np.abs(ops[ins, 3:]).max()
    assert np.abs(ps[ins, 3:] - ops[ins, 3:]).max() <= 1e-12 * vmax
    assert np.abs(s.part_pos_ref()[ins] - o.part_pos_ref()[ins]).max() <= 1e-12
    PS, oPS = s.part_source(), o.part_source()
    assert np.abs(PS - oPS).max() <= 1e-12 * np.abs(oPS).max()
    s.close()
