"""pic_adjoint on tensor grids of affine elements (factored position
derivative, affine interpolation) against the general path on the same mesh,
selected by PIC_SF_CARTESIAN=0 and PIC_AFFINE=0: exponents 2 to 4, step counts
that do and do not divide into the checkpoint interval.

Bar: the two differ in the order of sums of at most a few thousand terms per
gradient entry over at most 5 steps, some 1e-14 of the largest entry: 1e-11."""
import numpy as np
import pytest

from piclas_amd import adjoint as A
from piclas_amd import stage

pytestmark = pytest.mark.gpu


def _gradients(w, G, K, every):
    with stage.PICStage(w.mesh, w.N, max_particles=len(w.PartState), deposition=w.deposition, sf_radius=w.sf_radius,
                        sf_alpha=w.sf_alpha, charge=w.charge, mass=w.mass, mpf=w.mpf,
                        external_field=(0, 0, 0, 1e-4, -2e-4, 3e-4)) as s:
        s.set_field_operator(G)
        s.set_particles(w.PartState, elem=w.elem, species=w.species)
        loss, gx, gv = s.adjoint(w.dt, K, every)
        return loss, gx, gv, s.particles()[0], s.part_source()


@pytest.mark.parametrize("alpha,n_el,n,K,every", [(2, 5, 63, 1, 1), (3, 5, 4001, 5, 2), (4, 6, 3000, 3, 3),
                                                  (3, 7, 9000, 4, 10)])
def test_adjoint_paths_agree(monkeypatch, alpha, n_el, n, K, every):
    w, _ = A.landau_box(n_el=n_el, n_part=n, steps=K, sf_alpha=alpha)
    G = A.periodic_poisson_operator(w.mesh)
    print("case adjoint paths", alpha, n_el, n, K, every, flush=True)
    fast = _gradients(w, G, K, every)
    monkeypatch.setenv("PIC_SF_CARTESIAN", "0")
    monkeypatch.setenv("PIC_AFFINE", "0")
    ref = _gradients(w, G, K, every)
    assert abs(fast[0] - ref[0]) <= 1e-11 * abs(ref[0])
    for a, b in zip(fast[1:], ref[1:]):
        assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()
