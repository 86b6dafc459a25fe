"""pic_adjoint with and without the fields of its forward steps kept
(PIC_ADJOINT_FIELD_BYTES): a limit of nothing and one that is reached midway,
which gives back what was taken.  The second deposition of a step repeats the
first one's sums in their order, so everything agrees bit for bit."""
import numpy as np
import pytest
import torch

from piclas_amd import adjoint as A
from piclas_amd import stage

pytestmark = pytest.mark.gpu

LIMIT = "PIC_ADJOINT_FIELD_BYTES"


def _stage(w, G):
    s = stage.PICStage(w.mesh, w.N, max_particles=len(w.PartState), deposition=w.deposition, sf_radius=w.sf_radius,
                       sf_alpha=w.sf_alpha, charge=w.charge, mass=w.mass, mpf=w.mpf,
                       external_field=(0, 0, 0, 1e-4, -2e-4, 3e-4))
    s.set_field_operator(G)
    return s


def _run(s, w, K, every):
    s.set_particles(w.PartState, elem=w.elem, species=w.species)
    loss, gx, gv = s.adjoint(w.dt, K, every)
    return (np.float64(loss), gx, gv) + tuple(s.particles()) + (s.part_source(),)


def _same(a, b):
    assert all(np.array_equal(u, v) for u, v in zip(a, b))


@pytest.mark.parametrize("n_el,n,K,every", [(5, 3001, 1, 1), (5, 3001, 5, 1), (5, 3001, 5, 2), (6, 4003, 4, 4),
                                            (5, 2000, 3, 8)])
def test_fields_kept_or_not(monkeypatch, n_el, n, K, every):
    w, _ = A.landau_box(n_el=n_el, n_part=n, steps=K, sf_alpha=2)
    G = A.periodic_poisson_operator(w.mesh)
    print("case adjoint fields", n_el, n, K, every, flush=True)
    monkeypatch.delenv(LIMIT, raising=False)
    with _stage(w, G) as s:
        kept = _run(s, w, K, every)
    field = n_el ** 3 * (w.N + 1) ** 3 * 3 * 8
    for limit in (0, field * K - 1):
        monkeypatch.setenv(LIMIT, str(limit))
        with _stage(w, G) as s:
            _same(_run(s, w, K, every), kept)


def test_one_handle_with_and_without(monkeypatch):
    """More steps than the limit allows, on a handle that holds some fields, and fewer again."""
    w, _ = A.landau_box(n_el=5, n_part=3001, steps=6, sf_alpha=3)
    G = A.periodic_poisson_operator(w.mesh)
    print("case adjoint fields, one handle", flush=True)
    monkeypatch.delenv(LIMIT, raising=False)
    ref = {}
    for K in (2, 3, 6):
        with _stage(w, G) as s:
            ref[K] = _run(s, w, K, 2)
    with _stage(w, G) as s:
        _same(_run(s, w, 2, 2), ref[2])
        monkeypatch.setenv(LIMIT, str(5 * 125 * 64 * 24))
        _same(_run(s, w, 6, 2), ref[6])
        _same(_run(s, w, 3, 2), ref[3])
        monkeypatch.delenv(LIMIT)
        _same(_run(s, w, 6, 2), ref[6])


def test_limit_bounds_the_memory(monkeypatch):
    """40 steps of a mesh whose fields are 0.79 MB each, with states of 0.2 MB."""
    w, _ = A.landau_box(n_el=8, n_part=3000, steps=40, sf_alpha=2)
    G = A.periodic_poisson_operator(w.mesh)
    print("case adjoint memory", flush=True)
    monkeypatch.setenv(LIMIT, "0")
    with _stage(w, G) as s:
        s.set_particles(w.PartState, elem=w.elem, species=w.species)
        s.adjoint(w.dt, 1, 1)
        free = torch.cuda.mem_get_info()[0]
        s.adjoint(w.dt, 40, 7)
        taken = free - torch.cuda.mem_get_info()[0]
    # 13 states and 7 fields more than at first, each rounded up to 2 MB at the worst: 5 arrays a state
    assert taken <= 40 * 512 * 64 * 24 * 0.75, taken
