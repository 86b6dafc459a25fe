"""Shape-function deposition where several waves share a target element: mesh
sizes on both sides of the limits of 16, 8, 4 and 1 waves per target, with
ragged shapes, empty elements and fewer particles than lanes, against the
oracle."""
import numpy as np
import pytest

from piclas_amd import mesh as M
from piclas_amd import stage
from piclas_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha", [2, 3, 4])
@pytest.mark.parametrize("shape,n", [((4, 8, 8), 3), ((4, 8, 8), 4097), ((257, 1, 1), 900), ((16, 16, 8), 5000),
                                     ((9, 12, 19), 2500), ((16, 16, 16), 7001), ((17, 13, 19), 300000)])
def test_split_gather(oracle_mod, shape, n, alpha):
    print("case split gather", shape, n, alpha, flush=True)
    rng = np.random.Generator(np.random.PCG64(5))
    hi = np.array(shape) / 8.0
    mesh = M.cartesian_box(shape, hi=tuple(hi), periodic=tuple(s >= 4 for s in shape))
    pos = rng.uniform(0.0, 1.0, (n, 3)) ** 2 * hi     # crowded towards one corner
    part = np.hstack([pos, W.maxwellian(rng, n, 2.0, stage.ELECTRON_MASS)])
    kw = dict(deposition=stage.DEPO_SF, sf_radius=0.19, sf_alpha=alpha)
    with stage.PICStage(mesh, 3, max_particles=n, **kw) as s:
        s.set_particles(part, elem=mesh.element_of(pos))
        s.deposition()
        PS = s.part_source()
    o = oracle_mod.Oracle(mesh, 3, **kw)
    o.set_particles(part, elem=mesh.element_of(pos))
    o.deposition()
    ref = o.part_source()
    for c in (slice(0, 3), slice(3, 4)):
        assert np.abs(PS[..., c] - ref[..., c]).max() <= 1e-12 * np.abs(ref[..., c]).max()


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("kind,shape,n,alpha", [("box", (5, 4, 6), 701, 2), ("box", (3, 3, 3), 1, 3),
                                                ("deformed", (4, 4, 4), 1300, 4), ("annulus", (3, 12, 4), 2000, 2)])
def test_degrees(oracle_mod, kind, shape, n, alpha, N):
    """Every polynomial degree on the matrix cores: elements of less than 16 to
    512 DOFs (chunks of 64, the last one partly filled), on Cartesian, deformed
    and curved elements."""
    if N == 3 and kind == "box":
        pytest.skip("N = 3 boxes run the tensor-grid gather")
    print("case degrees", kind, shape, n, alpha, N, flush=True)
    rng = np.random.Generator(np.random.PCG64(7))
    if kind == "annulus":
        w = W.annulus_plasma(shape=shape, n_total=n)
        mesh, part, species = w.mesh, w.PartState, w.species
        kw = dict(tracking=stage.TRACK_REFMAPPING, refmapping_guess=2, sf_radius=0.11, charge=w.charge, mass=w.mass,
                  mpf=w.mpf)
    else:
        hi = np.array(shape) / 4.0
        mesh = M.cartesian_box(shape, hi=tuple(hi), periodic=tuple(s >= 4 for s in shape))
        if kind == "deformed":
            X = mesh.NodeCoords
            X += 0.02 * np.sin(2 * np.pi * X) * np.cos(2 * np.pi * np.roll(X, 1, axis=1))
        part = np.hstack([rng.uniform(0.0, 1.0, (n, 3)) * hi, W.maxwellian(rng, n, 2.0, stage.ELECTRON_MASS)])
        species, kw = np.ones(n, np.int32), dict(sf_radius=0.37)
    kw.update(deposition=stage.DEPO_SF, sf_alpha=alpha)
    with stage.PICStage(mesh, N, max_particles=n, **kw) as s:
        s.set_particles(part, species=species)
        s.deposition()
        PS = s.part_source()
        assert s.stats()["deposit_kernel"] == stage.KERNEL_SF_MATRIX
    o = oracle_mod.Oracle(mesh, N, **kw)
    o.set_particles(part, species=species)
    o.deposition()
    ref = o.part_source()
    for c in (slice(0, 3), slice(3, 4)):
        assert np.abs(PS[..., c] - ref[..., c]).max() <= 1e-12 * np.abs(ref[..., c]).max()
