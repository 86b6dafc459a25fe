"""Shape-function deposition on rows and sheets of elements, whose targets have
one and three to five runs of source elements: a wave takes a target of a row from
1,025 targets on, four or more share it elsewhere.  Tensor grids, deformed and
curved elements, degrees with one and with several chunks of 64 DOFs, against the
oracle."""
import numpy as np
import pytest

from piclas_amd import mesh as M
from piclas_amd import stage
from piclas_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha", [2, 3, 4])
@pytest.mark.parametrize("kind,shape,n,N", [("box", (1025, 1, 1), 9001, 3), ("box", (1024, 1, 1), 3000, 3),
                                            ("box", (33, 32, 1), 5000, 3), ("box", (1026, 1, 1), 4000, 1),
                                            ("box", (1, 1030, 1), 2000, 4), ("box", (1, 1, 150), 700, 7),
                                            ("deformed", (1027, 1, 1), 9001, 3), ("deformed", (1, 35, 33), 5003, 2),
                                            ("deformed", (40, 1, 3), 2001, 3), ("ring", (1, 1030, 1), 6001, 3),
                                            ("ring", (1, 1030, 1), 3000, 2), ("ring", (1, 300, 1), 3000, 7),
                                            ("annulus", (2, 40, 14), 6001, 3), ("annulus", (1, 24, 12), 3000, 5)])
def test_thin_meshes(oracle_mod, kind, shape, n, N, alpha):
    print("case thin gather", kind, shape, n, N, alpha, flush=True)
    rng = np.random.Generator(np.random.PCG64(11))
    if kind == "annulus":
        w = W.annulus_plasma(shape=shape, n_total=n)
        mesh, part, species = w.mesh, w.PartState, w.species
        kw = dict(tracking=stage.TRACK_REFMAPPING, refmapping_guess=2, sf_radius=0.02, charge=w.charge, mass=w.mass,
                  mpf=w.mpf)
    elif kind == "ring":     # curved elements; the radius reaches no periodic image in z
        mesh = M.annulus(shape, 0.5, 0.51, 0.01, NGeo=2)
        th, r = 2 * np.pi * rng.uniform(0.0, 1.0, n) ** 2, rng.uniform(0.5005, 0.5095, n)
        pos = np.stack([r * np.cos(th), r * np.sin(th), rng.uniform(0.0005, 0.0095, n)], 1)
        part = np.hstack([pos, W.maxwellian(rng, n, 2.0, stage.ELECTRON_MASS)])
        species = np.ones(n, np.int32)
        kw = dict(tracking=stage.TRACK_REFMAPPING, refmapping_guess=2, sf_radius=0.0006)
    else:
        hi = np.array(shape) / 8.0
        mesh = M.cartesian_box(shape, hi=tuple(hi), periodic=tuple(s >= 4 for s in shape))
        pos = rng.uniform(0.0, 1.0, (n, 3)) ** 2 * hi
        if kind == "deformed":
            X, X0 = mesh.NodeCoords, mesh.NodeCoords.copy()
            turn = np.where(np.array(shape) >= 4, 2.0, 1.0) * np.pi / hi
            for a in range(3):
                X[:, (a + 1) % 3] += 0.01 * np.sin(2 * np.pi * X0[:, a] / hi[a])
                X[:, a] += 0.01 * np.sin(2 * np.pi * X0[:, a] / hi[a]) * np.cos(turn * X0)[:, (a + 1) % 3]
        part = np.hstack([pos, W.maxwellian(rng, n, 2.0, stage.ELECTRON_MASS)])
        species, kw = np.ones(n, np.int32), dict(sf_radius=0.19)
    kw.update(deposition=stage.DEPO_SF, sf_alpha=alpha)
    with stage.PICStage(mesh, N, max_particles=n, **kw) as s:
        s.set_particles(part, species=species)
        elem = s.particles()[1]
        held = elem > 0                      # (the displaced walls leave some outside)
        assert held.sum() > n // 2
        part, species, elem = part[held], species[held], elem[held]
        s.set_particles(part, elem=elem, species=species)
        s.deposition()
        PS = s.part_source()
    o = oracle_mod.Oracle(mesh, N, **kw)
    o.set_particles(part, elem=elem, species=species)
    o.deposition()
    ref = o.part_source()
    for c in (slice(0, 3), slice(3, 4)):
        assert np.abs(PS[..., c] - ref[..., c]).max() <= 1e-12 * np.abs(ref[..., c]).max()
