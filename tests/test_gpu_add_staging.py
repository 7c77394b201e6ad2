"""Particle batches at the size limit of the context's staging: the same particles added in one copied
batch and in staged ones are the same state, with rejected particles and ids among them."""
import numpy as np
import pytest

from starfish_amd import deck as D

STAGE_MAX = 16384


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(1, STAGE_MAX), (STAGE_MAX - 1, 2), (5, STAGE_MAX - 4)])
@pytest.mark.parametrize("with_ids,rewind", [(True, False), (False, True)])
def test_staged_batches_equal_a_copied_one(sizes, with_ids, rewind):
    from starfish_amd.plugin import Simulation
    n = sum(sizes)
    assert n == STAGE_MAX + 1
    mesh = D.MeshSpec("XY", 33, 17, (0.0, 0.0), (1e-3, 1e-3), {f: ("OPEN", 0.0) for f in D.FACES})
    deck = D.Deck(mesh, boundaries=[], materials=[D.MaterialSpec("O+", "kinetic_hip", 16.0, 1.0, 1e4, 0.0)],
                  solver=None, num_it=1, dt=1e-7, seed=1)
    rng = np.random.default_rng(n)
    x, y = rng.uniform(-2e-3, 34e-3, n), rng.uniform(0, 16e-3, n)
    v = rng.normal(size=(n, 3)) * 1000.0
    v[::7, 1] = np.nan                       # dropped, like the particles outside of the mesh
    x[0], y[0], v[0] = 1e-3, 1e-3, 10.0
    ids = rng.permutation(n).astype(np.int32)
    got = []
    for batches in ((n,), sizes):
        sim = Simulation(deck, capacity=n + 64, track_ids=True)
        try:
            j, i = np.mgrid[0:17, 0:33]
            sim.set_efield((100.0 * i).ravel(), (50.0 * j).ravel())
            mat = sim.materials[0]
            a = 0
            for m in batches:
                s = slice(a, a + m)
                mat.add_particles(x[s], y[s], v[s, 0], v[s, 1], v[s, 2], ids=ids[s] if with_ids else None, rewind=rewind)
                a += m
            got.append(mat.particles(ids=True))
        finally:
            sim.close()
    assert 0 < len(got[0]["id"]) < n
    for k in ("id", "lc0", "lc1", "u", "v", "w"):
        assert np.array_equal(got[0][k], got[1][k]), k
