"""DSMC on the GPU (collisions/DSMC.java:167-430) against the oracle's restatement with the same
per-cell Philox streams and id-ordered cell lists: collisions, post-collision velocities,
sig_cr_max and the remainders, pass by pass; and at the full 512x256-cell / 5e7-particle N2
size, conservation of momentum and energy by one pass."""
import numpy as np
import pytest

from helpers import geometry, oracle_for
from starfish_amd import deck as D

N2 = dict(sigma="bird463", diam=(4.17e-10, 4.17e-10), ref_temp=(273.0, 273.0), visc_temp_index=(0.74, 0.74))


def _deck(two, spwt_b):
    mesh = D.MeshSpec("XY", 33, 17, (0.0, 0.0), (1e-4, 1e-4), {})
    mats = [D.MaterialSpec("N2", "kinetic_hip", 28.0, 0.0, 4e14, 0.0)]
    if two:
        mats.append(D.MaterialSpec("O2", "kinetic_hip", 32.0, 0.0, spwt_b, 0.0))
    return D.Deck(mesh, materials=mats, solver=None, num_it=3, dt=1e-8, seed=0)


def _particles(deck, n, seed, drift):
    m = deck.mesh
    rng = np.random.default_rng(seed)
    lc0 = rng.uniform(0, m.ni - 1, n).astype(np.float32).astype(np.float64)
    lc1 = rng.uniform(0, m.nj - 1, n).astype(np.float32).astype(np.float64)
    v = (rng.normal(size=(n, 3)) * 350.0 + drift).astype(np.float32).astype(np.float64)
    return m.x0[0] + lc0 * m.dh[0], m.x0[1] + lc1 * m.dh[1], v


def _vel_by_id(gp):
    o = np.argsort(gp["id"])
    return gp["id"][o], np.stack([gp["u"], gp["v"], gp["w"]], 1)[o]


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["vhs", "vss", "two_species", "dense_cells"])
def test_dsmc_matches_oracle(case):
    """dense_cells adds a cluster of 4000 particles over 2 x 2 cells (about 1000 per cell): cells
    longer than 512 particles go through the kernel copy with 2048-entry lists, the others through
    the 512-entry copy, in the same pass."""
    from starfish_amd.interactions import DsmcHip
    from starfish_amd.plugin import Simulation
    two = case == "two_species"
    deck = _deck(two, 8e14)
    geo, _ = geometry(deck)
    o = oracle_for(deck, geo)
    n = 20000
    vss = (1.4, 1.4) if case == "vss" else (1.0, 1.0)
    sim = Simulation(deck, capacity=2 * n + 4000, track_ids=True)
    dsmc = None
    try:
        mats = sim.materials
        for k, mat in enumerate(mats):
            x, y, v = _particles(deck, n // (k + 1), 7 + k, [200.0 * (1 - 2 * k), 0, 0])
            if case == "dense_cells":
                rng = np.random.default_rng(11)
                m = deck.mesh
                cx = rng.uniform(10, 12, 4000).astype(np.float32).astype(np.float64)
                cy = rng.uniform(6, 8, 4000).astype(np.float32).astype(np.float64)
                cv = (rng.normal(size=(4000, 3)) * 350.0).astype(np.float32).astype(np.float64)
                x = np.concatenate([x, m.x0[0] + cx * m.dh[0]])
                y = np.concatenate([y, m.x0[1] + cy * m.dh[1]])
                v = np.concatenate([v, cv])
            ids = np.arange(len(x), dtype=np.int32)
            mat.add_particles(x, y, v[:, 0], v[:, 1], v[:, 2], ids=ids, rewind=False)
            o.load_particles(k, np.stack([x, y, np.zeros(len(x))], 1), v, ids=ids, rewind=False)
        mb = mats[1] if two else mats[0]
        sb = 1 if two else 0
        dsmc = DsmcHip(sim, mats[0], mb, vss_alpha=vss, sig_cr_max=2e-16, seed=99, tag=1, **N2)
        ncell = (deck.mesh.ni - 1) * (deck.mesh.nj - 1)
        st = {"sig_cr_max": np.full(ncell, 2e-16), "rem": np.zeros(ncell)}
        acc = {"count_sum": np.zeros(sim.nn), "real_sum": np.zeros(sim.nn)}
        pair = {"sigma_type": 1, "diam": N2["diam"], "ref_temp": N2["ref_temp"],
                "visc_temp_index": N2["visc_temp_index"], "vss_alpha": vss}
        for it in (1, 2, 3):
            ng = dsmc.perform(it)
            no = o.dsmc_perform(0, sb, pair, 99, 1, it, 1, st, acc)
            errs = []
            for k, mat in enumerate(mats):
                gid, gv = _vel_by_id(mat.particles(ids=True))
                op = o.particles(k)
                oo = np.argsort(op["id"])
                assert np.array_equal(gid, op["id"][oo])
                errs.append(np.abs(gv - op["vel"][oo]).max() / np.abs(op["vel"]).max())
            print("%s pass %d: collisions gpu %d oracle %d, velocity error %.2e" % (case, it, ng, no, max(errs)),
                  flush=True)
            assert ng == no and ng > 100
            # The GPU rounds each collided velocity to FP32, the oracle keeps FP64; particles of
            # these dense cells collide about three times per pass.  VSS deflection divides by
            # sqrt(g_j^2 + g_k^2), which amplifies that rounding where g points along i, and the
            # amplification compounds over passes: 1e-5 on the first pass, 1e-4 after it for VSS.
            assert max(errs) < (1e-5 if (it == 1 or case != "vss") else 1e-4)
            assert np.allclose(dsmc.sig_cr_max(), st["sig_cr_max"], rtol=1e-6)
            assert np.array_equal(dsmc.field("col-count-sum"), acc["count_sum"])
            for mat in mats:
                mat.update()                   # ballistic push between passes (no field)
            o.move()
            for k in range(len(mats)):
                o.round_state_fp32(k)          # the GPU's stored state is FP32
        nu = dsmc.field("nu")
        assert np.allclose(nu, acc["real_sum"] / (3 * deck.dt), rtol=1e-12)
    finally:
        if dsmc is not None:
            dsmc.close()
        sim.close()


@pytest.mark.gpu
def test_dsmc_full_size_conservation():
    """512x256 cells at 1e-4 m, 5e7 N2 (VHS, d_ref 4.17e-10 m, omega 0.74, T_ref 273 K) preloaded
    at 300 K with a 500 m/s drift: one DSMC pass after the counting sort conserves the total
    momentum and energy of the FP32 particle state to 1e-6 and collides a fraction of the gas
    consistent with the NTC rate."""
    import time
    from starfish_amd.interactions import DsmcHip
    from starfish_amd.plugin import Simulation
    mesh = D.MeshSpec("XY", 513, 257, (0.0, 0.0), (1e-4, 1e-4), {})
    n = 50_000_000
    n_real = 1e22                                   # 1e22 m^-3 over the 5.12e-2 x 2.56e-2 m domain
    spwt = n_real * 512 * 256 * 1e-8 / n
    deck = D.Deck(mesh, materials=[D.MaterialSpec("N2", "kinetic_hip", 28.0, 0.0, spwt, 0.0)], solver=None,
                  num_it=1, dt=1e-8, seed=0)
    sim = Simulation(deck, capacity=n + 1_000_000, track_ids=True)
    dsmc = None
    try:
        mat = sim.materials[0]
        mat.preload(n, (500.0, 0.0, 0.0), 300.0, seed=5)
        ids0, v0 = _vel_by_id(mat.particles(ids=True))
        mom0, en0 = v0.sum(0), (v0 ** 2).sum()
        dsmc = DsmcHip(sim, mat, mat, sig_cr_max=1e-16, seed=3, **N2)
        t0 = time.perf_counter()
        ncol = dsmc.perform(1)
        sim.ctx.call("sf_ctx_synchronize")
        dt_ms = (time.perf_counter() - t0) * 1e3
        ids1, v1 = _vel_by_id(mat.particles(ids=True))
        assert np.array_equal(ids0, ids1)
        changed = np.mean(np.any(v1 != v0, axis=1))
        print("C5 DSMC pass: %d collisions, %.4f of the particles changed, %.1f ms" % (ncol, changed, dt_ms),
              flush=True)
        assert ncol > 10000
        assert abs(2 * ncol / n - changed) < 0.05 * changed + 1e-4
        assert np.abs(v1.sum(0) - mom0).max() <= 1e-6 * np.abs(v0).sum()
        assert abs((v1 ** 2).sum() / en0 - 1) < 1e-6
    finally:
        if dsmc is not None:
            dsmc.close()
        sim.close()


@pytest.mark.gpu
@pytest.mark.parametrize("two", [False, True])
def test_cell_orders_at_their_size_limits(two):
    """Cells of 1, 2, 63 .. 65, 127 .. 129, 255 .. 257, 511 .. 513, 1024 and 2048 particles, the
    lengths at which the pass changes how it orders a cell, the same lengths in the last cell column
    with five more particles on the last node line (not binned), and ids in random order: one pass
    matches the oracle collision for collision.  Velocities within the FP32 rounding of at most
    about ten collisions of one particle, 10 x 2^-24 of the largest, with a margin of ten."""
    from starfish_amd.interactions import DsmcHip
    from starfish_amd.plugin import Simulation
    deck = _deck(two, 8e14)
    m = deck.mesh
    geo, _ = geometry(deck)
    o = oracle_for(deck, geo)
    counts = [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1024, 2048]
    sim = Simulation(deck, capacity=40000, track_ids=True)
    dsmc = None
    try:
        for k, mat in enumerate(sim.materials):
            rng = np.random.default_rng(3 + k)
            lc = []
            for q, n in enumerate(counts):
                n = counts[-1 - q] if k else n
                for ci in (3, m.ni - 2):
                    lc.append(np.stack([ci + 0.999 * rng.random(n), q + 0.999 * rng.random(n)], 1))
                lc.append(np.stack([np.full(5, m.ni - 1.0), q + 0.999 * rng.random(5)], 1))
            lc = np.concatenate(lc).astype(np.float32).astype(np.float64)
            n = len(lc)
            v = (rng.normal(size=(n, 3)) * 350.0).astype(np.float32).astype(np.float64)
            x, y = lc[:, 0] * m.dh[0], lc[:, 1] * m.dh[1]
            ids = rng.permutation(n).astype(np.int32)
            mat.add_particles(x, y, v[:, 0], v[:, 1], v[:, 2], ids=ids, rewind=False)
            o.load_particles(k, np.stack([x, y, np.zeros(n)], 1), v, ids=ids, rewind=False)
        dsmc = DsmcHip(sim, sim.materials[0], sim.materials[-1], sig_cr_max=2e-16, seed=5, tag=1, **N2)
        ncell = (m.ni - 1) * (m.nj - 1)
        st = {"sig_cr_max": np.full(ncell, 2e-16), "rem": np.zeros(ncell)}
        acc = {"count_sum": np.zeros(sim.nn), "real_sum": np.zeros(sim.nn)}
        pair = {"sigma_type": 1, "diam": N2["diam"], "ref_temp": N2["ref_temp"],
                "visc_temp_index": N2["visc_temp_index"], "vss_alpha": (1.0, 1.0)}
        ng = dsmc.perform(1)
        no = o.dsmc_perform(0, len(sim.materials) - 1, pair, 5, 1, 1, 1, st, acc)
        assert ng == no and ng > 1000
        assert np.array_equal(dsmc.field("col-count-sum"), acc["count_sum"])
        assert np.allclose(dsmc.sig_cr_max(), st["sig_cr_max"], rtol=1e-6)
        for k, mat in enumerate(sim.materials):
            gid, gv = _vel_by_id(mat.particles(ids=True))
            op = o.particles(k)
            oo = np.argsort(op["id"])
            assert np.array_equal(gid, op["id"][oo])
            assert np.abs(gv - op["vel"][oo]).max() / np.abs(op["vel"]).max() < 100 * 2.0 ** -24
    finally:
        if dsmc is not None:
            dsmc.close()
        sim.close()


@pytest.mark.gpu
@pytest.mark.parametrize("ni,nj", [(2, 3), (5, 9), (9, 9), (17, 5), (33, 33), (46, 46), (65, 64)])
def test_cells_of_a_wave_match_oracle(ni, nj):
    """2, 32, 64, 64, 1024, 2025 and 4032 cells, which the collision loop takes 1 to 64 to a wave (whole
    and partial waves): two passes of a gas of about 30 particles a cell collide as the oracle does, cell
    for cell."""
    from starfish_amd.interactions import DsmcHip
    from starfish_amd.plugin import Simulation
    mesh = D.MeshSpec("XY", ni, nj, (0.0, 0.0), (1e-4, 1e-4), {f: ("SYMMETRY", 0.0) for f in D.FACES})
    ncell = (ni - 1) * (nj - 1)
    n = 30 * ncell
    deck = D.Deck(mesh, materials=[D.MaterialSpec("N2", "kinetic_hip", 28.0, 0.0, 1e22 * ncell * 1e-8 / n, 0.0)],
                  solver=None, num_it=1, dt=2e-7, seed=0)
    geo, _ = geometry(deck)
    o = oracle_for(deck, geo)
    rng = np.random.default_rng(ncell)
    lc = (rng.random((n, 2)) * [ni - 1, nj - 1] * 0.9999).astype(np.float32).astype(np.float64)
    v = (rng.normal(size=(n, 3)) * 400.0).astype(np.float32).astype(np.float64)
    x, y = lc[:, 0] * 1e-4, lc[:, 1] * 1e-4
    ids = np.arange(n, dtype=np.int32)
    sim = Simulation(deck, capacity=n + 16, track_ids=True)
    dsmc = None
    try:
        mat = sim.materials[0]
        mat.add_particles(x, y, v[:, 0], v[:, 1], v[:, 2], ids=ids, rewind=False)
        o.load_particles(0, np.stack([x, y, np.zeros(n)], 1), v, ids=ids, rewind=False)
        dsmc = DsmcHip(sim, mat, mat, sig_cr_max=2e-16, seed=9, tag=2, **N2)
        st = {"sig_cr_max": np.full(ncell, 2e-16), "rem": np.zeros(ncell)}
        acc = {"count_sum": np.zeros(sim.nn), "real_sum": np.zeros(sim.nn)}
        pair = {"sigma_type": 1, "diam": N2["diam"], "ref_temp": N2["ref_temp"],
                "visc_temp_index": N2["visc_temp_index"], "vss_alpha": (1.0, 1.0)}
        total = 0
        for it in (1, 2):
            ng = dsmc.perform(it)
            assert ng == o.dsmc_perform(0, 0, pair, 9, 2, it, 1, st, acc)
            assert np.array_equal(dsmc.field("col-count-sum"), acc["count_sum"])
            o.round_state_fp32(0)
            total += ng
        assert total > 0.1 * ncell
    finally:
        if dsmc is not None:
            dsmc.close()
        sim.close()
