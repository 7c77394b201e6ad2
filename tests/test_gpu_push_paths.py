"""The fast tile push (parts of tiles, moves of up to two cells, FP64 rotation and Boris in the tile)
against the general tile kernel that runs the reference loop for every particle (SF_NO_FAST_PUSH),
on the same particles: state, node fields and counts over six steps with a sort in between."""
import os

import numpy as np
import pytest

from starfish_amd import deck as D


def _run(domain, b, n, ni, nj, general):
    from starfish_amd.plugin import Simulation
    faces = {f: ("SYMMETRY", 0.0) for f in D.FACES}
    mesh = D.MeshSpec(domain, ni, nj, (0.0, 0.0), (1e-3, 1e-3), faces)
    Lx, Ly = (ni - 1) * 1e-3, (nj - 1) * 1e-3
    bnd = []
    if domain == "XY":
        bnd = [D.BoundarySpec("cylinder", "DIRICHLET", -100.0, D.circle_path(0.2 * Ly, 24, 0.5 * Lx, 0.5 * Ly), False, "SS")]
    deck = D.Deck(mesh, boundaries=bnd, materials=[D.MaterialSpec("O+", "kinetic_hip", 16.0, 1.0, 1e4, 0.0)],
                  solver=None, num_it=1, dt=1e-7, seed=1)
    rng = np.random.default_rng(n + ni)
    # half spread over the mesh, half in one 32 x 4-cell tile's corner; a quarter moves 1 to 2 cells a step
    lc = rng.random((n, 2)) * [ni - 1, nj - 1]
    lc[: n // 2] = [33, 4] + 4 * rng.random((n // 2, 2)) * [2, 1]
    if bnd:
        keep = np.hypot(lc[:, 0] * 1e-3 - 0.5 * Lx, lc[:, 1] * 1e-3 - 0.5 * Ly) > 0.22 * Ly
        lc = lc[keep]
    v = rng.normal(size=(len(lc), 3)) * 2000.0
    v[::4] = rng.choice([-1, 1], (len(v[::4]), 3)) * rng.uniform(8000, 21000, (len(v[::4]), 3))
    lc = lc.astype(np.float32).astype(np.float64)
    v = v.astype(np.float32).astype(np.float64)
    if general:
        os.environ["SF_NO_FAST_PUSH"] = "1"
    try:
        sim = Simulation(deck, capacity=n + 64, track_ids=True, vmax=4e4)
    finally:
        os.environ.pop("SF_NO_FAST_PUSH", None)
    try:
        y, x = np.mgrid[0:nj, 0:ni]
        sim.set_efield((3000 * np.cos(x / 9.0 + y / 5.0)).ravel(), (3000 * np.sin(x / 7.0 - y / 4.0)).ravel())
        if b:   # a field that is zero on half of the mesh: the electric kick there, Boris elsewhere
            sim.set_bfield(np.where(x > ni // 2, 0.3, 0.0).ravel(), np.where(x > ni // 2, -0.2, 0.0).ravel())
        mat = sim.materials[0]
        mat.add_particles(lc[:, 0] * 1e-3, lc[:, 1] * 1e-3, v[:, 0], v[:, 1], v[:, 2], rewind=False)
        for _ in range(6):
            mat.update()
        p = mat.particles(ids=True)
        o = np.argsort(p["id"])
        state = {k: p[k][o] for k in ("id", "lc0", "lc1", "u", "v", "w")}
        return state, {f: mat.field(f) for f in ("nd", "u", "v", "w", "uu-sum", "mpc-sum", "t")}, mat.stats()
    finally:
        sim.close()


@pytest.mark.gpu
@pytest.mark.parametrize("domain,b", [("XY", False), ("XY", True), ("RZ", False), ("RZ", True), ("ZR", False), ("ZR", True)])
@pytest.mark.parametrize("n,ni,nj", [(700, 67, 35), (60001, 131, 70)])
def test_fast_push_matches_the_general_kernel(domain, b, n, ni, nj):
    """FP64 paths repeat the general kernel's arithmetic: state within two FP32 roundings a step (a
    contraction may round an FP64 value the other way).  XY without B moves in FP32: within 1e-5 of the
    mesh and the largest speed, the bound of the parity tests.  Fields follow the state: within its
    relative error, 1e-5, of their maxima (the density of a mesh of 2000 to 9000 nodes)."""
    s0, f0, t0 = _run(domain, b, n, ni, nj, True)
    s1, f1, t1 = _run(domain, b, n, ni, nj, False)
    assert np.array_equal(s0["id"], s1["id"])
    f32 = domain == "XY" and not b
    for k, scale in (("lc0", ni), ("lc1", nj), ("u", None), ("v", None), ("w", None)):
        scale = scale or np.abs(s0[k]).max()
        bound = (1e-5 if f32 else 12 * 2.0 ** -23) * scale
        assert np.abs(s0[k] - s1[k]).max() <= bound, k
    for k in f0:
        assert np.abs(f0[k] - f1[k]).max() <= 1e-5 * max(np.abs(f0[k]).max(), 1e-300) * (20 if k == "t" else 1), k
    assert np.allclose(t0, t1, rtol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("v", [(12345.678, 3210.987, 777.77), (-10001.3, 17003.1, -2.5), (19000.7, -19000.7, 5000.9)])
def test_speed_sum_of_long_moves_is_double_precision(v):
    """The mover's speed sum of particles that move one to two cells a step, whose move the tile kernel
    evaluates in FP64: their speed is FP64 too, as in the reference loop.  Every particle has the same
    FP32 velocity, so a rounding of its speed to FP32 would not average out.  Bound: a contribution is
    rounded to a fixed-point quantum of at most 2 vmax 2^-40, half of that off, next to FP64's own."""
    from starfish_amd.plugin import Simulation
    vmax, n = 4e4, 3000
    mesh = D.MeshSpec("XY", 131, 70, (0.0, 0.0), (1e-3, 1e-3), {f: ("SYMMETRY", 0.0) for f in D.FACES})
    mat = D.MaterialSpec("O+", "kinetic_hip", 16.0, 1.0, 1e4, 0.0)
    sim = Simulation(D.Deck(mesh, materials=[mat], solver=None, num_it=1, dt=1e-7, seed=1), capacity=n, vmax=vmax)
    try:
        rng = np.random.default_rng(3)
        v = np.array(v, np.float32).astype(np.float64)
        x, y = 1e-3 * rng.uniform(40, 90, n), 1e-3 * rng.uniform(20, 50, n)
        sim.materials[0].add_particles(x, y, *[np.full(n, c) for c in v], rewind=False)
        for _ in range(3):   # the first push is of an unsorted population, by the reference loop
            sim.materials[0].update()
            s = sim.materials[0].stats()
            speed = np.sqrt((v * v).sum())
            err = abs(s[4] / s[0] / speed - 1)
            print("speed sum off by %.1e" % err, flush=True)
            assert err <= vmax / speed * 2.0 ** -40 + 1e-14
    finally:
        sim.close()


def _push_scene(domain, b, x0, faces, reverse, general):
    """Six steps of 20000 ions, a fifth of them one to two cells fast, around an object on 131 x 70 nodes;
    fifty more join after the third."""
    from starfish_amd.plugin import Simulation
    ni, nj, n = 131, 70, 20000
    mesh = D.MeshSpec(domain, ni, nj, x0, (1e-3, 7e-4), faces)
    Lx, Ly = (ni - 1) * 1e-3, (nj - 1) * 7e-4
    bnd = [D.BoundarySpec("c", "DIRICHLET", -100.0, D.circle_path(0.2 * Ly, 24, x0[0] + 0.5 * Lx, x0[1] + 0.5 * Ly), reverse,
                          "SS")]
    deck = D.Deck(mesh, boundaries=bnd, materials=[D.MaterialSpec("O+", "kinetic_hip", 16.0, 1.0, 1e4, 0.0)], solver=None,
                  num_it=1, dt=1e-7, seed=1)
    rng = np.random.default_rng(11)
    lc = rng.random((n, 2)) * [ni - 1, nj - 1]
    lc = lc[np.hypot((lc[:, 0] - 65) * 1e-3, (lc[:, 1] - 34.5) * 7e-4) > 0.22 * Ly]
    v = rng.normal(size=(len(lc), 3)) * 2000.0
    v[::5] = rng.choice([-1, 1], (len(v[::5]), 3)) * rng.uniform(8000, 14000, (len(v[::5]), 3))
    v = v.astype(np.float32).astype(np.float64)
    if general:
        os.environ["SF_NO_FAST_PUSH"] = "1"
    try:
        sim = Simulation(deck, capacity=n + 64, track_ids=True, vmax=4e4)
    finally:
        os.environ.pop("SF_NO_FAST_PUSH", None)
    try:
        y, x = np.mgrid[0:nj, 0:ni]
        sim.set_efield((3000 * np.cos(x / 9.0 + y / 5.0)).ravel(), (3000 * np.sin(x / 7.0 - y / 4.0)).ravel())
        if b:
            sim.set_bfield(np.where(x > ni // 2, 0.3, 0.0).ravel(), np.where(x > ni // 2, -0.2, 0.0).ravel())
        mat = sim.materials[0]
        add = lambda s: mat.add_particles(x0[0] + lc[s, 0] * 1e-3, x0[1] + lc[s, 1] * 7e-4, v[s, 0], v[s, 1], v[s, 2])  # noqa: E731
        add(slice(50, None))
        for k in range(6):
            mat.update()
            if k == 2:
                add(slice(0, 50))
        p = mat.particles(ids=True)
        o = np.argsort(p["id"])
        return {k: p[k][o] for k in ("id", "lc0", "lc1", "u", "v", "w")}, {f: mat.field(f) for f in ("nd", "u", "mpc-sum")}
    finally:
        sim.close()


@pytest.mark.gpu
@pytest.mark.parametrize("b", [False, True])
@pytest.mark.parametrize("faces", ["OPEN", "PERIODIC"])
@pytest.mark.parametrize("domain,x0,reverse", [("RZ", (0.02, -0.03), False), ("RZ", (5.0, 7.0), True),
                                               ("ZR", (-0.03, 0.013), False), ("ZR", (1.0, 0.4), True),
                                               ("XY", (-0.15, 0.3), False)])
def test_fast_push_away_from_the_axis_and_around_objects(domain, x0, reverse, faces, b):
    """The radial weights and the rotation of the tile kernel at an origin off the axis, near an object and
    with faces that absorb or wrap, against the general kernel: the same ions survive, with the bounds of
    the test above (state within two FP32 roundings a step, in XY without B within the parity tests')."""
    bc = {f: (faces, 0.0) for f in D.FACES} if faces == "PERIODIC" else {}
    s0, f0 = _push_scene(domain, b, x0, bc, reverse, True)
    s1, f1 = _push_scene(domain, b, x0, bc, reverse, False)
    assert len(s0["id"]) > 5000 and np.array_equal(s0["id"], s1["id"])
    f32 = domain == "XY" and not b
    for k, scale in (("lc0", 131), ("lc1", 70), ("u", None), ("v", None), ("w", None)):
        scale = scale or np.abs(s0[k]).max()
        assert np.abs(s0[k] - s1[k]).max() <= (1e-5 if f32 else 12 * 2.0 ** -23) * scale, k
    for k in f0:
        assert np.abs(f0[k] - f1[k]).max() <= 1e-5 * max(np.abs(f0[k]).max(), 1e-300), k


@pytest.mark.gpu
@pytest.mark.parametrize("general", [False, True])
def test_timings_name_the_kernel_that_pushed_appended_particles(general):
    """sf_last_push_timings: particles appended since the last sort are pushed in the slow-list kernel's
    launch, so their own interval is exactly zero; with the general tile kernel they have a kernel of
    their own, with a time.  The slots are counted either way."""
    import ctypes as C
    from starfish_amd.plugin import Simulation
    mesh = D.MeshSpec("XY", 131, 70, (0.0, 0.0), (1e-3, 1e-3), {f: ("SYMMETRY", 0.0) for f in D.FACES})
    mat = D.MaterialSpec("O+", "kinetic_hip", 16.0, 1.0, 1e4, 0.0)
    if general:
        os.environ["SF_NO_FAST_PUSH"] = "1"
    try:
        sim = Simulation(D.Deck(mesh, materials=[mat], solver=None, num_it=1, dt=1e-8, seed=1), capacity=30000, vmax=4e4)
    finally:
        os.environ.pop("SF_NO_FAST_PUSH", None)
    try:
        sim.ctx.call("sf_set_timing", 1)
        m = sim.materials[0]
        m.preload(20000, (100.0, 0.0, 0.0), 300.0, seed=1)
        m.update()
        one = np.full(300, 1000.0)
        m.add_particles(np.full(300, 0.05), np.full(300, 0.03), one, one, one)
        m.update()
        split, queue = np.zeros(3), np.zeros(2)
        dp = C.POINTER(C.c_double)
        sim.ctx.call("sf_last_push_timings", split.ctypes.data_as(dp))
        sim.ctx.call("sf_last_push_queue", queue.ctypes.data_as(dp))
        print(split, queue, flush=True)
        assert split[2] == 300 and split[0] > 0
        assert split[1] > 0 if general else split[1] == 0 and queue[0] > 0
    finally:
        sim.close()
