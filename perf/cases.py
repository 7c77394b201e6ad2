"""Performance cases of the ES-PIC path: what a user's program has the library do, at the sizes of
the repository's own decks, its benchmark's other workloads and between them.

Families (the "work" key of a case):
  loop   whole main-loop steps (injection, push + deposit + sort, rho, potential solve, E)
  push   push + deposit steps of one species in a given field, XY, RZ and ZR, with and without B
  solve  a potential solve for a host-owned rho, cold or from the previous step's potential
  mcc    collision passes of a species with a background gas
  dsmc   free flight and pairwise collisions of one gas, or of two
  cnn    the learned guess: training steps, gradients of one sample, and the guess itself

The potential of a solve or a step is determined by a relative residual of 1e-8, a few 1e-7 of its
values: it comes back in single precision, which holds those digits, as do the fields of whole
steps, which follow from it.  Fields of the push and the collisions alone are exact sums and come
back as the library gives them.
"""
import ctypes as C
import math

import numpy as np
import torch
import torch.nn.functional as F

from starfish_amd import _lib
from starfish_amd import deck as D
from starfish_amd.interactions import DsmcHip, MccHip
from starfish_amd.learned import LearnedGuess
from starfish_amd.plugin import Simulation

N_BEAM = 1e20 / 7000.0      # ion density of the inflowing O+ beam, m^-3
LX, LY = 1023e-3, 511e-3    # domain of the XY decks, m


def listed():
    return [
        # the reference's tutorial deck, one step at a time: launches and latency
        {"name": "loop_xy_81x41", "work": "loop", "ni": 81, "nj": 41, "particles": 20_000, "steps": 1,
         "device_sources": False},
        # the benchmark: one sort cycle of whole steps
        {"name": "loop_xy_1024x512", "work": "loop", "ni": 1024, "nj": 512, "particles": 20_000_000, "steps": 4,
         "device_sources": True},
        # the benchmark's population streaming through a periodic channel past the cylinder
        {"name": "push_xy_1024x512", "work": "push", "domain": "XY", "ni": 1024, "nj": 512, "particles": 20_000_000,
         "steps": 8, "b": False, "object": True},
        # the largest population: 1e8 Xe+ on the axisymmetric mesh
        {"name": "push_rz_2048x1024", "work": "push", "domain": "RZ", "ni": 2048, "nj": 1024,
         "particles": 100_000_000, "steps": 4, "b": False, "object": False},
        # a magnetised run with the axis along j, ragged mesh, few particles
        {"name": "push_zr_b_301x157", "work": "push", "domain": "ZR", "ni": 301, "nj": 157, "particles": 1_000_000,
         "steps": 4, "b": True, "object": False},
        # a host code that owns rho and phi calls the solver every step
        {"name": "solve_warm_xy_1024x512", "work": "solve", "domain": "XY", "ni": 1024, "nj": 512, "start": "warm",
         "linear": False, "object": True},
        {"name": "solve_warm_rz_2048x1024", "work": "solve", "domain": "RZ", "ni": 2048, "nj": 1024, "start": "warm",
         "linear": False, "object": False},
        # the initial solve of a run, from phi = 0
        {"name": "solve_cold_rz_1024x512", "work": "solve", "domain": "RZ", "ni": 1024, "nj": 512, "start": "cold",
         "linear": False, "object": False},
        # charge exchange of ions with a neutral background
        {"name": "mcc_cex_1024x512", "work": "mcc", "ni": 1024, "nj": 512, "particles": 40_000_000, "model": "CEX",
         "density": 1e19, "steps": 4},
        # a dense N2 gas: free flight, sort, collisions
        {"name": "dsmc_513x257", "work": "dsmc", "ni": 513, "nj": 257, "particles": 50_000_000, "pair": False,
         "steps": 2},
        # the learned guess: an Adam step at the benchmark's grid, and a guess on a ragged one
        {"name": "cnn_train_1024x512", "work": "cnn", "ni": 1024, "nj": 512, "mode": "train", "batch": 4},
        {"name": "cnn_guess_301x157", "work": "cnn", "ni": 301, "nj": 157, "mode": "guess", "batch": 1},
    ]


def _log_int(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    work = rng.choice(["loop", "push", "push", "solve", "solve", "mcc", "dsmc", "cnn"])
    if work == "cnn":
        mode = rng.choice(["train", "grads", "guess"])
        ni, nj = _log_int(rng, 40, 1024), _log_int(rng, 24, 512)
        return {"work": work, "ni": ni, "nj": nj, "mode": mode, "batch": rng.randint(1, 4) if mode == "train" else 1}
    ni = _log_int(rng, 65, 1024)
    nj = _log_int(rng, max(33, ni // 4), min(512, ni))
    cells = (ni - 1) * (nj - 1)
    if work == "loop":
        n = min(20_000_000, int(cells * rng.uniform(5, 50)))
        return {"work": work, "ni": ni, "nj": nj, "particles": n, "steps": rng.randint(1, 4),
                "device_sources": rng.random() < 0.7}
    if work == "push":
        n = min(40_000_000, int(cells * math.exp(rng.uniform(math.log(3), math.log(150)))))
        domain = rng.choice(["XY", "RZ", "ZR"])
        return {"work": work, "domain": domain, "ni": ni, "nj": nj, "particles": n, "steps": rng.randint(3, 9),
                "b": rng.random() < 0.3, "object": domain == "XY" and rng.random() < 0.5}
    if work == "solve":
        domain = rng.choice(["XY", "RZ", "ZR"])
        return {"work": work, "domain": domain, "ni": ni, "nj": nj, "start": rng.choice(["warm", "warm", "cold"]),
                "linear": rng.random() < 0.15, "object": domain == "XY" and rng.random() < 0.5}
    if work == "mcc":
        n = min(40_000_000, int(cells * math.exp(rng.uniform(math.log(5), math.log(150)))))
        return {"work": work, "ni": ni, "nj": nj, "particles": n, "model": rng.choice(["CEX", "MEX"]),
                "density": math.exp(rng.uniform(math.log(1e18), math.log(1e21))), "steps": rng.randint(1, 4)}
    ppc = math.exp(rng.uniform(math.log(15), math.log(500)))
    pair = rng.random() < 0.4
    return {"work": "dsmc", "ni": min(ni, 513), "nj": min(nj, 257),
            "particles": min(50_000_000, int((min(ni, 513) - 1) * (min(nj, 257) - 1) * ppc)), "pair": pair,
            "steps": rng.randint(1, 2)}


# ------------------------------------------------------------------------------------------
# what the program has in hand before the call
# ------------------------------------------------------------------------------------------
class State:
    """A running program's objects: the simulation, a collision object or network on it, its
    arrays.  Closing goes from the inside out."""

    def __init__(self, case):
        self.case = case
        self.it = 1
        self.sim = self.coll = self.net = self.ctx = None

    def __del__(self):
        for x in (self.coll, self.net, self.sim, self.ctx):
            if x is not None:
                try:
                    x.close()
                except Exception:
                    pass


def _dp(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def _waves(rng, ni, nj, terms, amp):
    """A smooth random field on the nodes, [nj, ni]: `terms` low-order cosine products, |f| <= amp."""
    x, y = np.linspace(0, 1, ni), np.linspace(0, 1, nj)
    f = np.zeros((nj, ni))
    for _ in range(terms):
        kx, ky = rng.integers(1, 6, 2)
        p, q = rng.uniform(0, 2 * math.pi, 2)
        f += np.outer(np.cos(2 * math.pi * ky * y + q), np.cos(2 * math.pi * kx * x + p))
    return f * (amp / terms)


def _mesh_xy(ni, nj, bc):
    return D.MeshSpec("XY", ni, nj, (-0.15, 0.0), (LX / (ni - 1), LY / (nj - 1)), bc)


def _cylinder():
    return D.BoundarySpec("cylinder", "DIRICHLET", -100.0, D.circle_path(0.05, 128), False, "SS")


def _axial_mesh(domain, ni, nj, bc):
    """The axisymmetric decks' 1e-4 m mesh at the axis, r along i (RZ) or j (ZR)."""
    return D.MeshSpec(domain, ni, nj, (0.0, 0.0), (1e-4, 1e-4), bc)


def _push_deck(case):
    n, ni, nj = case["particles"], case["ni"], case["nj"]
    if case["domain"] == "XY":
        mesh = _mesh_xy(ni, nj, {"LEFT": ("PERIODIC", 0.0), "RIGHT": ("PERIODIC", 0.0), "BOTTOM": ("SYMMETRY", 0.0),
                                 "TOP": ("SYMMETRY", 0.0)})
        # the benchmark's time step scaled with the cell, 0.7 cells a step at the beam's speed
        dt, drift, temp = 1e-7 * 1023 / (ni - 1), (7000.0, 0.0, 0.0), 1000.0
        mat = D.MaterialSpec("O+", "kinetic_hip", 16.0, 1.0, N_BEAM * LX * LY / n, 0.0)
    else:
        mesh = _axial_mesh(case["domain"], ni, nj, {f: ("SYMMETRY", 0.0) for f in D.FACES})
        dt, drift, temp = 1e-8, (0.0, 0.0, 0.0), 300.0
        mat = D.MaterialSpec("Xe+", "kinetic_hip", 131.0, 1.0, 1e4, 0.0)
    bnd = [_cylinder()] if case.get("object") else []
    deck = D.Deck(mesh, boundaries=bnd, materials=[mat], solver=None, num_it=1, dt=dt, seed=1)
    deck.preload = (n, drift, temp)
    return deck


def _set_waves(sim, rng, amp):
    m = sim.deck.mesh
    sim.set_efield(_waves(rng, m.ni, m.nj, 4, amp).ravel(), _waves(rng, m.ni, m.nj, 4, amp).ravel())


def _rho(case, seed):
    """(rho of the previous step, rho of this step) on the nodes: a plasma density with the noise of
    about 40 particles a cell, most of which a step keeps, and for a deck with the cylinder its
    wake, whose edges have moved by most of a cell."""
    ni, nj = case["ni"], case["nj"]
    rng = np.random.default_rng(seed)
    n0 = N_BEAM if case["domain"] == "XY" else 1e12
    if case["linear"]:
        n0 = 2e12 if case["domain"] == "XY" else 1e12
    base = n0 * (1.0 + _waves(rng, ni, nj, 4, 0.5))
    g1, g2 = rng.standard_normal((nj, ni)), rng.standard_normal((nj, ni))
    out = []
    for noise, shift in ((g1, 0.0), (0.8 * g1 + 0.6 * g2, 0.7)):
        n = base * np.maximum(1.0 + 0.16 * noise, 0.05)
        if case["object"]:
            # behind the cylinder: a wedge that narrows downstream, edges two cells wide
            dx, dy = LX / (ni - 1), LY / (nj - 1)
            x = (-0.15 + dx * np.arange(ni))[None, :]
            y = (dy * np.arange(nj))[:, None]
            half = 0.05 - 0.06 * (x - shift * dx)
            edge = np.clip((y - half) / (2 * dy), -30.0, 30.0)
            n *= np.where(x > 0.0, 0.02 + 0.98 / (1.0 + np.exp(-edge)), 1.0)
        out.append(D.QE * n.ravel())
    return out


def _solve_deck(case):
    ni, nj = case["ni"], case["nj"]
    lin = case["linear"]
    if case["domain"] == "XY":
        mesh = _mesh_xy(ni, nj, {"LEFT": ("DIRICHLET", 0.0), "BOTTOM": ("SYMMETRY", 0.0)})
        mat = D.MaterialSpec("O+", "kinetic_hip", 16.0, 1.0, 1e9, 0.0)
        solver = D.SolverSpec("poisson_hip", "GS", lin, 1e10, 2.0, 0.0)
    else:
        axis, ends = ("LEFT", ("BOTTOM", "TOP")) if case["domain"] == "RZ" else ("BOTTOM", ("LEFT", "RIGHT"))
        mesh = _axial_mesh(case["domain"], ni, nj, {axis: ("SYMMETRY", 0.0), ends[0]: ("DIRICHLET", 0.0),
                                                    ends[1]: ("DIRICHLET", -200.0)})
        mat = D.MaterialSpec("Xe+", "kinetic_hip", 131.0, 1.0, 1e4, 0.0)
        solver = D.SolverSpec("poisson_hip", "PCG", lin, 1e12, 2.0, 0.0)
    bnd = [_cylinder()] if case["object"] else []
    return D.Deck(mesh, boundaries=bnd, materials=[mat], solver=solver, num_it=1, dt=1e-8, seed=1)


def _cnn_params(seed):
    """He-initialised parameters of the network (the layout of LearnedGuess.params), FP32."""
    rng = np.random.default_rng(seed)
    out = []
    for kr, k, n in _CNN:
        w = np.zeros((9, n, k), np.float32)
        w[:, :, :kr] = rng.standard_normal((9, n, kr)) * math.sqrt(2.0 / (9 * kr))
        out += [w.ravel(), (0.02 * rng.standard_normal(n)).astype(np.float32)]
    out += [(rng.standard_normal(32) / math.sqrt(32)).astype(np.float32), np.zeros(1, np.float32)]
    return np.concatenate(out)


# the network's convolutions: real input channels, padded input channels, output channels
_CNN = [(4, 32, 32), (32, 32, 32), (32, 32, 64), (64, 64, 64), (64, 64, 128), (128, 128, 128), (192, 192, 64),
        (64, 64, 64), (96, 96, 32), (32, 32, 32)]


def _cnn_sample(rng, H, W):
    """A training sample with the network's input scales: rho, mask, boundary phi, inversion; target."""
    rho = 1.4 * (1.0 + _waves(rng, W, H, 4, 0.5)) * np.maximum(1 + 0.16 * rng.standard_normal((H, W)), 0.05)
    mask = np.zeros((H, W))
    mask[:, 0] = 1.0
    inv = 0.02 * np.log(np.maximum(rho * 1e6, 1.0))
    x4 = np.stack([rho, mask, np.zeros((H, W)), inv], -1).astype(np.float32)
    target = (inv * (1.0 - np.exp(-np.arange(W) / 6.0))[None, :]).astype(np.float32)
    return x4, target, (1 - mask).astype(np.uint8)


def _cnn_scene(case):
    """The deck whose rho the guess is made for."""
    return {"domain": "XY", "ni": case["ni"], "nj": case["nj"], "linear": False, "object": False}


def prepare(case, seed):
    s = State(case)
    work = case["work"]
    rng = np.random.default_rng(seed)
    if work == "loop":
        ni, nj, n = case["ni"], case["nj"], case["particles"]
        if (ni, nj) == (81, 41):
            deck = D.config_c1(seed=seed)
            deck.preload = (n, (7000.0, 0.0, 0.0), 1000.0)
        else:
            deck = D.config_c2(particles=n, ni=ni, nj=nj)
            deck.dt *= 1023 / (ni - 1)
            deck.seed = seed
        s.sim = Simulation(deck, capacity=int(1.6 * n) + 2_000_000, device_sources=case["device_sources"])
        s.sim.materials[0].preload(*deck.preload, seed=seed)
        s.sim.initial_solve()
        s.sim.run(2)
        nn = ni * nj
        s.buf = [np.ones(nn) for _ in range(2)]
        s.out = [np.ones(nn, np.float32) for _ in range(2)]
    elif work == "push":
        deck = _push_deck(case)
        n = case["particles"]
        s.sim = Simulation(deck, capacity=n + n // 64 + 1024)
        s.sim.materials[0].preload(*deck.preload, seed=seed)
        _set_waves(s.sim, rng, 100.0 if case["domain"] == "XY" else 1000.0)
        if case["b"]:
            m = deck.mesh
            s.sim.set_bfield(0.02 + _waves(rng, m.ni, m.nj, 3, 0.01).ravel(), _waves(rng, m.ni, m.nj, 3, 0.01).ravel())
        s.buf = [np.ones(s.sim.nn) for _ in range(4)]
    elif work == "solve":
        s.sim = Simulation(_solve_deck(case), capacity=16)
        before, s.rho = _rho(case, seed)
        s.guess = np.zeros(s.sim.nn)
        if case["start"] == "warm":
            s.sim.ctx.call("sf_rho_set", _dp(before))
            s.sim.ctx.call("sf_poisson_solve", _dp(s.guess), None)
        s.phi = np.ones(s.sim.nn)
        s.out = np.ones(s.sim.nn, np.float32)
        s.info = _lib.SolveInfo()
    elif work == "mcc":
        n = case["particles"]
        deck = _push_deck({"domain": "RZ", "ni": case["ni"], "nj": case["nj"], "particles": n})
        s.sim = Simulation(deck, capacity=n + 1024, track_ids=True)
        s.sim.materials[0].preload(n, (0.0, 2000.0, 0.0), 300.0, seed=seed)
        s.coll = MccHip(s.sim, s.sim.materials[0], case["model"], 5e-19, 131.0, seed=seed)
        f = lambda amp: _waves(rng, case["ni"], case["nj"], 3, amp).ravel()  # noqa: E731
        s.coll.set_target(case["density"] * (1.0 + f(0.5)), u=f(20.0), v=100.0 + f(20.0), w=f(5.0), temp=300.0 + f(50.0))
        s.buf = [np.ones(s.sim.nn) for _ in range(2)]
    elif work == "dsmc":
        ni, nj, n = case["ni"], case["nj"], case["particles"]
        mesh = D.MeshSpec("XY", ni, nj, (0.0, 0.0), (1e-4, 1e-4), {f: ("SYMMETRY", 0.0) for f in D.FACES})
        spwt = 1e22 * (ni - 1) * (nj - 1) * 1e-8 / n
        mats = [D.MaterialSpec("N2", "kinetic_hip", 28.0, 0.0, spwt, 0.0)]
        if case["pair"]:
            mats.append(D.MaterialSpec("Ar", "kinetic_hip", 40.0, 0.0, spwt, 0.0))
        deck = D.Deck(mesh, materials=mats, solver=None, num_it=1, dt=1e-8, seed=1)
        s.sim = Simulation(deck, capacity=n // len(mats) + 1024, track_ids=True, vmax=5000.0)
        for k, mat in enumerate(s.sim.materials):
            mat.preload(n // len(mats), (500.0, 0.0, 0.0), 300.0, seed=seed + k)
        a, b = s.sim.materials[0], s.sim.materials[-1]
        s.coll = DsmcHip(s.sim, a, b, sig_cr_max=1e-16, seed=seed, sigma="bird463",
                         diam=(4.17e-10, 4.17e-10), ref_temp=(273.0, 273.0), visc_temp_index=(0.74, 0.81)
                         if case["pair"] else (0.74, 0.74), vss_alpha=(1.36, 1.4) if case["pair"] else (1.0, 1.0))
        s.buf = [np.ones(s.sim.nn) for _ in range(5)]
    else:
        if case["mode"] == "guess":
            scene = _cnn_scene(case)
            s.sim = Simulation(_solve_deck(scene), capacity=16)
            s.sim.ctx.call("sf_rho_set", _dp(_rho(scene, seed)[1]))
            s.net = LearnedGuess(s.sim.ctx, max_batch=1, seed=seed)
            s.phi = np.ones(s.sim.nn)
            s.out = np.ones(s.sim.nn, np.float32)
        else:
            from starfish_amd.plugin import Context
            s.ctx = Context(0)
            s.net = LearnedGuess(s.ctx, ni=case["ni"], nj=case["nj"], max_batch=case["batch"], seed=seed)
            for _ in range(case["batch"]):
                s.net.add_sample(*_cnn_sample(rng, s.net.H, s.net.W))
        s.net.set_params(_cnn_params(seed))
    return s


# ------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------
def _fields(s, mat, names, bufs):
    """Species fields into the arrays that the program keeps for them."""
    for name, buf in zip(names, bufs):
        s.sim.ctx.call("sf_species_field", mat.index, _lib.FIELD[name], _dp(buf))


def run(s):
    case = s.case
    work = case["work"]
    if work == "loop":
        s.sim.run(case["steps"])
        s.sim.ctx.call("sf_phi_get", _dp(s.buf[0]))
        _fields(s, s.sim.materials[0], ["nd"], s.buf[1:])
        for a, b in zip(s.out, s.buf):
            np.copyto(a, b, casting="same_kind")
        return {"phi": s.out[0], "nd": s.out[1]}
    if work == "push":
        mat = s.sim.materials[0]
        for _ in range(case["steps"]):
            mat.update()
        _fields(s, mat, ["nd", "u", "v", "w"], s.buf)
        return {"nd": s.buf[0], "u": s.buf[1], "v": s.buf[2], "w": s.buf[3]}
    if work == "solve":
        np.copyto(s.phi, s.guess)
        s.sim.ctx.call("sf_rho_set", _dp(s.rho))
        s.sim.ctx.call("sf_poisson_solve", _dp(s.phi), C.byref(s.info))
        np.copyto(s.out, s.phi, casting="same_kind")
        return {"phi": s.out}
    if work == "mcc":
        n = 0
        for _ in range(case["steps"]):
            n += s.coll.perform(s.it, s.it * s.sim.deck.dt)
            s.it += 1
        for k, buf in zip((0, 4), s.buf):    # col-count-sum, the target's energy source
            s.coll._call("sf_mcc_field", k, _dp(buf))
        return {"collisions": n, "count": s.buf[0], "S": s.buf[1]}
    if work == "dsmc":
        n = 0
        for _ in range(case["steps"]):
            for mat in s.sim.materials:
                mat.update()
            n += s.coll.perform(s.it)
            s.it += 1
        s.coll._call("sf_dsmc_field", 0, _dp(s.buf[0]))
        mat = s.sim.materials[0]
        mat.update()                         # the collided velocities, as the next step's fields
        _fields(s, mat, ["nd", "u", "v", "w"], s.buf[1:])
        return {"collisions": n, "count": s.buf[0], "nd": s.buf[1], "u": s.buf[2], "v": s.buf[3], "w": s.buf[4]}
    if case["mode"] == "train":
        loss = s.net.train(1, batch=case["batch"], lr=1e-3)
        return {"loss": np.float32(loss), "params": s.net.params()}
    if case["mode"] == "grads":
        loss, y, g = s.net.loss_and_grads(0)
        return {"loss": np.float32(loss), "y": y, "grads": g}
    s.net.predict(s.sim)
    s.sim.ctx.call("sf_phi_get", _dp(s.phi))
    np.copyto(s.out, s.phi, casting="same_kind")
    return {"phi": s.out}


def work(case):
    nn = case["ni"] * case["nj"]
    w = case["work"]
    if w == "loop":      # state read and written, seven sums read and written, rho, phi, E; fields out
        return {"bytes": case["steps"] * (48.0 * case["particles"] + nn * (7 * 16 + 8 * 8)) + 16.0 * nn,
                "flops": case["steps"] * (150.0 * case["particles"] + 20.0 * nn)}
    if w == "push":
        return {"bytes": case["steps"] * (48.0 * case["particles"] + nn * (7 * 16 + 4 * 8 + 8)) + 32.0 * nn,
                "flops": case["steps"] * 150.0 * case["particles"]}
    if w == "solve":     # rho and the guess in, phi out (iterations are not counted)
        return {"bytes": 24.0 * nn, "flops": 40.0 * nn}
    if w == "mcc":       # cell, position, velocity and id of every particle read
        return {"bytes": case["steps"] * 28.0 * case["particles"] + 16.0 * nn, "flops": case["steps"] * 60.0 * case["particles"]}
    if w == "dsmc":      # one push, one counting sort and the collision pass a step
        return {"bytes": case["steps"] * (48.0 + 56.0 + 28.0) * case["particles"] + 48.0 * case["particles"],
                "flops": case["steps"] * 200.0 * case["particles"]}
    H, W = (case["nj"] + 3) // 4 * 4, (case["ni"] + 3) // 4 * 4
    div = [1, 1, 2, 2, 4, 4, 2, 2, 1, 1]
    fwd = sum(2.0 * 9 * kr * n * (H // d) * (W // d) for (kr, _, n), d in zip(_CNN, div)) * case["batch"]
    par = sum(9 * k * n + n for _, k, n in _CNN) + 33
    if case["mode"] == "guess":
        return {"bytes": 16.0 * nn + 4.0 * par, "flops": fwd}
    out = 16.0 * par if case["mode"] == "train" else 4.0 * par + 4.0 * H * W
    return {"bytes": 13.0 * H * W * case["batch"] + 4.0 * par + out, "flops": 3.0 * fwd}


# ------------------------------------------------------------------------------------------
# the same results in 64 bits
# ------------------------------------------------------------------------------------------
def _exact_phi(case, rho):
    """The discrete Boltzmann-electron Poisson problem on a rectangle without objects, by Newton
    with diagonally preconditioned conjugate gradients in FP64 on the reduced system: interior
    nodes are unknowns, Dirichlet faces are known, the other faces (zero normal gradient) take the
    value of their inner neighbour; the row of a node is scaled by its control volume."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    deck = _solve_deck(case)
    m = deck.mesh
    ni, nj, (hx, hy) = m.ni, m.nj, m.dh
    eps, kte, n0 = 8.85418782e-12, deck.solver.Te0, deck.solver.n0
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
    i, j = t(np.arange(1, ni - 1, dtype=float))[None, :], t(np.arange(1, nj - 1, dtype=float))[:, None]
    one = torch.ones((nj - 2, ni - 2), dtype=torch.float64, device=dev)
    if case["domain"] == "RZ":
        cE, cW, cN, cS, V = (i + 0.5) * hy * one, (i - 0.5) * hy * one, i * hx * hx / hy * one, None, 2 * math.pi * hx * hy * i * hx * one
    elif case["domain"] == "ZR":
        cN, cS, cE, cW, V = (j + 0.5) * hx * one, (j - 0.5) * hx * one, j * hy * hy / hx * one, None, 2 * math.pi * hx * hy * j * hy * one
    else:
        cE, cW, cN, cS, V = hy / hx * one, None, hx / hy * one, None, hx * hy * one
    cW = cE if cW is None else cW
    cS = cN if cS is None else cS
    sides = {"RIGHT": (cE, (slice(None), -1)), "LEFT": (cW, (slice(None), 0)), "TOP": (cN, (-1, slice(None))),
             "BOTTOM": (cS, (0, slice(None)))}
    # a face that is not Dirichlet: its node equals the inner one, so the link drops out
    links = {f: c.clone() for f, (c, _) in sides.items()}
    fix, value = torch.zeros_like(one), {}
    for f, (_, at) in sides.items():
        kind, val = m.mesh_bc.get(f, ("OPEN", 0.0))
        value[f] = val if kind == "DIRICHLET" else None
        if kind == "DIRICHLET":
            fix[at] += links[f][at] * val
        else:
            links[f][at] = 0.0
    diag = links["RIGHT"] + links["LEFT"] + links["TOP"] + links["BOTTOM"]
    lx, ly = links["RIGHT"][:, :-1], links["TOP"][:-1, :]

    def L(x):
        y = diag * x
        y[:, :-1] -= lx * x[:, 1:]
        y[:, 1:] -= lx * x[:, :-1]
        y[:-1, :] -= ly * x[1:, :]
        y[1:, :] -= ly * x[:-1, :]
        return y

    r = t(rho.reshape(nj, ni))[1:-1, 1:-1]
    lin = case["linear"]
    f = V * r / eps + fix
    Cn0 = 0.0 if lin else D.QE * n0 / eps
    x = torch.zeros_like(one) if lin else kte * torch.log(torch.clamp(r / (D.QE * n0), min=1e-8))
    for it in range(60):
        b = torch.zeros_like(x) if lin else Cn0 * torch.exp(x / kte)
        res = f - L(x) - V * b
        dj = diag + V * b / kte
        P = V * b / kte
        d, q = torch.zeros_like(one), res.clone()
        z = q / dj
        p, rz = z.clone(), (q * z).sum()
        stop = (1e-14 if lin else 1e-9) ** 2 * (q * q).sum()
        for k in range(40000):
            Ap = L(p) + P * p
            a = rz / (p * Ap).sum().clamp(min=1e-300)   # (a residual that is zero already stays zero)
            d += a * p
            q -= a * Ap
            z = q / dj
            new = (q * z).sum()
            if k % 32 == 31 and bool((q * q).sum() <= stop):
                break
            p = z + (new / rz.clamp(min=1e-300)) * p
            rz = new
        if not lin:
            d = torch.where(d > kte, kte * (1 + torch.log(torch.clamp(d / kte, min=1.0))), torch.clamp(d, min=-10 * kte))
        x = x + d
        if lin and it >= 1 or float(d.abs().max()) < 1e-11 * float(x.abs().max()):
            break
    phi = torch.zeros((nj, ni), dtype=torch.float64, device=dev)
    phi[1:-1, 1:-1] = x
    # a corner follows the left or right face's row, so those faces go last
    for f, at, inner in (("BOTTOM", (0, slice(1, -1)), (1, slice(1, -1))), ("TOP", (-1, slice(1, -1)), (-2, slice(1, -1))),
                         ("LEFT", (slice(None), 0), (slice(None), 1)), ("RIGHT", (slice(None), -1), (slice(None), -2))):
        phi[at] = phi[inner] if value[f] is None else value[f]
    for f, at in (("BOTTOM", (0, slice(None))), ("TOP", (-1, slice(None))), ("LEFT", (slice(None), 0)), ("RIGHT", (slice(None), -1))):
        if value[f] is not None:
            phi[at] = value[f]
    return phi.reshape(-1).cpu().numpy()


def _exact_net(params, x4):
    """The network in FP64: convolutions 3x3 with ReLU, three levels, skips, a 1x1 head on top of the
    input's fourth channel.  x4 [H, W, 4]; returns [H, W] and the parameter leaves."""
    leaves, ws, at = [], [], 0
    for kr, k, n in _CNN:
        w = torch.tensor(params[at:at + 9 * n * k].astype(np.float64).reshape(9, n, k), requires_grad=True)
        at += 9 * n * k
        b = torch.tensor(params[at:at + n].astype(np.float64), requires_grad=True)
        at += n
        leaves += [w, b]
        ws.append((w.reshape(3, 3, n, k).permute(2, 3, 0, 1)[:, :kr], b))
    hw = torch.tensor(params[at:at + 32].astype(np.float64), requires_grad=True)
    hb = torch.tensor(params[at + 32:].astype(np.float64), requires_grad=True)
    leaves += [hw, hb]
    conv = lambda x, k: torch.relu(F.conv2d(x, ws[k][0], ws[k][1], padding=1))  # noqa: E731
    up = lambda x: x.repeat_interleave(2, 2).repeat_interleave(2, 3)  # noqa: E731
    x = torch.tensor(x4.astype(np.float64)).permute(2, 0, 1)[None]
    e1 = conv(conv(x, 0), 1)
    e2 = conv(conv(F.avg_pool2d(e1, 2), 2), 3)
    e3 = conv(conv(F.avg_pool2d(e2, 2), 4), 5)
    d2 = conv(conv(torch.cat([up(e3), e2], 1), 6), 7)
    d1 = conv(conv(torch.cat([up(d2), e1], 1), 8), 9)
    return (d1 * hw[None, :, None, None]).sum(1)[0] + hb + x[0, 3], leaves


def exact(case, seed):
    if case["work"] == "solve" and not case["object"]:
        return {"phi": _exact_phi(case, _rho(case, seed)[1])}
    if case["work"] != "cnn" or case["mode"] == "train" or case["ni"] * case["nj"] > 200_000:
        return None
    H, W = (case["nj"] + 3) // 4 * 4, (case["ni"] + 3) // 4 * 4
    if case["mode"] == "grads":
        x4, target, mask = _cnn_sample(np.random.default_rng(seed), H, W)
        y, leaves = _exact_net(_cnn_params(seed), x4)
        e = (y - torch.tensor(target.astype(np.float64))) * torch.tensor(mask.astype(np.float64))
        loss = (e * e).sum() / (H * W)
        loss.backward()
        return {"loss": float(loss.detach()), "y": y.detach().numpy(),
                "grads": torch.cat([v.grad.reshape(-1) for v in leaves]).numpy()}
    ni, nj = case["ni"], case["nj"]
    rho = _rho(_cnn_scene(case), seed)[1].reshape(nj, ni)
    x4 = np.zeros((H, W, 4))
    x4[:nj, :ni, 0] = rho / (D.QE * 1e16)
    x4[:nj, 0, 1] = 1.0                                        # the Dirichlet face, at 0 V
    x4[:nj, :ni, 3] = 2.0 * np.log(np.maximum(rho / (D.QE * 1e10), 1.0)) / 100.0
    with torch.no_grad():
        y, _ = _exact_net(_cnn_params(seed), x4)
    return {"phi": 100.0 * y[:nj, :ni].numpy().reshape(-1)}
