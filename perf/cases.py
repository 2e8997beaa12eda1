"""Timed workloads of the engine: the calls that a user's program makes, over
the sizes and options it makes them with.

Three families, each through its public entry points:

* ``run``: molecular dynamics of a batch of windows (``Engine.run``), the
  production and pilot runs of free-energy ladders;
* ``score``: pair lists, energies and gradients of given frames
  (``Engine.set_state`` + ``Engine.evaluate``), as rescoring stored frames does;
* ``mlp_*``: the overlap predictor of the learned lambda schedule
  (``MLP.forward``, ``forward_device``, ``grad``, ``train``).

A case is a dict of plain values; ``prepare`` makes the inputs and the handle
that a program keeps, ``run`` is one pass.  The synthetic systems are seeded;
the seed of a case sets the Maxwell velocities, the frames, the network and
its rows.
"""
from __future__ import annotations

import functools
import math
import os
import tempfile

import numpy as np
import torch

from q_amd import synth
from q_amd.engine import Engine
from q_amd.mlp import MLP

# step count in the windows' input files: further than any program here goes
INP_STEPS = 2_000_000
# Coulomb constant of the topologies
COULOMB = 332.0716
# convention for counted work: FP operations per interacting pair or term
FLOP_WW, FLOP_PAIR, FLOP_Q, FLOP_LRF = 200, 32, 36, 90


def listed():
    return [
        # the schedule's call for one leg: 10 intervals of an 11-point pilot grid
        dict(name="mlp_predict_grid", kind="mlp_forward", n_in=34, hidden=128, rows=10),
        # the whole training set of the shipped network at once
        dict(name="mlp_predict_set", kind="mlp_forward", n_in=34, hidden=128, rows=7960),
        # a serving loop on device buffers and the caller's stream, ragged batch
        dict(name="mlp_serve_777", kind="mlp_device", n_in=35, hidden=128, rows=777),
        # loss and gradient over the training set, before and after a training
        dict(name="mlp_grad_set", kind="mlp_grad", n_in=34, hidden=128, rows=7960),
        # part of a training: one pass of minibatches of 256
        dict(name="mlp_train_2100", kind="mlp_train", n_in=34, hidden=128, rows=2100, batch=256),
        # rescoring frames: the smallest system (pure water, no LRF), and
        # a few windows of the largest one
        dict(name="score_droplet", kind="score", config="water", radius=15.0, windows=1),
        dict(name="score_protein_4", kind="score", config="protein", radius=25.0, windows=4),
        # one window per engine, as `qmi-qdyn <input>` runs it: either leg
        dict(name="run_ligwat_1", kind="run", config="ligwat", radius=20.0, windows=1, steps=100, energy=10, output=5),
        dict(name="run_protein_1", kind="run", config="protein", radius=25.0, windows=1, steps=100, energy=10,
             output=5),
        # the pilot grid of one leg: energies every 5 steps, no log summaries
        dict(name="run_pilots_11", kind="run", config="ligwat", radius=20.0, windows=11, steps=50, energy=5,
             output=INP_STEPS),
        # a short ladder with the 3-atom water model, small sphere
        dict(name="run_tip3_5", kind="run", config="ligtip3", radius=18.0, windows=5, steps=50, energy=10, output=50),
        # both legs of a perturbation in one engine, the throughput workload
        dict(name="run_ladder_64", kind="run", config="both", radius=25.0, windows=64, steps=50, energy=10, output=5),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "score", "mlp_forward", "mlp_device", "mlp_grad", "mlp_train"])
    if kind.startswith("mlp"):
        c = dict(kind=kind, n_in=rng.randint(8, 64), hidden=rng.choice([64, 96, 100, 128, 128, 128]))
        cap = 1_048_576 // (4 * c["hidden"] + 1) if kind == "mlp_device" else 7960
        c["rows"] = max(1, min(cap, round(_log_uniform(rng, 3, 7960))))
        if kind == "mlp_train":
            c["rows"] = 64 + c["rows"] // 3
            c["batch"] = rng.randint(32, 256)
        return c
    if kind == "score":
        c = dict(kind=kind, config=rng.choice(["water", "ligwat", "protein"]))
    else:
        c = dict(kind=kind, config=rng.choice(["water", "ligwat", "ligwat", "ligtip3", "ligarithlibq", "ligrestr",
                                               "protein", "both"]))
    big = c["config"] in ("protein", "both")
    c["radius"] = 25.0 if big else round(rng.uniform(14.0, 22.0), 1)
    if kind == "score":
        c["windows"] = max(1, round(_log_uniform(rng, 1, 4 if big else 12)))
        return c
    c["windows"] = max(2 if c["config"] == "both" else 1, round(_log_uniform(rng, 1, 30 if big else 60)))
    c["steps"] = rng.choice([25, 37, 50])
    c["energy"] = rng.choice([5, 10, 20])
    c["output"] = rng.choice([5, 50, INP_STEPS])
    return c


# ------------------------------------------------------------- molecules --
@functools.lru_cache(maxsize=None)
def _system(config, radius):
    """The synthetic system, which a program has as topology files: the
    ligand is the same for every radius, water fills the sphere."""
    builder, kw, _ = synth.CONFIGS[config]
    kw = dict(kw, radius=radius)
    return builder(seed=2 if config == "protein" else 0, **kw)


def _legs(case):
    """(config, radius, windows) of each leg of the case"""
    if case["config"] == "both":
        half = case["windows"] // 2
        return [("ligwat", 20.0, case["windows"] - half), ("protein", case["radius"], half)]
    return [(case["config"], case["radius"], case["windows"])]


def _engine(case, seed, folder, **inp):
    """An engine with the case's windows, prepared: lambda spread evenly over
    each leg's windows, a Maxwell seed per window."""
    e = Engine(0)
    sizes = []
    for leg, (config, radius, n) in enumerate(_legs(case)):
        system = _system(config, radius)
        d = os.path.join(folder, config)
        for k in range(n):
            path = synth.make_window(config, d, seed=0, md_seed=1 + (1000 * seed + 100 * leg + k) % 900_000,
                                     lam=k / (n - 1) if n > 1 else 0.5, steps=INP_STEPS,
                                     energy=case.get("energy", 10), output=case.get("output", 5),
                                     tag=f"w{k:02d}", system=system if k == 0 else None, **inp)
            w = e.add_window(path)
            if case.get("output", 5) == INP_STEPS:
                e.set_log(w, None)
            sizes.append((w, system.natom, len(system.qatoms) > 0))
    e.prepare()
    return e, sizes


def _frame(config, radius, seed, k):
    """A stored frame of window k: the system's coordinates with thermal
    displacements, waters moved as rigid bodies."""
    s = _system(config, radius)
    x = np.asarray(s.x, np.float64).reshape(-1, 3).copy()
    rng = np.random.default_rng([seed, k])
    x[:s.nat_solute] += rng.normal(0.0, 0.01, (s.nat_solute, 3))
    x[s.nat_solute:] += np.repeat(rng.normal(0.0, 0.1, ((len(x) - s.nat_solute) // 3, 3)), 3, axis=0)
    return x


# --------------------------------------------------------------- network --
def _rows(rng, n, n_in):
    """Predictor rows: a normalised histogram of the centred reduced work
    (160 samples, so far bins are empty), lambda, and the soft-core alpha."""
    bins = np.linspace(-1.0, 1.0, n_in - 2)
    mu = rng.normal(0.0, 0.05, (n, 1))
    sd = np.exp(rng.normal(-1.6, 0.6, (n, 1)))
    h = np.exp(-0.5 * ((bins - mu) / sd) ** 2) * np.exp(rng.normal(0.0, 0.2, (n, n_in - 2)))
    h /= h.sum(axis=1, keepdims=True)
    h = np.round(160 * h) / 160
    tail = np.stack([rng.integers(0, 11, n) / 10.0, np.ones(n)], axis=1)
    return np.concatenate([h, tail], axis=1).astype(np.float32)


def _network_inputs(case, seed):
    """(parameters, rows, targets) of the case, from the seed alone"""
    rng = np.random.default_rng([seed, case["n_in"], case["rows"]])
    n_in, H = case["n_in"], case["hidden"]
    parts = [rng.normal(0, (2 / n_in) ** 0.5, H * n_in), rng.normal(0, 0.1, H), rng.normal(0, (2 / H) ** 0.5, H * H),
             rng.normal(0, 0.1, H), rng.normal(0, (1 / H) ** 0.5, H), rng.normal(0, 0.1, 1)]
    x = _rows(rng, case["rows"], n_in)
    t = rng.beta(5.0, 2.0, case["rows"]).astype(np.float32)
    return np.concatenate(parts).astype(np.float32), x, t


# ------------------------------------------------------------ interface --
def prepare(case, seed):
    kind = case["kind"]
    if kind.startswith("mlp"):
        params, x, t = _network_inputs(case, seed)
        net = MLP(case["n_in"], case["hidden"], seed=0)
        net.params = params
        st = dict(case=case, net=net, x=x, t=t, seed=seed)
        if kind == "mlp_device":
            st["dx"] = torch.from_numpy(x).cuda()
            st["dy"] = torch.zeros(case["rows"], device="cuda")
            st["stream"] = torch.cuda.Stream()
        return st
    folder = tempfile.TemporaryDirectory(prefix="qmi_cases_")
    inp = {}
    if case["config"] == "water":
        inp["polarization"] = False
    e, sizes = _engine(case, seed, folder.name, **inp)
    st = dict(case=case, engine=e, sizes=sizes, folder=folder)
    if kind == "score":
        frames, w = [], 0
        for config, radius, n in _legs(case):
            for _ in range(n):
                frames.append(_frame(config, radius, seed, w))
                w += 1
        st["frames"] = frames
    return st


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    if kind == "mlp_forward":
        return st["net"].forward(st["x"])
    if kind == "mlp_device":
        st["net"].forward_device(st["dx"].data_ptr(), case["rows"], st["dy"].data_ptr(),
                                 st["stream"].cuda_stream)
        return st["dy"]
    if kind == "mlp_grad":
        loss, g = st["net"].grad(st["x"], st["t"])
        return {"loss": loss, "grad": g}
    if kind == "mlp_train":
        loss = st["net"].train(st["x"], st["t"], epochs=1, batch=case["batch"], lr=1e-3, seed=st["seed"])
        return {"loss": loss, "params": st["net"].params}
    e = st["engine"]
    if kind == "score":
        for (w, _, _), x in zip(st["sizes"], st["frames"]):
            e.set_state(w, x=x)
        e.evaluate(rebuild_lists=True)
        if case["windows"] == 1:
            out = {"energies": e.energies(0), "forces": e.forces(0)}
            if st["sizes"][0][2]:
                out["q_energies"] = e.q_energies(0)
            return out
        return {"energies": np.array([list(e.energies(w).values()) for w, _, _ in st["sizes"]]),
                "q_energies": np.concatenate([np.zeros((0, 15))] + [e.q_energies(w) for w, _, q in st["sizes"] if q]),
                "forces": np.concatenate([e.forces(w) for w, _, _ in st["sizes"]])}
    # molecular dynamics: the next `steps` steps of every window.  Positions
    # and velocities come back as the FP32 frames that trajectory files hold,
    # the energies with the digits of the log.
    e.run(case["steps"], finalize=False)
    x = np.concatenate([e.coords(w) for w, _, _ in st["sizes"]]).astype(np.float32)
    v = np.concatenate([e.velocities(w) for w, _, _ in st["sizes"]]).astype(np.float32)
    energies = np.array([list(e.energies(w).values()) for w, _, _ in st["sizes"]], np.float32)
    out = {"x": x, "v": v, "energies": energies}
    with_q = [e.q_energies(w) for w, _, q in st["sizes"] if q]
    if with_q:
        out["q_energies"] = np.concatenate(with_q).astype(np.float32)
    return out


# ----------------------------------------------------------------- work --
@functools.lru_cache(maxsize=None)
def _counts(config, radius):
    """Per window: atoms, water-water molecule pairs, solute-water and
    solute-solute pairs, q pairs, LRF source terms (target groups x charges)"""
    s = _system(config, radius)
    ikw = synth.CONFIGS[config][2]
    x = np.asarray(s.x, np.float32).reshape(-1, 3)
    isq = np.zeros(len(x), bool)
    isq[[a - 1 for a in s.qatoms]] = True
    o = x[s.nat_solute::3]
    p = x[:s.nat_solute][~isq[:s.nat_solute]]
    rcs, rcw = ikw.get("rc_solute", 11.0), 10.0

    def within(a, b, rc):
        n = 0
        for k in range(0, len(a), 256):
            d2 = ((a[k:k + 256, None, :] - b[None, :, :]) ** 2).sum(-1)
            n += int((d2 <= rc * rc).sum())
        return n

    ww = (within(o, o, rcw) - len(o)) // 2
    pw = 3 * within(p, o, rcs)
    pp = (within(p, p, rcs) - len(p)) // 2
    nq = int(isq.sum())
    q = 2 * nq * (len(x) - nq) + nq * nq
    lrf = len(s.cgps) * (len(x) - nq) if ikw.get("lrf", True) else 0
    return len(x), ww, pw, pp, q, lrf


def work(case):
    kind = case["kind"]
    if kind.startswith("mlp"):
        n, n_in, H = case["rows"], case["n_in"], case["hidden"]
        np_ = H * n_in + H * H + 3 * H + 1
        if kind == "mlp_train":
            n = n // case["batch"] * case["batch"]
            # per minibatch: parameters and both Adam moments read and written
            return {"bytes": 4.0 * n * (n_in + 1) + 24.0 * np_ * (n // case["batch"]), "flops": 6.0 * n * np_}
        if kind == "mlp_grad":
            return {"bytes": 4.0 * n * (n_in + 1) + 6.0 * np_, "flops": 6.0 * n * np_}
        return {"bytes": 4.0 * n * (n_in + 1) + 2.0 * np_, "flops": 2.0 * n * np_}
    atoms = flops = lrf = 0.0
    for config, radius, n in _legs(case):
        a, ww, pw, pp, q, l = _counts(config, radius)
        atoms += n * a
        flops += n * (FLOP_WW * ww + FLOP_PAIR * (pw + pp) + FLOP_Q * q + 100.0 * a)
        lrf += n * FLOP_LRF * l
    if kind == "score":
        return {"bytes": 48.0 * atoms, "flops": flops + lrf}
    # positions and velocities in and out; lists and LRF expansions every 25
    # steps
    return {"bytes": 96.0 * atoms, "flops": flops * case["steps"] + lrf * case["steps"] / 25.0}


# ---------------------------------------------------------------- exact --
def _bf16(a):
    return torch.from_numpy(a).to(torch.bfloat16).to(torch.float64)


def _exact_network(case, seed, with_grad):
    params, x, t = _network_inputs(case, seed)
    n_in, H = case["n_in"], case["hidden"]
    sizes = [H * n_in, H, H * H, H, H, 1]
    w1, b1, w2, b2, w3, b3 = np.split(params, np.cumsum(sizes)[:-1])
    w1, w2, w3 = _bf16(w1).reshape(H, n_in), _bf16(w2).reshape(H, H), _bf16(w3).reshape(1, H)
    b1, b2, b3 = (torch.from_numpy(b).double() for b in (b1, b2, b3))
    leaf = [v.requires_grad_(with_grad) for v in (w1, b1, w2, b2, w3, b3)]
    xd, td = torch.from_numpy(x).double(), torch.from_numpy(t).double()
    h = torch.nn.functional.silu(xd @ w1.T + b1)
    h = torch.nn.functional.silu(h @ w2.T + b2)
    y = torch.sigmoid(h @ w3.T + b3)[:, 0]
    if not with_grad:
        return y.numpy()
    loss = ((y - td) ** 2).mean()
    loss.backward()
    return {"loss": loss.detach().numpy(), "grad": np.concatenate([v.grad.numpy().ravel() for v in leaf])}


def _exact_water_energies(case, seed):
    """Electrostatic and LJ energy of the water-water pairs of the frame: O-O
    distances within the cut-off, all nine sites, LJ between the oxygens;
    charges in single precision and LJ columns with the digits of a topology
    file, as the engine reads them"""
    x = _frame(case["config"], case["radius"], seed, 0)
    o = x[0::3]
    ow = synth.LJ_TYPES[synth.T_OW - 1]
    ra, rb = synth.lj_sqrt(ow[1], ow[2])
    lj_a, lj_b = round(ra, 4) ** 2, round(rb, 5) ** 2
    sq = np.float32(math.sqrt(COULOMB))
    c = np.array([synth.SPC_QO, -synth.SPC_QO / 2, -synth.SPC_QO / 2], np.float32) * sq
    el = vdw = 0.0
    for i in range(len(o) - 1):
        d = o[i + 1:] - o[i]
        j = np.nonzero((d ** 2).sum(1) <= 100.0)[0] + i + 1
        for a in range(3):
            for b in range(3):
                r = np.sqrt(((x[3 * j + b] - x[3 * i + a]) ** 2).sum(1))
                el += float((np.float64(c[a] * c[b]) / r).sum())
                if a == 0 and b == 0:
                    vdw += float((lj_a / r ** 12 - lj_b / r ** 6).sum())
    return {"ww.el": el, "ww.vdw": vdw}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mlp_forward", "mlp_device"):
        return _exact_network(case, seed, False)
    if kind == "mlp_grad":
        return _exact_network(case, seed, True)
    if kind == "score" and case["config"] == "water" and case["windows"] == 1:
        return {"energies": _exact_water_energies(case, seed), "forces": None}
    # trajectories are chaotic, a training's shuffles and rounded weights are
    # its own, and a whole force field of a solvated solute is the library
    return None
