"""The framework's work as cases that can be timed and compared.

Five kinds of case, each through the package's public entry points:

* ``box``: one engine on a graded or uniform grid (PEC walls, CPML or
  openEMS PML layers, dielectric blocks, dispersive spheres), fields already
  everywhere, a soft source and voltage probes; a pass runs ``steps`` time
  steps, the last of them with the energy check of the run loop.
* ``scatter``: the composite model (CPML, Lorentz and Drude spheres, a
  conformal PEC cylinder with its reduced currents, a TF/SF plane wave).
* ``sweep``: many patch antennas stepped together, then one energy check of
  all of them and their port traces.
* ``train``: Adam steps of the early-stop network on traces held by the
  device.
* ``predict``: the network's prediction of a sweep's late traces from host
  arrays.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import ems_amd as E
from ems_amd import workloads as W
from ems_amd.learn import _batch_engines

F = E.Face


def listed():
    box = {"kind": "box", "layers": "pec", "cells": 8, "graded": False, "blocks": 0, "spheres": 0,
           "openems": False}
    return [
        # The smoke model, stepped one step at a time by a program that looks
        # at the fields after each step: launches and latency are all of it.
        {**box, "name": "box_24_single_steps", "nx": 24, "ny": 24, "nz": 24, "steps": 1},
        # The reference's own bench (50^3 vacuum, PEC): one check interval.
        {**box, "name": "box_50_vacuum", "nx": 50, "ny": 50, "nz": 50, "steps": 50},
        # An ordinary antenna-sized model: odd sizes, graded mesh, dielectric
        # blocks, CPML on every face; two check intervals.
        {**box, "name": "box_cpml_mid", "nx": 131, "ny": 97, "nz": 74, "steps": 100,
         "layers": "cpml", "graded": True, "blocks": 8},
        # The same with Lorentz spheres (pole updates beside the fused step).
        {**box, "name": "box_lorentz", "nx": 120, "ny": 110, "nz": 96, "steps": 100,
         "layers": "cpml", "graded": False, "blocks": 2, "spheres": 4},
        # An openEMS model run as openEMS runs it: its curl order, PML_8 on
        # every face, its energy measure at its check.
        {**box, "name": "box_openems_pml", "nx": 141, "ny": 112, "nz": 90, "steps": 60,
         "layers": "pml", "graded": True, "blocks": 4, "openems": True},
        # The benchmark's box: 512^3 cells, 8-cell CPML, 64 FR-4 blocks.
        {**box, "name": "box_cpml_512", "nx": 512, "ny": 512, "nz": 512, "steps": 50,
         "layers": "cpml", "graded": True, "blocks": 64},
        # The dispersive / conformal / plane-wave model at half the
        # benchmark's size along each axis: one check interval.
        {"kind": "scatter", "name": "scatter_192", "nx": 192, "ny": 192, "nz": 128, "pml": 10,
         "lorentz": 8, "drude": 4, "radius": 20, "steps": 50},
        # A few antennas of a design under work.
        {"kind": "sweep", "name": "sweep_8", "models": 8, "steps": 50},
        # The benchmark's sweep: 256 uneven models, one check interval.
        {"kind": "sweep", "name": "sweep_256", "models": 256, "steps": 50},
        # The early-stop network's training as learn.train runs it (with the
        # spectral loss term): eight Adam steps of 32 traces.
        {"kind": "train", "name": "train_32", "batch": 32, "T": 512, "channels": 64, "steps": 8},
        # One model's prediction while its solve waits.
        {"kind": "predict", "name": "predict_1", "batch": 1, "T": 512, "channels": 64},
        # The predictions of a whole sweep.
        {"kind": "predict", "name": "predict_256", "batch": 256, "T": 512, "channels": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["box"] * 5 + ["scatter", "sweep", "sweep", "train", "predict", "predict"])
    if kind == "box":
        layers = rng.choice(["pec", "cpml", "cpml", "pml"])
        hi = 180 if layers == "pml" else 330
        n = [_log(rng, 24, hi) for _ in range(3)]
        # short runs of large grids, long ones of small grids
        most = min(200, int(2.0e9 / (n[0] * n[1] * n[2])))
        return {"kind": "box", "layers": layers, "cells": rng.choice([6, 8, 10]),
                "graded": rng.random() < 0.6, "blocks": rng.randrange(0, 12),
                "spheres": rng.choice([0, 0, 0, 3]) if layers == "cpml" and min(n) > 60 else 0,
                "openems": layers == "pml" or rng.random() < 0.15,
                "nx": n[0], "ny": n[1], "nz": n[2], "steps": _log(rng, 1, max(2, most))}
    if kind == "scatter":
        n = [rng.randrange(96, 200) for _ in range(2)]
        return {"kind": "scatter", "nx": n[0], "ny": n[1], "nz": rng.randrange(72, 140),
                "pml": rng.choice([6, 8, 10]), "lorentz": rng.randrange(2, 6),
                "drude": rng.randrange(1, 4), "radius": rng.randrange(8, 15),
                "steps": rng.randrange(10, 60)}
    if kind == "sweep":
        return {"kind": "sweep", "models": _log(rng, 2, 200), "steps": rng.randrange(20, 60)}
    if kind == "train":
        return {"kind": "train", "batch": _log(rng, 4, 48), "T": rng.choice([256, 384, 500, 512]),
                "channels": rng.choice([32, 48, 64]), "steps": rng.randrange(1, 9)}
    return {"kind": "predict", "batch": _log(rng, 1, 400), "T": rng.randrange(200, 600),
            "channels": rng.choice([32, 48, 64, 64])}


# ---------------------------------------------------------------- models --

_kept = {}


def _model(key, build):
    """The compiled arrays of the last few geometries (a program that tries
    other excitations on a geometry compiles it once)."""
    if key not in _kept:
        while len(_kept) >= 3:
            _kept.pop(next(iter(_kept)))
        _kept[key] = build()
    return _kept[key]


def _nodes(c):
    return c["nx"] + 1, c["ny"] + 1, c["nz"] + 1


def _spheres(c):
    """Cell masks of the seeded dispersive spheres: (radius, centre) each."""
    rng = np.random.default_rng(77)
    n = (c["nx"], c["ny"], c["nz"])
    mask = np.zeros(n, dtype=bool)
    for _ in range(c["spheres"]):
        r = float(rng.uniform(4.0, 8.0))
        lo = c["cells"] + 2 + r
        p = [float(rng.uniform(lo, n[a] - lo)) for a in range(3)]
        box = [slice(int(p[a] - r) - 1, int(p[a] + r) + 2) for a in range(3)]
        ax = [np.arange(s.start, s.stop) + 0.5 - p[a] for a, s in enumerate(box)]
        mask[tuple(box)] |= (ax[0][:, None, None] ** 2 + ax[1][None, :, None] ** 2 +
                             ax[2][None, None, :] ** 2) < r * r
    return mask


def _box_model(c):
    """Grid, time step and coefficient lanes of a box."""
    rng = np.random.default_rng(2026)
    n = (c["nx"], c["ny"], c["nz"])
    if c["graded"]:
        g = E.Grid([W.graded_lines(q, rng) for q in n])
    else:
        g = E.Grid.uniform(n, [1e-3] * 3)
    m = E.CellMaterials.vacuum(g)
    fr4 = E.Material.dielectric(4.3).with_kappa(0.02)
    edge = c["cells"] + 2
    for _ in range(c["blocks"]):
        lo, hi = [], []
        for a in range(3):
            free = n[a] - 2 * edge
            if free < 2:
                break
            size = int(rng.integers(min(10, free), min(60, free) + 1))
            lo.append(edge + int(rng.integers(0, free - size + 1)))
            hi.append(lo[-1] + size)
        if len(lo) == 3:
            m.fill_box(list(zip(lo, hi)), fr4)
    mask = None
    if c["spheres"]:
        mask = _spheres(c)
        m.ids[mask] = m._id(E.Material.dielectric(2.0))
    dt = E.TimeStep.courant(0.99).resolve(g)
    lanes = E.coefficients(g, m, [E.FaceCondition.Pec] * 6, dt,
                           1 if c["openems"] else 0)
    return g, dt, lanes, mask


def _fields(n, seed, comps):
    """Smooth-enough voltages everywhere inside the walls, separable so that
    the largest grid's are made quickly."""
    rng = np.random.default_rng([1009, seed])
    out = {}
    for a in range(3):
        v = [rng.standard_normal(q).astype(np.float32) for q in n]
        for t in range(3):
            v[t][0] = v[t][-1] = 0.0
            if t == a and n[t] > 2:
                v[t][-2] = 0.0
        if a in comps:
            out[a] = 1e-3 * v[0][:, None, None] * (v[1][:, None] * v[2][None, :])[None]
    return out


def _points(n, seed, count):
    rng = np.random.default_rng([2003, seed])
    return [[int(rng.integers(2, max(3, q - 2))) for q in n] for _ in range(count)]


class _Box:
    pass


def _prepare_box(c, seed):
    key = tuple(sorted((k, v) for k, v in c.items() if k not in ("name", "steps")))
    g, dt, lanes, mask = _model(key, lambda: _box_model(c))
    n = g.nodes()
    s = _Box()
    s.case = c
    s.engine = e = E.Engine(g, dt, lanes, curl_order=1 if c["openems"] else 0)
    s.pml = s.cpml = s.poles = None
    if c["layers"] == "cpml":
        s.cpml = E.CpmlBoundary.new(e, [(f, E.Cpml.with_cells(min(c["cells"], (min(n) - 1) // 3)))
                                        for f in F])
        e.add_operator(s.cpml)
    if mask is not None:
        s.poles = E.Dispersive.new()
        w0 = 2.0 * math.pi * 8e9
        s.poles.fill_mask(g, mask, E.Field.Electric,
                          [E.Pole.lorentz(math.sqrt(3.0) * w0, w0, 2.0 * math.pi * 1e9)])
        e.add_operator(s.poles)
    if c["layers"] == "pml":
        s.pml = E.OpenEmsPml.new(e, [(f, min(c["cells"], (min(n) - 1) // 3)) for f in F])
        e.add_operator(s.pml)
    comps = (2,) if g.num_nodes() > 20_000_000 else (0, 1, 2)
    s.start = _fields(n, seed, comps)
    for a, v in s.start.items():
        e.set_component(0, a, v)
    s.source = (_points(n, seed, 1)[0], E.Waveform.gaussian(5e9, 4e9), 1e-2 * (1 + seed % 7))
    e.add_operator(E.EdgeSource(s.source[1]).edge(E.Axis.Z, s.source[0], s.source[2]))
    # the benchmark's 16 points in all components on a large grid, a few
    # points on a small one (whose fields are read whole)
    s.whole = g.num_nodes() <= 2_500_000
    s.at = _points(n, 17, 2 if s.whole else 16)
    s.probes = [e.add_operator(E.Probe.voltage(a, p)) for p in s.at for a in range(3)]
    s.lanes = e.coefficients()
    e.release_dense_lanes()
    s.taken = 0
    return s


def _run_box(s):
    c, e = s.case, s.engine
    if c["steps"] > 1:
        e.run(c["steps"] - 1)
    if c["openems"]:
        e.run(1)
        w = e.energy_openems()
    else:
        w = e.step_with_energy()
    out = {"energy": np.array([w])}
    if s.whole:  # the program looks at the fields
        out["u"] = [e.u_component(a) for a in range(3)]
        out["i"] = [e.i_component(a) for a in range(3)]
    else:        # the program takes the traces since its last look
        v = [p.values() for p in s.probes]
        out["probes"] = np.stack([x[s.taken:] for x in v])
        s.taken = v[0].size
    return out


def _scatter_model(c):
    return W.dispersive_box((c["nx"], c["ny"], c["nz"]), pml=c["pml"], lorentz=c["lorentz"],
                            drude=c["drude"], cylinder_cells=float(c["radius"]),
                            radii=(4.0, 8.0), skip_stability=True)


def _prepare_scatter(c, seed):
    key = tuple(sorted((k, v) for k, v in c.items() if k not in ("name", "steps")))
    wl = _model(key, lambda: _scatter_model(c))
    s = _Box()
    s.case = c
    s.engine = e = E.Engine(wl.grid, wl.dt, wl.lanes)
    s.probes = wl.build_ops(e)
    for a, v in _fields(wl.grid.nodes(), seed, (0, 1, 2)).items():
        e.set_component(0, a, np.where(e.coefficients()[3 + a] == 0.0, np.float32(0.0), v))
    e.release_dense_lanes()
    s.whole, s.taken = wl.grid.num_nodes() <= 2_500_000, 0
    s.case = {**c, "openems": False}
    return s


def _prepare_sweep(c, seed):
    models = W.patch_sweep(c["models"], seed=4242 + seed)
    s = _Box()
    s.case, s.models = c, models
    s.engines, s.ports = _batch_engines(models)
    s.batch = E.EngineBatch(s.engines)
    s.batch.set_schedule(7, 16, packed=True)
    s.taken = 0
    return s


def _run_sweep(s):
    s.batch.run(s.case["steps"])
    w = E.energy_many(s.engines)
    v = [p.voltage() for p in s.ports]
    i = [p.current() for p in s.ports]
    out = {"energy": np.array(w), "v": np.stack([x[s.taken:] for x in v]),
           "i": np.stack([x[s.taken:] for x in i])}
    s.taken = v[0].size
    return out


# ---------------------------------------------------------------- network --

_DIL = (1, 2, 4, 8, 16, 32)


def _traces(c, seed, count):
    """Network sequences of port traces: decaying two-tone ringing after a
    Gaussian pulse, observed over the first quarter; [n][4][T], [n][2][T]."""
    rng = np.random.default_rng([3001, seed])
    T, N = c["T"], c["T"] // 4
    t = np.arange(T)
    src = (np.exp(-((t - 0.15 * T) / (0.05 * T)) ** 2) * np.cos(0.35 * (t - 0.15 * T)))
    y = np.zeros((count, 2, T))
    for ch in range(2):
        a, f, d, ph = (rng.uniform(lo, hi, (count, 2, 1)) for lo, hi in
                       ((0.1, 0.5), (0.2, 0.5), (3.0 / T, 12.0 / T), (0.0, 6.28)))
        ring = (a * np.exp(-d * np.maximum(t - 0.15 * T, 0.0)) *
                np.cos(f * t + ph) * (t > 0.1 * T)).sum(axis=1)
        y[:, ch] = 0.5 * src + ring
    x = np.zeros((count, 4, T), np.float32)
    x[:, 0, :N], x[:, 1, :N], x[:, 2, :N], x[:, 3] = y[:, 0, :N], y[:, 1, :N], 1.0, src
    return x, y.astype(np.float32)


def _params(c, seed):
    """Weights as a net under training has them (its start's scale)."""
    rng = np.random.default_rng([4001, seed])
    C, L = c["channels"], len(_DIL)
    p = []
    for l in range(L):
        ci, co = (4 if l == 0 else C), (2 if l == L - 1 else C)
        p.append((rng.standard_normal(co * ci * 9) / math.sqrt(9 * ci)).astype(np.float32))
        p.append((0.05 * rng.standard_normal(co)).astype(np.float32))
    return np.concatenate(p)


def _net(c, seed):
    net = E.ConvNet(4, 2, c["channels"], _DIL)
    net.set_params(_params(c, seed))
    return net


def _spectral(c):
    """A spectral loss matrix over the predicted samples, of the scale of
    learn.spectral_matrix."""
    n = c["T"] - c["T"] // 4
    d = np.arange(n)[:, None] - np.arange(n)[None, :]
    K = np.zeros((n, n))
    for q in range(24):
        K += np.cos((0.15 + 0.02 * q) * d)
    return (K / (24 * n)).astype(np.float32)


_CLIP = 0.5
_RATE = 6e-4


def _batches(c, seed):
    rng = np.random.default_rng([5003, seed])
    return [rng.integers(0, 128, c["batch"]) for _ in range(c["steps"])]


def _prepare_train(c, seed):
    s = _Box()
    s.case, s.net = c, _net(c, seed)
    s.net.set_data(*_traces(c, seed, 128))
    s.net.set_spectral(_spectral(c), c["T"] // 4, 4.0)
    s.batches = _batches(c, seed)
    return s


def _run_train(s):
    loss, norm = [], []
    for idx in s.batches:
        loss.append(s.net.train_batch(idx, s.case["T"] // 4, _RATE, _CLIP))
        norm.append(s.net.last_grad_norm)
    return {"loss": np.array(loss), "norm": np.array(norm), "params": s.net.params()}


def _prepare_predict(c, seed):
    s = _Box()
    s.case, s.net = c, _net(c, seed)
    s.x = _traces(c, seed, c["batch"])[0]
    return s


def _run_predict(s):
    return s.net.forward(s.x)


_PREPARE = {"box": _prepare_box, "scatter": _prepare_scatter, "sweep": _prepare_sweep,
            "train": _prepare_train, "predict": _prepare_predict}
_RUN = {"box": _run_box, "scatter": _run_box, "sweep": _run_sweep, "train": _run_train,
        "predict": _run_predict}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s.kind = case["kind"]
    return s


def run(state):
    return _RUN[state.kind](state)


# ------------------------------------------------------ what it amounts to --

def work(case):
    """One pass. A time step reads and writes every voltage and current once
    (48 bytes a node) and reads the coefficients that differ from node to
    node (cb and db, 24 bytes, on a graded grid or among materials; rows of
    one value cost nothing), CPML and PML state is read and written once."""
    k = case["kind"]
    if k in ("box", "scatter"):
        n = _nodes(case)
        N = n[0] * n[1] * n[2]
        per = 48.0 + (24.0 if case.get("graded") else 0.0)
        flops = 36.0
        lay = case.get("layers", "cpml")
        if lay != "pec":
            d = case.get("cells", case.get("pml", 0))
            share = 1.0 - math.prod(max(0.0, 1.0 - 2.0 * d / q) for q in n)
            # CPML: four psi of a node per normal; PML: flux and value of six
            # edges and their four coefficients
            per += share * (32.0 if lay == "cpml" else 6 * 32.0)
            flops += share * (24.0 if lay == "cpml" else 36.0)
        return {"bytes": N * per * case["steps"] + N * 24.0, "flops": N * flops * case["steps"]}
    if k == "sweep":
        # 20 to 60 mm square substrates of 0.5 mm cells, 12 to 24 cells high,
        # 8-cell layers on five faces: on average 81 x 81 x 19 nodes
        N = 81.0 * 81.0 * 19.0 * 1.1 * case["models"]
        return {"bytes": N * (48.0 + 24.0) * case["steps"] + N * 24.0,
                "flops": N * 50.0 * case["steps"]}
    C, T, B, L = case["channels"], case["T"], case["batch"], len(_DIL)
    macs = B * T * 9.0 * (4 * C + (L - 2) * C * C + 2 * C)
    P = 9.0 * (4 * C + (L - 2) * C * C + 2 * C) + (L - 1) * C + 2
    if k == "predict":
        return {"bytes": 4.0 * B * T * 6 + 2.0 * P, "flops": 2.0 * macs}
    spec = 2.0 * B * 2 * (T - T // 4) ** 2
    # forward, both gradients; parameters, moments and gradient once a step
    return {"bytes": case["steps"] * (4.0 * B * T * 6 + 30.0 * P),
            "flops": case["steps"] * (6.0 * macs + spec)}


def tolerance(case):
    # Fields, probes, port traces and energies are the reference engine's to
    # the bit in every schedule.
    if case["kind"] in ("box", "scatter", "sweep"):
        return "exact"
    # Sums of 9 * channels f32 products in another order, six layers deep
    # (measured against 64 bits: 4.5e-7).
    if case["kind"] == "predict":
        return {"rel": 5e-6}
    # The same through the gradient and Adam (whose first steps turn small
    # gradients into whole learning-rate steps; measured: 5.5e-6).
    return {"rel": 5e-5}


# ------------------------------------------------------------ in 64 bits --

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Slab64:
    def __init__(self, s, dev):
        self.s = s
        self.e, self.c, n = s["e_side"], s["comp"], s["normal"]
        self.n = n
        self.sign, self.o = ((1.0, (self.c + 2) % 3) if n == (self.c + 1) % 3
                             else (-1.0, (self.c + 1) % 3))
        self.box = tuple(slice(lo, hi) for lo, hi in zip(s["lo"], s["hi"]))
        shape = [1, 1, 1]
        shape[n] = -1
        self.b, self.a, self.k = (torch.from_numpy(s[x]).to(dev).double().reshape(shape)
                                  for x in "bak")
        self.psi = torch.zeros([hi - lo for lo, hi in zip(s["lo"], s["hi"])],
                               dtype=torch.float64, device=dev)

    def apply(self, src, dst, cf):
        if not self.psi.numel():
            return
        x = src[self.o]
        lo, hi = self.s["lo"][self.n], self.s["hi"][self.n]
        near = list(self.box)
        if self.e:  # x[node] - x[node - 1], 0 before the grid
            near[self.n] = slice(max(lo - 1, 0), hi - 1)
            d = x[self.box].clone()
            part = [slice(None)] * 3
            part[self.n] = slice(1 if lo == 0 else 0, None)
            d[tuple(part)] -= x[tuple(near)]
        else:
            near[self.n] = slice(lo + 1, hi + 1)
            d = x[tuple(near)] - x[self.box]
        d = self.sign * d
        self.psi = self.b * self.psi + self.a * d
        dst[self.c][self.box] += (1.0 if self.e else -1.0) * cf[self.c][self.box] * (self.k * d +
                                                                                     self.psi)


def _h64(u, i, da, db):
    i[0][:, :-1, :-1] = da[0][:, :-1, :-1] * i[0][:, :-1, :-1] - db[0][:, :-1, :-1] * (
        (u[2][:, 1:, :-1] - u[2][:, :-1, :-1]) - (u[1][:, :-1, 1:] - u[1][:, :-1, :-1]))
    i[1][:-1, :, :-1] = da[1][:-1, :, :-1] * i[1][:-1, :, :-1] - db[1][:-1, :, :-1] * (
        (u[0][:-1, :, 1:] - u[0][:-1, :, :-1]) - (u[2][1:, :, :-1] - u[2][:-1, :, :-1]))
    i[2][:-1, :-1] = da[2][:-1, :-1] * i[2][:-1, :-1] - db[2][:-1, :-1] * (
        (u[1][1:, :-1] - u[1][:-1, :-1]) - (u[0][:-1, 1:] - u[0][:-1, :-1]))


def _back(x, axis):
    """x[node] - x[node - 1] along an axis, 0 before the grid."""
    d = x.clone()
    at, to = [slice(None)] * 3, [slice(None)] * 3
    at[axis], to[axis] = slice(1, None), slice(0, -1)
    d[tuple(at)] -= x[tuple(to)]
    return d


def _e64(u, i, ca, cb):
    for a in range(3):
        b, c = (a + 1) % 3, (a + 2) % 3
        at = [slice(None)] * 3
        at[a] = slice(0, -1)
        at = tuple(at)
        d = _back(i[c], b) - _back(i[b], c)
        u[a][at] = ca[a][at] * u[a][at] + cb[a][at] * d[at]


def _energy64(u, i, L, dt):
    """dt/4 of the sum of (1 + a) x x' / b over every edge, x' the next
    current of an H edge (read-only)."""
    nxt = [x.clone() for x in i]
    _h64(u, nxt, L[6:9], L[9:12])
    w = torch.zeros((), dtype=torch.float64, device=u[0].device)
    for a in range(3):
        for c, d, p in ((L[a], L[3 + a], u[a] * u[a]), (L[6 + a], L[9 + a], i[a] * nxt[a])):
            w += torch.where(d != 0, (1.0 + c) * p / torch.where(d != 0, d, 1.0), 0.0).sum()
    return 0.25 * dt * float(w)


def _exact_box(c, seed):
    s = _prepare_box(c, seed)
    dev, e = _dev(), s.engine
    n = e.grid.nodes()
    L = [torch.from_numpy(np.ascontiguousarray(s.lanes[l])).to(dev).double() for l in range(12)]
    u = [torch.zeros(n, dtype=torch.float64, device=dev) for _ in range(3)]
    i = [torch.zeros(n, dtype=torch.float64, device=dev) for _ in range(3)]
    for a, v in s.start.items():
        u[a][:] = torch.from_numpy(v).to(dev).double()
    slabs = [_Slab64(x, dev) for x in s.cpml.slabs] if s.cpml else []
    layers = {}
    if s.pml is not None:
        for side, (ax, nd, co) in ((1, s.pml.e), (0, s.pml.h)):
            for a in range(3):
                sel = ax == a
                q = torch.from_numpy(np.ascontiguousarray(nd[sel]).astype(np.int64)).to(dev)
                layers[side, a] = [tuple(q[:, t] for t in range(3)),
                                   torch.from_numpy(co[sel]).to(dev).double(),
                                   torch.zeros(len(q), dtype=torch.float64, device=dev),
                                   torch.zeros(len(q), dtype=torch.float64, device=dev)]

    def pml(stage):  # the flux update of one side, the other side's start values
        for (side, a), st in layers.items():
            x = (u if side else i)[a]
            at, co, flux, v = st
            if side == (1 if stage == 0 else 0):
                st[3] = x[at]
            else:
                f1 = co[:, 0] * flux + x[at]
                st[2], new = f1, (co[:, 1] * v - co[:, 3] * flux) + co[:, 2] * f1
                st[3] = new
                x[at] = new
    pole = None
    if s.poles is not None:
        plan = s.poles._installed[2]
        sd = plan["sides"][0]
        end = np.array(sd["pole_end"])
        k = np.array(plan["consts"])[np.array(sd["cidx"])]
        ax, nd = np.array(sd["axis"]), np.array(sd["nodes"])
        flat = torch.from_numpy(((nd[:, 0] * n[1] + nd[:, 1]) * n[2] + nd[:, 2]) +
                                ax * n[0] * n[1] * n[2]).to(dev)
        pole = dict(at=flat, edge=torch.from_numpy(np.repeat(np.arange(len(end)), np.diff(end,
                    prepend=0))).to(dev), siz=torch.tensor(sd["sum_inv_z"], device=dev).double(),
                    a=torch.from_numpy(k[:, 0]).to(dev), ic=torch.from_numpy(k[:, 1]).to(dev),
                    iz=torch.from_numpy(k[:, 2]).to(dev), j=0.0, q=0.0,
                    cb=torch.stack(L[3:6]).reshape(-1)[flat])
    amp = s.source[1].values(e.dt, 0.5, c["steps"] + 1) * s.source[2]
    w, rec = None, []
    for step in range(c["steps"]):
        if step == c["steps"] - 1 and not c["openems"]:
            w = _energy64(u, i, L, e.dt)
            if pole is not None and step:
                h = torch.from_numpy(k[:, 3]).to(dev)
                w += float((h * pole["j"] ** 2 + 0.5 * pole["ic"] * pole["q"] ** 2).sum())
        _h64(u, i, L[6:9], L[9:12])
        pml(0)
        for x in slabs:
            if not x.e:
                x.apply(u, i, L[9:12])
        old = torch.stack(u).reshape(-1)[pole["at"]] if pole is not None else None
        _e64(u, i, L[0:3], L[3:6])
        pml(1)
        for x in slabs:
            if x.e:
                x.apply(i, u, L[3:6])
        if pole is not None:
            d = pole
            all_u = torch.stack(u).reshape(-1)
            kk = d["a"] * d["j"] - d["q"] * d["ic"] + 0.5 * old[d["edge"]]
            tot = torch.zeros_like(old).index_add_(0, d["edge"], kk * d["iz"])
            new = (all_u[d["at"]] - d["cb"] * tot) / (1.0 + 0.5 * d["cb"] * d["siz"])
            jb = (kk + 0.5 * new[d["edge"]]) * d["iz"]
            d["j"], d["q"] = 2.0 * jb - d["j"], d["q"] + e.dt * jb
            all_u[d["at"]] = new
            u = list(all_u.reshape(3, *n))
        p = s.source[0]
        u[2][p[0], p[1], p[2]] += float(amp[step])
        rec.append([float(u[a][p[0], p[1], p[2]]) for p in s.at for a in range(3)]
                   if not s.whole else None)
    out = {"energy": None if w is None else np.array([w])}
    if s.whole:
        out["u"] = [x.cpu().numpy() for x in u]
        out["i"] = [x.cpu().numpy() for x in i]
    else:
        out["probes"] = np.array(rec).T.copy()
    e.close()
    return out


def _unpack(p, C):
    out, at, L = [], 0, len(_DIL)
    for l in range(L):
        ci, co = (4 if l == 0 else C), (2 if l == L - 1 else C)
        w = p[at:at + co * ci * 9].reshape(co, ci, 9)
        at += co * ci * 9
        out.append((w, p[at:at + co]))
        at += co
    return out


def _forward64(p, C, x):
    """The network in f64 on bf16-rounded weights, taps as matrix products."""
    h = x
    for l, (w, b) in enumerate(_unpack(p, C)):
        w = w + (w.float().bfloat16().double() - w).detach()
        T = h.shape[2]
        z = b[None, :, None]
        for k in range(9):
            lag = _DIL[l] * (8 - k)
            if lag < T:
                y = torch.einsum("oi,bit->bot", w[:, :, k], h[:, :, :T - lag])
                z = z + torch.nn.functional.pad(y, (lag, 0))
        if l == len(_DIL) - 1:
            return z
        a = torch.tanh(z)
        h = a if l == 0 else h + a


def _exact_predict(c, seed):
    x = torch.from_numpy(_traces(c, seed, c["batch"])[0]).double()
    p = torch.from_numpy(_params(c, seed)).double()
    with torch.no_grad():
        return _forward64(p, c["channels"], x).numpy()


def _exact_train(c, seed):
    x, y = (torch.from_numpy(v).double() for v in _traces(c, seed, 128))
    p = torch.from_numpy(_params(c, seed)).double()
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    K = torch.from_numpy(_spectral(c)).double()
    t0 = c["T"] // 4
    losses, norms = [], []
    for step, idx in enumerate(_batches(c, seed), 1):
        q = p.clone().requires_grad_(True)
        d = (_forward64(q, c["channels"], x[idx]) - y[idx])[:, :, t0:]
        loss = (d * d).mean() + 4.0 / (d.shape[0] * 2) * ((d @ K) * d).sum()
        loss.backward()
        g = q.grad
        norm = float(g.norm())
        losses.append(float(loss.detach()))
        norms.append(norm)
        g = g * min(1.0, _CLIP / norm)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - _RATE * (m / (1 - 0.9 ** step)) / ((v / (1 - 0.999 ** step)).sqrt() + 1e-8)
    return {"loss": np.array(losses), "norm": np.array(norms), "params": p.numpy()}


def exact(case, seed):
    """None for the composite model (its reduced currents are thousands of
    triangular solves per step) and for the sweeps (hundreds of models one
    after the other)."""
    if case["kind"] == "box":
        return _exact_box(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, seed)
    if case["kind"] == "predict":
        return _exact_predict(case, seed)
    return None
