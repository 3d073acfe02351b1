"""The measured workloads: what a user of the framework has it do, through its public entry points.

A case is a plain dict: ``kind`` (the sort of simulation, below), the mesh lines ``nx``, ``ny``, ``nz``, the
``steps`` of one pass and the options of its kind.  ``prepare`` builds what a program holds before it
advances (the operator, the engine with its extensions, probes and dumps: ``Simulation``, ``BatchEngine`` or
``DesignProblem``); ``run`` advances it and reads what it recorded, as the host program of a running
simulation does between two chunks of its timestep loop.

Kinds:
  cavity      PEC box, uniform mesh, Gaussian source: resonators, and the reference's first benchmark
  bricks      dielectric bricks, UPML on all faces, a 50 Ohm lumped port, port probes, an E and an H
              frequency-domain plane: antennas and boards, the headline workload.  ``mesh``: "graded" (fine
              core, graded towards the faces), "uniform", or "varied" (every line spacing its own: no two
              cells share coefficients, so the operator cannot be compressed)
  layers      dielectric layers, Mur ABC on all faces, sinusoidal sheet source: memory-scale runs; ``steady``:
              with the steady-state detection a periodic source gets by default
  mixed       Mur, UPML, PMC and PEC faces on one mesh, the reference's engine cross-check
  wires       wire antenna of polyline curves in UPML
  dispersive  Drude, Lorentz and Debye boxes and lumped RLC elements in UPML
  batch       a parameter sweep of uneven UPML meshes advanced together
  adjoint     objective and its gradient for a design region
"""
import math

import numpy as np
import torch

from openems_amd import scenes
from openems_amd.adjoint import DesignProblem
from openems_amd.batch import BatchEngine
from openems_amd.simulation import Simulation

#: passes whose probe and dump samples a state has room for
PASSES = 24
#: cell updates of the largest pass
MOST = 4.6e9


def listed():
    return [
        # the smallest runs: a few thousand cells, where launches and their gaps are the time
        {"name": "mixed_27x11x33", "kind": "mixed", "nx": 27, "ny": 11, "nz": 33, "steps": 400, "fields": True},
        {"name": "wires_47", "kind": "wires", "nx": 47, "ny": 47, "nz": 47, "pml": 6, "steps": 400, "fields": True},
        # dispersive materials and lumped elements: many extensions, each with hooks in every step
        {"name": "dispersive_72", "kind": "dispersive", "nx": 72, "ny": 72, "nz": 72, "pml": 8, "steps": 300, "fields": False},
        # the reference's plain benchmark box
        {"name": "cavity_64", "kind": "cavity", "nx": 64, "ny": 64, "nz": 64, "steps": 2000, "fields": True},
        # a metal box larger than the caches, sides of no round size
        {"name": "cavity_253x209x178", "kind": "cavity", "nx": 253, "ny": 209, "nz": 178, "steps": 200, "fields": False},
        # ordinary open-region runs: odd sides, and a mesh that cannot be compressed
        {"name": "bricks_109x97x131", "kind": "bricks", "nx": 109, "ny": 97, "nz": 131, "mesh": "graded", "pml": 8, "steps": 600, "fields": False},
        {"name": "bricks_varied_140x121x104", "kind": "bricks", "nx": 140, "ny": 121, "nz": 104, "mesh": "varied", "pml": 8, "steps": 300, "fields": False},
        # the headline workload
        {"name": "bricks_256", "kind": "bricks", "nx": 256, "ny": 256, "nz": 256, "mesh": "graded", "pml": 8, "steps": 270, "fields": False},
        # Mur faces: a small box with the default steady-state detection, and the memory-scale layers at a
        # size that can be prepared quickly
        {"name": "layers_96x90x70", "kind": "layers", "nx": 96, "ny": 90, "nz": 70, "steady": True, "steps": 300, "fields": False},
        {"name": "layers_512x384x320", "kind": "layers", "nx": 512, "ny": 384, "nz": 320, "steady": False, "steps": 72, "fields": False},
        # the parameter sweep of uneven meshes
        {"name": "batch_12", "kind": "batch", "count": 12, "lo": 48, "hi": 160, "steps": 200},
        # inverse design: objective, and its gradient backwards in time
        {"name": "adjoint_96x88x72", "kind": "adjoint", "nx": 96, "ny": 88, "nz": 72, "pml": 8, "design": 16, "steps": 600},
    ]


def draw(rng):
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["cavity", "cavity", "bricks", "bricks", "bricks", "layers", "layers", "mixed", "wires", "dispersive", "batch", "adjoint"])
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(4, 12), "lo": rng.randint(40, 60), "hi": rng.randint(80, 160), "steps": rng.randint(80, 200)}
    if kind == "adjoint":
        return {"kind": kind, "nx": side(64, 96), "ny": side(64, 88), "nz": side(56, 72), "pml": 8, "design": rng.randint(8, 16), "steps": rng.randint(200, 600)}
    c = {"kind": kind}
    if kind == "wires":
        c["nx"] = c["ny"] = c["nz"] = side(36, 96)
        c["pml"] = 6
    elif kind == "dispersive":
        c["nx"] = c["ny"] = c["nz"] = side(48, 96)
        c["pml"] = rng.choice([6, 8])
    elif kind == "mixed":
        c["nx"], c["ny"], c["nz"] = side(27, 80), side(11, 60), side(33, 80)
    elif kind == "cavity":
        c["nx"], c["ny"], c["nz"] = side(30, 260), side(30, 260), side(30, 260)
    elif kind == "bricks":
        c["nx"], c["ny"], c["nz"] = side(64, 256), side(64, 256), side(64, 256)
        c["mesh"] = rng.choice(["graded", "graded", "uniform", "varied"])
        c["pml"] = rng.choice([6, 8, 8])
        if c["mesh"] == "varied":       # twelve coefficients a cell: as many cells as a plain operator is used for
            c["nx"], c["ny"], c["nz"] = side(64, 160), side(64, 160), side(64, 160)
    else:
        c["nx"], c["ny"], c["nz"] = side(64, 512), side(64, 384), side(64, 320)
        c["steady"] = rng.choice([True, False])
    cells = c["nx"] * c["ny"] * c["nz"]
    small = 400 if kind == "mixed" else 300 if kind in ("dispersive", "layers") else 800
    c["steps"] = max(40, min(small, int(0.8 * MOST / cells)))
    c["fields"] = kind in ("mixed", "wires") or cells < 150000
    return c


# ---- scenes ---------------------------------------------------------------------------------------------


def _bricks(case, rng):
    n = [case["nx"], case["ny"], case["nz"]]
    pml = case["pml"]
    if case["mesh"] == "graded":
        lines = [scenes.graded_lines(k, 0.5, 10, 1.2) for k in n]
    elif case["mesh"] == "uniform":
        lines = [np.arange(k) * 0.5 for k in n]
    else:
        lines = [np.concatenate([[0.0], np.cumsum(rng.uniform(0.4, 0.6, k - 1))]) for k in n]
    mats = []
    for k in range(40):
        lo, hi = [], []
        for a in range(3):
            s = int(rng.integers(max(2, n[a] // 32), max(4, n[a] // 5)))
            i = int(rng.integers(pml + 3, n[a] - 4 - pml - s))
            lo.append(lines[a][i])
            hi.append(lines[a][i + s])
        mats.append({"eps": float(rng.uniform(1.0, 10.0)), "kappa": float(rng.uniform(0.0, 0.05)), "priority": k + 1,
                     "start": tuple(lo), "stop": tuple(hi)})
    c = [k // 2 for k in n]
    x, y, z = (lines[a][c[a] - 1:c[a] + 1] for a in range(3))
    z0, z1 = lines[2][c[2] - 2], lines[2][c[2] + 2]
    xm, ym, zm = 0.5 * (x[0] + x[1]), 0.5 * (y[0] + y[1]), 0.5 * (z0 + z1)
    start, stop = (x[0], y[0], z0), (x[1], y[1], z1)
    plane = {"start": (lines[0][0], lines[1][0], lines[2][c[2]]), "stop": (lines[0][-1], lines[1][-1], lines[2][c[2]])}
    wall = {"start": (lines[0][c[0]], lines[1][0], lines[2][0]), "stop": (lines[0][c[0]], lines[1][-1], lines[2][-1])}
    freqs = [5e9, 10e9, 15e9]
    return {
        "lines": lines, "delta_unit": 1e-3, "bc": [3] * 6, "pml_size": [pml] * 6, "materials": mats,
        "lumped": [{"dir": 2, "R": 50.0, "C": 0.0, "L": 0.0, "caps": True, "type": "parallel", "priority": 0, "start": start, "stop": stop}],
        "excitations": [{"type": 0, "val": (0.0, 0.0, -1.0), "start": start, "stop": stop, "priority": 0}],
        "signal": {"type": "gauss", "f0": 0.0, "fc": 20e9}, "oversampling": 4,
        "probes": [scenes._probe(0, (xm, ym, z0), (xm, ym, z1), weight=-1.0, name="ut"),
                   scenes._probe(1, (x[0], y[0], zm), (x[1], y[1], zm), norm_dir=2, name="it")],
        "dumps": [dict(plane, type=0, freqs=freqs, name="Ef"), dict(wall, field="H", interp=2, freqs=freqs, name="Hf")],
    }


def _cavity(case, rng):
    n = [case["nx"], case["ny"], case["nz"]]
    at = [int(rng.integers(k // 3, 2 * k // 3)) for k in n]
    to = [int(rng.integers(k // 4, 3 * k // 4)) for k in n]
    return {
        "lines": [np.arange(k, dtype=np.float64) for k in n], "delta_unit": 1e-3, "bc": [0] * 6,
        "signal": {"type": "gauss", "f0": 0.0, "fc": float(rng.uniform(9e9, 11e9))}, "oversampling": 4,
        "excitations": [{"type": 0, "val": (0.0, 0.0, float(rng.uniform(0.5, 2.0))), "start": tuple(at),
                         "stop": (at[0], at[1], at[2] + 1), "priority": 0}],
        "probes": [scenes._probe(2, to, to, name="et"), scenes._probe(0, (to[0], to[1], 0), (to[0], to[1], n[2] - 1), name="ut")],
    }


def _mixed(case, rng):
    n = [case["nx"], case["ny"], case["nz"]]
    at = [n[0] // 3, n[1] // 2, n[2] // 2]
    return {
        "lines": [np.arange(k) * 1.0 for k in n], "delta_unit": 1e-3, "bc": [2, 3, 1, 0, 0, 0], "pml_size": [8] * 6,
        "materials": [{"eps": float(rng.uniform(2.0, 5.0)), "start": (3, 2, 5), "stop": (n[0] // 2, n[1] - 3, n[2] // 2), "priority": 1}],
        "excitations": [{"type": 0, "val": (0.0, 1.0, 1.0), "start": tuple(at), "stop": (at[0], at[1] + 1, at[2] + 1)}],
        "signal": {"type": "gauss", "f0": 10e9, "fc": 8e9}, "oversampling": 4,
        "probes": [scenes._probe(2, (n[0] // 2, n[1] // 2, n[2] // 4), (n[0] // 2, n[1] // 2, n[2] // 4), name="et"),
                   scenes._probe(0, (n[0] // 2, 0, n[2] // 2), (n[0] // 2, n[1] - 1, n[2] // 2), name="ut")],
    }


def _layers(case, rng):
    n = [case["nx"], case["ny"], case["nz"]]
    lines = [np.arange(k) * 0.25 for k in n]
    cuts = [k * (n[2] - 1) // 8 for k in range(9)]
    mats = [{"eps": float(rng.uniform(1.5, 6.0)) if k else 1.0, "priority": k + 1,      # vacuum first: it sets the timestep
             "start": (-1.0, -1.0, lines[2][cuts[k]]), "stop": (lines[0][-1] + 1.0, lines[1][-1] + 1.0, lines[2][cuts[k + 1]])}
            for k in range(8)]
    z = n[2] // 2 - 5
    at = [(lines[0][i * n[0] // 5], lines[1][j * n[1] // 5], lines[2][n[2] // 2]) for i in range(1, 5) for j in range(1, 5)]
    return {
        "lines": lines, "delta_unit": 1e-3, "bc": [2] * 6, "materials": mats,
        "excitations": [{"type": 0, "val": (float(rng.uniform(0.5, 2.0)), 0.0, 0.0), "start": (lines[0][0], lines[1][0], lines[2][z]),
                         "stop": (lines[0][-1], lines[1][-1], lines[2][z]), "priority": 0}],
        "signal": {"type": "sinus", "f0": 15e9}, "oversampling": 4,
        "probes": [scenes._probe(2, p, p, name="e%d" % k) for k, p in enumerate(at)]
        + [scenes._probe(0, (at[9][0], at[9][1], lines[2][0]), (at[9][0], at[9][1], lines[2][-1]), name="ut")],
    }


def _scene(case, seed):
    rng = np.random.default_rng([seed, 11])
    kind, steps = case["kind"], case["steps"]
    if kind == "cavity":
        s = _cavity(case, rng)
    elif kind == "bricks":
        s = _bricks(case, rng)
    elif kind == "mixed":
        s = _mixed(case, rng)
    elif kind == "layers":
        s = _layers(case, rng)
        s["steady_state"] = case["steady"]
    elif kind == "wires":
        s = scenes.wire_antenna(case["nx"], steps, case["pml"])
        s["materials"][0]["eps"] = float(rng.uniform(2.0, 5.0))
    else:
        s = scenes.dispersive_rlc(case["nx"], steps, case["pml"])
        s["materials"][2]["eps"] = float(rng.uniform(2.0, 5.0))
        s["materials"][0]["kappa"] = float(rng.uniform(0.005, 0.02))
    s["nrts"] = PASSES * steps
    return s


def _batch_scenes(case, seed):
    scs = scenes.batched_sweep(count=case["count"], nrts=PASSES * case["steps"], seed=20260204, lo=case["lo"], hi=case["hi"])
    rng = np.random.default_rng([seed, 12])
    for s in scs:      # the same meshes, other materials
        for m in s["materials"]:
            m["eps"] = float(rng.uniform(1.0, 12.0))
    return scs


def _design(case, seed):
    scene, probes, freq = scenes.adjoint_design(case["nx"], case["ny"], case["nz"], pml=case["pml"], design=(case["design"], case["design"], 6),
                                                nrts=case["steps"], seed=seed)
    g = scene["materials"][0]["grid"]
    return scene, probes, freq, g["eps"].copy(), np.zeros_like(g["eps"])


# ---- what is measured -----------------------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        b = BatchEngine(_batch_scenes(case, seed))
        b.autotune(steps=4)
        return {"case": case, "batch": b}
    if kind == "adjoint":
        scene, probes, freq, eps, kappa = _design(case, seed)
        p = DesignProblem(scene, probes, freq, case["steps"], checkpoint_every=128)
        return {"case": case, "problem": p, "eps": eps, "kappa": kappa}
    return {"case": case, "sim": Simulation(_scene(case, seed))}


def _recorded(sim, fields):
    out = {p.name: list(sim.eng.probe_results(p.pid)) for p in sim.probes}
    for d in sim.dumps:
        out[d.name] = d.collect(sim.eng)
    out["energy"] = sim.eng.energy()      # what the end criterion samples
    if fields:
        out["volt"], out["curr"] = sim.eng.get_volt(), sim.eng.get_curr()
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        state["batch"].iterate(case["steps"])
        return [_recorded(s, False) for s in state["batch"].sims]
    if case["kind"] == "adjoint":
        J, d_eps, d_kappa = state["problem"].value_and_grad(state["eps"], state["kappa"])
        return {"J": np.array([J]), "d_eps": d_eps, "d_kappa": d_kappa}
    state["sim"].run(case["steps"])
    return _recorded(state["sim"], case["fields"])


def _pml_cells(n, pml):
    return n[0] * n[1] * n[2] - max(0, n[0] - 2 * pml) * max(0, n[1] - 2 * pml) * max(0, n[2] - 2 * pml)


def work(case):
    """Of one timestep: the fields read and written once (48 bytes a cell), its coefficients (an index of two
    bytes, or twelve floats where no two cells share them), and at UPML positions the fluxes read and written
    and the coefficients' index (52 bytes, or 120); 18 operations for each of a cell's two updates, and 9 more
    for each at a UPML position.  An adjoint pass is three such runs (forward, its replay, backward)."""
    if case["kind"] == "batch":
        scs = scenes.batched_sweep(count=case["count"], nrts=1, seed=20260204, lo=case["lo"], hi=case["hi"])
        meshes = [([len(l) for l in s["lines"]], 6) for s in scs]
    else:
        n = [case["nx"], case["ny"], case["nz"]]
        meshes = [(n, case.get("pml", 0))]
    plain = case.get("mesh") == "varied"
    total, flops = 0.0, 0.0
    for n, pml in meshes:
        cells = n[0] * n[1] * n[2]
        shell = cells - (n[0] - 9) * cells // n[0] if case["kind"] == "mixed" else _pml_cells(n, pml) if pml else 0
        total += cells * (96.0 if plain else 50.0) + shell * (120.0 if plain else 52.0)
        flops += cells * 36.0 + shell * 18.0
    runs = case["steps"] * (3 if case["kind"] == "adjoint" else 1)
    return {"bytes": total * runs, "flops": flops * runs}


def tolerance(case):
    # Four times the largest error measured against exact().  What the 32-bit fields of a pass lose is largest
    # where a source leaves a static field behind, in which the remaining waves are small: the currents of a
    # closed box (4e-4) and of wires and lumped elements (2.5e-4); elsewhere 2e-5 at most.
    if case["kind"] == "cavity":
        return {"rel": 2e-3}
    if case["kind"] in ("wires", "dispersive"):
        return {"rel": 1e-3}
    return {"rel": 1e-4}


# ---- the same in 64 bits --------------------------------------------------------------------------------


class _Steps64:
    """The timestep of an operator in float64, written out with torch."""

    def __init__(self, op, ade=True):
        dev = "cuda"
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).double()  # noqa: E731
        self.dev, self.N, self.op = dev, op.N, op
        self.vv, self.vi, self.ii, self.iv = (t(op.coeff(k)) for k in ("vv", "vi", "ii", "iv"))
        self.V = torch.zeros((3,) + tuple(op.N), dtype=torch.float64, device=dev)
        self.I = torch.zeros_like(self.V)
        self.slabs = []
        for s in op.upml_slabs():
            box = (slice(None),) + tuple(slice(a, a + k) for a, k in zip(s["start"], s["num"]))
            k = {n: t(s[n]) for n in ("vv", "vvfo", "vvfn", "ii", "iifo", "iifn")}
            self.slabs.append((box, k, torch.zeros_like(k["vv"]), torch.zeros_like(k["vv"])))
        self.mur = [(f["ny"], f["line"], f["line_shift"], t(f["coeff_nyP"]), t(f["coeff_nyPP"]), f["start_ts"]) for f in op.mur_faces()]
        self.sig = [s.astype(np.float64) for s in op.signal()]
        self.period, self.exc = op.period_steps, [op.excitation(False), op.excitation(True)]
        self.lor = [o for o in op.lorentz_tables() if o["pos"].shape[1] and (o["volt"] or o["curr"])] if ade else []
        for o in self.lor:
            o["at"] = [torch.from_numpy(o["pos"][a].astype(np.int64)).to(dev) for a in range(3)]
            for k in ("v_int", "v_ext", "v_lor", "i_int", "i_ext", "i_lor"):
                o[k] = None if o[k] is None else t(o[k])
            o["state"] = {c: [torch.zeros_like(o["v_int"]), torch.zeros_like(o["v_int"])] for c in "vi"}
        r = op.rlc_table() if ade else None
        self.rlc = None
        if r is not None:
            c = [t(r[k]) for k in ("i2v", "ilv", "vvd", "vv2", "vj1", "vj2", "ib0", "b1", "b2")]
            z = torch.zeros_like(c[0])
            ix = tuple(torch.from_numpy(a.astype(np.int64)).to(dev) for a in (r["dir"], *r["pos"]))
            self.rlc = {"c": c, "ix": ix, "il": z, "vd": [z, z, z], "jn": [z, z, z]}
        self.ts = 0

    @staticmethod
    def _down(F, a):
        """F minus its lower neighbour along a (0 at the first line)"""
        d = torch.zeros_like(F)
        d.narrow(a, 1, F.shape[a] - 1).copy_(torch.diff(F, dim=a))
        return d

    def _excite(self, F, which):
        e = self.exc[which]
        if not len(e["dir"]):
            return
        s, n = self.sig[which], self.ts
        at = n - e["delay"].astype(np.int64)
        at = np.where(at > 0, at, 0) % (self.period if self.period > 0 else n + 1)
        at = np.where(at < len(s), at, 0)
        v = torch.from_numpy(e["amp"].astype(np.float64) * s[at]).to(self.dev)
        ix = tuple(torch.from_numpy(a.astype(np.int64)).to(self.dev) for a in (e["dir"], *e["index"]))
        F.index_put_(ix, v, accumulate=True)

    def _ade_pre(self, F, c):
        for o in self.lor:
            if o["volt" if c == "v" else "curr"]:
                ade, lor = o["state"][c]
                f = F[:, o["at"][0], o["at"][1], o["at"][2]]
                if o[c + "_lor"] is not None:
                    lor += o[c + "_lor"] * ade
                    f = f - lor
                ade.mul_(o[c + "_int"]).add_(o[c + "_ext"] * f)

    def _ade_apply(self, F, c):
        for o in self.lor:
            if o["volt" if c == "v" else "curr"]:
                F[:, o["at"][0], o["at"][1], o["at"][2]] -= o["state"][c][0]

    def _face(self, F, n, line, c):
        return F[c].select(n, line) if (n + 1) % 3 < (n + 2) % 3 else F[c].select(n, line).transpose(0, 1)

    def step(self):
        V, I, Nx, Ny, Nz = self.V, self.I, *self.N
        mur = [m for m in self.mur if self.ts >= m[5]]
        held = []
        for n, line, near, cP, cPP, _ in mur:
            held.append([self._face(V, n, near, c) - k * self._face(V, n, line, c) for c, k in (((n + 1) % 3, cP), ((n + 2) % 3, cPP))])
        self._ade_pre(V, "v")
        if self.rlc:
            r = self.rlc
            r["vd"], r["jn"] = r["vd"][-1:] + r["vd"][:-1], r["jn"][-1:] + r["jn"][:-1]
            r["il"] = r["il"] + r["c"][0] * r["c"][1] * r["vd"][1]
        keep = []
        for box, k, F, _ in self.slabs:
            keep.append(k["vv"] * V[box] - k["vvfo"] * F)
            V[box] = F
        d = self._down
        curl = torch.stack([d(I[(n + 2) % 3], (n + 1) % 3) - d(I[(n + 1) % 3], (n + 2) % 3) for n in range(3)])
        self.V = V = V * self.vv + self.vi * curl
        for (box, k, F, _), kept in zip(self.slabs, keep):
            F.copy_(V[box])
            V[box] = kept + k["vvfn"] * F
        for (n, line, near, cP, cPP, _), h in zip(mur, held):
            h[0] = h[0] + cP * self._face(V, n, near, (n + 1) % 3)
            h[1] = h[1] + cPP * self._face(V, n, near, (n + 2) % 3)
        if self.rlc:
            r = self.rlc
            c, v = r["c"], V[r["ix"]]
            v = c[2] * (v - r["il"] + c[3] * r["vd"][2] + c[4] * r["jn"][1] + c[5] * r["jn"][2])
            r["vd"][0] = v
            r["jn"][0] = c[6] * (v - r["vd"][2] - c[7] * r["jn"][1] - c[8] * r["jn"][2])
            V[r["ix"]] = v
        self._ade_apply(V, "v")
        for (n, line, near, cP, cPP, _), h in reversed(list(zip(mur, held))):
            self._face(V, n, line, (n + 1) % 3).copy_(h[0])
            self._face(V, n, line, (n + 2) % 3).copy_(h[1])
        self._excite(V, 0)
        self._ade_pre(I, "i")
        keep = []
        for box, k, _, F in self.slabs:
            keep.append(k["ii"] * I[box] - k["iifo"] * F)
            I[box] = F
        m = (slice(0, Nx - 1), slice(0, Ny - 1), slice(0, Nz - 1))
        for n in range(3):
            a, b = (n + 1) % 3, (n + 2) % 3
            curl = torch.diff(V[a], dim=b).narrow(a, 0, self.N[a] - 1).narrow(n, 0, self.N[n] - 1)
            curl = curl - torch.diff(V[b], dim=a).narrow(b, 0, self.N[b] - 1).narrow(n, 0, self.N[n] - 1)
            I[n][m] = I[n][m] * self.ii[n][m] + self.iv[n][m] * curl
        for (box, k, _, F), kept in zip(self.slabs, keep):
            F.copy_(I[box])
            I[box] = kept + k["iifn"] * F
        self._ade_apply(I, "i")
        self._excite(I, 1)
        self.ts += 1


def _plane64(d, F, op):
    """The dump's field on its box, [3][nx][ny][nz] (E with node, H with cell interpolation)"""
    out = []
    for n in range(3):
        el = torch.from_numpy(op.edge_lengths(n, d.field == 1)).to(F.device)
        shape = [1, 1, 1]
        shape[n] = -1
        E = torch.where(el.view(shape) != 0, F[n] / el.view(shape), 0.0)
        W = torch.zeros_like(E)
        k = E.shape[n]
        if d.field == 0:
            rel = (el[1:-1] / (el[1:-1] + el[:-2])).view(shape)
            W.narrow(n, 1, k - 2).copy_(E.narrow(n, 1, k - 2) * (1 - rel) + E.narrow(n, 0, k - 2) * rel)
            W.narrow(n, 0, 1).copy_(E.narrow(n, 0, 1))
            W.narrow(n, k - 1, 1).copy_(E.narrow(n, k - 2, 1))
        else:
            rel = (el[:-1] / (el[:-1] + el[1:])).view(shape)
            W.narrow(n, 0, k - 1).copy_(E.narrow(n, 0, k - 1) * (1 - rel) + E.narrow(n, 1, k - 1) * rel)
        out.append(W[tuple(slice(a, b + 1) for a, b in zip(d.start, d.stop))])
    return torch.stack(out)


def _exact_sim(sim, steps, fields):
    op = sim.op
    S = _Steps64(op)
    taken = {p.name: ([], []) for p in sim.probes}
    planes = {}

    def sample():
        for p in sim.probes:
            if p.due(S.ts):
                F = S.I if p.ptype in (1, 3) else S.V
                x = F[[torch.tensor(v, device=S.dev) for v in (p.comp, *zip(*p.pos))]]
                if p.ptype in (0, 1):
                    x = torch.stack([(x * torch.tensor(p.sign, device=S.dev)).sum(), *x.new_zeros(2)])
                else:
                    x = x / torch.tensor(p.div, dtype=torch.float64, device=S.dev)
                taken[p.name][0].append(S.ts)
                taken[p.name][1].append(x)
        for d in sim.dumps:
            if S.ts % d.fd_interval == 0:
                E = _plane64(d, S.I if d.field else S.V, op)
                T = (S.ts + (0.5 if d.dual_time else 0.0)) * op.dT
                w = torch.tensor([2 * op.dT * d.fd_interval * np.exp(-2j * math.pi * f * T) for f in d.freqs], device=S.dev)
                planes[d.name] = planes.get(d.name, 0) + w.view(-1, 1, 1, 1, 1) * E

    sample()
    for _ in range(steps):
        S.step()
        sample()
    out = {k: [np.array(ts, np.uint32), torch.stack(v).cpu().numpy()] for k, (ts, v) in taken.items()}
    out.update({k: v.cpu().numpy() for k, v in planes.items()})
    inner = tuple(slice(0, k - 1) for k in op.N)
    out["energy"] = float(8.85418781762e-12 * S.V[(slice(None),) + inner].square().sum() + 4e-7 * math.pi * S.I[(slice(None),) + inner].square().sum())
    if fields:
        out["volt"], out["curr"] = S.V.cpu().numpy(), S.I.cpu().numpy()
    return out


def _exact_adjoint(case, seed):
    """J and its gradient by torch's own differentiation of the float64 steps"""
    scene, probes, freq, eps, kappa = _design(case, seed)
    sim = Simulation(dict(scene, probes=[]))
    op, S = sim.op, None
    S = _Steps64(op)
    g = scene["materials"][0]["grid"]
    lo, nc = [int(v) for v in g["cell0"]], [int(v) for v in g["ncells"]]
    e = torch.from_numpy(eps).to(S.dev).double().requires_grad_()
    k = torch.from_numpy(kappa).to(S.dev).double().requires_grad_()
    # edge values of the box around the design cells on the uniform mesh: the mean of the four cells
    # around an edge times the spacing
    d, eps0, dT = (scene["lines"][0][1] - scene["lines"][0][0]) * 1e-3, 8.85418781762e-12, op.dT
    pad = lambda a, v: torch.nn.functional.pad(a.permute(2, 1, 0), (1, 1, 1, 1, 1, 1), value=v)  # noqa: E731
    ce, ck = pad(e, 1.0), pad(k, 0.0)
    box = [slice(a, a + n + 1) for a, n in zip(lo, nc)]

    def mean4(c, n):
        c = c.narrow(n, 1, c.shape[n] - 1)
        for a in ((n + 1) % 3, (n + 2) % 3):
            c = 0.5 * (c.narrow(a, 0, c.shape[a] - 1) + c.narrow(a, 1, c.shape[a] - 1))
        return c
    vi, vv = [], []
    for n in range(3):
        C, G = eps0 * d * mean4(ce, n), d * mean4(ck, n)
        vi.append(dT / (C + dT * G / 2))
        vv.append((2 * C - dT * G) / (2 * C + dT * G))
    vi = torch.stack(vi)
    vv = torch.stack(vv)
    leaf_vi, leaf_vv = vi.detach().requires_grad_(), vv.detach().requires_grad_()
    b = (slice(None), *box)
    S.vi[b], S.vv[b] = leaf_vi.detach(), leaf_vv.detach()
    # forward, keeping every step's box fields; then the transposed steps by torch's differentiation
    pc = [torch.tensor(v, device=S.dev) for v in ([c for c, _ in probes], *zip(*[p for _, p in probes]))]
    div = torch.tensor([op.edge_length(c, p[c]) for c, p in probes], dtype=torch.float64, device=S.dev)
    F = torch.zeros(len(probes), dtype=torch.complex128, device=S.dev)
    saved = []
    state = lambda: [S.V, S.I] + [x for s in S.slabs for x in s[2:]]  # noqa: E731
    every = 20
    for n in range(case["steps"]):
        if n % every == 0:
            saved.append([x.clone() for x in state()])
        S.step()
        F += (S.V[tuple(pc)] / div) * np.exp(-2j * math.pi * freq * (n + 1) * dT) * dT
    J = F.abs().square().sum()
    # segments from last to first
    gF = (2 * F).conj()
    grads = [torch.zeros_like(x) for x in state()]
    g_vi, g_vv = torch.zeros_like(leaf_vi), torch.zeros_like(leaf_vv)
    main_vi, main_vv = S.vi, S.vv
    for j in reversed(range(len(saved))):
        start = [x.detach().requires_grad_() for x in saved[j]]
        with torch.enable_grad():
            S.vi, S.vv = main_vi.clone(), main_vv.clone()
            S.vi[b], S.vv[b] = leaf_vi, leaf_vv
            S.V, S.I = start[0].clone(), start[1].clone()
            S.slabs = [(s[0], s[1], start[2 + 2 * m].clone(), start[3 + 2 * m].clone()) for m, s in enumerate(S.slabs)]
            S.ts = j * every
            got = 0.0
            for n in range(j * every, min(case["steps"], (j + 1) * every)):
                S.step()
                w = gF * np.exp(-2j * math.pi * freq * (n + 1) * dT) * dT
                got = got + ((S.V[tuple(pc)] / div) * w.real).sum()
            end = state()
            total = got + sum((x * y).sum() for x, y in zip(end, grads))
            res = torch.autograd.grad(total, start + [leaf_vi, leaf_vv], allow_unused=True)
        grads = [torch.zeros_like(x) if r is None else r for x, r in zip(start, res)]
        g_vi, g_vv = g_vi + res[-2], g_vv + res[-1]
    d_eps, d_kappa = torch.autograd.grad((vi * g_vi).sum() + (vv * g_vv).sum(), [e, k])
    sim.close()
    return {"J": J.detach().reshape(1).cpu().numpy(), "d_eps": d_eps.cpu().numpy(), "d_kappa": d_kappa.cpu().numpy()}


def exact(case, seed):
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, seed)
    if case["kind"] == "batch":
        out = []
        for s in _batch_scenes(case, seed):
            sim = Simulation(s)
            out.append(_exact_sim(sim, case["steps"], False))
            sim.close()
        return out
    sim = Simulation(_scene(case, seed))
    out = _exact_sim(sim, case["steps"], case["fields"])
    sim.close()
    return out
