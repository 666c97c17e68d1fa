"""What a user of this framework has it do: the sweeps, single runs, coupled
stacks and arrays of its configurations, tests and benchmark, each through
the entry point that a program calls.

listed() / draw(rng)   cases: dicts of plain values
prepare(case, seed)    what a program holds before the call, from the seed
run(state)             one pass; returns every output whole
work(case)             bytes and operations a pass cannot do without
exact(case, seed)      the outputs in 64 bits from a plain numpy integrator
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cmtj_amd import (AxialDriver, CVector, Junction, Layer, NullDriver, SolverMode, constantDriver, sineDriver,
                      stepDriver, workloads)
from cmtj_amd.batch import JunctionBatch
from cmtj_amd.reservoir import GroupInteraction, computeDipoleInteraction, computeDipoleInteractionNoumra
from cmtj_amd.stack import ParallelStack, SeriesStack

DT = 1e-13
DP_STEP = 1e-11  # first adaptive step: long enough that its error estimate is no rounding residue
TRAPEZOID = 6  # the driver kind's number
T_TO_AM = 795774.715459


# --- the cases ----------------------------------------------------------------

def listed() -> list:
    return [
        # the benchmark's sweep: pulse-induced spectra of 4096 two-layer
        # junctions, uneven durations, every step logged (the FFT's input)
        {"name": "pimm_sweep", "kind": "pimm", "points": 4096, "t_min": 2e-9, "t_max": 20e-9, "every": 1,
         "precision": "fp32"},
        # the same sweep wider than the chip, shorter and decimated
        {"name": "pimm_wide", "kind": "pimm", "points": 65536, "t_min": 0.2e-9, "t_max": 2e-9, "every": 10,
         "precision": "fp32"},
        # hysteresis loop: 101 fields, one layer, binary64, strip resistances
        {"name": "rh_loop", "kind": "rh", "points": 101, "steps": 50000, "precision": "fp64"},
        # spin-torque oscillator current sweep asked for in the bulk mode
        {"name": "sto_sweep", "kind": "sto", "points": 512, "steps": 50000, "precision": "fp32"},
        # thermal switching ensemble (currents x seeds), final state only: the
        # chip full of stochastic instances
        {"name": "cims_ensemble", "kind": "cims", "currents": 256, "seeds": 512, "steps": 10000,
         "precision": "fp32"},
        # spin-diode map: fields x frequencies, sine drive, resistance logged
        # every step in binary64 (what the mixing voltage is taken from)
        {"name": "vsd_map", "kind": "vsd", "fields": 31, "freqs": 33, "steps": 10000, "precision": "fp64"},
        # the smallest call: one junction, one short run, log read back
        {"name": "dropin_short", "kind": "dropin", "device": "pimm", "steps": 1000, "every": 1},
        # every field term at once (full demagnetisation and dipole tensors,
        # second-order anisotropy, both exchange terms, IDMI, a driven coupling)
        {"name": "all_terms", "kind": "terms", "points": 257, "steps": 5000, "precision": "fp64"},
        # a ragged batch of unlike requests: 1-4 layers, RK4 and Euler-Heun,
        # step, sine and trapezoid drives, time steps from 1e-14 to 1e-13 s
        {"name": "mixed_requests", "kind": "mixed", "requests": 96, "t_min": 0.05e-9, "t_max": 0.5e-9},
        # adaptive steps: a stability diagram, fields x currents (a last step
        # cut to a short remainder has an error estimate at rounding level,
        # which the controller answers with its smallest or largest factor)
        {"name": "dp_diagram", "kind": "dp", "fields": 45, "currents": 45, "total_time": 3e-9},
        # eight oscillators in series sharing one current, logs read back
        {"name": "stack_series", "kind": "stack", "members": 8, "steps": 10000, "series": True, "kcl": True},
        # an 8 x 8 dipole-coupled array, logs read back
        {"name": "dipole_array", "kind": "array", "side": 8, "steps": 10000, "interaction": "kanao"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """One more case: sizes over the logarithm of each range; a case's passes
    stay below the largest listed one's."""
    kind = rng.choice(["pimm", "pimm", "rh", "sto", "cims", "vsd", "dropin", "terms", "mixed", "dp", "stack", "array"])
    if kind == "pimm":
        n = _log_int(rng, 2, 65536)
        t_max = min(20e-9, 8e-6 / n) * rng.uniform(0.3, 1.0)
        return {"kind": kind, "points": n, "t_min": t_max * rng.uniform(0.1, 0.9), "t_max": t_max,
                "every": rng.choice([1, 10]) if n <= 8192 else 10, "precision": rng.choice(["fp32", "fp32", "fp64"])}
    if kind == "rh":
        return {"kind": kind, "points": _log_int(rng, 11, 4001), "steps": _log_int(rng, 2000, 50000),
                "precision": rng.choice(["fp32", "fp64"])}
    if kind == "sto":
        return {"kind": kind, "points": _log_int(rng, 8, 4096), "steps": _log_int(rng, 2000, 50000),
                "precision": rng.choice(["fp32", "fp64"])}
    if kind == "cims":
        return {"kind": kind, "currents": _log_int(rng, 4, 256), "seeds": _log_int(rng, 4, 512),
                "steps": _log_int(rng, 1000, 10000), "precision": rng.choice(["fp32", "fp32", "fp64"])}
    if kind == "vsd":
        return {"kind": kind, "fields": _log_int(rng, 3, 40), "freqs": _log_int(rng, 3, 60),
                "steps": _log_int(rng, 2000, 20000), "precision": rng.choice(["fp32", "fp64"])}
    if kind == "dropin":
        return {"kind": kind, "device": rng.choice(["pimm", "rh", "sto", "vsd", "terms"]),
                "steps": _log_int(rng, 100, 10000), "every": rng.choice([1, 10, 100])}
    if kind == "terms":
        return {"kind": kind, "points": _log_int(rng, 3, 3000), "steps": _log_int(rng, 1000, 8000),
                "precision": rng.choice(["fp32", "fp64"])}
    if kind == "mixed":
        t = rng.uniform(0.2e-9, 0.5e-9)
        return {"kind": kind, "requests": _log_int(rng, 8, 200), "t_min": t * 0.1, "t_max": t}
    if kind == "dp":
        return {"kind": kind, "fields": _log_int(rng, 4, 64), "currents": _log_int(rng, 4, 48),
                "total_time": rng.uniform(1e-9, 3e-9)}
    if kind == "stack":
        return {"kind": kind, "members": rng.randint(2, 12), "steps": _log_int(rng, 500, 20000),
                "series": rng.random() < 0.5, "kcl": rng.random() < 0.7}
    return {"kind": kind, "side": rng.randint(2, 8), "steps": _log_int(rng, 500, 10000),
            "interaction": rng.choice(["kanao", "nomura"])}


# --- devices that the workload module does not already build --------------------

EXOTIC_DEMAG = [[0.02, 0.001, 0.0005], [0.001, 0.03, 0.0002], [0.0005, 0.0002, 0.95]]
EXOTIC_DIPOLE = [[0.01, 0.002, 0.0], [0.002, 0.015, 0.001], [0.0, 0.001, -0.02]]


def _rows(t) -> list:
    return [CVector(*r) for r in t]


def _terms_junction() -> Junction:
    """Two layers with every field term of the engine (the parity tests'
    exotic bilayer with a biquadratic coupling)."""
    a = Layer("a", mag=CVector(0.1, 0.2, 1), anis=CVector(0, 0, 1), Ms=1.2, thickness=1.5e-9, cellSurface=1e-16,
              demagTensor=_rows(EXOTIC_DEMAG), damping=0.05)
    b = Layer("b", mag=CVector(1, 0.1, 0), anis=CVector(1, 0, 0), Ms=0.9, thickness=2e-9, cellSurface=1e-16,
              demagTensor=_rows(EXOTIC_DEMAG), damping=0.06)
    a.setTopDipoleTensor(_rows(EXOTIC_DIPOLE))
    b.setBottomDipoleTensor(_rows(EXOTIC_DIPOLE))
    j = Junction([a, b])
    j.setLayerAnisotropyDriver("a", constantDriver(4e5))
    j.setLayerAnisotropyDriver("b", constantDriver(2e4))
    j.setLayerSecondOrderAnisotropyDriver("a", constantDriver(-3e4))
    j.setIDMIDriver("a", "b", AxialDriver(1e-4, -2e-4, 5e-5))
    j.setIECDriver("a", "b", sineDriver(1e-4, 5e-5, 2e9, 0))
    j.setQuadIECDriver("a", "b", constantDriver(-2e-5))
    j.setLayerHdmiDriver("all", AxialDriver(1e3, 0, -2e3))
    j.setLayerExternalFieldDriver("b", AxialDriver(100e3, 0, 0))
    return j


def _rh_junction() -> Junction:
    l = Layer("free", mag=CVector(1, 0, 0), anis=CVector(1, 0, 0), Ms=1.2, thickness=2e-9, cellSurface=1e-16,
              demagTensor=_rows(np.diag([0.00024, 0.0022, 0.99756]).tolist()), damping=0.01)
    j = Junction([l], [100.0], [0.0], [1.0], [0.0], [0.0], [0.0], [0.0])
    j.setLayerAnisotropyDriver("free", constantDriver(5e3))
    return j


def _stack_member(q: int, m0) -> Junction:
    l = Layer.createSTTLayer("free", mag=CVector(*m0), anis=CVector(1, 0, 0), Ms=1.65 - 0.02 * q, thickness=3e-9,
                             cellSurface=7e-14, demagTensor=_rows(np.diag([0.0, 0.0, 1.0]).tolist()), damping=0.005,
                             SlonczewskiSpacerLayerParameter=1.0, beta=0.1, spinPolarisation=0.6)
    l.setReferenceLayer(CVector(1, 0, 0))
    j = Junction([l], 100, 200)
    j.setLayerAnisotropyDriver("free", constantDriver(1.05e3))
    return j


def _array_element(m0, h: float) -> Junction:
    l = Layer("free", mag=CVector(*m0), anis=CVector(0, 0, 1), Ms=1.2, thickness=1.5e-9,
              cellSurface=math.pi * (25e-9) ** 2, demagTensor=_rows(np.diag([0.04, 0.04, 0.92]).tolist()),
              damping=0.01)
    j = Junction([l])
    j.setLayerAnisotropyDriver("free", constantDriver(8e5))
    j.setLayerExternalFieldDriver("all", AxialDriver(h, 0.0, 0.0))
    return j


def _dp_junction(Hx: float, Hz: float, fl: float, dl: float, m0) -> Junction:
    p = 0.017
    l = Layer("free", mag=CVector(*m0), anis=CVector(0, 0, 1), Ms=1.12, thickness=1e-9,
              cellSurface=math.pi * (300e-9) ** 2,
              demagTensor=_rows(np.diag([p, p, math.sqrt(1 - 2 * p * p)]).tolist()), damping=0.01)
    l.setReferenceLayer(CVector(0, 0, 1))
    l.setSecondOrderAnisotropyDriver(constantDriver(-30e3))
    l.setAnisotropyDriver(constantDriver(563e3))
    j = Junction([l])
    j.setLayerExternalFieldDriver("free", AxialDriver(Hx, 0, Hz))
    j.setLayerFieldLikeTorqueDriver("free", stepDriver(0, fl, 0, 1e-9))
    j.setLayerDampingLikeTorqueDriver("free", stepDriver(0, dl, 0, 1e-9))
    return j


# --- inputs from the seed (shared by prepare and exact) -------------------------

def _unit(v: np.ndarray) -> np.ndarray:
    return v / np.linalg.norm(v, axis=-1, keepdims=True)


def _inputs(case: dict, seed: int) -> dict:
    """The numbers a case draws: fields, currents, starting directions."""
    rng = np.random.default_rng([seed, 20])
    k = case["kind"]
    if k == "pimm":
        n = case["points"]
        h = np.sort(rng.uniform(0, 600e3, n))
        phi = math.radians(30)
        # the durations shape the log: the case's own, whatever the seed
        return {"T": np.random.default_rng(n).uniform(case["t_min"], case["t_max"], n),
                "H": np.stack([h * math.cos(phi), h * math.sin(phi), np.zeros(n)], axis=1)}
    if k == "rh":
        n = case["points"]
        th, ph = rng.uniform(0.01, 0.03, n), rng.uniform(0, 2 * math.pi, n)  # about 1 degree off the easy axis
        H = np.zeros((n, 3))
        H[:, 0] = np.linspace(-800e3, 800e3, n)
        return {"H": H, "m": _unit(np.stack([np.cos(th), np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph)], axis=1))}
    if k == "sto":
        n = case["points"]
        return {"I": np.linspace(-2e11, -2e10, n) * rng.uniform(0.99, 1.01, n)}
    if k == "cims":
        n = case["currents"] * case["seeds"]
        j = np.repeat(np.logspace(10, 12, case["currents"]), case["seeds"])
        return {"I": j, "seeds": rng.integers(0, 2 ** 63, n, dtype=np.uint64)}
    if k == "vsd":
        H = np.repeat(rng.uniform(50e3, 400e3, case["fields"]), case["freqs"])
        f = np.tile(np.linspace(1e9, 20e9, case["freqs"]), case["fields"])
        return {"H": np.stack([H * math.sqrt(0.5), 0 * H, H * math.sqrt(0.5)], axis=1), "f": f,
                "m": _unit(np.array([0.5, 0.0, 0.866]) + rng.normal(0, 1e-3, (len(H), 3)))}
    if k == "terms":
        n = case["points"]
        H = np.zeros((n, 3))
        H[:, 0] = rng.uniform(20e3, 200e3, n)
        return {"H": H}
    if k == "dropin":
        two = case["device"] in ("pimm", "sto", "terms")
        base = {"pimm": [[0.866, 0.5, 0.05], [1, 0, 0]], "sto": [[1, 0, 0], [1, 0.1, 0.1]],
                "terms": [[0.1, 0.2, 1], [1, 0.1, 0]], "rh": [[1, 0.02, 0.02]], "vsd": [[0.5, 0, 0.866]]}
        m = np.array(base[case["device"]], dtype=np.float64)
        return {"m": _unit(m + rng.normal(0, 1e-3, m.shape)), "h": float(rng.uniform(100e3, 300e3)), "two": two}
    if k == "dp":
        Hz, jd = np.meshgrid(np.linspace(-4e5, 4e5, case["fields"]), np.linspace(0.0, 0.3, case["currents"]),
                             indexing="ij")
        Hz, jd = Hz.ravel(), jd.ravel()
        m = _unit(np.array([0.1, 0.1, 0.99]) + rng.normal(0, 1e-2, (len(Hz), 3)))
        return {"Hx": 0.1 * np.abs(Hz) + 1e3, "Hz": Hz, "fl": 0.7 * T_TO_AM * 1e-3 * jd ** 2,
                "dl": 0.7 * T_TO_AM * 16e-3 * jd, "m": m}
    if k == "stack":
        n = case["members"]
        m = np.stack([0.1 * np.arange(n), np.full(n, 0.2), np.ones(n)], axis=1)
        return {"m": _unit(m + rng.normal(0, 1e-2, (n, 3))), "I": float(rng.uniform(2e11, 5e11)),
                "c": float(rng.uniform(0.02, 0.08))}
    if k == "array":
        n = case["side"] ** 2
        th = 0.2 + 0.01 * np.arange(n)
        m = np.stack([np.sin(th), 0 * th, np.cos(th)], axis=1)
        pos = np.stack([(np.arange(n) % case["side"]) * 60e-9, (np.arange(n) // case["side"]) * 60e-9, 0 * th], axis=1)
        return {"m": _unit(m + rng.normal(0, 1e-2, (n, 3))), "h": rng.uniform(1e4, 5e4, n), "pos": pos}
    return {}


# --- prepare --------------------------------------------------------------------

def _single(case: dict, x: dict) -> Junction:
    """The junction of a single run, its field from the inputs."""
    d, h = case["device"], x["h"]
    if d == "pimm":
        j = workloads.pimm_junction()
        j.setLayerExternalFieldDriver("all", AxialDriver(h * math.cos(math.pi / 6), h * math.sin(math.pi / 6), 0))
    elif d == "rh":
        j = _rh_junction()
        j.setLayerExternalFieldDriver("all", AxialDriver(h, 0, 0))
    elif d == "sto":
        j = workloads.sto_junction()
        j.setLayerCurrentDriver("free", constantDriver(-1e11))
    elif d == "vsd":
        j = workloads.vsd_junction(h, 5e9)
    else:
        j = _terms_junction()
        j.setLayerExternalFieldDriver("b", AxialDriver(h, 0, 0))
    return j


def prepare(case: dict, seed: int) -> dict:
    k, x = case["kind"], _inputs(case, seed)
    s = {"case": case, "x": x}
    if k == "pimm":
        b = JunctionBatch.replicate(workloads.pimm_junction(), case["points"], x["T"], DT, case["every"] * 1.0001 * DT,
                                    SolverMode.RK4, precision=case["precision"], log="mx")
        b.set_external_field("all", x["H"])
    elif k == "rh":
        b = JunctionBatch.replicate(_rh_junction(), case["points"], (case["steps"] + 0.5) * DT, DT, 1e-12,
                                    SolverMode.RK4, precision=case["precision"], log="full")
        b.set_external_field("all", x["H"])
        b.set_magnetisation("free", x["m"])
    elif k == "sto":
        b = workloads.sto(case["points"], (case["steps"] + 0.5) * DT, DT, precision=case["precision"])
        b.set_driver("free", "current", "constant", x["I"])
    elif k == "cims":
        T = (case["steps"] + 0.5) * 1e-14
        n = case["currents"] * case["seeds"]
        b = JunctionBatch.replicate(workloads.cims_junction(), n, T, 1e-14, T, SolverMode.EulerHeun,
                                    precision=case["precision"], log="none")
        b.set_driver("free", "current", "type", np.full(n, TRAPEZOID, dtype=np.int32))
        b.set_driver("free", "current", "amplitude", x["I"])
        b.set_driver("free", "current", "edge_time", np.full(n, T / 5))
        b.set_driver("free", "current", "steady_time", np.full(n, T / 5))
        b.set_seeds(x["seeds"])
    elif k == "vsd":
        b = JunctionBatch.replicate(workloads.vsd_junction(), len(x["f"]), (case["steps"] + 0.5) * 5e-13, 5e-13, 5e-13,
                                    SolverMode.RK4, precision=case["precision"], log="r", log_dtype="f64")
        b.set_external_field("all", x["H"])
        b.set_magnetisation("free", x["m"])
        f = np.zeros((len(x["f"]), 3))
        f[:, 1] = x["f"]
        b.set_driver("all", "oersted", "frequency", f)
    elif k == "terms":
        b = JunctionBatch.replicate(_terms_junction(), case["points"], (case["steps"] + 0.5) * DT, DT, 1e-12,
                                    SolverMode.RK4, precision=case["precision"], log="m")
        b.set_external_field("b", x["H"])
    elif k == "mixed":
        # structures and durations shape the log: the case's own; starting
        # directions and noise streams are the seed's
        specs = workloads.serving_mix(case["requests"], case["requests"], case["t_min"], case["t_max"])
        rng = np.random.default_rng([seed, 21])
        for q in specs:
            for l in q[1].layers:
                l.setMagnetisation(CVector(*(np.array([l.mag.x, l.mag.y, l.mag.z]) + rng.normal(0, 1e-2, 3)).tolist()))
            q[1].setNoiseSeed(int(rng.integers(0, 2 ** 62)))
        b = JunctionBatch.from_junctions([q[1] for q in specs], [q[2] for q in specs], [q[3] for q in specs],
                                         [q[4] for q in specs], [q[5] for q in specs], precision="fp32", log="m")
    elif k == "dp":
        js = [_dp_junction(*map(float, v[:4]), v[4].tolist()) for v in
              zip(x["Hx"], x["Hz"], x["fl"], x["dl"], x["m"])]
        b = JunctionBatch.from_junctions(js, case["total_time"], DP_STEP, 1e-11, SolverMode.DormandPrince,
                                         precision="fp64", log="none")
    elif k == "dropin":
        return dict(s, junction=_single(case, x))
    elif k == "stack":
        st = (SeriesStack if case["series"] else ParallelStack)(
            [_stack_member(q, m) for q, m in enumerate(x["m"].tolist())], useKCL=case["kcl"])
        st.setCouplingStrength(x["c"])
        st.setCoupledCurrentDriver(constantDriver(x["I"]))
        return dict(s, stack=st)
    else:
        g = GroupInteraction(_rows(x["pos"].tolist()),
                             [_array_element(m, float(h)) for m, h in zip(x["m"].tolist(), x["h"])])
        g.setInteractionFunction(computeDipoleInteraction if case["interaction"] == "kanao"
                                 else computeDipoleInteractionNoumra)
        return dict(s, group=g)
    b.plan()  # descriptors on the GPU, as a program that executes a sweep again keeps them
    b._buffers("cuda")
    return dict(s, batch=b)


# --- run ------------------------------------------------------------------------

def _log_of(junction: Junction) -> dict:
    return {k: np.asarray(v) for k, v in junction.getLog().items()}


def run(state: dict):
    case, x = state["case"], state["x"]
    k = case["kind"]
    if k == "dropin":  # one point as the procedures run it: clear, set m, run, read the log
        j = state["junction"]
        j.clearLog()
        for lid, m in zip(j.getLayerIds(), x["m"].tolist()):
            j.setLayerMagnetisation(lid, CVector(*m))
        dt = 5e-13 if case["device"] == "vsd" else DT
        j.runSimulation((case["steps"] + 0.5) * dt, dt, case["every"] * 1.0001 * dt)
        return _log_of(j)
    if k == "stack":
        st = state["stack"]
        st.clearLogs()
        for q, m in enumerate(x["m"].tolist()):
            st.setMagnetisation(q, "free", CVector(*m))
        st.runSimulation((case["steps"] + 0.5) * DT, DT, 1e-12)
        logs = [_log_of(st.getJunction(q)) for q in range(case["members"])]
        lg = st.getLog()
        return {"m": np.stack([[lo["free_mx"], lo["free_my"], lo["free_mz"]] for lo in logs]),
                "R": np.stack([lo["R"] for lo in logs]), "stack": {q: np.asarray(v) for q, v in lg.items()}}
    if k == "array":
        g = state["group"]
        g.clearLogs()
        for q, m in enumerate(x["m"].tolist()):
            g.junctionList[q].setLayerMagnetisation("free", CVector(*m))
        g.runSimulation((case["steps"] + 0.5) * DT, DT, 1e-12)
        logs = [_log_of(j) for j in g.junctionList]
        return np.stack([[lo["free_mx"], lo["free_my"], lo["free_mz"]] for lo in logs])
    b = state["batch"]
    r = b.execute()
    if k == "dp":  # the reached state and the step counts
        return {"m": r.final_m, "status": r.status_dev}
    # a program of the bulk mode goes on in binary32, as its log entries are
    m = r.final_m if case.get("precision") == "fp64" else r.final_m.to(torch.float32)
    return {"m": m} if k == "cims" else {"log": r.log, "m": m}


# --- work -----------------------------------------------------------------------

# algorithmic operations of one junction step: the reference's formulas with
# the active terms only, a fused multiply-add counted as two
_FLOP = {"pimm": 666, "rh": 297, "sto": 746, "cims": 450, "vsd": 330, "terms": 1300, "stack": 420}
_LAYER, _JUNCTION = 3056, 528


def work(case: dict) -> dict:
    k = case["kind"]
    if k == "pimm":
        n, T = case["points"], 0.5 * (case["t_min"] + case["t_max"])
        steps = n * T / DT
        size = 4 if case["precision"] == "fp32" else 8
        return {"bytes": n * (_JUNCTION + 2 * _LAYER) + 3 * size * steps / case["every"], "flops": 666 * steps}
    if k == "cims":
        n = case["currents"] * case["seeds"]
        return {"bytes": n * (_JUNCTION + 2 * _LAYER + 48), "flops": _FLOP[k] * n * case["steps"]}
    if k in ("rh", "sto", "vsd", "terms"):
        n = case["fields"] * case["freqs"] if k == "vsd" else case["points"]
        layers = 1 if k in ("rh", "vsd") else 2
        entries = case["steps"] / {"rh": 10, "sto": 100, "vsd": 1, "terms": 10}[k]
        channels = {"rh": 5, "sto": 7, "vsd": 1, "terms": 6}[k]
        size = 4 if case["precision"] == "fp32" and k != "vsd" else 8
        return {"bytes": n * (_JUNCTION + layers * _LAYER + channels * entries * size),
                "flops": _FLOP[k] * n * case["steps"]}
    if k == "mixed":  # mean steps of a request: its duration over a time step log-uniform in 1e-14..1e-13 s
        n, T = case["requests"], 0.5 * (case["t_min"] + case["t_max"])
        return {"bytes": n * (_JUNCTION + 2 * _LAYER + 6 * 4 * T / 1e-12), "flops": 700 * n * T / 3e-14}
    if k == "dp":  # about 7 evaluations of 75 operations and the step control per step of about 5 ps
        n = case["fields"] * case["currents"]
        return {"bytes": n * (_JUNCTION + _LAYER + 40), "flops": 700 * n * case["total_time"] / 5e-12}
    if k == "dropin":
        flop = _FLOP[case["device"]]
        layers, channels = (2, 7) if case["device"] in ("pimm", "sto", "terms") else (1, 4)
        return {"bytes": _JUNCTION + layers * _LAYER + 8 * channels * case["steps"] / case["every"],
                "flops": flop * case["steps"]}
    n = case["members"] if k == "stack" else case["side"] ** 2
    per = _FLOP["stack"] if k == "stack" else 333 + 26 * n
    return {"bytes": n * (_JUNCTION + _LAYER + 6 * 8 * case["steps"] / 10), "flops": per * n * case["steps"]}


# --- exact: the reference's equations in plain numpy, 64 bits --------------------

MU0, GYRO, HBAR, ECHARGE, KB = 12.566e-7, 220880.0, 6.62607015e-34 / (2.0 * math.pi), 1.60217662e-19, 1.380649e-23


def _cross(a, b):
    return (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _mat(N, m):
    return tuple(N[r][0] * m[0] + N[r][1] * m[1] + N[r][2] * m[2] for r in range(3))


class _L:
    """One layer of every instance: constants, and its applied field and
    torque current as functions of time."""

    def __init__(self, Ms, t, alpha, anis, K, N, K2=0.0, H=(0.0, 0.0, 0.0), field=None, **kw):
        self.Ms, self.t, self.alpha, self.anis, self.K, self.K2, self.H, self.field = Ms, t, alpha, anis, K, K2, H, field
        N = np.asarray(N, dtype=np.float64)
        self.N, self.diag = N, not np.any(N - np.diag(np.diag(N)))
        self.Jt = self.Jb = self.stt = self.sot = self.D = self.Nb = self.Nt = None
        self.J2t = self.J2b = 0.0
        self.__dict__.update(kw)

    def heff(self, t, m, bot, top):
        H = self.H if self.field is None else self.field(t)
        N, s = self.N, self.Ms / MU0
        u = _dot(self.anis, m)
        ha = 2 * self.K * u / self.Ms
        if self.K2:
            ha = ha + 4 * self.K2 * u ** 3 / self.Ms
        d = (N[0, 0] * m[0], N[1, 1] * m[1], N[2, 2] * m[2]) if self.diag else _mat(N, m)
        out = [H[q] + self.anis[q] * ha - s * d[q] for q in range(3)]
        for nb, J, J2, D, T in ((bot, self.Jb, self.J2b, self.D, self.Nb), (top, self.Jt, self.J2t, self.D, self.Nt)):
            if nb is None:
                continue
            if J is not None:
                w = (J(t) + 2 * J2 * _dot(nb, m)) / (self.Ms * self.t)
                out = [out[q] + nb[q] * w for q in range(3)]
            if D is not None:
                c = _cross(D, nb)
                out = [out[q] - c[q] / (self.Ms * self.t) for q in range(3)]
            if T is not None:
                c = _mat(T, nb)
                out = [out[q] - s * c[q] for q in range(3)]
        return out

    def rhs(self, t, m, bot, top, I=None):
        P = _cross(m, self.heff(t, m, bot, top))
        Q = _cross(m, P)
        a = self.alpha
        g = -GYRO / (1 + a * a)
        if self.stt is not None:  # Slonczewski torque: polarisation, beta, polariser
            pol, beta, ref = self.stt
            ref = bot if ref == "bottom" else ref
            w = GYRO * HBAR * (self.I if I is None else I) / (ECHARGE * self.Ms * self.t) * pol / 2
            F = _cross(m, ref)
            G = _cross(m, F)
            return [g * (P[q] + a * Q[q]) + w * (beta * F[q] - G[q]) / (1 + a * a) for q in range(3)]
        if self.sot is not None:  # field- and damping-like amplitudes at t, polariser
            fl, dl = self.sot(t)
            F = _cross(m, self.ref)
            G = _cross(m, F)
            return [g * (P[q] + a * Q[q] + (fl - a * dl) * F[q] + (dl + a * fl) * G[q]) for q in range(3)]
        return [g * (P[q] + a * Q[q]) for q in range(3)]


def _normal(m):
    r = np.sqrt(m[0] * m[0] + m[1] * m[1] + m[2] * m[2])
    return [m[0] / r, m[1] / r, m[2] / r]


def _rk4(layers, m, steps, dt, every, observe, before=None):
    """Fixed-step RK4, neighbours frozen at the start of a step; observe(m)
    after the steps that are logged; before(m): what a step takes from every
    instance's m at its start (a stack's currents, an array's field)."""
    out = []
    n = len(layers)
    for i in range(steps):
        t = i * dt
        I = before(m) if before is not None else None
        new = []
        for l, L in enumerate(layers):
            x, b, u = m[l], (m[l - 1] if l else None), (m[l + 1] if l + 1 < n else None)
            f = lambda ts, y: L.rhs(ts, y, b, u, I)  # noqa: E731
            k1 = f(t, x)
            k2 = f(t + 0.5 * dt, [x[q] + 0.5 * dt * k1[q] for q in range(3)])
            k3 = f(t + 0.5 * dt, [x[q] + 0.5 * dt * k2[q] for q in range(3)])
            k4 = f(t + dt, [x[q] + dt * k3[q] for q in range(3)])
            new.append(_normal([x[q] + dt / 6 * (k1[q] + 2 * (k2[q] + k3[q]) + k4[q]) for q in range(3)]))
        m = new
        if i % every == 0:
            out.append(observe(m))
    return m, np.asarray(out)


def _philox(c, k):
    """Philox4x32-10 on uint64 arrays of 32-bit words."""
    lo = np.uint64(0xFFFFFFFF)
    s = np.uint64(32)
    k0, k1 = k
    for r in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> s) ^ c[1] ^ k0, p1 & lo, (p0 >> s) ^ c[3] ^ k1, p0 & lo]
        k0, k1 = (k0 + np.uint64(0x9E3779B9)) & lo, (k1 + np.uint64(0xBB67AE85)) & lo
    return c


def _normals(seeds, streams, step, layer):
    lo, s = np.uint64(0xFFFFFFFF), np.uint64(32)
    o = _philox([np.full_like(seeds, step), np.full_like(seeds, layer), streams & lo, streams >> s],
                (seeds & lo, seeds >> s))
    u = [(w.astype(np.float64) + 0.5) * 2.0 ** -32 for w in o]
    r0, r1 = np.sqrt(-2 * np.log(u[0])), np.sqrt(-2 * np.log(u[2]))
    return r0 * np.cos(2 * math.pi * u[1]), r0 * np.sin(2 * math.pi * u[1]), r1 * np.cos(2 * math.pi * u[3])


def _euler_heun(layers, m, steps, dt, sigma, seeds):
    streams = np.arange(len(seeds), dtype=np.uint64)
    n = len(layers)
    for i in range(steps):
        new = []
        for l, L in enumerate(layers):
            x = m[l]
            f = L.rhs(i * dt, x, m[l - 1] if l else None, m[l + 1] if l + 1 < n else None)
            g = -GYRO / (1 + L.alpha ** 2)
            dW = [sigma[l] * z for z in _normals(seeds, streams, i, l)]

            def noise(y):
                c1 = _cross(y, dW)
                c2 = _cross(y, c1)
                return [g * (c1[q] + L.alpha * c2[q]) for q in range(3)]

            g0 = noise(x)
            g1 = noise([x[q] + math.sqrt(dt) * g0[q] for q in range(3)])
            new.append(_normal([x[q] + dt * f[q] + 0.5 * math.sqrt(dt) * (g0[q] + g1[q]) for q in range(3)]))
        m = new
    return m


_C = (0.0, 1 / 5, 3 / 10, 4 / 5, 8 / 9, 1.0, 1.0)
_A = ((), (1 / 5,), (3 / 40, 9 / 40), (44 / 45, -56 / 15, 32 / 9),
      (19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729),
      (9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656),
      (35 / 384, 0.0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84))
_B4 = (5179 / 57600, 0.0, 7571 / 16695, 393 / 640, -92097 / 339200, 187 / 2100, 1 / 40)


def _dormand_prince(L, m, T, h0):
    """Every instance on its own steps, with the reference's clock (it
    advances by the step proposed for the next attempt)."""
    n = len(m[0])
    t, h, steps = np.zeros(n), np.full(n, h0), np.zeros(n, dtype=np.int64)
    for _ in range(100000):
        on = t < T
        if not on.any():
            break
        h = np.where(t + h > T, T - t, h)
        h = np.where(h > 0, h, h0)
        k = []
        for s in range(7):
            y = [m[q] + sum(h * a * k[j][q] for j, a in enumerate(_A[s]) if a) for q in range(3)]
            k.append(L.rhs(t + _C[s] * h, y, None, None))
        m5 = y
        e = [m5[q] - m[q] - h * sum(b * k[j][q] for j, b in enumerate(_B4) if b) for q in range(3)]
        ratio = np.sqrt(_dot(e, e)) / (1e-6 + 1e-3 * np.sqrt(_dot(m, m)))
        with np.errstate(divide="ignore"):
            fac = 0.9 * (1.0 / ratio) ** 0.2
        fac = np.maximum(np.minimum(np.where(np.isfinite(fac), fac, 0.1), 5.0), 0.1)
        nh = h * fac
        ok = on & (ratio <= 1.0)
        forced = on & ~ok & (nh < 1e-15)
        new = _normal(m5)
        m = [np.where(ok, new[q], m[q]) for q in range(3)]
        h = np.where(on, nh, h)
        adv = ok | forced
        t = np.where(adv, t + h, t)
        steps += adv
    return m, steps


THIN = np.diag([0.0, 0.0, 1.0])
X, Z = (1.0, 0.0, 0.0), (0.0, 0.0, 1.0)


def _plain(case: dict, x: dict, device: str):
    """(layers, starting m, dt) of a device with the inputs' fields."""
    if device == "pimm":
        H = x["H"].T if "H" in x else x["h"] * np.array([[math.cos(math.pi / 6)], [math.sin(math.pi / 6)], [0.0]])
        on = 3 * DT
        field = lambda t: (H[0], H[1] + (1e3 if 0 <= t <= on else 0.0), H[2])  # noqa: E731
        J = lambda t: -1e-4  # noqa: E731
        Ls = [_L(1.0, 1e-9, 0.01, Z, 1.5e5, THIN, field=field, Jt=J), _L(1.6, 3e-9, 0.01, X, 1e4, THIN, field=field,
                                                                         Jb=J)]
        return Ls, [[math.cos(math.pi / 6), math.sin(math.pi / 6), 0.05], X], DT
    if device == "rh":
        H = x["H"].T if "H" in x else (x["h"], 0.0, 0.0)
        return [_L(1.2, 2e-9, 0.01, X, 5e3, np.diag([0.00024, 0.0022, 0.99756]), H=H)], [X], DT
    if device == "sto":
        I = x["I"] if "I" in x else -1e11
        Hz = (0.0, 0.0, 200e3)
        return [_L(1.2, 3e-9, 0.02, X, 1e5, THIN, H=Hz),
                _L(0.8, 2e-9, 0.005, X, 2e3, THIN, H=Hz, stt=(0.6, 0.0, "bottom"), I=I)], [X, (1.0, 0.1, 0.1)], DT
    if device == "vsd":
        H = x["H"].T if "H" in x else (x["h"] * math.sqrt(0.5), 0.0, x["h"] * math.sqrt(0.5))
        f = x["f"] if "f" in x else 5e9
        field = lambda t: (H[0], H[1] + 500.0 * np.sin(2 * math.pi * t * f), H[2])  # noqa: E731
        return [_L(1.0, 1.5e-9, 0.02, Z, 1e5, THIN, field=field)], [(0.5, 0.0, 0.866)], 5e-13
    if device == "cims":
        T = (case["steps"] + 0.5) * 1e-14
        e, hdl = T / 5, 1e-12 * T_TO_AM

        def sot(t):
            w = t / e if t <= e else 1.0 if t <= 2 * e else 1 - (t - 2 * e) / e if t <= 3 * e else 0.0
            return 0.3 * hdl * x["I"] * w, hdl * x["I"] * w

        H = (-20e3, 0.0, 0.0)
        return [_L(1.1, 1.2e-9, 0.02, Z, 3e5, np.zeros((3, 3)), H=H, sot=sot, ref=(0.0, 1.0, 0.0)),
                _L(1.2, 3e-9, 0.02, X, 1e5, THIN, H=H)], [Z, X], 1e-14
    Hb = x["H"][:, 0] if "H" in x else x["h"]
    J = lambda t: 1e-4 + 5e-5 * math.sin(2 * math.pi * t * 2e9)  # noqa: E731
    D = (1e-4, -2e-4, 5e-5)
    return [_L(1.2, 1.5e-9, 0.05, Z, 4e5, EXOTIC_DEMAG, K2=-3e4, H=(1e3, 0.0, -2e3), Jt=J, J2t=-2e-5, D=D,
               Nt=EXOTIC_DIPOLE),
            _L(0.9, 2e-9, 0.06, X, 2e4, EXOTIC_DEMAG, H=(1e3 + Hb, 0.0, -2e3), Jb=J, J2b=-2e-5, D=D,
               Nb=EXOTIC_DIPOLE)], [(0.1, 0.2, 1.0), (1.0, 0.1, 0.0)], DT


def _resistance(device: str, m) -> list:
    if device == "rh":
        rx = 100.0 + m[0][0] * m[0][0]
        return [rx, np.zeros_like(rx)]  # Ry: no transverse coefficient
    if device in ("pimm", "sto"):
        return [100 + 50 * (1 - _dot(m[0], m[1]))]
    return [100 + 50 * (1 - m[0][0])] if device == "vsd" else []


def _cost(n: int, steps: int, ops: float) -> float:
    """Seconds of the numpy integrator: operations of a step, per call and per element."""
    return steps * ops * (1.2e-6 + 1.5e-9 * n)


def exact(case: dict, seed: int):
    k, x = case["kind"], _inputs(case, seed)
    ops = {"pimm": 520, "rh": 230, "sto": 620, "vsd": 240, "terms": 1500}
    if k in ("pimm", "rh", "sto", "vsd", "terms"):
        n = len(x["f"]) if k == "vsd" else case["points"]
        steps = None if k == "pimm" else case["steps"]
        # a ragged sweep would be as many runs as it has points
        if k == "pimm" or _cost(n, steps, ops[k]) > 20:
            return None
        Ls, m0, dt = _plain(case, x, k)
        m = [[np.full(n, v) for v in w] for w in m0]
        if "m" in x:
            m = [[x["m"][:, q].copy() for q in range(3)]]
        keep = (lambda m: _resistance(k, m)) if k == "vsd" else \
            (lambda m: [c for w in m for c in w] + (_resistance(k, m) if k != "terms" else []))
        m, log = _rk4(Ls, m, steps, dt, {"rh": 10, "sto": 100, "vsd": 1, "terms": 10}[k], keep)
        final = np.zeros((n, 8, 3))
        for l, w in enumerate(m):
            final[:, l] = np.stack(w, axis=1)
        if k == "rh":  # Ry = 1 / (1 / 0): the reference's infinite conductance gives 0
            log[:, 4] = 0.0
        return {"log": np.ascontiguousarray(log.transpose(2, 1, 0)).ravel(), "m": final}
    if k == "cims":
        n = case["currents"] * case["seeds"]
        if _cost(n, case["steps"], 900) > 20:
            return None
        Ls, m0, dt = _plain(case, x, k)
        S = (50e-9) ** 2 * math.pi
        sigma = [math.sqrt(2 * L.alpha * KB * 300.0 / (L.Ms * S * L.t * GYRO)) for L in Ls]
        m = _euler_heun(Ls, [[np.full(n, v) for v in w] for w in m0], case["steps"], dt, sigma, x["seeds"])
        final = np.zeros((n, 8, 3))
        for l, w in enumerate(m):
            final[:, l] = np.stack(w, axis=1)
        return {"m": final}
    if k == "dropin":
        d = case["device"]
        Ls, _, dt = _plain(case, x, d)
        m = [[np.full(1, v) for v in w] for w in x["m"]]
        _, log = _rk4(Ls, m, case["steps"], dt, case["every"],
                      lambda m: [c for w in m for c in w] + _resistance(d, m))
        log = log[:, :, 0].T
        ids = {"pimm": ["free", "ref"], "sto": ["pinned", "free"], "terms": ["a", "b"]}.get(d, ["free"])
        out = {f"{i}_m{c}": log[3 * l + q] for l, i in enumerate(ids) for q, c in enumerate("xyz")}
        out["time"] = np.arange(log.shape[1]) * case["every"] * dt
        if d == "rh":
            out.update(Rx=log[3], Ry=np.zeros_like(log[3]), Rz=np.zeros_like(log[3]))
        elif d == "vsd":
            out["R"] = log[3]
        elif d in ("pimm", "sto"):
            out[f"R_{ids[0]}_{ids[1]}"] = log[6]
        return out
    if k == "dp":
        H = (x["Hx"], np.zeros_like(x["Hx"]), x["Hz"])
        p = 0.017
        L = _L(1.12, 1e-9, 0.01, Z, 563e3, np.diag([p, p, math.sqrt(1 - 2 * p * p)]), K2=-30e3, H=H, ref=Z,
               sot=lambda t: (np.where(t <= 1e-9, x["fl"], 0.0), np.where(t <= 1e-9, x["dl"], 0.0)))
        m, steps = _dormand_prince(L, [x["m"][:, q].copy() for q in range(3)], case["total_time"], DP_STEP)
        final = np.zeros((len(steps), 8, 3))
        final[:, 0] = np.stack(m, axis=1)
        return {"m": final, "status": None}
    if k == "stack":
        n = case["members"]
        L = _L(1.65 - 0.02 * np.arange(n), 3e-9, 0.005, X, 1.05e3, THIN, stt=(0.6, 0.1, X))
        rec = []

        def before(m):
            d = m[0][0]  # m . p, the polariser along x
            C = x["c"] * (d[:-1] + d[1:] if case["series"] else d[:-1] - d[1:])
            if case["kcl"]:
                I, shown = np.full(n, x["I"] * (1 + C.sum())), C
            else:
                I = x["I"] * np.concatenate([[1.0], np.cumprod(1 + C)])
                shown = (I[:-1] / x["I"]) * (1 + C)
            rec.append((I, shown))
            return I

        _, log = _rk4([L], [[x["m"][:, q].copy() for q in range(3)]], case["steps"], DT, 10, lambda m: m[0], before)
        R = 100 + 50 * (1 - log[:, 0])
        lg = {"Resistance": R.sum(axis=1) if case["series"] else 1 / (1 / R).sum(axis=1)}
        for q in range(n):
            lg[f"I_{q}"] = np.array([r[0][q] for r in rec[::10]])
            if q < n - 1:
                lg[f"C_{q}_{q + 1}"] = np.array([r[1][q] for r in rec[::10]])
        lg["time"] = np.arange(len(log)) * 10 * DT
        return {"m": log.transpose(2, 1, 0).copy(), "R": R.T.copy(), "stack": lg}
    if k == "array":
        n = case["side"] ** 2
        r = x["pos"][:, None] - x["pos"][None]
        d = np.linalg.norm(r, axis=-1) + np.eye(n)
        w = 1.2 / MU0 * 1.5e-9 * math.pi * (25e-9) ** 2 / (1 if case["interaction"] == "kanao" else 4 * math.pi)
        T = w * (3 * r[:, :, :, None] * r[:, :, None, :] / d[:, :, None, None] ** 5 -
                 np.eye(3) / d[:, :, None, None] ** 3) * (1 - np.eye(n))[:, :, None, None]
        T = T.transpose(2, 3, 0, 1).copy()
        L = _L(1.2, 1.5e-9, 0.01, Z, 8e5, np.diag([0.04, 0.04, 0.92]))

        def before(m):  # the field of the other elements at the start of the step
            g = [sum(T[a, b] @ m[0][b] for b in range(3)) for a in range(3)]
            L.H = (x["h"] + g[0], g[1], g[2])

        _, log = _rk4([L], [[x["m"][:, q].copy() for q in range(3)]], case["steps"], DT, 10, lambda m: m[0], before)
        return log.transpose(2, 1, 0).copy()
    return None
