"""One layer per lane for the exact feature sets (RK4 chains under field
steps, Euler-Heun switching devices under trapezoid drives) against the
oracle: 2-4 layers, drive windows inside and across blocks of 64 steps, every
scalar slot a trapezoid can feed there, a polariser taken from the neighbour,
log intervals, steps too long for the length correction's series, NaN stops
and runs cut into slices."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from cmtj_amd import (AxialDriver, CVector, Junction, Layer, NullDriver, Reference, SolverMode, _lib, constantDriver,
                      stepDriver, trapezoidDriver, workloads)
from cmtj_amd.batch import JunctionBatch

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-8, "fp32": 1e-4}  # the drop-in's bar; the bulk mode's
STEPS = np.array([1, 2, 63, 64, 65, 129, 300, 301])


def _chain(nl, q, dt):
    j = workloads.chain_junction(nl, 100e3 + 20e3 * q) if nl > 2 else workloads.pimm_junction()
    if nl == 2:
        j.setLayerExternalFieldDriver("all", AxialDriver(50e3 * (q + 1), 20e3, 0))
    j.setLayerOerstedFieldDriver("all", AxialDriver(NullDriver(), stepDriver(0, 2e3, 60.25 * dt, 67.25 * dt),
                                                    NullDriver()))
    return j


def _check(js, dt, w, solver, precision, steps=STEPS):
    b = JunctionBatch.from_junctions(js, (steps + 0.5) * dt, dt, w * 1.0001 * dt, solver, precision=precision,
                                     log="full", log_dtype="f64").set_lanes("per_layer")
    kname = b.plan().info.kernel_name.decode()
    assert "k_junction_ll" in kname and "waves" in kname and b.plan().info.n_kernels == 1, kname
    r = b.run()
    olog, omag, ost = oracle.run_batch(b.js, b.layers, _lib.constants_get(), b.tables, b.log_elements)
    st = r.status()
    for f in ("code", "steps_done", "entries_done", "nan_layer"):
        assert (st[f] == ost[f]).all(), (f, st[f], ost[f])
    g, gm = r.log.cpu().numpy(), r.final_m.cpu().numpy()
    nl = int(b.js[0]["n_layers"])
    worst = 0.0
    for i in range(len(js)):
        ne, off = int(b.js[i]["n_entries"]), int(b.js[i]["log_offset"])
        n = int(ost[i]["entries_done"])
        nch = _lib.n_channels(nl, int(b.js[i]["mr_mode"]), int(b.js[i]["log_mask"]))
        x, y = (v[off:off + nch * ne].reshape(nch, ne)[:, :n] for v in (g, olog))
        worst = max(worst, float(np.max(np.abs(x - y) / np.maximum(1.0, np.abs(y)), initial=0.0)))
    ok = np.isfinite(omag[:, :nl])
    assert np.array_equal(np.isfinite(gm[:, :nl]), ok)
    worst = max(worst, float(np.max(np.abs(gm[:, :nl][ok] - omag[:, :nl][ok]))))
    print(f"[layer lanes] {kname} w={w}: {worst:.2e}", flush=True)
    assert worst <= TOL[precision]
    if (st["code"] == 0).all():
        # (the same noise streams: packing the junctions again would take new ones)
        s = b.subset(np.arange(len(js)), log_dtype="f64").run_sliced(77)
        np.testing.assert_array_equal(s.log.cpu().numpy(), g)
        np.testing.assert_array_equal(s.final_m.cpu().numpy(), gm)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("w", [1, 3, 1000])
@pytest.mark.parametrize("nl", [2, 3, 4])
def test_chains_match_the_oracle(nl, w, precision):
    dt = 2e-13
    _check([_chain(nl, q, dt) for q in range(len(STEPS))], dt, w, SolverMode.RK4, precision)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_long_steps_and_a_nan(precision):
    """gamma H dt of about 0.7 takes the length correction out of its series;
    an infinite drive from step 70 on stops one instance."""
    dt = 2.5e-12
    js = [_chain(2, q, dt) for q in range(len(STEPS))]
    for q, j in enumerate(js):
        j.setLayerExternalFieldDriver("all", AxialDriver(1e5, 0, 1.2e6 if q % 2 else 1e5))
        j.setLayerOerstedFieldDriver("all", AxialDriver(
            NullDriver(), stepDriver(0, float("inf") if q == 6 else 2e3, 70.25 * dt, 1e-6), NullDriver()))
    _check(js, dt, 1, SolverMode.RK4, precision)


def _device(kind, q, dt):
    T = 300 * dt
    trap = lambda a: trapezoidDriver(0, a, 10.3 * dt, 40 * dt, 100 * dt)  # noqa: E731
    j = workloads.cims_junction(300.0)
    j.setNoiseSeed(100 + q)
    jc = 2e11 * (q + 1)
    if kind == "fl_dl":
        l = Layer("free", mag=CVector(0.1, 0, 1), anis=CVector(0, 0, 1), Ms=1.1, thickness=1.2e-9, cellSurface=1e-15,
                  demagTensor=[CVector(0, 0, 0)] * 3, damping=0.02)
        l.setReferenceLayer(CVector(0, 1, 0))
        j = Junction([l, j.getLayer("pinned")], 100, 200)
        j.setNoiseSeed(100 + q)
        j.setLayerAnisotropyDriver("free", constantDriver(3e5))
        j.setLayerPrimaryTorqueDrivers("free", trap(2e4 + 1e3 * q), trap(1e5))
        j.setLayerTemperatureDriver("all", constantDriver(300.0))
        return j
    j.setLayerCurrentDriver("free", trap(jc))
    if kind == "two_currents":
        j.setLayerCurrentDriver("pinned", trapezoidDriver(0, 1e11, 0, T / 5, T / 7))
    elif kind == "temperature":
        j.setLayerTemperatureDriver("pinned", trapezoidDriver(100.0, 300.0, 0, T / 3, T / 9))
    elif kind == "anisotropy":
        j.setLayerAnisotropyDriver("free", trapezoidDriver(3e5, -5e4, 20 * dt, 64 * dt, 64 * dt))
    elif kind == "polariser_neighbour":
        j.setLayerReferenceType("free", Reference.top)
    elif kind == "sharp":
        j.setLayerCurrentDriver("free", trapezoidDriver(1e10, jc, 64 * dt, 1e-3 * dt, 63 * dt))
    return j


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("kind", ["current", "two_currents", "temperature", "anisotropy", "fl_dl",
                                  "polariser_neighbour", "sharp"])
def test_switching_devices_match_the_oracle(kind, precision):
    dt = 1e-14
    _check([_device(kind, q, dt) for q in range(len(STEPS))], dt, 3, SolverMode.EulerHeun, precision)
