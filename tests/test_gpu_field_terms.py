"""Every field term on one lane per component in binary64 (the set without
spin torques, and the general set where a record is no sine): couplings and
anisotropies that a drive moves against those kept in the step's constant
matrix and base field, records beyond the two kept in registers, off-diagonal
tensors, one to four layers, against the oracle.  Tolerance: the drop-in's
bar, 1e-8 (500 steps round at 1e-16 each)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from cmtj_amd import (AxialDriver, CVector, Junction, Layer, SolverMode, _lib, constantDriver, sineDriver, stepDriver)
from cmtj_amd.batch import JunctionBatch

pytestmark = pytest.mark.gpu

DEMAG = [CVector(0.02, 0.001, 0.0005), CVector(0.001, 0.03, 0.0002), CVector(0.0005, 0.0002, 0.95)]
DIPOLE = [CVector(0.01, 0.002, 0.0), CVector(0.002, 0.015, 0.001), CVector(0.0, 0.001, -0.02)]


def _junction(nl, kind, q):
    ls = []
    for l in range(nl):
        a = Layer(f"l{l}", mag=CVector(0.1 + 0.3 * l, 0.2, 1 - 0.2 * l), anis=CVector(l % 2, 0.1, 1 - l % 2),
                  Ms=1.2 - 0.1 * l, thickness=1.5e-9, cellSurface=1e-16, demagTensor=DEMAG, damping=0.05)
        if l + 1 < nl:
            a.setTopDipoleTensor(DIPOLE)
        if l:
            a.setBottomDipoleTensor(DIPOLE)
        ls.append(a)
    j = Junction(ls)
    wave = (lambda c, a, k: sineDriver(c, a, 3e9 + 1e9 * k, 0.2 * k + 0.1 * q))
    if "step" in kind:
        wave = (lambda c, a, k: stepDriver(c, a, 3e-12 + 1e-12 * k, 3e-11))
    j.setLayerAnisotropyDriver("all", wave(4e5, 1e5, 1) if "k1" in kind else constantDriver(4e5))
    j.setLayerSecondOrderAnisotropyDriver("all", wave(-3e4, 1e4, 2) if "k2" in kind else constantDriver(-3e4))
    j.setLayerExternalFieldDriver("l0", AxialDriver(wave(1e4, 5e3, 0), wave(0, 4e3, 1), wave(2e3, 3e3, 2))
                                  if "h" in kind.split("_") else AxialDriver(1e4 * (q + 1), 2e3, 0))
    for l in range(nl - 1):
        a, b = f"l{l}", f"l{l + 1}"
        j.setIECDriver(a, b, wave(1e-4, 5e-5, 3) if "iec" in kind else constantDriver(1e-4))
        j.setQuadIECDriver(a, b, wave(-2e-5, 1e-5, 1) if "quad" in kind else constantDriver(-2e-5))
        j.setIDMIDriver(a, b, AxialDriver(wave(1e-4, 3e-5, 0), wave(-2e-4, 5e-5, 1), wave(5e-5, 2e-5, 2))
                        if "idmi" in kind else AxialDriver(1e-4, -2e-4, 5e-5))
    return j


@pytest.mark.parametrize("kind", ["const", "k1", "k2", "h", "iec", "quad", "idmi", "h_iec_quad_k1_k2_idmi",
                                  "step_iec_k1", "step_quad_idmi"])
@pytest.mark.parametrize("nl", [1, 2, 3, 4])
def test_field_terms(nl, kind):
    if nl == 1 and set(kind.split("_")) & {"iec", "quad", "idmi"}:
        pytest.skip("no neighbour to couple to")
    js = [_junction(nl, kind, q) for q in range(5)]
    steps = np.array([1, 63, 64, 130, 500])
    b = JunctionBatch.from_junctions(js, (steps + 0.5) * 1e-13, 1e-13, 3.0003e-13, SolverMode.RK4, precision="fp64",
                                     log="m", log_dtype="f64").set_lanes("per_component")
    kname = b.plan().info.kernel_name.decode()
    want = f"k_junction_cl<double,{4 if nl > 2 else nl}," + ("FM_STTC" if "step" in kind else "FM_FIELD")
    assert kname.startswith(want) and b.plan().info.n_kernels == 1, kname
    r = b.run()
    olog, omag, ost = oracle.run_batch(b.js, b.layers, _lib.constants_get(), b.tables, b.log_elements)
    g, gm = r.log.cpu().numpy(), r.final_m.cpu().numpy()
    worst = max(float(np.max(np.abs(g - olog))), float(np.max(np.abs(gm[:, :nl] - omag[:, :nl]))))
    print(f"[field terms] {kname} {kind}: {worst:.2e}", flush=True)
    assert worst <= 1e-8


def test_a_drive_that_is_not_finite_stays_with_its_layer():
    """An infinite field amplitude on layer 0 of two uncoupled layers from step
    70 on stops the run there, layer 1's last m finite."""
    js = []
    for q in range(3):
        ls = [Layer(f"l{l}", mag=CVector(0.1, 0.2, 1), anis=CVector(0, 0, 1), Ms=1.2, thickness=1.5e-9, cellSurface=1e-16,
                    demagTensor=DEMAG, damping=0.05) for l in range(2)]
        j = Junction(ls)
        j.setLayerAnisotropyDriver("all", sineDriver(4e5, 1e5, 3e9, 0.1))
        j.setLayerExternalFieldDriver("l1" if q == 1 else "l0", AxialDriver(
            stepDriver(0, float("inf") if q else 1e3, 7e-12, 1e-9), constantDriver(0), constantDriver(1e4)))
        j.setLayerExternalFieldDriver("l0" if q == 1 else "l1", AxialDriver(
            stepDriver(0, 1e3, 7e-12, 1e-9), constantDriver(0), constantDriver(1e4)))
        js.append(j)
    b = JunctionBatch.from_junctions(js, 2e-11, 1e-13, 3.0003e-13, SolverMode.RK4, precision="fp64", log="m",
                                     log_dtype="f64").set_lanes("per_component")
    r = b.execute()
    olog, omag, ost = oracle.run_batch(b.js, b.layers, _lib.constants_get(), b.tables, b.log_elements)
    st, gm = r.status(), r.final_m.cpu().numpy()
    for f in ("code", "steps_done", "entries_done", "nan_layer"):
        assert (st[f] == ost[f]).all(), (f, st[f], ost[f])
    assert np.array_equal(np.isfinite(gm[:, :2]), np.isfinite(omag[:, :2]))
