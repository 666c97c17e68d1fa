"""Component and layer lanes with a diagonal field matrix (anisotropy along an axis) and
with a full one: each against the oracle, and an instance's bits the same
whether its wave holds tilted axes beside it or not.  Tolerances: the
drop-in's bar in FP64, the bulk mode's in FP32."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from cmtj_amd import AxialDriver, CVector, Junction, Layer, NullDriver, SolverMode, _lib, constantDriver, stepDriver
from cmtj_amd.batch import JunctionBatch

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-8, "fp32": 1e-4}
AXES = [(0, 0, 1), (1, 0, 0), (0, 1, 0), (0.6, 0, 0.8), (0.48, 0.64, 0.6), (0, -1, 0), (0, 0.8, -0.6), (0, 0, -1)]


def _junction(nl, q, tilted, stt):
    axis = AXES[q % 8] if tilted else AXES[[0, 1, 2, 5, 7][q % 5]]
    ls = []
    for l in range(nl):
        make = Layer.createSTTLayer if stt else Layer
        kw = dict(SlonczewskiSpacerLayerParameter=1.0, beta=0.1, spinPolarisation=0.5) if stt else {}
        y = make(f"l{l}", mag=CVector(0.1 + 0.1 * q, 0.3, 0.9), anis=CVector(*axis), Ms=1.2, thickness=1.5e-9,
                 cellSurface=1e-15, demagTensor=[CVector(0.02, 0, 0), CVector(0, 0.05, 0), CVector(0, 0, 0.93)],
                 damping=0.03, **kw)
        if stt:
            y.setReferenceLayer(CVector(0, 0.6, 0.8))
        ls.append(y)
    j = Junction(ls, 100, 200) if nl == 2 else Junction(ls)
    j.setLayerAnisotropyDriver("all", constantDriver(4e5))
    if stt:
        j.setLayerCurrentDriver("l0", constantDriver(3e10))
    else:
        j.setLayerOerstedFieldDriver("all", AxialDriver(NullDriver(), stepDriver(0, 2e3, 3e-12, 9e-12), NullDriver()))
    for l in range(nl - 1):
        j.setIECDriver(f"l{l}", f"l{l + 1}", constantDriver(2e-5))
    j.setLayerExternalFieldDriver("all", AxialDriver(3e4 * (q + 1), 1e4, 2e4))
    return j


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("nl,stt,lanes", [(1, False, "per_component"), (2, False, "per_component"),
                                          (4, False, "per_component"), (2, True, "per_component"),
                                          (2, False, "per_layer"), (4, False, "per_layer")])
def test_axes(nl, stt, lanes, precision):
    out = {}
    for tilted in (False, True):
        js = [_junction(nl, q, tilted, stt) for q in range(16)]
        b = JunctionBatch.from_junctions(js, 2.005e-11, 1e-13, 1e-13, SolverMode.RK4, precision=precision, log="m",
                                         log_dtype="f64").set_lanes(lanes)
        assert ("k_junction_cl" if lanes == "per_component" else "waves 3") in b.plan().info.kernel_name.decode() and b.plan().info.n_kernels == 1
        r = b.run()
        olog, omag, _ = oracle.run_batch(b.js, b.layers, _lib.constants_get(), b.tables, b.log_elements)
        worst = float(np.max(np.abs(r.log.cpu().numpy() - olog)))
        print(f"[axes] {b.plan().info.kernel_name.decode()} tilted={tilted}: {worst:.2e}", flush=True)
        assert worst <= TOL[precision]
        out[tilted] = b, r.final_m.cpu().numpy()
    # alone (or among axis-aligned ones) and beside tilted axes
    b, m = out[True]
    for q in (0, 1, 2, 5):
        a = b.subset(np.array([q]), log_dtype="f64").set_lanes(lanes)
        np.testing.assert_array_equal(a.run().final_m.cpu().numpy()[0, :nl], m[q, :nl])
