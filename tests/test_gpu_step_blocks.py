"""The component-lane step loop's blocks of 64 steps against the oracle:
lengths of runs and log intervals around a block's edges, steps so long that
the length correction leaves its series' range (every block is then taken
again step by step), sine drives whose phase is carried from stage to stage,
and runs cut into slices inside a block."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from cmtj_amd import AxialDriver, CVector, Junction, Layer, SolverMode, _lib, constantDriver, posSineDriver, workloads
from cmtj_amd.batch import JunctionBatch

pytestmark = pytest.mark.gpu

# binary64 kernels: the drop-in's bar; binary32 increments: the bulk mode's
TOL = {"fp64": 1e-8, "fp32": 1e-4}


def _junction(kind, q):
    if kind == "sine":
        return workloads.vsd_junction(100e3 + 5e3 * q, 3e9 + 1e9 * q)
    if kind == "half_and_pos_sine":
        j = workloads.vsd_junction(100e3 + 5e3 * q, 3e9)
        j.setLayerExternalFieldDriver("all", AxialDriver(posSineDriver(5e4, 2e4, 2.5e9 + 1e8 * q, 0.4),
                                                         constantDriver(1e3), constantDriver(7e4)))
        return j
    # gamma H dt is about 0.7 q: the length changes by up to a few percent a step
    l = Layer("free", mag=CVector(0.6, 0.1, 0.8), anis=CVector(0, 0, 1), Ms=1.0, thickness=1e-9, cellSurface=1e-16,
              demagTensor=[CVector(0, 0, 0), CVector(0, 0, 0), CVector(0, 0, 1)], damping=0.1)
    l.setReferenceLayer(CVector(1, 0, 0))
    j = Junction([l], 100, 200)
    j.setLayerAnisotropyDriver("free", constantDriver(1e5))
    j.setLayerExternalFieldDriver("all", AxialDriver(1e5, 0, 1.2e6 * q))
    return j


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("w", [1, 3, 64, 1000])
@pytest.mark.parametrize("kind", ["sine", "half_and_pos_sine", "long_steps"])
def test_blocks_match_the_oracle(kind, w, precision):
    dt = 2.5e-12 if kind == "long_steps" else 5e-13
    steps = np.array([1, 2, 63, 64, 65, 128, 129, 301])
    js = [_junction(kind, q % 3) for q in range(len(steps))]
    b = JunctionBatch.from_junctions(js, (steps + 0.5) * dt, dt, w * 1.0001 * dt, SolverMode.RK4, precision=precision,
                                     log="full", log_dtype="f64").set_lanes("per_component")
    assert "k_junction_cl" in b.plan().info.kernel_name.decode()
    r = b.run()
    olog, omag, ost = oracle.run_batch(b.js, b.layers, _lib.constants_get(), b.tables, b.log_elements)
    st = r.status()
    assert (st["steps_done"] == steps).all() and (st["entries_done"] == ost["entries_done"]).all()
    g = r.log.cpu().numpy()
    d = float(np.max(np.abs(g - olog) / np.maximum(1.0, np.abs(olog))))
    dm = float(np.max(np.abs(r.final_m.cpu().numpy()[:, :1] - omag[:, :1])))
    print(f"[blocks] {kind} w={w} {precision}: log {d:.2e}, m {dm:.2e}", flush=True)
    assert d <= TOL[precision] and dm <= TOL[precision]
    # the same run in slices of a block and a part: bit for bit
    s = JunctionBatch.from_junctions(js, (steps + 0.5) * dt, dt, w * 1.0001 * dt, SolverMode.RK4, precision=precision,
                                     log="full", log_dtype="f64").set_lanes("per_component").run_sliced(77)
    np.testing.assert_array_equal(s.log.cpu().numpy(), g)
    np.testing.assert_array_equal(s.final_m.cpu().numpy(), r.final_m.cpu().numpy())
