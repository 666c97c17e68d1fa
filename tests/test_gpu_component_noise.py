"""Stochastic solvers on one lane per component: the normals of four steps at a
time shared by a quad (binary32 normals in FP32 batches), drives on straight
pieces of a trapezoid, the length correction's series and the root beyond it,
against the oracle on the same noise streams: step counts around blocks of 4
and 64, one to four layers, Euler-Heun and Heun, and runs cut into slices at a
step that is no multiple of 4.

Tolerances: the drop-in's bar in FP64; in FP32 the normals carry 1.3e-7 each
and a step's kick is below 1e-2, so 300 steps stay within 1e-5 (the bulk mode's
bar is 1e-4)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from cmtj_amd import SolverMode, _lib, constantDriver, workloads
from cmtj_amd.batch import JunctionBatch
from test_gpu_layer_lanes_exact import _device

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-8, "fp32": 1e-5}
STEPS = np.array([1, 2, 3, 4, 5, 63, 64, 65, 129, 300])


def _check(js, dt, solver, precision, exact, w=3):
    b = JunctionBatch.from_junctions(js, (STEPS + 0.5) * dt, dt, w * 1.0001 * dt, solver, precision=precision,
                                     log="full", log_dtype="f64")
    kname = b.plan().info.kernel_name.decode()
    assert kname.startswith("k_junction_cl<" + ("double" if precision == "fp64" else "normals f32"))
    # (FP32: by the automatic choice only)
    assert ("FM_CIMS" in kname) == exact and b.plan().info.n_kernels == 1, kname
    r = b.run()
    olog, omag, ost = oracle.run_batch(b.js, b.layers, _lib.constants_get(), b.tables, b.log_elements)
    g, gm = r.log.cpu().numpy(), r.final_m.cpu().numpy()
    nl = int(b.js[0]["n_layers"])
    assert (r.status()["code"] == 0).all()
    worst = float(np.max(np.abs(g - olog) / np.maximum(1.0, np.abs(olog))))
    worst = max(worst, float(np.max(np.abs(gm[:, :nl] - omag[:, :nl]))))
    print(f"[component noise] {kname}: {worst:.2e}", flush=True)
    assert worst <= TOL[precision]
    s = b.subset(np.arange(len(js)), log_dtype="f64").run_sliced(77)
    np.testing.assert_array_equal(s.log.cpu().numpy(), g)
    np.testing.assert_array_equal(s.final_m.cpu().numpy(), gm)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("kind", ["current", "temperature", "anisotropy", "only_temperature", "only_anisotropy",
                                  "polariser_neighbour", "sharp"])
def test_switching_devices(kind, precision):
    dt = 1e-14
    js = [_device(kind.replace("only_", ""), q, dt) for q in range(len(STEPS))]
    if kind.startswith("only_"):  # the trapezoid feeds that slot alone
        for j in js:
            j.setLayerCurrentDriver("free", constantDriver(4e11))
    # (a second record takes the general set)
    _check(js, dt, SolverMode.EulerHeun, precision, exact=kind not in ("temperature", "anisotropy"))


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("solver", [SolverMode.EulerHeun, SolverMode.Heun])
@pytest.mark.parametrize("nl", [1, 2, 3, 4])
def test_general_sets(nl, solver, precision):
    js = []
    for q in range(len(STEPS)):
        j = workloads.chain_junction(nl, 1e5 + 1e4 * q) if nl > 1 else workloads.vsd_junction()
        # the last instances leave the series' range: kicks of several percent
        j.setLayerTemperatureDriver("all", constantDriver(300.0 if q < 7 else 3e5))
        j.setNoiseSeed(7 + q)
        js.append(j)
    _check(js, 1e-13, solver, precision, exact=False)
