"""FP32 batches with binary32 log entries, the default: the component-lane
kernels that carry the sine phases (their names end in "log f32"), one to four
layers, every sine kind, sines beside steps, records beyond the two kept in
registers, runs that end around blocks of 64 steps and are cut inside one,
against the oracle.

Tolerance: a step's increments are binary32, below 0.1 of m each and rounded a
dozen times at 6e-8: 1e-7 a step at the very most, 3e-5 over 301 steps if all
of them added up.  1e-5 for m holds since they do not; entries round once more
at 6e-8 of their size."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from cmtj_amd import (AxialDriver, NullDriver, SolverMode, _lib, constantDriver, posSineDriver, sineDriver, stepDriver,
                      workloads)
from cmtj_amd.batch import JunctionBatch
from test_gpu_component_lanes import _chain

pytestmark = pytest.mark.gpu

TOL = 1e-5
DT = 5e-13
STEPS = np.array([1, 2, 63, 64, 65, 128, 129, 301])


def _junction(kind, nl, q):
    j = _chain(nl, mr="none") if nl > 1 else workloads.vsd_junction(100e3 + 5e3 * q, 3e9 + 1e9 * q)
    step = stepDriver(0, 2e3, 20.25 * DT, 67.25 * DT)
    if kind == "sine":
        x, o = (constantDriver(1e5), sineDriver(0, 500, 3e9 + 1e9 * q, 0.1 * q), constantDriver(2e4)), None
    elif kind == "pos_sine":
        x, o = (posSineDriver(5e4, 2e4, 2.5e9 + 1e8 * q, 0.4), constantDriver(1e3), constantDriver(7e4)), None
    elif kind == "sine_step":
        x, o = (sineDriver(5e4, 2e4, 3e9, 0.3), constantDriver(0), constantDriver(1e5)), step
    else:  # four records
        x, o = (sineDriver(5e4, 2e4, 3e9, 0.3), sineDriver(0, 3e3, 2e9 + 1e8 * q, 0),
                posSineDriver(1e5, 4e3, 4e9, 0.2)), step
    j.setLayerExternalFieldDriver("all", AxialDriver(*x))
    j.setLayerOerstedFieldDriver("all", AxialDriver(NullDriver(), o or NullDriver(), NullDriver()))
    return j


@pytest.mark.parametrize("w", [1, 3])
@pytest.mark.parametrize("kind", ["sine", "pos_sine", "sine_step", "four"])
@pytest.mark.parametrize("nl", [1, 2, 3, 4])
def test_binary32_entries(nl, kind, w):
    js = [_junction(kind, nl, q % 3) for q in range(len(STEPS))]
    b = JunctionBatch.from_junctions(js, (STEPS + 0.5) * DT, DT, w * 1.0001 * DT, SolverMode.RK4, log="full")
    kname = b.plan().info.kernel_name.decode()
    assert kname.startswith("k_junction_cl<") and "log f32" in kname and b.plan().info.n_kernels == 1, kname
    r = b.run()
    olog, omag, ost = oracle.run_batch(b.js, b.layers, _lib.constants_get(), b.tables, b.log_elements)
    st = r.status()
    assert (st["steps_done"] == STEPS).all() and (st["entries_done"] == ost["entries_done"]).all()
    g, gm = r.log.cpu().numpy(), r.final_m.cpu().numpy()
    assert g.dtype == np.float32
    d = float(np.max(np.abs(g - olog) / np.maximum(1.0, np.abs(olog))))
    dm = float(np.max(np.abs(gm[:, :nl] - omag[:, :nl])))
    print(f"[f32 entries] {kname} {kind} w={w}: log {d:.2e}, m {dm:.2e}", flush=True)
    assert dm <= TOL and d <= TOL + 1.2e-7
    s = b.subset(np.arange(len(js))).run_sliced(77)
    np.testing.assert_array_equal(s.log.cpu().numpy(), g)
    np.testing.assert_array_equal(s.final_m.cpu().numpy(), gm)
