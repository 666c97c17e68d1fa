"""A switching step adds its drift and its thermal kick to m in binary64 also
in FP32 batches: at a temperature where the kick (1e-10) lies below the
spacing of binary32 numbers at the drift (0.004), one step with and one
without the kick differ by it as they do in FP64.

Tolerance: the normals and the kick's products are binary32, some ten
roundings of 6e-8 of its size; the difference of two unit vectors adds 4e-16.
2e-6 of the largest kick and 2e-15 cover both."""
from __future__ import annotations

import numpy as np
import pytest

from cmtj_amd import SolverMode, constantDriver, trapezoidDriver, workloads
from cmtj_amd.batch import JunctionBatch

pytestmark = pytest.mark.gpu

DT = 1e-12


def _final(T, two, precision):
    js = []
    for q in range(64):
        j = workloads.cims_junction(T)
        j.setNoiseSeed(100 + q)
        j.setLayerCurrentDriver("free", trapezoidDriver(0, 2e10 * (q + 1), 0, 10 * DT, 10 * DT))
        if two:
            j.setLayerCurrentDriver("pinned", trapezoidDriver(0, 1e11, 0, 5 * DT, 5 * DT))
        js.append(j)
    b = JunctionBatch.from_junctions(js, 1.5 * DT, DT, 1e-9, SolverMode.EulerHeun, precision=precision,
                                     log="none").set_lanes("per_layer")
    assert "waves" in b.plan().info.kernel_name.decode() and b.plan().info.n_kernels == 1
    return b.run().final_m.cpu().numpy()[:, :2]


@pytest.mark.parametrize("two", [False, True])
def test_a_small_kick_is_kept(two):
    T = 1e-13
    kick = {p: _final(T, two, p) - _final(0.0, two, p) for p in ("fp64", "fp32")}
    big = float(np.max(np.abs(kick["fp64"])))
    off = float(np.max(np.abs(kick["fp32"] - kick["fp64"])))
    print(f"[kick] two={two}: largest kick {big:.2e}, FP32 off by {off:.2e}", flush=True)
    assert 1e-11 < big < 1e-9
    assert off <= 2e-6 * big + 2e-15
