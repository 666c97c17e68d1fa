"""Full-chip sweeps of uneven lengths laid out in workgroups that hold a CU's
share of waves (pair_waves): every instance runs once, in whichever slot, with
the bits it has in a small batch; one instance past a full round, part-filled
last rounds and waves, two and three rounds, two- and four-layer lanes, a
resume in slices and a NaN."""
from __future__ import annotations

import numpy as np
import pytest

from cmtj_amd import AxialDriver, NullDriver, SolverMode, stepDriver, workloads
from cmtj_amd.batch import JunctionBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nl,n", [(2, 32769), (2, 45000), (2, 65536), (2, 65537), (2, 98304), (3, 16385), (4, 40000)])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_every_instance_runs_once(nl, n, precision):
    import torch

    rng = np.random.default_rng(n)
    steps = rng.integers(1, 70, n)
    steps[0], steps[1] = 130, 1
    dt = 2e-13
    j = workloads.pimm_junction() if nl == 2 else workloads.chain_junction(nl, 1e5)
    j.setLayerOerstedFieldDriver("all", AxialDriver(NullDriver(), stepDriver(0, 2e3, 5 * dt, 20 * dt), NullDriver()))
    b = JunctionBatch.replicate(j, n, (steps + 0.5) * dt, dt, 3.0003 * dt, SolverMode.RK4, precision=precision, log="full")
    H = rng.normal(0, 5e4, (n, 3))
    H[7] = np.inf  # stops at its first step
    b.set_external_field("all", H)
    assert "waves 3" in b.plan().info.kernel_name.decode()
    log, mag, st = b._buffers("cuda")
    log.fill_(float("nan"))
    mag.fill_(float("nan"))
    st.fill_(0xFF)
    r = b.execute()
    torch.cuda.synchronize()
    s = r.status()
    bad = np.arange(n) == 7
    assert (s["steps_done"][~bad] == steps[~bad]).all() and (s["code"][~bad] == 0).all() and s["code"][7] != 0
    pick = np.unique(np.concatenate([[0, 1, 7, n - 1], rng.integers(0, n, 300)]))
    q = b.subset(pick).set_lanes("per_layer")
    rq = q.execute()
    torch.cuda.synchronize()
    np.testing.assert_array_equal(r.final_m.cpu().numpy()[pick][:, :nl], rq.final_m.cpu().numpy()[:, :nl])
    for i, p in enumerate(pick):
        if p == 7:
            continue
        x, y = r.instance_log(int(p)), rq.instance_log(i)
        for k in x:
            np.testing.assert_array_equal(x[k], y[k])
    if n == 45000:
        want = r.final_m.clone()
        np.testing.assert_array_equal(b.subset(np.arange(n)).run_sliced(37).final_m.cpu().numpy()[:, :nl],
                                      want.cpu().numpy()[:, :nl])
