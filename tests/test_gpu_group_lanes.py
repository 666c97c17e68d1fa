"""Point-dipole groups on one lane per component (k_junction_cl's group form)
against the oracle's group runner, at the edges of its workgroups: one
element, partial and full octets and waves, one- and two-layer elements,
constant and time-dependent drives, positions off the plane, and a NaN in the
last wave, which ends the group's run in every wave at the same step.

Tolerance: a step rounds a handful of times at 1e-16 relative and 500 damped
steps add at most their sum, so 1e-10 leaves three orders of magnitude."""
from __future__ import annotations

import numpy as np
import pytest

from cmtj_amd import AxialDriver, CVector, Junction, constantDriver, sineDriver, stepDriver
from cmtj_amd import _lib, reservoir
from cmtj_amd.reservoir import GroupInteraction, run_groups
from oracle_backend import OracleGroupInteraction
from test_group_cpu import _elements

pytestmark = pytest.mark.gpu


def _positions(n, k=0):
    rng = np.random.default_rng(100 * n + k)
    side = int(np.ceil(np.sqrt(n)))
    return [CVector(*(np.array([q % side, q // side, 0.0]) * 70e-9 + rng.uniform(-9e-9, 9e-9, 3)).tolist())
            for q in range(n)]


def _build(G, n, two, driven, k=0, bad=-1):
    js = _elements(Junction, n, two)
    for q, j in enumerate(js):
        if driven:
            j.setLayerExternalFieldDriver("all", AxialDriver(sineDriver(0, 2e3 + 10 * q, 3e9, 0.1 * q),
                                                             constantDriver(1e3), constantDriver(5e3)))
        if bad >= 0:
            amp = float("inf") if q == bad else 1e3
            j.setLayerExternalFieldDriver("all", AxialDriver(stepDriver(0, amp, 2.2e-11, 1e-9), constantDriver(0),
                                                             constantDriver(5e3)))
    g = G(_positions(n, k), js)
    g.setInteractionFunction(reservoir.computeDipoleInteractionNoumra if k % 2 else reservoir.computeDipoleInteraction)
    return g


def _worst(a, b, n):
    w = 0.0
    for q in range(n):
        la, lb = a.getLog(q), b.getLog(q)
        assert la.keys() == lb.keys()
        for key in la:
            x, y = np.asarray(la[key]), np.asarray(lb[key])
            assert x.shape == y.shape, key
            if y.size:
                w = max(w, float(np.max(np.abs(x - y))) / max(1.0, float(np.max(np.abs(y)))))
    return w


@pytest.mark.parametrize("driven", [False, True])
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 16, 17, 32, 33, 63, 64])
def test_group_sizes(n, two, driven):
    g = [_build(GroupInteraction, n, two, driven, k) for k in range(2)]
    o = [_build(OracleGroupInteraction, n, two, driven, k) for k in range(2)]
    run_groups(g, 0.05e-9, 1e-13, 7e-13)
    (name,) = _lib.last_kernels()
    assert name.startswith("k_junction_cl<double," + ("2," if two else "1,")) and "group of" in name
    worst = 0.0
    for a, b in zip(g, o):
        b.runSimulation(0.05e-9, 1e-13, 7e-13)
        worst = max(worst, _worst(a, b, n))
    print(f"[group lanes] n={n} two={two} driven={driven}: {worst:.3e}", flush=True)
    assert worst <= 1e-10


@pytest.mark.parametrize("n,two", [(12, False), (40, False), (20, True), (60, True)])
def test_nan_ends_the_group_in_every_wave(n, two):
    """The bad element sits in the last wave; 220 steps in, in the middle of a
    block of steps."""
    g = [_build(GroupInteraction, n, two, False, k, bad=n - 1 if k == 1 else n) for k in range(3)]
    o = [_build(OracleGroupInteraction, n, two, False, k, bad=n - 1 if k == 1 else n) for k in range(3)]
    with pytest.raises(RuntimeError, match="NAN magnetisation"):
        run_groups(g, 0.05e-9, 1e-13, 1e-13)
    for k, b in enumerate(o):
        if k == 1:
            with pytest.raises(RuntimeError, match="NAN magnetisation"):
                b.runSimulation(0.05e-9, 1e-13, 1e-13)
        else:
            b.runSimulation(0.05e-9, 1e-13, 1e-13)
        assert _worst(g[k], b, n) <= 1e-10
    assert 0 < len(g[1].getLog(0)["time"]) < len(g[0].getLog(0)["time"])
