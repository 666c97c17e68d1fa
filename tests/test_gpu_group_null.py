"""Uncoupled groups in a launch with dipole-coupled ones: nothing is checked
about an uncoupled group's positions, so elements may share a point, and a
coordinate may be infinite or no number; its elements run as they do alone.
Sizes at the edges of octets and waves, one- and two-layer elements, against
the oracle.  Tolerance as in test_gpu_group_lanes.py: 500 damped steps of
roundings at 1e-16, 1e-10 leaves three orders of magnitude."""
from __future__ import annotations

import math

import numpy as np
import pytest

from cmtj_amd import CVector, Junction, _lib, reservoir
from cmtj_amd.reservoir import GroupInteraction, run_groups
from oracle_backend import OracleGroupInteraction
from test_gpu_group_lanes import _build, _worst

pytestmark = pytest.mark.gpu

PLACES = {"one_point": lambda n: [CVector(0, 0, 0)] * n,
          "infinite": lambda n: [CVector(math.inf if q % 2 else -math.inf, 0, 7e-8 * q) for q in range(n)],
          "no_number": lambda n: [CVector(math.nan, 7e-8 * q, 0) for q in range(n)]}


@pytest.mark.parametrize("place", list(PLACES))
@pytest.mark.parametrize("n,two", [(2, False), (9, False), (33, False), (2, True), (9, True), (64, True)])
def test_uncoupled_beside_coupled(n, two, place):
    def groups(G):
        gs = [_build(G, n, two, True, k) for k in range(4)]
        for g in gs[1:3]:  # between a Kanao and a Nomura group
            g.setInteractionFunction(reservoir.nullDipoleInteraction)
            g.coordinateMatrix = PLACES[place](n)
        return gs

    g, o = groups(GroupInteraction), groups(OracleGroupInteraction)
    run_groups(g, 0.05e-9, 1e-13, 7e-13)
    (name,) = _lib.last_kernels()
    assert "group of" in name  # one lane per component
    worst = 0.0
    for a, b in zip(g, o):
        b.runSimulation(0.05e-9, 1e-13, 7e-13)
        worst = max(worst, _worst(a, b, n))
        for q in range(n):
            m = np.array(a.junctionList[q].getLayerMagnetisation("free").tolist())
            w = np.array(b.junctionList[q].getLayerMagnetisation("free").tolist())
            assert np.isfinite(m).all()
            worst = max(worst, float(np.max(np.abs(m - w))))
    print(f"[null group] n={n} two={two} {place}: {worst:.3e}", flush=True)
    assert worst <= 1e-10
