"""KCL stacks on component lanes: the sum over the members by lane moves
(half rows, rows, row pairs, halves of the wave) at every lane count a stack
can take, against the oracle: 2 to 16 one-layer and 2 to 8 two-layer members
(partly filled lane groups included), constant and time-dependent currents,
several stacks of a wave, series and parallel coupling.  Tolerance 1e-8, the
drop-in's bar."""
from __future__ import annotations

import pytest

from cmtj_amd import ScalarDriver, _lib
from cmtj_amd.stack import ParallelStack, SeriesStack, run_stacks
from oracle_backend import OracleParallelStack, OracleSeriesStack
from test_gpu_stack import _compare, _members
from test_stack_cpu import _single, _two

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sine", [False, True])
@pytest.mark.parametrize("series", [True, False])
@pytest.mark.parametrize("member,n", [(_single, n) for n in (2, 3, 4, 5, 8, 9, 16)] + [(_two, n) for n in (2, 3, 4, 5, 8)])
def test_member_counts(member, n, series, sine):
    def build(k, cls):
        s = cls(_members(member, n), useKCL=True)
        s.setCouplingStrength([0.05 * (-1) ** q * (1 + k) / (1 + q) for q in range(n - 1)])
        s.setCoupledCurrentDriver(ScalarDriver.getSineDriver(8e11, 5e11, 3e9, 0.4) if sine
                                  else ScalarDriver.getConstantDriver(8e11 + 1e10 * k))
        return s

    g = [build(k, SeriesStack if series else ParallelStack) for k in range(5)]
    o = [build(k, OracleSeriesStack if series else OracleParallelStack) for k in range(5)]
    run_stacks(g, 0.02e-9, 1e-13, 3e-13)
    (name,) = _lib.last_kernels()
    assert name.startswith("k_junction_cl<double") and "stack" in name
    worst = 0.0
    for a, b in zip(g, o):
        b.runSimulation(0.02e-9, 1e-13, 3e-13)
        worst = max(worst, _compare(a, b))
    print(f"[stack sum] {member.__name__} n={n} series={series} sine={sine}: {worst:.2e}", flush=True)
    assert worst <= 1e-8
