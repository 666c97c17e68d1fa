"""Devices of anisotropy, bilinear coupling and constant or sine fields take the
lean binary64 sets on component lanes, not the one with every field term: one
to four layers, axes along a component and tilted ones, records beyond the two
kept in registers, against the oracle; and the same bits in slices.
Tolerance: the drop-in's bar, 1e-8 (500 steps round at 1e-16 each)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from cmtj_amd import AxialDriver, CVector, Junction, Layer, SolverMode, _lib, constantDriver, sineDriver, stepDriver
from cmtj_amd.batch import JunctionBatch

pytestmark = pytest.mark.gpu

FIELDS = {"const": lambda q: (constantDriver(1e5 + 1e4 * q), constantDriver(0), constantDriver(2e4)),
          "sine": lambda q: (constantDriver(1e5), sineDriver(0, 5e3, 5e9 + 1e8 * q, 0), constantDriver(0)),
          "sines": lambda q: (sineDriver(1e5, 5e3, 5e9 + 1e8 * q, 0.3), sineDriver(0, 4e3, 3e9, 0.1 * q),
                              sineDriver(2e3, 3e3, 2e9, 1.0)),
          "sine_step": lambda q: (sineDriver(1e5, 5e3, 5e9, 0.1 * q), stepDriver(0, 2e3, 3e-12, 9e-12),
                                  constantDriver(1e4))}


def _junction(nl, fields, q):
    axis = CVector(0.6, 0, 0.8) if q % 2 else CVector(0, 0, 1)
    ls = [Layer(f"l{l}", mag=CVector(0.1 + 0.3 * l, 0.2, 1 - 0.2 * l), anis=axis, Ms=1.2 - 0.1 * l, thickness=1.5e-9,
                cellSurface=1e-16, demagTensor=[CVector(0.02, 0, 0), CVector(0, 0.03, 0), CVector(0, 0, 0.95)],
                damping=0.03) for l in range(nl)]
    j = Junction(ls)
    j.setLayerAnisotropyDriver("all", constantDriver(4e5))
    for l in range(nl - 1):
        j.setIECDriver(f"l{l}", f"l{l + 1}", constantDriver(-1e-4))
    j.setLayerExternalFieldDriver("all", AxialDriver(*FIELDS[fields](q)))
    return j


@pytest.mark.parametrize("tilted", [False, True])
@pytest.mark.parametrize("fields", list(FIELDS))
@pytest.mark.parametrize("nl", [1, 2, 3, 4])
def test_lean_devices(nl, fields, tilted):
    steps = np.array([1, 63, 64, 130, 500])
    js = [_junction(nl, fields, 2 * q + int(tilted and q % 2 == 0)) for q in range(len(steps))]
    b = JunctionBatch.from_junctions(js, (steps + 0.5) * 1e-13, 1e-13, 3.0003e-13, SolverMode.RK4, precision="fp64",
                                     log="m", log_dtype="f64")
    kname = b.plan().info.kernel_name.decode()
    assert kname.startswith("k_junction_cl<double") and b.plan().info.n_kernels == 1, kname
    assert "FM_FIELD" not in kname and "FM_STTC" not in kname, kname
    r = b.run()
    olog, omag, ost = oracle.run_batch(b.js, b.layers, _lib.constants_get(), b.tables, b.log_elements)
    g, gm = r.log.cpu().numpy(), r.final_m.cpu().numpy()
    worst = max(float(np.max(np.abs(g - olog))), float(np.max(np.abs(gm[:, :nl] - omag[:, :nl]))))
    print(f"[lean sets] {kname} {fields} tilted={tilted}: {worst:.2e}", flush=True)
    assert worst <= 1e-8
    s = b.subset(np.arange(len(js)), log_dtype="f64").run_sliced(77)
    np.testing.assert_array_equal(s.log.cpu().numpy(), g)
    np.testing.assert_array_equal(s.final_m.cpu().numpy(), gm)
