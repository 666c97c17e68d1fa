"""Groups of one execute side by side (launch_spread): a batch of several
small groups equals each group run alone, bit for bit, in stream order with
the work around it, on several streams and threads at once, with more
executes in flight than there are stream sets, and under capture."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from cmtj_amd.batch import JunctionBatch
from test_gpu_graph import _mixed, _snapshot

pytestmark = pytest.mark.gpu


def _fill(b):
    log, mag, st = b._buffers("cuda")
    log.fill_(float("nan"))
    mag.fill_(float("nan"))
    st.fill_(0xFF)


def _same(want, got):
    for lw, lg in zip(want[0], got[0]):
        assert lw.keys() == lg.keys()
        for k in lw:
            np.testing.assert_array_equal(lw[k], lg[k])
    for mw, mg in zip(want[1], got[1]):
        np.testing.assert_array_equal(mw, mg)
    assert want[2].tobytes() == got[2].tobytes()


def _alone(b):
    """Every instance in a batch of its own: one group, one launch."""
    logs, mags, sts = [], [], []
    for i in range(len(b.js)):
        q = b.subset(np.array([i]))
        l, m, s = _snapshot(q.run(), q)
        logs += l
        mags += m
        sts.append(s)
    return logs, mags, np.concatenate(sts)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_groups_side_by_side_equal_groups_alone(precision):
    import torch

    b = _mixed(precision)
    assert b.plan().info.n_kernels >= 4 and int(b.js["n_steps"].sum()) >= 4000
    want = _alone(b)
    s = torch.cuda.Stream()
    for st in (torch.cuda.current_stream(), s):
        with torch.cuda.stream(st):
            _fill(b)
            r = b.execute()
            # ordered after the execute on its stream, with no synchronisation
            log, mag, status = (t.clone() for t in b._bufs)
            _fill(b)
        torch.cuda.synchronize()
        for t, c in zip(b._bufs, (log, mag, status)):
            t.copy_(c)
        _same(want, _snapshot(r, b))
    # a captured execute keeps its launches on the capturing stream
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        r = b.execute()
    for _ in range(3):
        _fill(b)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        _same(want, _snapshot(r, b))


def test_threads_and_many_executes_in_flight():
    import torch

    bs = [_mixed("fp32") for _ in range(6)]
    want = _alone(bs[0])
    for b in bs:
        b.plan()
        _fill(b)
    torch.cuda.synchronize()
    errors = []

    def work(mine):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for _ in range(4):
                    for b in mine:
                        b.execute()
            s.synchronize()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    ts = [threading.Thread(target=work, args=(bs[q::3],)) for q in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors
    from cmtj_amd.batch import BatchResult
    for b in bs:
        _same(want, _snapshot(BatchResult(b, *b._bufs), b))
