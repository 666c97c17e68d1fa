"""Which stream set an execute of several small groups takes: a caller's stream
keeps its own while its work is pending; another caller's stream takes one
that is free, and with every set in use its groups follow one another on it;
the per-thread stream, one handle for every thread's own stream, is a stream
of each thread's own.  The results are the same on every route."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from cmtj_amd import SolverMode, _lib, constantDriver, workloads
from cmtj_amd.batch import BatchResult, JunctionBatch
from test_gpu_graph import _snapshot
from test_gpu_side_streams import _fill, _same

pytestmark = pytest.mark.gpu

PER_THREAD = 2  # hipStreamPerThread
SETS = 4


def _batch(n_steps):
    """Four groups of one to four layers, some 0.3 us per step each."""
    js = []
    for nl in range(1, 5):
        j = workloads.chain_junction(nl) if nl > 1 else workloads.vsd_junction()
        j.setLayerTemperatureDriver("all", constantDriver(300.0))
        js.append(j)
    b = JunctionBatch.from_junctions(js, (n_steps + 0.5) * 1e-13, 1e-13, 1e-11, SolverMode.EulerHeun,
                                     precision="fp64", log="m")
    b.set_seeds(np.arange(4, dtype=np.uint64))
    b.js["stream"] = 0  # (packing gives every batch streams of its own)
    assert b.plan().info.n_kernels == 4
    _fill(b)
    return b


def _results(bs):
    return [_snapshot(BatchResult(b, *b._bufs), b) for b in bs]


def test_more_callers_than_sets():
    import torch

    bs = [_batch(100000) for _ in range(SETS + 2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in bs]
    assert len({s.cuda_stream for s in streams}) == len(streams)
    sets = []
    for b, s in zip(bs, streams):
        b.execute(stream=s)
        sets.append(_lib.last_side_set())
    # a stream whose own set is in use goes on with it
    bs[0].execute(stream=streams[0])
    again = _lib.last_side_set()
    bs[-1].execute(stream=streams[-1])
    last = _lib.last_side_set()
    pending = not streams[0].query()
    torch.cuda.synchronize()
    print(f"[stream sets] {sets}, again {again}, beyond {last}", flush=True)
    assert pending  # (else the sets were free again)
    assert sorted(sets[:SETS]) == list(range(SETS)) and sets[SETS:] == [-1] * 2
    assert again == sets[0] and last == -1
    want, *rest = _results(bs)
    for got in rest:
        _same(want, got)


def test_per_thread_streams_are_streams_of_their_own():
    import torch

    bs = [_batch(300000) for _ in range(2)]
    torch.cuda.synchronize()
    sets, errors = [(), ()], []
    first, second = threading.Event(), threading.Event()

    def work(q):
        try:
            if q == 1:
                first.wait(60)
            for _ in range(2):  # (the second: the thread's own set again)
                bs[q].execute(stream=PER_THREAD)
                sets[q] += (_lib.last_side_set(),)
        except Exception as e:  # noqa: BLE001
            errors.append(e)
        finally:
            (first, second)[q].set()
        second.wait(60)
        torch.cuda.ExternalStream(PER_THREAD).synchronize()  # (the stream ends with its thread)

    ts = [threading.Thread(target=work, args=(q,)) for q in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    print(f"[stream sets] per thread {sets}", flush=True)
    assert not errors
    assert sets[0][0] == sets[0][1] >= 0 and sets[1][0] == sets[1][1] >= 0
    assert sets[0][0] != sets[1][0]
    want, got = _results(bs)
    _same(want, got)


def test_one_group_stays_on_the_callers_stream():
    b = workloads.pimm(n_points=16, t_min=1e-10, t_max=2e-10, precision="fp64")
    b.execute()
    assert _lib.last_side_set() == -1
