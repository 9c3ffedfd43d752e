"""The batch's default schedule (launches per stack in order or in lanes, or the persistent kernel, chosen by the work)
and an explicit persistent schedule: every stack against the oracle, eager and over three graph replays with eager work
in between; stacks that share one C pool."""
import numpy as np
import pytest

import libxstream_amd as lx
import oracle
from libxstream_amd.workload import make_mixed_batch
from tests.test_gpu_batch import Resident, check_all

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def stream():
    lx.init()
    s = lx.Stream("schedule")
    yield s
    s.close()
    lx.finalize()


# the persistent kernel, in order, lanes under replay; one stack; persistent by request
@pytest.mark.parametrize("count,lengths,params", [(60, (1, 20), None), (6, (20, 400), None), (40, (1500, 3000), None),
                                                  (1, (700, 700), None), (12, (1, 2000), (0, 4, 0)),
                                                  (12, (1, 2000), (20000, 0, 0))])
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
def test_batch_schedules(stream, count, lengths, params, dtype):
    works = make_mixed_batch(count, seed=count, dtype=dtype, len_range=lengths, c_init="uniform")
    res = Resident(works, stream)
    try:
        batch = lx.Batch(lx.typeid(dtype), res.items, None if params is None else lx.BatchParams(*params))
        c_ref = [w.c.ravel().copy() for w in works]
        for step in range(4):
            if 0 == step:
                batch.process(stream)
            else:
                batch.replay(stream)
            stream.sync()
            expected = [oracle.stack_dd(w.m, w.n, w.k, w.stack, w.a, w.b, c_in=c) for w, c in zip(works, c_ref)]
            check_all(res, expected)
            c_ref = [res.download(i).ravel().copy() for i in range(count)]
        batch.close()
    finally:
        res.free()


def test_batch_shared_c(stream):
    """24 launches that update the same C blocks: in lanes they overlap"""
    from libxstream_amd.workload import make_stack_workload

    w = make_stack_workload(23, 23, 23, 9000, nc=300, dtype=np.float64, seed=3, c_init="uniform")
    res = Resident([w], stream)
    try:
        batch = lx.Batch(lx.REAL_8, res.items * 24)
        batch.replay(stream)
        stream.sync()
        stack = np.concatenate([w.stack] * 24)
        expected = [oracle.stack_dd(w.m, w.n, w.k, stack, w.a, w.b, c_in=w.c.ravel())]
        check_all(res, expected)
        batch.close()
    finally:
        res.free()
