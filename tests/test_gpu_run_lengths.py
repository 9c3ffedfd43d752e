"""Stacks of other run lengths than 30: the configuration that libsmm_acc_process chooses against the built-in heuristic's,
which takes every shape the same way whatever the stack, and results where a piece spans several work-groups."""
import time

import numpy as np
import pytest

import libxstream_amd as lx
import oracle
from libxstream_amd.workload import make_stack_workload
from tests.helpers import run_stack, tol

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def stream():
    lx.init()
    s = lx.Stream("runs")
    yield s
    s.close()
    lx.finalize()


def _stack(w, lengths):
    stack = w.stack.copy()
    stack[:, 2] = np.repeat(np.arange(len(lengths), dtype=np.int64), lengths)[:len(stack)] * (w.m * w.n) + 1
    return stack


def _time(call, stream):
    call()
    stream.sync()
    best = np.inf
    for _ in range(5):
        t = time.perf_counter()
        for _ in range(20):
            call()
        stream.sync()
        best = min(best, (time.perf_counter() - t) / 20)
    return best


# single entries in small blocks, and runs of 100 in blocks that keep a CU busy
@pytest.mark.parametrize("dtype,shape,entries,run", [(np.float32, (5, 5, 5), 10000, 1), (np.float32, (5, 5, 5), 15000, 2),
                                                    (np.float32, (8, 8, 8), 4000, 1), (np.float64, (23, 23, 23), 7000, 100),
                                                    (np.float64, (45, 45, 13), 7000, 100)],
                         ids=lambda v: getattr(v, "__name__", str(v)))
def test_time_over_run_lengths(stream, dtype, shape, entries, run):
    m, n, k = shape
    tid = lx.typeid(dtype)
    nc = entries // run
    w = make_stack_workload(m, n, k, entries, nc=nc, na=500, nb=500, dtype=dtype, seed=run)
    bufs = [lx.DeviceBuffer.from_array(x) for x in (_stack(w, [run] * nc), w.a, w.b_device_layout(), w.c)]
    heuristic = lx.default_config(tid, m, n, k)
    try:
        own = _time(lambda: lx.process(bufs[0], entries, tid, *bufs[1:], m, n, k, stream), stream)
        ref = _time(lambda: lx.process_config(heuristic, bufs[0], entries, tid, *bufs[1:], m, n, k, stream), stream)
    finally:
        for b in bufs:
            b.free()
    assert own <= 1.5 * ref, (own, ref)


# below and at the lines between pieces of 2 to 32 entries, and more than 256 work-groups, which then take segments that
# lie apart; runs that end at, before and after the multiples of a piece
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", [(23, 23, 23), (17, 33, 5), (40, 40, 70), (13, 13, 13), (6, 7, 9), (5, 5, 5)],
                         ids=lambda s: "%dx%dx%d" % s)
def test_pieces(stream, shape, dtype):
    m, n, k = shape
    for entries in (60, 511, 1300, 2600, 4099):
        lengths = [1, 7, 8, 9, 16, 17, 31, 32, 33, 40, 41, 64, 65, 130]
        lengths = (lengths * (entries // sum(lengths) + 1))
        nc = int(np.searchsorted(np.cumsum(lengths), entries)) + 1
        w = make_stack_workload(m, n, k, entries, nc=nc, na=64, nb=64, dtype=dtype, seed=entries, c_init="uniform")
        stack = _stack(w, lengths[:nc])
        out = run_stack(stream, w, device_transpose=False, stack=stack)
        ref = oracle.stack_dd(m, n, k, stack, w.a, w.b, c_in=w.c.ravel())
        assert oracle.error(out.ravel(), *ref)[0] <= tol(dtype), entries
