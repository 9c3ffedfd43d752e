"""The Ozaki stack kernel where its wavefronts' tiles (32 x 16), its DMA (16 rows) and its two entry buffers end: bit
for bit equal to the oracle, as the digits, level sums and the order of the entries define the result.
"""
import numpy as np
import pytest

import libxstream_amd as lx
import oracle
from libxstream_amd.workload import make_stack_workload
from tests.test_gpu_ozaki_stack import _run

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16, 64), (17, 15, 1), (32, 33, 63), (33, 48, 16), (49, 1, 17), (1, 64, 5), (64, 49, 64)]
RUNS = [1, 2, 1, 3, 64, 65, 1, 20]  # one and two entries (no entry to load ahead), past a ballot of 64


@pytest.fixture(scope="module")
def stream():
    lx.init()
    s = lx.Stream("edges")
    yield s
    s.close()
    lx.finalize()


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("s", range(1, 9))
def test_stack_edges(stream, s, dtype):
    f64 = dtype == np.float64
    for i, (m, n, k) in enumerate(SHAPES):
        trim = (0, s - 1, s // 2)[(i + s) % 3]  # all pairs, the triangle, a cutoff taken at run time
        w = make_stack_workload(m, n, k, sum(RUNS), nc=len(RUNS), dtype=dtype, seed=10 * s + i, c_init="random")
        stack = w.stack.copy()
        stack[:, 2] = np.repeat(np.arange(len(RUNS), dtype=np.int32), RUNS) * (m * n) + 1
        out, bl = _run(stream, w, s, trim, use_double=f64, stack=stack)
        ref = oracle.ozaki_stack(m, n, k, stack, w.a, bl, w.c, s, trim=trim, dtype=dtype)
        assert np.array_equal(out, ref), (m, n, k, trim)
