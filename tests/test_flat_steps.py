"""The flat k-steps of the entry-parallel stack kernels: the k of a run's entries as one sequence, split over the
wavefronts of a work-group in whole steps (smm_mfma.hip).

CPU: index arithmetic of every k: each (entry, k) is fed exactly once, by one wavefront and lane, and the quotient
by multiplication is exact. GPU: parity where a step, a stage, a table of 64 entries or the multiplier's range ends.
"""
import numpy as np
import pytest

import libxstream_amd as lx
import oracle
from libxstream_amd.workload import make_stack_workload
from tests.helpers import run_stack, tol

WE = 64  # entries of a table


@pytest.mark.parametrize("kw,ep", [(4, 2), (4, 4), (4, 8), (16, 4), (16, 8)])
def test_flat_index_covers_every_k_once(kw, ep):
    for k in list(range(1, 90)) + [127, 128, 129, 255, 300, 511, 512, 513, 700]:
        we = WE if k <= 512 else 1
        ksh = 20 if k <= 128 else 24
        kinv = ((1 << ksh) + k - 1) // k if k <= 512 else 0
        assert kinv < 1 << 24 and (we * k - 1) * kinv < 1 << 32  # 24-bit factors, 32-bit product
        f = np.arange(we * k, dtype=np.int64)
        assert np.array_equal((f * kinv) >> ksh, f // k), k
        for entries in sorted({1, 2, 3, 13, 30, 31, 33, we} & set(range(1, we + 1))):
            flen = entries * k
            steps = -(-flen // kw)
            seen = np.zeros(flen, dtype=np.int64)
            for q in range(ep):
                s0, s1 = steps * q // ep, steps * (q + 1) // ep
                if s0 < s1:
                    flast = min(kw * s1, flen) - 1
                    fed = np.arange(kw * s0, kw * s1)
                    np.add.at(seen, fed[fed <= flast], 1)
                    # only the last step of the range holds anything past it, and only that stage is masked
                    assert np.all(fed[:-kw] <= flast)
            assert np.all(seen == 1), (k, entries)


SHAPES = [(5, 5, 1), (23, 23, 3), (9, 20, 17), (16, 16, 64), (33, 18, 129), (13, 13, 512), (7, 12, 513)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%dx%d" % s)
def test_flat_steps_parity(shape, dtype):
    m, n, k = shape
    tid = lx.typeid(dtype)
    runs = [64, 1, 65, 2, 63, 130, 3, 31, 33]  # below, at and past the 64 entries of a table
    lx.init()
    stream = lx.Stream("flat")
    try:
        w = make_stack_workload(m, n, k, sum(runs), nc=len(runs), dtype=dtype, seed=sum(shape), c_init="uniform")
        stack = w.stack.copy()
        stack[:, 2] = np.repeat(np.arange(len(runs), dtype=np.int32), runs) * (m * n) + 1
        ref = oracle.stack_dd(m, n, k, stack, w.a, w.b, c_in=w.c.ravel())
        for variant, tm, tn, nt, kt in lx.kernel_candidates(tid, m, n, k):
            if variant not in (2, 3, 4):
                continue
            for bs, split in ((16, 4), (32, 64)):  # runs cut, and kept whole
                cfg = lx.SmmConfig(variant=variant, tm=tm, tn=tn, nt=nt, kt=kt, bs=bs, flush=2, split=split)
                out = run_stack(stream, w, config=cfg, device_transpose=False, stack=stack)
                assert oracle.error(out.ravel(), *ref)[0] <= tol(dtype), cfg
    finally:
        stream.close()
        lx.finalize()
