"""Kernel choice by shape and stack size for untuned shapes, and the pieces that short stacks are cut into (smm.c):
libsmm_acc_process against the oracle on both sides of every line, and the kernels of one and two wavefronts per run.
"""
import numpy as np
import pytest

import libxstream_amd as lx
import oracle
from libxstream_amd.workload import make_stack_workload
from tests.helpers import run_stack, tol

# 4 | 5 blocks of 4x4, 11 | 12 blocks, k of 1, 2 and 4 wavefronts, one | two tiles, 8 | 9 tiles and 16 | 20
SHAPES = [(8, 8, 6), (8, 9, 7), (4, 16, 18), (4, 16, 19), (12, 12, 40), (16, 11, 3), (16, 17, 5), (32, 64, 9), (48, 48, 8),
          (64, 65, 4), (5, 5, 5), (23, 23, 23)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%dx%d" % s)
def test_process_by_stack_size(shape, dtype):
    m, n, k = shape
    lx.init()
    stream = lx.Stream("rule")
    try:
        for entries in (1, 999, 1001, 1999, 7999, 8001, 16383, 16384):
            w = make_stack_workload(m, n, k, entries, nc=max(1, entries // 30), dtype=dtype, seed=entries, c_init="uniform")
            ref = oracle.stack_dd(m, n, k, w.stack, w.a, w.b, c_in=w.c.ravel())
            out = run_stack(stream, w, device_transpose=False)
            assert oracle.error(out.ravel(), *ref)[0] <= tol(dtype), entries
    finally:
        stream.close()
        lx.finalize()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("nt", [64, 128, 256])
def test_small_blocks_few_wavefronts(nt, dtype):
    tid = lx.typeid(dtype)
    runs = [64, 1, 65, 2, 130, 3, 31]
    lx.init()
    stream = lx.Stream("small")
    try:
        for m, n, k in [(1, 1, 1), (5, 5, 5), (16, 16, 65), (13, 3, 16), (4, 9, 129), (7, 16, 513)]:
            w = make_stack_workload(m, n, k, sum(runs), nc=len(runs), dtype=dtype, seed=nt + k, c_init="uniform")
            stack = w.stack.copy()
            stack[:, 2] = np.repeat(np.arange(len(runs), dtype=np.int32), runs) * (m * n) + 1
            ref = oracle.stack_dd(m, n, k, stack, w.a, w.b, c_in=w.c.ravel())
            cands = [c for c in lx.kernel_candidates(tid, m, n, k) if c[0] == 4 and c[3:] == (nt, 64)]
            assert cands
            for variant, tm, tn, _, kt in cands:
                for bs, split in ((1, 1), (4, 2), (24, 64)):  # pieces, runs cut, runs whole
                    cfg = lx.SmmConfig(variant=variant, tm=tm, tn=tn, nt=nt, kt=kt, bs=bs, flush=2, split=split)
                    out = run_stack(stream, w, config=cfg, device_transpose=False, stack=stack)
                    assert oracle.error(out.ravel(), *ref)[0] <= tol(dtype), cfg
    finally:
        stream.close()
        lx.finalize()
