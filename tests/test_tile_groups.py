"""Grouped tiles of the entry-parallel kernels (lxs_mfma.h): up to 16 bytes of consecutive rows or columns per lane.

CPU: every row of a block is written by exactly one lane and tile, and every load stays inside the block. GPU: parity
at the edges of the groups, and for grids with more tiles than the block has rows or columns.
"""
import numpy as np
import pytest

import libxstream_amd as lx
import oracle
from libxstream_amd.workload import make_stack_workload
from tests.helpers import run_stack, tol


@pytest.mark.parametrize("size", [4, 8])
def test_every_row_once(size):
    v = 16 // size
    for ntiles in range(1, 6):
        for extent in range(min(ntiles, v), 16 * ntiles + 1):
            rows = []
            for t in range(ntiles):
                c, x = t // v, t % v
                g = min(v, ntiles - c * v)
                for lane in range(16):
                    base = 16 * v * c + g * lane
                    s = min(base, extent - g)
                    assert 0 <= s and s + g <= extent
                    if s + x >= base:
                        rows.append(s + x)
            assert sorted(rows) == list(range(extent)), (ntiles, extent)


SHAPES = [(1, 33, 5), (3, 40, 17), (33, 17, 9), (45, 48, 13), (48, 3, 16), (64, 2, 30), (49, 64, 3), (2, 2, 5), (17, 16, 4),
          (34, 63, 21), (65, 20, 8)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
def test_grouped_tiles_parity(dtype):
    tid = lx.typeid(dtype)
    lx.init()
    stream = lx.Stream("groups")
    try:
        for m, n, k in SHAPES:
            w = make_stack_workload(m, n, k, 500, nc=20, dtype=dtype, seed=m + n + k, c_init="uniform")
            ref = oracle.stack_dd(m, n, k, w.stack, w.a, w.b, c_in=w.c.ravel())
            ti, tj = (m + 15) // 16, (n + 15) // 16
            grids = {(a, b) for a in range(ti, 6) for b in range(tj, 6) if a * b <= 16}
            ran = 0
            for tm, tn in sorted(grids):
                for nt in (128, 256, 512):
                    cfg = lx.SmmConfig(variant=2, tm=tm, tn=tn, nt=nt, kt=16, bs=16, flush=2, split=4)
                    if not lx.config_valid(tid, m, n, k, cfg):
                        continue
                    out = run_stack(stream, w, config=cfg, device_transpose=False)
                    assert oracle.error(out.ravel(), *ref)[0] <= tol(dtype), cfg
                    ran += 1
            assert ran > 0
    finally:
        stream.close()
        lx.finalize()
