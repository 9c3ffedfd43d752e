"""Scheme I with all levels of an output tile in registers (ozaki_pairs.h): every slice count over the triangle and over
all pairs, tile edges, work-groups that share a tile's k, planes without a nonzero digit, and a K whose level sums
would not fit int32 (the level GEMM's partials again). Bar: bit for bit the oracle."""
import numpy as np
import pytest

import libxstream_amd as lx
import oracle

pytestmark = pytest.mark.gpu


def _gemm(m, n, k, s, trim, values, dtype=np.float64, beta=0.5):
    rng = np.random.default_rng(m + 5 * n + 11 * k + s)
    a, b = values(rng, (k, m)).astype(dtype), values(rng, (n, k)).astype(dtype)  # column-major op N
    c = rng.uniform(-1, 1, (n, m)).astype(dtype)
    lx.init()
    stream = lx.Stream("pairs")
    oz = lx.Ozaki(use_double=dtype == np.float64, nslices=s, trim=trim)
    try:
        da, db, dc = (lx.DeviceBuffer.from_array(x) for x in (a, b, c))
        oz.gemm("N", "N", m, n, k, 1.5, da, m, db, k, beta, dc, m, stream=stream)
        stream.sync()
        out = np.empty_like(c)
        dc.download(out)
        for buf in (da, db, dc):
            buf.free()
    finally:
        oz.close()
        stream.close()
        lx.finalize()
    ref = oracle.ozaki_gemm("N", "N", m, n, k, 1.5, a.ravel(), m, b.ravel(), k, beta, c.ravel(), m, s, trim=trim)
    return out.ravel(), ref


def _scaled(rng, shape):
    return rng.uniform(-1, 1, shape) * np.exp2(rng.integers(-20, 21, shape))


@pytest.mark.parametrize("s", range(1, 9))
@pytest.mark.parametrize("full", [False, True], ids=["triangle", "all"])
def test_slices(s, full):
    out, ref = _gemm(129, 66, 190, s, 0 if full else s - 1, _scaled)
    assert np.array_equal(out, ref)


@pytest.mark.parametrize("shape", [(1, 1, 128), (64, 64, 129), (65, 1, 1024), (128, 63, 1100), (30, 300, 2050)],
                         ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
def test_edges_and_shared_k(shape, dtype):
    out, ref = _gemm(*shape, 8 if dtype == np.float64 else 4, 0, _scaled, dtype=dtype)
    assert np.array_equal(out, ref)


def test_empty_planes():
    out, ref = _gemm(70, 80, 300, 8, 0, lambda rng, shape: rng.integers(-3, 4, shape).astype(float))
    assert np.array_equal(out, ref)


def test_long_k():
    out, ref = _gemm(20, 30, 16700, 8, 0, _scaled)
    assert np.array_equal(out, ref)
