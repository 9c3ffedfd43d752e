"""Native FP64 GEMM (ozaki_dgemm_native): tiles of 128 and 64, k split over four groups of wavefronts, and every edge:
one row or column, odd extents, a last stage that is not full, padded leading dimensions, all four transposes.
Reference: extended precision; bound: the rounding of K products and sums, (K + 4) 2^-53 (|alpha| |A| |B| + |beta C|)."""
import numpy as np
import pytest

import libxstream_amd as lx

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (1, 70, 33), (70, 1, 16), (2, 2, 17), (63, 65, 15), (64, 64, 64), (129, 127, 50), (640, 650, 19),
         (2560, 2500, 18)]  # the last two: 64 x 64 tiles with one group, 128 x 128 tiles


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("ta,tb", ["NN", "NT", "TN", "TT"])
def test_dgemm_edges(size, ta, tb):
    m, n, k = size
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    pad = 3
    a = rng.uniform(-1, 1, ((k, m + pad) if "N" == ta else (m, k + pad)))  # (columns, leading dimension)
    b = rng.uniform(-1, 1, ((n, k + pad) if "N" == tb else (k, n + pad)))
    c = rng.uniform(-1, 1, (n, m + pad))
    alpha, beta = 1.5, -0.5
    opa = (a[:, :m].T if "N" == ta else a[:, :k])  # m x k
    opb = (b[:, :k].T if "N" == tb else b[:, :n])  # k x n
    rows = np.unique(np.r_[0:min(m, 40), max(0, m - 40):m, rng.integers(0, m, 20)])
    ext = opa[rows].astype(np.longdouble) @ opb.astype(np.longdouble)
    ref = alpha * ext + beta * c[:, rows].T.astype(np.longdouble)
    bound = (k + 4) * 2.0**-53 * (abs(alpha) * (np.abs(opa[rows]) @ np.abs(opb)) + abs(beta) * np.abs(c[:, rows].T))
    lx.init()
    stream = lx.Stream("dgemm")
    try:
        da, db, dc = (lx.DeviceBuffer.from_array(x) for x in (a, b, c))
        lx.dgemm_native(ta, tb, m, n, k, alpha, da, a.shape[1], db, b.shape[1], beta, dc, c.shape[1], stream=stream)
        stream.sync()
        out = np.empty_like(c)
        dc.download(out)
        for buf in (da, db, dc):
            buf.free()
    finally:
        stream.close()
        lx.finalize()
    assert np.array_equal(out[:, m:], c[:, m:])  # the rows past m of the leading dimension stay
    assert np.all(np.abs(out[:, rows].T - ref) <= bound)
