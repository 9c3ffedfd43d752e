"""Native FP64 GEMM (ozaki_dgemm_native) over several stages of k and past its 32-bit offsets: the one-group kernels' steady
state (64 x 64 and 128 x 128 tiles) with odd extents and a last stage that is not full, and leading dimensions at and
above 2^21 elements, from which on operands go through the LDS element by element; all four transposes.
Reference: extended precision; bound: the rounding of K products and sums, (K + 4) 2^-53 (|alpha| |A| |B| + |beta C|)."""
import numpy as np
import pytest

import libxstream_amd as lx

pytestmark = pytest.mark.gpu

LD = 1 << 21  # the largest leading dimension of the 32-bit byte offsets
TRANS = ["NN", "NT", "TN", "TT"]


def run(m, n, k, ta, tb, lda, ldb):
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a = np.zeros((k if "N" == ta else m, lda))  # (columns, leading dimension)
    b = np.zeros((n if "N" == tb else k, ldb))
    va, vb = a[:, :m if "N" == ta else k], b[:, :k if "N" == tb else n]
    va[:] = rng.uniform(-1, 1, va.shape)
    vb[:] = rng.uniform(-1, 1, vb.shape)
    ldc, alpha, beta = m + 3, 1.5, -0.5
    c = rng.uniform(-1, 1, (n, ldc))
    opa, opb = (va.T if "N" == ta else va), (vb.T if "N" == tb else vb)
    rows = np.unique(np.r_[0:min(m, 40), max(0, m - 40):m, rng.integers(0, m, 20)])
    ref = alpha * (opa[rows].astype(np.longdouble) @ opb.astype(np.longdouble)) + beta * c[:, rows].T.astype(np.longdouble)
    bound = (k + 4) * 2.0**-53 * (abs(alpha) * (np.abs(opa[rows]) @ np.abs(opb)) + abs(beta) * np.abs(c[:, rows].T))
    lx.init()
    stream = lx.Stream("dgemm")
    try:
        da, db, dc = (lx.DeviceBuffer.from_array(x) for x in (a, b, c))
        lx.dgemm_native(ta, tb, m, n, k, alpha, da, lda, db, ldb, beta, dc, ldc, stream=stream)
        stream.sync()
        out = np.empty_like(c)
        dc.download(out)
        for buf in (da, db, dc):
            buf.free()
    finally:
        stream.close()
        lx.finalize()
    assert np.array_equal(out[:, m:], c[:, m:])
    assert np.all(np.abs(out[:, rows].T - ref) <= bound)


# one group: 64 x 64 tiles, 128 x 128 tiles; 1 to 6 full stages of 16 with 0, 1, 3 and 15 more
@pytest.mark.parametrize("size", [(641, 651, 83), (650, 640, 48), (639, 705, 33), (2561, 2499, 83), (2560, 2435, 111)],
                         ids=lambda s: "%dx%dx%d" % s)
@pytest.mark.parametrize("ta,tb", TRANS)
def test_stages(size, ta, tb):
    m, n, k = size
    run(m, n, k, ta, tb, (m if "N" == ta else k) + 3, (k if "N" == tb else n) + 5)


# both operands, A alone and B alone past the limit; at the limit
@pytest.mark.parametrize("extra", [(8, 8), (9, None), (None, 9), (0, 0)],
                         ids=["both", "a", "b", "at"])
@pytest.mark.parametrize("ta,tb", TRANS)
def test_leading_dimension(ta, tb, extra):
    m, n, k = 66, 35, 37
    own = ((m if "N" == ta else k) + 1, (k if "N" == tb else n) + 1)
    run(m, n, k, ta, tb, *(own[x] if extra[x] is None else LD + extra[x] for x in (0, 1)))
