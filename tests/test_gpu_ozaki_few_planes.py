"""Scheme I on operands that need few of the slices (whole numbers, short mantissas), in products large enough that a
call leaves its pairs either to the kernel of all planes or to the level GEMM by the planes that hold digits: the same
bits as the columns computed by small calls, which are compared with the oracle elsewhere; and the time, which has to
follow the digits and not the slices."""
import ctypes
import time

import numpy as np
import pytest
import torch

import libxstream_amd as lx

pytestmark = pytest.mark.gpu


class Memory:
    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


@pytest.fixture(scope="module")
def stream():
    torch.cuda.init()
    lx.init()
    s = lx.Stream("few")
    yield s
    s.close()
    lx.finalize()


def _values(gen, shape, bits, dtype):
    if bits is None:
        return torch.rand(shape, generator=gen, dtype=dtype, device="cuda").sub_(0.5)
    return torch.randint(1 - (1 << bits), 1 << bits, shape, generator=gen, device="cuda").to(dtype)


# one plane per 7 bits; A and B alike, A with fewer, the last: 23 of 36 pairs, around the line
@pytest.mark.parametrize("bits", [(7, 7), (28, 28), (35, 28), (7, 49), (49, 49), (None, None)], ids=str)
@pytest.mark.parametrize("s,trim,size", [(8, 7, (2050, 2100, 3700)), (8, 0, (2050, 2100, 2000)), (3, 0, (4000, 4100, 4096))],
                         ids=["8 triangle", "8 all", "3 all"])
def test_large_products(stream, bits, s, trim, size):
    m, n, k = size
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m + s)
    a, b = _values(gen, (k, m), bits[0], torch.float64), _values(gen, (n, k), bits[1], torch.float64)  # column-major
    c = _values(gen, (n, m), None, torch.float64)
    oz = lx.Ozaki(use_double=True, nslices=s, trim=trim)
    try:
        full, parts = c.clone(), []
        torch.cuda.synchronize()
        oz.gemm("N", "N", m, n, k, 1.5, Memory(a), m, Memory(b), k, 0.5, Memory(full), m, stream=stream)
        for j, w in ((0, 70), (n - 66, 66)):
            part = c[j:j + w].clone()
            torch.cuda.synchronize()
            oz.gemm("N", "N", m, w, k, 1.5, Memory(a), m, Memory(b[j:j + w]), k, 0.5, Memory(part), m, stream=stream)
            parts.append((j, w, part))
        stream.sync()
        for j, w, part in parts:
            assert torch.equal(full[j:j + w], part), j
    finally:
        oz.close()


def test_time_follows_the_digits(stream):
    """4096^3 with 8 slices: whole numbers of one plane against values that fill all eight"""
    n = 4096
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1)
    oz = lx.Ozaki(use_double=True, nslices=8, trim=7)
    taken = []
    try:
        for bits in (7, None):
            a, b = (Memory(_values(gen, (n, n), bits, torch.float64)) for _ in range(2))
            c = Memory(torch.zeros((n, n), dtype=torch.float64, device="cuda"))
            torch.cuda.synchronize()
            best = np.inf
            for _ in range(4):
                t = time.perf_counter()
                for _ in range(4):
                    oz.gemm("N", "N", n, n, n, 1.0, a, n, b, n, 0.0, c, n, stream=stream)
                stream.sync()
                best = min(best, time.perf_counter() - t)
            taken.append(best)
    finally:
        oz.close()
    assert taken[0] < 0.5 * taken[1], taken
