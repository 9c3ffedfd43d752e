"""Scheme I over the triangle of few slices: which of the two ways of a large product is taken (the kernel of all planes,
or the level GEMM with int32 partials in scratch memory, which is faster where a long k meets few pairs per plane), and the
same bits either way."""
import ctypes

import pytest
import torch

import libxstream_amd as lx

pytestmark = pytest.mark.gpu


class Memory:
    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())
        self.nbytes = tensor.numel() * tensor.element_size()

    def __bool__(self):
        return True


@pytest.fixture(scope="module")
def stream():
    torch.cuda.init()
    lx.init()
    s = lx.Stream("slices")
    yield s
    s.close()
    lx.finalize()


# below and above the lines in k, and a product too small for the choice; all planes hold digits but the last two of 6 in
# FP32 (multiples of 2^-24, 4 planes), whose 15 of 21 pairs go to the level GEMM
@pytest.mark.parametrize("s,size,partials", [(3, (3000, 3100, 15500), True), (3, (6500, 6400, 2050), False),
                                            (3, (4000, 3900, 4100), False), (4, (4100, 4200, 8100), True),
                                            (4, (5000, 5100, 4000), False), (6, (3000, 3100, 9000), False)], ids=str)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
def test_way_and_bits(stream, s, size, partials, dtype):
    m, n, k = size
    partials = partials or (torch.float32 == dtype and 6 == s)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(s)
    a, b, c = (torch.rand(shape, generator=gen, dtype=dtype, device="cuda").sub_(0.5) for shape in ((k, m), (n, k), (n, m)))
    oz = lx.Ozaki(use_double=torch.float64 == dtype, nslices=s, trim=s - 1)
    try:
        scratch = torch.full((oz.scratch_size("N", "N", m, n, k, m, k, m),), 0x5A, dtype=torch.uint8, device="cuda")
        oz.scratch_set(Memory(scratch))
        full = c.clone()
        torch.cuda.synchronize()
        oz.gemm("N", "N", m, n, k, 1.5, Memory(a), m, Memory(b), k, 0.5, Memory(full), m, stream=stream)
        stream.sync()
        up = lambda x, t: (x + t - 1) // t * t
        begin = s * (up(m, 256) + up(n, 256)) * up(k, 128) + (1 << 20)  # past the planes, exponents and flags
        assert bool((scratch[begin:begin + (1 << 20)] != 0x5A).any()) == partials
        for j, w in ((0, 70), (n - 66, 66)):
            part = c[j:j + w].clone()
            torch.cuda.synchronize()
            oz.gemm("N", "N", m, w, k, 1.5, Memory(a), m, Memory(b[j:j + w]), k, 0.5, Memory(part), m, stream=stream)
            stream.sync()
            assert torch.equal(full[j:j + w], part), j
    finally:
        oz.scratch_set(None)
        oz.close()
