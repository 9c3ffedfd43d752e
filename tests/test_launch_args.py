"""The launches that the host layer makes (CPU): tests/native/launches.c prints them instead of making them."""
import os
import shutil
import subprocess

import pytest

import libxstream_amd as lx

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "libxstream_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HOST = ["runtime", "dbcsr", "smm", "batch", "ozaki", "mlp"]
HIP = ["smm_stack_f64", "smm_stack_f32", "smm_mfma_f64", "smm_mfma_f32", "smm_batch", "lxs_launch", "ozaki_dev",
       "ozaki_stack_dev", "mlp_dev"]


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    """commands -> a list of (launches, configuration, result) per command"""
    if shutil.which("gcc") is None:
        pytest.skip("gcc not available")
    objects = [os.path.join(LIB, "_build", x + ".o") for x in HOST + HIP]
    if not all(os.path.exists(x) for x in objects):
        pytest.skip("libxstream_amd not built (its objects are linked in)")
    path = tmp_path_factory.mktemp("launches")
    exe = str(path / "launches")
    subprocess.run(["gcc", "-O1", "-std=gnu11", "-D__HIP_PLATFORM_AMD__", "-I" + ROCM + "/include",
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "native", "launches.c"), *objects,
                    "-o", exe, "-L" + ROCM + "/lib", "-Wl,-rpath," + ROCM + "/lib", "-lamdhip64", "-lstdc++", "-lpthread",
                    "-ldl", "-lm"], check=True)
    os.symlink(os.path.join(LIB, "params"), str(path / "params"))  # found next to the program, as next to the library

    def run(commands, **env):
        full = {k: v for k, v in os.environ.items() if not k.startswith(("OPENCL_LIBSMM", "LIBXSTREAM"))}
        out = subprocess.run([exe], input="\n".join(commands) + "\n", capture_output=True, text=True, timeout=120,
                             env={**full, **env})
        assert out.returncode == 0, out.stderr[-2000:]
        result, made, config = [], [], None
        for line in out.stdout.splitlines():
            word, *values = line.split()
            if word == "launch":
                made.append(dict(zip(("groups", "nt", "bs", "k", "kt", "tsplit", "atomic", "a", "b"), map(int, values))))
            elif word == "config":
                config = tuple(map(int, values))
            elif word == "rc":
                result.append((made, config, int(values[0])))
                made, config = [], None
        assert len(result) == len(commands)
        return result

    return run


def umul24(a, b):
    """the kernels' product: the low 24 bits of each factor, 32 bits of the result"""
    return ((a & 0xffffff) * (b & 0xffffff)) & 0xffffffff


@pytest.mark.parametrize("tid", [lx.REAL_8, lx.REAL_4])
@pytest.mark.parametrize("k", [(1 << 24) - 1, 1 << 24, (1 << 24) + 5, (1 << 30) + 7])
def test_long_k_in_parts(launches, tid, k):
    """one launch of an entry-parallel kernel takes at most the k that its 24-bit products hold; the parts cover k"""
    m = n = 1
    (made, _, rc), (explicit, _, rc2) = launches(["process %d %d %d %d 2" % (tid, m, n, k),
                                                  "config %d %d %d %d 2 2 1 1 256 1 16 2 0 0 0 0" % (tid, m, n, k)])
    size = 8 if tid == lx.REAL_8 else 4
    assert 0 == rc and 0 == rc2
    for launch in (made, explicit):
        k0 = 0
        for part in launch:
            assert part["a"] == size * m * k0 and part["b"] == size * n * k0
            last = part["k"] - 1
            for f in (0, 1, 511, 512, last // 2, last):  # the flat index of one entry is its k
                assert umul24(f, m) == f * m
            steps, wavefronts = (part["k"] + 3) // 4, part["nt"] // 64
            assert steps * wavefronts < 1 << 31
            k0 += part["k"]
        assert k0 == k


@pytest.mark.gpu
@pytest.mark.parametrize("tid", [lx.REAL_8, lx.REAL_4])
def test_long_k_result(tid):
    """m = n = 1, k just above 2^24, whole numbers: the sum is exact in any order"""
    import numpy as np

    k = (1 << 24) + 5
    rng = np.random.default_rng(k)
    dtype = lx.nptype(tid)
    a, b = (rng.integers(-1, 2, (2, k)).astype(dtype) for _ in range(2))
    a[:, 0] = b[:, 0] = 0  # a k that wraps to the start of the block would lose the last terms
    a[:, 1 << 24:] = b[:, 1 << 24:] = 3
    c = np.array([5.0], dtype=dtype)
    stack = np.array([[1, 1, 1], [k + 1, k + 1, 1]], dtype=np.int32)
    expected = 5 + int(np.sum(a.astype(np.int64) * b.astype(np.int64)))
    lx.init()
    stream = lx.Stream("long")
    try:
        bufs = [lx.DeviceBuffer.from_array(x) for x in (stack, a, b, c)]
        assert 0 == lx.process(bufs[0], 2, tid, bufs[1], bufs[2], bufs[3], 1, 1, k, stream)
        stream.sync()
        out = np.empty_like(c)
        bufs[3].download(out)
        for x in bufs:
            x.free()
    finally:
        stream.close()
        lx.finalize()
    assert out[0] == expected
