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
                made.append(dict(zip(("groups", "nt", "bs", "k", "kt", "tsplit", "atomic", "a", "b", "piece"), map(int, values))))
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


# variant tm tn nt bs kt flush s split bs_short split_short
TUNED = {"23x23x23": (lx.REAL_8, 23, 23, 23, "2 2 2 512 32 16 2 30000 3 0 0"), "5x5x5": (lx.REAL_4, 5, 5, 5, "4 2 2 64 24 64 2 30000 2 0 0")}


def scaled(bs, stack_size, s):
    """bs for a stack shorter than the s it was chosen for (smm_kernel.c:463-473)"""
    return min(bs, max(1, -(-stack_size * max(bs, 32) // (s - 1)))) if s > 1 and stack_size < s else bs


@pytest.mark.parametrize("name", sorted(TUNED))
@pytest.mark.parametrize("entries", [300, 3000, 12000, 16383])
def test_explicit_configurations_are_launched(launches, tmp_path, name, entries):
    """what the caller sets (process_config, config_set, a file, the environment) is launched in short stacks: bs scaled
    by s, its own cut factor, threads and k per stage"""
    tid, m, n, k, text = TUNED[name]
    _, _, _, nt, bs, kt, _, s, split, _, _ = map(int, text.split())
    shape = "%d %d %d %d" % (tid, m, n, k)
    path = tmp_path / "mine.csv"
    v, tm, tn, _, _, _, fl, _, _, bss, sps = text.split()
    path.write_text("DEVICE;TYPEID;M;N;K;S;GFLOPS;VARIANT;TM;TN;NT;BS;KT;FLUSH;SPLIT;BSS;SPLITS\n"
                    "MI355X;%d;%d;%d;%d;%d;1.0;%s;%s;%s;%d;%d;%d;%s;%d;%s;%s\n" % (tid, m, n, k, s, v, tm, tn, nt, bs, kt, fl,
                                                                                split, bss, sps))
    process = "process %s %d" % (shape, entries)
    made = [launches(["config %s %d %s" % (shape, entries, text)])[0][0],
            launches(["set %s %s" % (shape, text), process])[1][0],
            launches([process], OPENCL_LIBSMM_SMM_PARAMS=str(path))[0][0]]
    expected = scaled(bs, entries, s)
    for one in made:
        assert len(one) == 1 and (one[0]["nt"], one[0]["kt"], one[0]["bs"]) == (nt, kt, expected), made
        assert one[0]["tsplit"] == split * expected and one[0]["groups"] == -(-entries // expected)
    env = launches([process], OPENCL_LIBSMM_SMM_BS="20")[0][0][0]
    assert env["bs"] == scaled(20, entries, s)


@pytest.mark.parametrize("entries", [300, 12000])
def test_short_stack_pair_is_launched(launches, entries):
    """bs_short and split_short of a configuration, for stacks of at most s entries"""
    text = "2 2 2 512 32 16 2 16000 3 9 2"
    for command in (["config 3 23 23 23 %d %s" % (entries, text)],
                    ["set 3 23 23 23 " + text, "process 3 23 23 23 %d" % entries]):
        (made,), _, rc = launches(command)[-1]
        assert 0 == rc and made["bs"] == scaled(9, entries, 16000) and made["tsplit"] == 2 * made["bs"]


@pytest.mark.parametrize("tid", [lx.REAL_8, lx.REAL_4])
@pytest.mark.parametrize("entries", [300, 500, 750, 1500, 1800, 5000])
def test_cut_follows_the_launched_wavefronts(launches, tid, entries):
    """5x5x5: the shipped row (one wavefront per run at 30000 entries, four in short stacks) and the rule for shapes
    without a row launch the same threads, so they cut the stack alike"""
    commands = ["process %d 5 5 5 %d" % (tid, entries)]
    row = launches(commands)[0][0][0]
    rule = launches(commands, OPENCL_LIBSMM_SMM_PARAMS="0")[0][0][0]
    assert row["nt"] == rule["nt"] == 256
    assert (row["bs"], row["tsplit"]) == (rule["bs"], rule["tsplit"])


# without a row in the shipped file, up to 16 tiles of 16x16
@pytest.mark.parametrize("shape", [(7, 9, 11), (16, 16, 5), (40, 20, 33), (60, 64, 9), (3, 4, 700)], ids=str)
@pytest.mark.parametrize("tid", [lx.REAL_8, lx.REAL_4])
def test_configuration_reported_and_predictor_switches(launches, tid, shape):
    """config_get tells what process launches; the predictor switched off, cleared or held to a threshold that it misses
    leads to the heuristic, as it does for larger blocks"""
    name = "%d %d %d %d" % (tid, *shape)
    commands = ["get " + name, "process %s 30000" % name, "process %s 500000" % name]
    heuristic = lx.default_config(tid, *shape)
    for env, clear in (({}, 0), (dict(LIBXSTREAM_LEARNED="0"), 0), (dict(LIBXSTREAM_LEARNED_CONF="1.5"), 0), ({}, 1)):
        got, *made = launches(["clear"] * clear + commands, **env)[clear:]
        source, variant, tm, tn, nt, bs, kt, flush, s, split, _, _ = got[1]
        assert 0 == source and 30000 == s and 0 == got[2]
        if env or clear:
            assert (variant, tm, tn, nt, bs, kt) == (heuristic.variant, heuristic.tm, heuristic.tn, heuristic.nt,
                                                     heuristic.bs, heuristic.kt)
        for (one,), _, rc in made:
            assert 0 == rc and (one["nt"], one["bs"]) == (nt, bs) and one["kt"] == (kt or one["kt"])
            assert one["tsplit"] == max((split or 2) * bs, 64)


@pytest.mark.parametrize("tid", [lx.REAL_8, lx.REAL_4])
@pytest.mark.parametrize("shape", [(23, 23, 23), (13, 13, 13), (5, 5, 5), (45, 45, 13), (17, 3, 40), (6, 7, 70)],
                         ids=lambda s: "%dx%dx%d" % s)
def test_short_stacks_in_pieces(launches, tid, shape):
    """short stacks: few entries per work-group, which begin the pieces of longer runs"""
    sizes = (30, 300, 1000, 2000, 4000, 7000, 10000, 15000, 16383)
    runs = launches(["process %d %d %d %d %d" % (tid, *shape, s) for s in sizes])
    for size, (made, _, rc) in zip(sizes, runs):
        assert 0 == rc and 1 == len(made)
        launch = made[0]
        assert 1 <= launch["bs"] <= 16 and launch["groups"] == (size + launch["bs"] - 1) // launch["bs"]
        assert 0 == launch["piece"] % launch["bs"] and 1 <= launch["piece"] <= 32 and 0 < launch["tsplit"] <= 40
    # an explicit configuration's own segments
    for made, _, rc in launches(["config %d %d %d %d 4000 2 2 2 256 12 16 2 2 0 0 0" % (tid, *shape)]):
        assert rc or (12 == made[0]["bs"] == made[0]["piece"])
