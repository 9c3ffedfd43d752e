"""Performance cases of the framework: what they compute, on which inputs, and what they cannot do without.

Each case is one call of a public entry point of ``libxstream_amd`` on device memory that the caller holds (torch
tensors here, passed by address), on one stream the program keeps:

    stack         libsmm_acc_process: C[c_i] += A[a_i] B[b_i] over a parameter stack sorted by C
    transpose     libsmm_acc_transpose: the blocks of a pool transposed in place
    batch         libsmm_acc_batch_replay: stacks of mixed shapes planned once and replayed from a graph
    ozaki_gemm    ozaki_gemm: a GEMM emulated with int8 products (scheme 1: slices, scheme 2: CRT)
    ozaki_stack   ozaki_stack: the parameter stack with emulated products
    dgemm         ozaki_dgemm_native: the native FP64 matrix-core GEMM

``listed()`` are the fixed cases, ``draw(rng)`` gives others of the same ranges, ``prepare`` makes a case's inputs and
handles, ``run`` is one pass, ``work`` its unavoidable bytes and operations and ``exact`` its result in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

import libxstream_amd as lx

NP = {"f64": np.float64, "f32": np.float32}
TORCH = {"f64": torch.float64, "f32": torch.float32}
SIZE = {"f64": 8, "f32": 4}


def listed():
    return [
        # the headline of the reference's benchmark: 30000 entries over 1000 C blocks, water-like 23x23 blocks
        _stack("stack_f64_23_30k", "f64", 23, 23, 23, 30000),
        # the same blocks with pools that exceed the last-level cache: a large DBCSR multiplication
        _stack("stack_f64_23_500k", "f64", 23, 23, 23, 500000),
        # large blocks, where the matrix cores rather than memory set the pace
        _stack("stack_f64_64_100k", "f64", 64, 64, 64, 100000),
        # the smallest blocks of the stack workloads, single precision, many entries
        _stack("stack_f32_5_500k", "f32", 5, 5, 5, 500000),
        # a flat k with odd extents, single precision
        _stack("stack_f32_45x45x13_100k", "f32", 45, 45, 13, 100000),
        # a short stack: what one thread hands over while a sparse multiplication is being assembled
        _stack("stack_f64_13_1k", "f64", 13, 13, 13, 1000),
        # the B pool of the large 23x23 stack brought into the kernel's layout
        {"name": "transpose_f64_23_33k", "kind": "transpose", "dtype": "f64", "m": 23, "n": 23, "blocks": 33334},
        # 24 stacks of log-uniform shapes in 4..64 and lengths in 1000..200000, replayed from one graph
        {"name": "batch_f64_24", "kind": "batch", "dtype": "f64", "count": 24, "shapes": 25071975, "dim_lo": 4,
         "dim_hi": 64, "len_lo": 1000, "len_hi": 200000},
        # FP64 GEMM by the CRT scheme at the size of the DGEMM benchmark
        _gemm("ozaki2_f64_8192", "ozaki_gemm", "f64", 8192, 8192, 8192, "N", "N", 2),
        # the slice scheme with its default slices on an ordinary, ragged, transposed GEMM
        _gemm("ozaki1_f64_1000x1100x900", "ozaki_gemm", "f64", 1000, 1100, 900, "T", "N", 1),
        # emulated products over a parameter stack of 64x64 blocks, default slices
        {"name": "ozaki_stack_f64_64_100k", "kind": "ozaki_stack", "dtype": "f64", "m": 64, "n": 64, "k": 64,
         "entries": 100000, "slices": 0},
        # the native FP64 GEMM that the emulation is an alternative to
        _gemm("dgemm_f64_4096", "dgemm", "f64", 4096, 4096, 4096, "N", "N", 0),
    ]


def _stack(name, dtype, m, n, k, entries):
    case = {"name": name, "kind": "stack", "dtype": dtype, "m": m, "n": n, "k": k, "entries": entries}
    return {key: v for key, v in case.items() if v is not None}


def _gemm(name, kind, dtype, m, n, k, ta, tb, scheme, beta=0.0):
    case = {"name": name, "kind": kind, "dtype": dtype, "m": m, "n": n, "k": k, "ta": ta, "tb": tb, "beta": beta}
    if "ozaki_gemm" == kind:
        case["scheme"] = scheme
    return {key: v for key, v in case.items() if v is not None}


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["stack"] * 6 + ["transpose", "batch", "ozaki_gemm", "ozaki_gemm", "ozaki_stack", "dgemm"])
    dtype = rng.choice(["f64", "f64", "f32"])
    if "stack" == kind:
        return _stack(None, dtype, log(4, 64), log(4, 64), log(4, 64), log(300, 300000))
    if "transpose" == kind:
        return {"kind": kind, "dtype": dtype, "m": log(4, 64), "n": log(4, 64), "blocks": log(300, 40000)}
    if "batch" == kind:
        return {"kind": kind, "dtype": dtype, "count": rng.randint(2, 24), "shapes": rng.randrange(1 << 30), "dim_lo": 4,
                "dim_hi": 64, "len_lo": 1000, "len_hi": 200000}
    if "ozaki_stack" == kind:
        return {"kind": kind, "dtype": dtype, "m": log(8, 64), "n": log(8, 64), "k": log(8, 64),
                "entries": log(1000, 100000), "slices": rng.randint(3, 8)}
    ta, tb, beta = rng.choice("NT"), rng.choice("NT"), rng.choice([0.0, 0.0, 1.0])
    m, n, k = log(64, 4096), log(64, 4096), log(64, 4096)
    return _gemm(None, kind, "f64" if "dgemm" == kind else dtype, m, n, k, ta, tb, rng.choice([1, 2]), beta)


# ---- inputs -------------------------------------------------------------------------------------


def _uniform(gen, shape, dtype):
    """Uniform in [-1, 1), the block values of the stack workloads."""
    return torch.rand(shape, generator=gen, dtype=TORCH[dtype], device="cuda").mul_(2).sub_(1)


def _scaled(gen, rows, cols, dtype, by_row):
    """+-[1, 2) mantissas times 2^x with x uniform in -10..10 per row (by_row) or per column: a rows x cols matrix."""
    value = torch.rand((rows, cols), generator=gen, dtype=TORCH[dtype], device="cuda").add_(1)
    value.mul_(torch.randint(0, 2, (rows, cols), generator=gen, device="cuda", dtype=torch.int8).mul_(2).sub_(1))
    x = torch.randint(-10, 11, (rows, 1) if by_row else (1, cols), generator=gen, device="cuda").to(TORCH[dtype])
    return value.mul_(torch.exp2(x))


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _indices(rng, entries, na, nb, nc):
    """(a, b, c) block indices of a stack sorted by c: runs of about entries / nc, the last one takes the rest."""
    avg = max(1, int(round(entries / nc)))
    lengths = rng.integers(max(1, avg - 4), avg + 5, size=nc)
    c = np.repeat(np.arange(nc, dtype=np.int64), lengths)[:entries]
    c = np.concatenate([c, np.full(entries - c.size, nc - 1, dtype=np.int64)])
    return np.stack([rng.integers(0, na, size=entries), rng.integers(0, nb, size=entries), c], axis=1)


def _pools(case):
    """Blocks of the A, B and C pools of a stack: about 30 updates per C block, as in the stack workloads."""
    nc = max(1, int(round(case["entries"] / 30.0)))
    return 2 * nc, 2 * nc, nc


def _stack_inputs(case, seed):
    """Block indices on the host; A (na, k, m), B (nb, k, n), C (nc, n, m) and the stack of 1-based offsets on the GPU."""
    m, n, k, dtype = case["m"], case["n"], case["k"], case["dtype"]
    na, nb, nc = _pools(case)
    idx = _indices(np.random.default_rng(seed), case["entries"], na, nb, nc)
    stack = (idx * np.array([m * k, k * n, m * n]) + 1).astype(np.int32)
    gen = _generator(seed)
    a, b, c = (_uniform(gen, shape, dtype) for shape in ((na, k, m), (nb, k, n), (nc, n, m)))
    return idx, a, b, c, torch.from_numpy(stack).cuda()


def _batch_stacks(case):
    """The (m, n, k, entries) of a batch: its shapes are the case's, its values the seed's."""
    rng = np.random.default_rng(case["shapes"])
    dims = np.rint(np.exp(rng.uniform(math.log(case["dim_lo"]), math.log(case["dim_hi"]), size=(case["count"], 3))))
    lens = np.rint(np.exp(rng.uniform(math.log(case["len_lo"]), math.log(case["len_hi"]), size=case["count"])))
    return [{"dtype": case["dtype"], "m": int(d[0]), "n": int(d[1]), "k": int(d[2]), "entries": int(s)}
            for d, s in zip(dims, lens)]


def _gemm_inputs(case, seed):
    """Stored operands, column-major: a tensor of shape (columns, rows) holds them."""
    m, n, k, dtype = case["m"], case["n"], case["k"], case["dtype"]
    gen = _generator(seed)
    # op(A) is scaled by row and op(B) by column; the tensors are the transposes of the stored matrices
    a = _scaled(gen, k, m, dtype, False) if "N" == case["ta"] else _scaled(gen, m, k, dtype, True)
    b = _scaled(gen, n, k, dtype, True) if "N" == case["tb"] else _scaled(gen, k, n, dtype, False)
    c = _uniform(gen, (n, m), dtype)
    return a, b, c


# ---- the program's handles and one pass ---------------------------------------------------------


class _Memory:
    """A tensor's device memory as the framework takes it: an address and a size."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())
        self.nbytes = tensor.numel() * tensor.element_size()


class _Batch:
    """A planned batch and the buffers it works on."""

    def __init__(self, dtype, stacks):
        self.batch, self.stacks = lx.Batch(lx.typeid(NP[dtype]), stacks), stacks

    def __del__(self):
        self.batch.close()


_program = {}


def _stream():
    """The library initialised and the program's stream, once per process."""
    if "stream" not in _program:
        torch.cuda.init()
        lx.init()
        _program["stream"] = lx.Stream("cases")
    return _program["stream"]


def _context(dtype, scheme, slices=0):
    """The emulation's context of these settings, which a program keeps for all of its products."""
    key = (dtype, scheme, slices)
    if key not in _program:
        _program[key] = lx.Ozaki(use_double="f64" == dtype, kind=scheme, nslices=slices)
    return _program[key]


def prepare(case, seed):
    state = {"case": case, "stream": _stream()}
    kind, dtype = case["kind"], case["dtype"]
    if kind in ("stack", "ozaki_stack"):
        _, a, b, c, stack = _stack_inputs(case, seed)
        state.update(a=_Memory(a), b=_Memory(b), c=_Memory(c), stack=_Memory(stack))
        if "ozaki_stack" == kind:
            state["context"] = _context(dtype, 1, case["slices"])
    elif "transpose" == kind:
        m, n = case["m"], case["n"]
        data = _uniform(_generator(seed), (case["blocks"], n, m), dtype)
        offsets = torch.arange(case["blocks"], dtype=torch.int32, device="cuda").mul_(m * n)
        state.update(data=_Memory(data), offsets=_Memory(offsets))
    elif "batch" == kind:
        stacks = []
        for i, one in enumerate(_batch_stacks(case)):
            _, a, b, c, stack = _stack_inputs(one, seed + 7919 * i)
            stacks.append((_Memory(stack), one["entries"], one["m"], one["n"], one["k"], _Memory(a), _Memory(b), _Memory(c)))
        state["batch"] = _Batch(dtype, stacks)
    else:
        a, b, c = _gemm_inputs(case, seed)
        state.update(a=_Memory(a), b=_Memory(b), c=_Memory(c))
        if "ozaki_gemm" == kind:
            state["context"] = _context(dtype, case["scheme"])
    return state


def run(state):
    case, stream = state["case"], state["stream"]
    kind, tid = case["kind"], lx.typeid(NP[case["dtype"]])
    if "stack" == kind:
        code = lx.process(state["stack"], case["entries"], tid, state["a"], state["b"], state["c"], case["m"], case["n"],
                          case["k"], stream)
        if 0 != code:
            raise RuntimeError("libsmm_acc_process left the stack to the host")
        return state["c"].tensor
    if "transpose" == kind:
        lx.transpose(state["offsets"], 0, case["blocks"], state["data"], tid, case["m"], case["n"], stream)
        return state["data"].tensor
    if "batch" == kind:
        state["batch"].batch.replay(stream)
        return [s[7].tensor for s in state["batch"].stacks]
    m, n, k = case["m"], case["n"], case["k"]
    if "ozaki_stack" == kind:
        na, nb, _ = _pools(case)
        state["context"].stack(state["stack"], case["entries"], m, n, k, state["a"], na, state["b"], nb, state["c"], stream)
        return state["c"].tensor
    lda, ldb = (m if "N" == case["ta"] else k), (k if "N" == case["tb"] else n)
    args = (case["ta"], case["tb"], m, n, k, 1.0, state["a"], lda, state["b"], ldb, case["beta"], state["c"], m, stream)
    if "ozaki_gemm" == kind:
        state["context"].gemm(*args)
    else:
        lx.dgemm_native(*args)
    return state["c"].tensor


# ---- what a pass cannot do without, and its result in 64 bits -----------------------------------


def _stack_work(case):
    m, n, k = case["m"], case["n"], case["k"]
    na, nb, nc = _pools(case)
    return {"bytes": SIZE[case["dtype"]] * (na * m * k + nb * k * n + 2 * nc * m * n) + 12 * case["entries"],
            "flops": 2.0 * m * n * k * case["entries"]}


def work(case):
    kind = case["kind"]
    if kind in ("stack", "ozaki_stack"):
        return _stack_work(case)
    if "transpose" == kind:
        return {"bytes": case["blocks"] * (2 * SIZE[case["dtype"]] * case["m"] * case["n"] + 4), "flops": 0}
    if "batch" == kind:
        each = [_stack_work(one) for one in _batch_stacks(case)]
        return {key: sum(w[key] for w in each) for key in ("bytes", "flops")}
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": SIZE[case["dtype"]] * (m * k + k * n + (1 if 0 == case["beta"] else 2) * m * n),
            "flops": 2.0 * m * n * k}


def _stack_exact(case, seed):
    idx, a, b, c, _ = _stack_inputs(case, seed)
    idx = torch.from_numpy(idx).cuda()
    a, bt, c = a.double(), b.double().transpose(1, 2).contiguous(), c.double()
    step = max(1, (1 << 27) // (case["m"] * case["k"] + case["k"] * case["n"] + case["m"] * case["n"]))
    for e in range(0, case["entries"], step):
        i = idx[e:e + step]
        c.index_add_(0, i[:, 2], torch.bmm(bt[i[:, 1]], a[i[:, 0]]))  # (n, k) (k, m): the block's columns
    return c


def exact(case, seed):
    kind = case["kind"]
    if kind in ("stack", "ozaki_stack"):
        return _stack_exact(case, seed)
    if "transpose" == kind:
        data = _uniform(_generator(seed), (case["blocks"], case["n"], case["m"]), case["dtype"]).double()
        return data.transpose(1, 2).contiguous().view(data.shape)
    if "batch" == kind:
        return [_stack_exact(one, seed + 7919 * i) for i, one in enumerate(_batch_stacks(case))]
    a, b, c = (x.double() for x in _gemm_inputs(case, seed))
    a, b = (a if "N" == case["ta"] else a.t().contiguous()), (b if "N" == case["tb"] else b.t().contiguous())
    return b @ a + case["beta"] * c  # column-major C: (n, k) (k, m)
