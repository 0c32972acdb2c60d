"""Cases that a user of the library runs, for timing and for comparing two builds of it.

A program that uses the library multiplies column-major matrices of one of four element types:
data that is already in device memory (`Handle.device_gemm`, the library's tile product on its
own), data in host memory (`Handle.gemm`, the out-of-core call), or a batch of host matrices of
uneven sizes (`Handle.gemm_batched`). A FP64 handle may be switched to the INT8 emulation (Ozaki
scheme II) by its modulus count. A case is a dict of plain values:

  kind    "device", "host" or "batch"
  dtype   "d", "s", "z", "c": double, float, complex double, complex float
  ops     two of N, T, C
  m, n, k, pad   sizes, and rows by which every leading dimension exceeds its minimum
  beta    0 or 1; with 1 the product is added to the C of the state (alpha is 1)
  moduli  INT8 emulation with so many moduli (0: native matrix cores)
  pinned  host memory is page-locked (host and batch)
  count, low, high, mix   batch: problems, the range of their edges, the seed of their sizes
"""
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tiled-mm_amd"))
import tiledmm  # noqa: E402

TORCH = {"s": torch.float32, "d": torch.float64, "c": torch.complex64, "z": torch.complex128}
NUMPY = {"s": np.float32, "d": np.float64, "c": np.complex64, "z": np.complex128}
CODE = {"s": tiledmm.F32, "d": tiledmm.F64, "c": tiledmm.C32, "z": tiledmm.C64}
BYTES = {"s": 4, "d": 8, "c": 8, "z": 16}


def _device(dtype, ops, m, n, k, pad=0, beta=0, moduli=0):
    return {"kind": "device", "dtype": dtype, "ops": ops, "m": m, "n": n, "k": k, "pad": pad, "beta": beta,
            "moduli": moduli}


def _host(dtype, ops, m, n, k, pad, beta, pinned):
    return {"kind": "host", "dtype": dtype, "ops": ops, "m": m, "n": n, "k": k, "pad": pad, "beta": beta,
            "moduli": 0, "pinned": pinned}


def _batch(count, low, high, mix, ops):
    return {"kind": "batch", "dtype": "d", "ops": ops, "count": count, "low": low, "high": high, "mix": mix,
            "pinned": True}


def listed():
    named = {
        # one small block of a larger program: the call's latency, and a k that is no multiple of 8
        "dgemm small": _device("d", "TN", 300, 200, 260),
        # the smallest of the reference's square test sizes
        "dgemm square": _device("d", "NN", 1000, 1000, 1000),
        # its small non-square test size: an odd n and an odd k, both operands row-contiguous
        "dgemm ragged": _device("d", "NT", 1234, 4567, 1357),
        # overlap (Gram-like) matrices: a short C and a long inner dimension
        "dgemm long k": _device("d", "TN", 500, 600, 40000),
        # one block of an out-of-core product, added to the C of the earlier blocks
        "dgemm large": _device("d", "TN", 8192, 8192, 8192, pad=64, beta=1),
        # the ordinary square size in single precision
        "sgemm": _device("s", "NN", 2048, 2048, 2048),
        # complex types with a conjugated operand, as electronic-structure codes call them
        "cgemm": _device("c", "CN", 1500, 1300, 2000),
        "zgemm": _device("z", "CN", 1000, 1100, 1200),
        # FP64 on the INT8 matrix cores
        "dgemm emulated": _device("d", "NN", 2048, 2048, 2048, moduli=16),
        # an ordinary call on ordinary (pageable) host memory
        "host dgemm": _host("d", "NN", 1234, 4567, 1357, 0, 0, False),
        # the largest square test size of the reference, pinned and padded as the benchmark has it
        "host dgemm large": _host("d", "TN", 10000, 10000, 10000, 64, 1, True),
        # many small products of uneven size in one call
        "batch": _batch(48, 64, 1024, 1, "NN"),
    }
    return [dict(case, name=name) for name, case in named.items()]


def _log(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    what = rng.random()
    pad = rng.choice([0, 0, 1, 8, 64])
    beta = rng.choice([0, 0, 1])
    if what < 0.45:  # device products of every type, small to ordinary
        t = rng.choice("ddszc")
        ops = "".join(rng.choice("NTC" if t in "cz" else "NT") for _ in range(2))
        top = 4500 if t in "ds" else 3000
        return _device(t, ops, _log(rng, 100, top), _log(rng, 100, top), _log(rng, 100, top), pad, beta)
    if what < 0.55:  # a short C and a long inner dimension
        ops = rng.choice(["TN", "TN", "NN", "NT"])
        return _device(rng.choice("ds"), ops, _log(rng, 200, 1000), _log(rng, 200, 1000), _log(rng, 8000, 40000), pad, beta)
    if what < 0.65:  # blocks of an out-of-core product
        return _device("d", rng.choice(["TN", "NN", "NT", "TT"]), _log(rng, 4500, 8192), _log(rng, 4500, 8192),
                       _log(rng, 2000, 8192), pad, beta)
    if what < 0.77:  # emulated
        return _device("d", rng.choice(["NN", "TN", "NT"]), _log(rng, 500, 4096), _log(rng, 500, 4096),
                       _log(rng, 500, 4096), pad, beta, rng.choice([14, 16, 18]))
    if what < 0.9:  # host memory
        t = rng.choice("ddszc")
        top = 5000 if t in "ds" else 3000
        return _host(t, rng.choice(["NN", "TN", "NT"]), _log(rng, 400, top), _log(rng, 400, top), _log(rng, 400, top),
                     pad, beta, rng.random() < 0.5)
    return _batch(rng.randint(8, 60), 64, _log(rng, 400, 1400), rng.randint(2, 1 << 20), rng.choice(["NN", "TN", "NT"]))


# A program keeps one handle per element type and setting.
_handles = {}


def _handle(case):
    moduli = case.get("moduli", 0)
    key = (case["dtype"], moduli)
    if key not in _handles:
        h = tiledmm.Handle(CODE[case["dtype"]], 2, 8192, 8192, 8192)
        if moduli:
            h.set_option(tiledmm.OPT_OZAKI_MODULI, moduli)
        _handles[key] = h
    return _handles[key]


def _uniform(gen, dtype, rows, cols, ld):
    """Column-major rows x cols of uniform [-1, 1) values on the GPU: a (cols, ld) tensor."""
    real = torch.float32 if dtype in "sc" else torch.float64
    width = ld * (2 if dtype in "cz" else 1)
    x = torch.rand(cols, width, generator=gen, dtype=real, device="cuda").mul_(2).sub_(1)
    return torch.view_as_complex(x.view(cols, ld, 2)) if dtype in "cz" else x


def _stored(op, rows, cols):
    """Rows and columns of the stored matrix whose op() is rows x cols."""
    return (rows, cols) if op == "N" else (cols, rows)


def _operands(case, seed):
    """A, B, C of a device or host case on the GPU, each with its leading dimension."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    m, n, k, pad, t = case["m"], case["n"], case["k"], case["pad"], case["dtype"]
    out = []
    for rows, cols in (_stored(case["ops"][0], m, k), _stored(case["ops"][1], k, n), (m, n)):
        out.append(_uniform(gen, t, rows, cols, rows + pad))
    return out


def _edges(case):
    """Sizes (m, n, k) of a batch's problems, uneven and of the case alone."""
    r = random.Random(case["mix"])
    return [tuple(_log(r, case["low"], case["high"]) for _ in range(3)) for _ in range(case["count"])]


def _to_host(x, pinned):
    """A (cols, ld) tensor's values in host memory: a column-major (ld, cols) array."""
    cols, ld = x.shape
    dtype = NUMPY[{v: k for k, v in TORCH.items()}[x.dtype]]
    a = tiledmm.pinned_empty((ld, cols), dtype) if pinned else np.empty((ld, cols), dtype, order="F")
    torch.from_numpy(a.T).copy_(x)
    return a


def prepare(case, seed):
    state = {"case": case, "handle": _handle(case)}
    if case["kind"] == "batch":
        gen = torch.Generator(device="cuda").manual_seed(seed)
        problems = []
        for m, n, k in _edges(case):
            shapes = (_stored(case["ops"][0], m, k), _stored(case["ops"][1], k, n), (m, n))
            problems.append([_to_host(_uniform(gen, "d", r, c, r), case["pinned"]) for r, c in shapes])
        state["sizes"], state["problems"] = _edges(case), problems
    elif case["kind"] == "host":
        state["abc"] = [_to_host(x, case["pinned"]) for x in _operands(case, seed)]
    else:
        state["abc"] = _operands(case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    case, h = state["case"], state["handle"]
    ta, tb = case["ops"]
    if case["kind"] == "batch":
        ms, ns, ks = zip(*state["sizes"])
        a, b, c = zip(*state["problems"])
        count = len(ms)
        h.gemm_batched(ta, tb, ms, ns, ks, [1.0] * count, a, [x.shape[0] for x in a], b, [x.shape[0] for x in b],
                       [0.0] * count, c, [x.shape[0] for x in c])
        return list(c)
    a, b, c = state["abc"]
    m, n, k = case["m"], case["n"], case["k"]
    if case["kind"] == "host":
        h.gemm(ta, tb, m, n, k, 1.0, a, a.shape[0], b, b.shape[0], float(case["beta"]), c, c.shape[0])
        return c[:m]
    h.device_gemm(ta, tb, m, n, k, 1.0, a, a.shape[1], b, b.shape[1], float(case["beta"]), c, c.shape[1])
    return c[:, :m]


def work(case):
    per = 8 if case["dtype"] in "cz" else 2
    total, flops = 0, 0
    for m, n, k in _edges(case) if case["kind"] == "batch" else [(case["m"], case["n"], case["k"])]:
        total += BYTES[case["dtype"]] * (m * k + k * n + m * n * (1 + case.get("beta", 0)))
        flops += per * m * n * k
    return {"bytes": total, "flops": flops}


def _product(ops, a, b):
    """(op(A) op(B))^T = op(B)^T op(A)^T in 64 bits; a (cols, rows) tensor of a matrix X is X^T."""
    def transposed(x, op):
        x = x.to(torch.complex128 if x.is_complex() else torch.float64)
        return x if op == "N" else x.T if op == "T" else x.conj().T

    return transposed(b, ops[1]) @ transposed(a, ops[0])


def exact(case, seed):
    if case["kind"] == "batch":
        gen = torch.Generator(device="cuda").manual_seed(seed)
        out = []
        for m, n, k in _edges(case):
            shapes = (_stored(case["ops"][0], m, k), _stored(case["ops"][1], k, n), (m, n))
            a, b, _ = (_uniform(gen, "d", r, c, r) for r, c in shapes)
            out.append(_product(case["ops"], a, b).T.cpu())
        return out
    a, b, c = (x[:, :x.shape[1] - case["pad"]] for x in _operands(case, seed))
    r = _product(case["ops"], a, b)
    if case["beta"]:
        r += c
    return r if case["kind"] == "device" else r.T.cpu()
