"""Batched host-to-host DGEMM at the edges of its 64 x 64 tiles and 8-wide inner-dimension stages.

Integer data, so the products are exact in FP64 in any order of the sums: no tolerance.
"""
import itertools

import numpy as np
import pytest

import tiledmm

pytestmark = pytest.mark.gpu

EDGES = (1, 15, 63, 64, 65, 129)
KS = (0, 1, 7, 8, 9, 31, 32, 33, 65, 257)


@pytest.mark.parametrize("flags", ["NN", "TN", "NT", "TT"])
def test_batched_tile_edges_exact(torch_gpu, flags):
    """Every pair of row and column counts around a tile's edge, over inner dimensions that leave a
    wave without a stage, with a partial one, or with several; problems without inner dimension
    scale C."""
    rng = np.random.default_rng(21)
    ks = itertools.cycle(KS)
    probs = []
    for m, n in itertools.product(EDGES, EDGES):
        k = next(ks)
        a, b = rng.integers(-9, 10, (m, k)).astype(float), rng.integers(-9, 10, (k, n)).astype(float)
        c = rng.integers(-9, 10, (m, n)).astype(float)
        probs.append((m, n, k, a, b, c))

    def stored(x, op, pad):
        x = x if op == "N" else x.T
        out = tiledmm.pinned_empty((max(1, x.shape[0]) + pad, max(1, x.shape[1])), np.float64)
        out[...] = np.nan
        out[:x.shape[0], :x.shape[1]] = x
        return out

    A = [stored(p[3], flags[0], i % 3) for i, p in enumerate(probs)]
    B = [stored(p[4], flags[1], (i + 1) % 3) for i, p in enumerate(probs)]
    C = [stored(p[5], "N", (i + 2) % 3) for i, p in enumerate(probs)]
    ms, ns, ks_ = ([p[j] for p in probs] for j in range(3))
    with tiledmm.Handle(tiledmm.F64, 2) as h:
        h.set_option(tiledmm.OPT_BATCH_BODY, 1)
        h.gemm_batched(flags[0], flags[1], ms, ns, ks_, [2.0] * len(probs), A, [x.shape[0] for x in A], B,
                       [x.shape[0] for x in B], [3.0] * len(probs), C, [x.shape[0] for x in C])
        assert h.stats()["batch_body"] == 1
    for (m, n, k, a, b, c), out in zip(probs, C):
        np.testing.assert_array_equal(out[:m], 2 * (a @ b) + 3 * c, err_msg=f"{m} x {n} x {k}")
        assert np.isnan(out[m:]).all()


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("pad,shift", [(0, 0), (0, 1), (1, 0), (2, 1)])
def test_batched_copies_exact(torch_gpu, pad, shift, graph):
    """A batch whose copies run by kernel: matrices on both sides of the 4096 elements of its pieces and
    of 16-byte alignment; contiguous and padded; nothing beyond the matrices is written."""
    rng = np.random.default_rng(22)
    sizes = [(362, 362, 362), (363, 362, 361), (1, 1, 1), (64, 64, 64), (4095, 3, 5), (4096, 2, 3), (4097, 3, 2),
             (3, 4099, 2), (17, 9, 4101)]

    def stored(x):
        flat = tiledmm.pinned_empty((shift + (x.shape[0] + pad) * x.shape[1] + 1,), np.float64)
        flat[...] = np.nan
        out = flat[shift:-1].reshape((x.shape[0] + pad, x.shape[1]), order="F")
        out[:x.shape[0]] = x
        return flat, out

    mats = [[rng.integers(-9, 10, s).astype(float) for s in ((m, k), (k, n), (m, n))] for m, n, k in sizes]
    held = [[stored(x) for x in group] for group in mats]
    A, B, C = ([group[j][1] for group in held] for j in range(3))
    ms, ns, ks = zip(*sizes)
    count = len(sizes)
    with tiledmm.Handle(tiledmm.F64, 2) as h:
        h.set_option(tiledmm.OPT_BATCH_GRAPH, graph)
        for _ in range(2):  # the second call reads the C that the first one left
            h.gemm_batched("N", "N", ms, ns, ks, [1.0] * count, A, [x.shape[0] for x in A], B,
                           [x.shape[0] for x in B], [1.0] * count, C, [x.shape[0] for x in C])
        assert h.stats()["batch_graph"] == graph
    for (a, b, c), group, size in zip(mats, held, sizes):
        flat, out = group[2]
        np.testing.assert_array_equal(out[:size[0]], 2 * (a @ b) + c, err_msg=str(size))
        assert np.isnan(out[size[0]:]).all() and np.isnan(flat[:shift]).all() and np.isnan(flat[-1])


def test_batched_long_columns_take_the_other_body(torch_gpu):
    """Columns of more than 256 MB are beyond the direct-to-LDS body's 32-bit lane offsets: the batch
    runs on the register-staged one. Ones and twos: the sum is exact."""
    k = (1 << 25) + 9
    a, b = tiledmm.pinned_empty((k, 1)), tiledmm.pinned_empty((k, 1))
    a[...], b[...] = 1.0, 2.0
    small = np.asfortranarray(np.arange(6.0).reshape(3, 2))
    C = [tiledmm.pinned_empty((1, 1)), tiledmm.pinned_empty((2, 2))]
    A, B = [a, tiledmm.pinned_empty((3, 2))], [b, tiledmm.pinned_empty((3, 2))]
    A[1][...], B[1][...] = small, small
    with tiledmm.Handle(tiledmm.F64, 2) as h:
        h.set_option(tiledmm.OPT_BATCH_BODY, 1)
        h.gemm_batched("T", "N", [1, 2], [1, 2], [k, 3], [1.0] * 2, A, [k, 3], B, [k, 3], [0.0] * 2, C, [1, 2])
        assert h.stats()["batch_body"] == 0
    assert C[0][0, 0] == 2.0 * k
    np.testing.assert_array_equal(C[1], small.T @ small)
