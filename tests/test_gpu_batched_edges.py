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
