"""A batch of small page-locked matrices, whose copies run by kernel, is enqueued on the queues by itself; as
a graph, when that is asked for, its copies are the graph's copy nodes. Integer data, exact."""
import numpy as np
import pytest

import tiledmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("option,graph", [(-1, 0), (0, 0), (1, 1)])
def test_small_batches_run_on_queues(torch_gpu, option, graph):
    rng = np.random.default_rng(3)
    sizes = [(100, 90, 80), (33, 44, 55), (200, 10, 300), (1, 1, 1), (64, 64, 64)]

    def pinned(rows, cols):
        x = tiledmm.pinned_empty((rows, cols))
        x[...] = rng.integers(-9, 10, (rows, cols))
        return x

    A, B, C = ([pinned(*f(s)) for s in sizes] for f in (lambda s: (s[0], s[2]), lambda s: (s[2], s[1]), lambda s: s[:2]))
    ms, ns, ks = zip(*sizes)
    with tiledmm.Handle(tiledmm.F64, 2) as h:
        h.set_option(tiledmm.OPT_BATCH_GRAPH, option)
        for beta in (0.0, 1.0, 1.0):
            h.gemm_batched("N", "N", ms, ns, ks, [1.0] * 5, A, [x.shape[0] for x in A], B, [x.shape[0] for x in B],
                           [beta] * 5, C, [x.shape[0] for x in C])
        assert h.stats()["batch_graph"] == graph
    for a, b, c in zip(A, B, C):
        np.testing.assert_array_equal(c, 3 * (a @ b))
