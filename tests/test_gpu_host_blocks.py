"""Block sizes that a host-to-host call runs on, by the statistics of the call."""
import numpy as np
import pytest

import tiledmm

pytestmark = pytest.mark.gpu

M, N, K, TILE, BLOCKS = 3000, 2900, 300, 1500, 2  # complex float: coarsened to 3000 x 1536 blocks of C


def _array(shape, pinned, rng):
    x = tiledmm.pinned_empty(shape, np.complex64) if pinned else np.empty(shape, np.complex64, order="F")
    x[...] = rng.integers(-4, 5, shape) + 1j * rng.integers(-4, 5, shape)
    return x


def _call(pinned_ab, pinned_c, beta, coarsen=1):
    rng = np.random.default_rng(5)
    a, b, c = _array((M, K), pinned_ab, rng), _array((K, N), pinned_ab, rng), _array((M, N), pinned_c, rng)
    exact = (a @ b + beta * c).astype(np.complex64)  # small integers
    with tiledmm.Handle(tiledmm.C32, 2, TILE, TILE, TILE) as h:
        h.set_option(tiledmm.OPT_COARSEN, coarsen)
        h.gemm("N", "N", M, N, K, 1.0, a, M, b, K, beta, c, M)
        np.testing.assert_array_equal(c, exact)
        return h.stats()


@pytest.mark.parametrize("pinned_ab,pinned_c,beta,cut", [
    (True, True, 1.0, True), (True, True, 0.0, True),
    (False, True, 1.0, True),   # C itself is copied without the host's threads
    (False, False, 0.0, True),
    (False, False, 1.0, False), (True, False, 1.0, False),
])
def test_blocks_with_a_pageable_c_read_are_not_cut(torch_gpu, pinned_ab, pinned_c, beta, cut):
    st = _call(pinned_ab, pinned_c, beta)
    assert st["k_chunks"] == 1
    assert (st["gemm_launches"] > BLOCKS) == cut, st
    assert cut or st["gemm_launches"] == BLOCKS, st


@pytest.mark.parametrize("coarsen", [0, 1])
@pytest.mark.parametrize("pinned", [False, True])
def test_statistics_report_the_blocks_that_ran(torch_gpu, pinned, coarsen):
    st = _call(pinned, pinned, 0.0, coarsen)
    blocks = -(-M // int(st["tile_m"])) * -(-N // int(st["tile_n"]))
    assert st["gemm_launches"] == blocks * st["k_chunks"], st
    assert blocks > BLOCKS, st  # without coarsening 2 x 2 tiles, with it cut blocks
