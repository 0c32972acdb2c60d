"""What the search for block sizes of a host-to-host call costs (pipeline_panels in tiled-mm_amd/csrc/tmm_plan.cpp): it runs on
the caller's thread in every call, so a long inner dimension in many k-chunks must not multiply it."""
import ctypes

import pytest

import tiledmm


def steps(m, n, k, tiles, beta=0, first=0, es=8, rate=70e12):
    L = ctypes.CDLL(tiledmm.HOST_PATH)
    i, l, d = ctypes.c_int, ctypes.c_long, ctypes.c_double
    f = L.tmmh_pipeline_panels_steps
    f.argtypes, f.restype = [i] * 8 + [l, i, d, ctypes.POINTER(i)], l
    out = (i * 4)()
    return f(m, n, k, beta, *tiles, first, 0, es, rate, out), tuple(out)


@pytest.mark.parametrize("m,n,k,tiles,beta", [
    (2000, 2000, 20000, (2000, 2000, 1024), 0),
    (2000, 2000, 100000, (2000, 2000, 1024), 0),
    (2000, 2000, 100000, (2000, 2000, 1024), 1),
    (4000, 500, 60000, (4000, 500, 1024), 0),
])
def test_long_inner_dimension_is_not_searched(m, n, k, tiles, beta):
    """No cut gains 3% here: at most the present blocks and a few cuts are walked through."""
    chunks = -(-k // tiles[2])
    walked, out = steps(m, n, k, tiles, beta)
    assert out == tiles + (0,)
    assert chunks <= walked <= 50 * chunks


@pytest.mark.parametrize("m,n,k,tiles,beta,first", [
    (1234, 4567, 1357, (1234, 4567, 1357), 0, 0),
    (10000, 10000, 10000, (5120, 5120, 5000), 1, 624),
    (16000, 16000, 12000, (8064, 8064, 6000), 0, 744),
])
def test_search_of_calls_that_gain(m, n, k, tiles, beta, first):
    walked, out = steps(m, n, k, tiles, beta, first)
    assert out[:2] != tiles[:2] and walked <= 8000
