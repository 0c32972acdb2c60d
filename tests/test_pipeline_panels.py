"""Block sizes of host-to-host calls to which the host link matters (pipeline_panels in
tiled-mm_amd/csrc/tmm_plan.cpp), on the CPU: what must stay as it is stays, and cuts lie on the
kernels' grid and inside the work pool."""
import ctypes

import pytest

import tiledmm

RATE = 70e12  # FP64 flop/s


def panels(m, n, k, tiles, beta=0, first=0, budget=0, es=8, rate=RATE):
    L = ctypes.CDLL(tiledmm.HOST_PATH)
    i, l, d = ctypes.c_int, ctypes.c_long, ctypes.c_double
    L.tmmh_pipeline_panels.argtypes = [i] * 8 + [l, i, d, ctypes.POINTER(i)]
    out = (i * 4)()
    assert L.tmmh_pipeline_panels(m, n, k, beta, *tiles, first, budget, es, rate, out) == 0
    return tuple(out)


@pytest.mark.parametrize("m,n,k,tiles,first", [
    (500, 500, 500, (500, 500, 500), 0),              # 6 MB: copies cost more apart
    (40000, 40000, 40000, (8064, 8064, 8000), 1000),  # products take 2.7 times the link's time
    (3000, 3000, 0, (3000, 3000, 1), 0),              # no product
])
def test_blocks_that_stay(m, n, k, tiles, first):
    assert panels(m, n, k, tiles, beta=1, first=first) == tiles + (first,)


@pytest.mark.parametrize("m,n,k,tiles,beta,first", [
    (1976, 2631, 2728, (1976, 2631, 2728), 0, 0),
    (1234, 4567, 1357, (1234, 4567, 1357), 0, 0),
    (4000, 300, 4000, (4000, 300, 4000), 1, 0),
    (10000, 10000, 10000, (5120, 5120, 5000), 1, 624),
    (16000, 16000, 12000, (8064, 8064, 6000), 0, 744),
])
def test_cuts(m, n, k, tiles, beta, first):
    tm, tn, tk, fc = panels(m, n, k, tiles, beta, first)
    assert (tm, tn) != tiles[:2] and tm <= tiles[0] and tn <= tiles[1] and tk <= tiles[2]
    for t, whole in ((tm, tiles[0]), (tn, tiles[1])):
        assert t == whole or (t % 64 == 0 and t >= 128)
    assert (tk, fc) == (tiles[2], first) or (fc == 0 and tk % 8 == 0 and 2 * tk >= k)
    blocks = -(-m // tm) * -(-n // tn)
    assert 1 < blocks <= 128
    # a work pool that holds the present blocks only just: the cut ones must fit it too
    need = lambda a, b, c: 2 * c * (-(-m // a) * a + -(-n // b) * b) + (1 + beta) * -(-m // a) * a * -(-n // b) * b
    budget = need(*tiles)
    got = panels(m, n, k, tiles, beta, first, budget=budget)
    assert got == tiles + (first,) or need(*got[:3]) <= budget
