"""The residue of an int32 sum in the epilogue of the INT8 product kernel (residue_of_sum in
tiled-mm_amd/csrc/tmm_ozaki.hip), modelled in FP32 on the CPU: for every modulus and every value that
the folded sum t can take (and so for every sum up to 2^30 in magnitude) it must be the exact
remainder in [0, modulus)."""
import numpy as np
import pytest

from crt_model import MODULI


@pytest.mark.parametrize("m", MODULI)
def test_residue_of_every_folded_sum(m):
    c16 = 65536 % m
    c16 = c16 - m if c16 > m // 2 else c16
    assert abs(c16) <= 128
    top = 16384 * 128 + 65535  # |hi| <= 2^14 for |sum| <= 2^30, lo < 2^16
    inv = np.float32(1) / np.float32(m)
    for lo in range(-top, top + 1, 1 << 20):
        t = np.arange(lo, min(lo + (1 << 20), top + 1))
        f = t.astype(np.float32)
        assert np.array_equal(f.astype(np.int64), t)
        # fma(f, inv, inv / 2): the products and the sum fit 53 bits, one rounding to FP32
        q = np.floor((f.astype(np.float64) * np.float64(inv) + np.float64(np.float32(0.5) * inv)).astype(np.float32))
        r = f.astype(np.float64) - q.astype(np.float64) * m
        assert np.array_equal(r.astype(np.int64), t % m)


def test_folding_keeps_the_residue():
    rng = np.random.default_rng(5)
    s = np.concatenate([rng.integers(-2 ** 30, 2 ** 30 + 1, 100000), [-2 ** 30, -1, 0, 1, 65535, 65536, 2 ** 30]])
    for m in MODULI:
        c16 = 65536 % m
        c16 = c16 - m if c16 > m // 2 else c16
        t = (s >> 16) * c16 + (s & 0xffff)
        assert np.array_equal(t % m, s % m) and np.abs(t).max() <= 16384 * 128 + 65535
