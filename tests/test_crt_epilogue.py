"""The residue of an int32 sum in the epilogue of the INT8 product kernel (residues_of_sums in
tiled-mm_amd/csrc/tmm_ozaki.hip), modelled in integers on the CPU: for every modulus and sums up to 2^30
in magnitude it must be congruent to the sum and lie in [0, modulus], where the byte it is stored in
holds it (modulus 256: [0, 255])."""
import numpy as np
import pytest

from crt_model import MODULI


def _residue(s, m):
    magic = -(-2 ** 38 // m)
    assert magic < 2 ** 31  # a signed 32-bit factor
    h = (s * magic) >> 32
    q = (h & 0xffff) >> 6  # 16-bit lanes from here on
    return ((q * ((-m) & 0xffff) + (s & 0xffff)) & 0xffff) & 0xff


@pytest.mark.parametrize("m", MODULI)
def test_residue_of_a_sum(m):
    assert 129 <= m <= 256
    rng = np.random.default_rng(m)
    top = 2 ** 30
    near = (np.arange(-top // m, top // m + 1, 997, dtype=np.int64)[:, None] * m + np.arange(-2, 3)).ravel()
    ends = np.concatenate([np.arange(-top, -top + 5000), np.arange(-5000, 5000), np.arange(top - 5000, top + 1)])
    for s in (rng.integers(-top, top + 1, 2000000), near[np.abs(near) <= top], ends):
        r = _residue(s.astype(np.int64), m)
        assert np.array_equal(r % m, s % m)
        assert r.min() >= 0 and r.max() <= min(m, 255)
