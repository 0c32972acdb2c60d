"""Size of the pieces in which pageable memory passes through the staging slots (stage_piece in tiled-mm_amd/csrc/tmm_plan.hpp):
small enough for a small call's pieces to overlap, and no smaller, since every piece waits for the host's threads once."""
import ctypes

import pytest

import tiledmm

MIB = 1 << 20


def piece(call_bytes, whole):
    f = ctypes.CDLL(tiledmm.HOST_PATH).tmmh_stage_piece
    f.argtypes, f.restype = [ctypes.c_long, ctypes.c_int], ctypes.c_long
    return f(call_bytes, whole)


@pytest.mark.parametrize("whole,parts", [(1, 64), (0, 8)])
@pytest.mark.parametrize("call_bytes", [0, 1, MIB, 63 * MIB, 64 * MIB, 65 * MIB, 200 * MIB, 917 * 10**6, 1 << 30, 1 << 34, 1 << 40])
def test_pieces(call_bytes, whole, parts):
    p = piece(call_bytes, whole)
    assert 8 * MIB <= p <= 128 * MIB
    pieces = -(-call_bytes // p)
    if p < 128 * MIB:
        assert pieces <= parts + 1  # and what the division leaves
    if call_bytes >= 8 * parts * MIB:
        assert pieces >= parts


def test_calls_of_several_blocks_keep_large_pieces():
    """A call of several blocks that moves 917 MB in and 633 MB out: 8 pieces each way, not 64."""
    assert piece(917 * 10**6, 0) == 917 * 10**6 // 8 and piece(633 * 10**6, 0) == 633 * 10**6 // 8
    assert piece(2 * 10**9, 0) == 128 * MIB
