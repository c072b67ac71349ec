"""The prefill GEMM's block map (gemm.h), on the CPU: every (row group, token
tile) pair runs in exactly one block and the eight XCDs get equal shares, for
every count of row groups and tiles up to the 256 blocks of a launch's first
round and for launches of more tiles."""
import ctypes as ct

import pytest


def _fns(hip):
    blocks, place = hip._Z18draco_gemmh_blocksii, hip._Z17draco_gemmh_placeiii
    blocks.restype, blocks.argtypes = ct.c_uint, [ct.c_int] * 2
    place.restype, place.argtypes = ct.c_int, [ct.c_int] * 3
    return blocks, place


def _check(hip, M, m):
    blocks, place = _fns(hip)
    n = blocks(M, m)
    at = [place(M, m, b) for b in range(n)]
    assert sorted(a for a in at if a >= 0) == list(range(M * m)), (M, m)
    per = [sum(a >= 0 for a in at[x::8]) for x in range(8)]
    assert n == 8 * -(-M * m // 8) and max(per) == n // 8, (M, m, per)
    for x in range(8):  # the majors of whole eights stay on one XCD
        assert all(a // m % 8 == x for a in at[x::8] if 0 <= a < (M & ~7) * m)


@pytest.mark.parametrize("M", [1, 2, 3, 7, 8, 9, 12, 16, 28, 63, 64, 82, 104, 255, 256])
def test_blocks_cover_the_pairs_evenly(hip, M):
    for m in range(1, max(1, 256 // M) + 1):
        _check(hip, M, m)


@pytest.mark.parametrize("M,m", [(1, 257), (2, 300), (9, 129), (300, 3), (1000, 1), (21, 40)])
def test_more_than_one_round(hip, M, m):
    _check(hip, M, m)
