"""The prefill GEMM's block map (gemm.h), on the CPU: every (row group, token
tile) pair runs in exactly one block and the eight XCDs get equal shares, for
every count of row groups and tiles up to the 256 blocks of a launch's first
round and for launches of more tiles; and the plan of a single matrix."""
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


def _plan(hip, n_out, n_in, T):
    f = hip._Z16draco_gemmh_planiiiPi
    f.restype, f.argtypes = None, [ct.c_int] * 3 + [ct.POINTER(ct.c_int)]
    out = (ct.c_int * 4)()
    f(n_out, n_in, T, out)
    return list(out)


@pytest.mark.parametrize("n_in", [32, 256, 960, 1056, 2048, 2304, 4096, 6400, 8192, 8224, 14336, 16384])
def test_plan_covers_the_rows(hip, n_in):
    for n_out in (1, 33, 320, 512, 2048, 4096, 8192, 14336, 128256):
        for T in (1, 2, 32, 33, 64, 100, 256, 289, 1024, 4096, 9000):
            nsb, rpb, ksp, pps = _plan(hip, n_out, n_in, T)
            nb, rts, ntt = -(-n_in // 256), -(-n_out // 32), -(-T // 32)
            passes, rg = -(-nb // nsb), -(-rts // (rpb * (8 // nsb)))
            assert nsb in (4, 8) and (ksp - 1) * pps < passes <= ksp * pps  # every split has a pass
            assert rg * ntt * ksp <= 256 or (rg == 1 and ksp == 1)           # one block a CU
            assert ksp == 1 or ksp * T * n_out <= 1 << 25


@pytest.mark.parametrize("n_out,n_in,T", [(512, 14336, 1), (512, 8192, 128), (2048, 8192, 32), (4096, 14336, 16),
                                          (1024, 14336, 64)])
def test_long_rows_of_few_tiles_use_the_chip(hip, n_out, n_in, T):
    """Products whose (row, token) tiles are at most half the CUs and whose
    rows take four passes or more: a block each ran them in series, 1.1 to 1.8
    times the time of a split over blocks."""
    _, rpb, ksp, pps = _plan(hip, n_out, n_in, T)
    tiles = -(-n_out // 32) * -(-T // 32)
    assert rpb == 1 and tiles * ksp > 128 or pps == 1
