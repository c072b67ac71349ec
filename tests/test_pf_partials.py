"""The chunk attention's partial rows (prefill.hip), on the CPU: the host
function that sizes their buffer.  The kernels store and load a row's o as
float4, so a row must be a whole number of 16-byte units and hold o, m and l."""
import ctypes as ct

import pytest


@pytest.mark.parametrize("hd", [64, 128, 256])
def test_partial_rows_are_16_byte_units(hip, hd):
    f = hip._Z14pf_part_floatsiiii  # size_t pf_part_floats(int NH, int T, int HD, int nspl)
    f.restype, f.argtypes = ct.c_size_t, [ct.c_int] * 4
    row = f(1, 1, hd, 1)
    assert row % 4 == 0 and row >= hd + 2
    assert f(3, 5, hd, 7) == 3 * 5 * 7 * row
