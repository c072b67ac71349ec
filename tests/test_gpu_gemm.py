"""Prefill GEMM on the GPU: m5_gemm / m5_gemm_auto (src/m5/m5_gemm.c:249-272,
src/m5/m5_gemm_fused.c:231-241) vs the oracle's or_gemm (pinned as "equals
stacked GEMVs").  Bar: max|dY| <= 1e-5 * max|Y_ref| over the whole output.
"""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _case(code, T, n_out, n_in, seed):
    from dracohip import lib
    rng = np.random.default_rng(seed)
    W = lib.quantize(code, rng.standard_normal((n_out, n_in), dtype=np.float32) * np.float32(0.02))
    X = rng.standard_normal((T, n_in)).astype(np.float32)
    X[0, :7] = 0.0           # zeros, a large value and a tiny one in one super-block
    if n_in > 300:
        X[-1, 300] = 80.0
        X[-1, 301] = 1e-30
    return W, X


@pytest.mark.parametrize("code", [5, 4, 0, 3])
@pytest.mark.parametrize("T,n_out,n_in", [(1, 16, 256), (7, 40, 512), (37, 96, 2048), (256, 2048, 2048),
                                          (64, 8192, 2048), (100, 2048, 8192), (9, 48, 768),
                                          # the ragged last prefill chunk on the K-split products, 3 super-blocks
                                          # per row with n_out off the 16-row tile, n_in at the 16384 cap
                                          (191, 512, 2048), (191, 2048, 8192), (33, 1000, 768), (255, 130, 4096),
                                          (32, 16, 16384)])
def test_gemm_vs_oracle(hip, oracle, code, T, n_out, n_in):
    from dracohip import lib
    W, X = _case(code, T, n_out, n_in, T + n_out + code)
    Y = np.zeros((T, n_out), np.float32)
    wbuf = np.zeros(8, np.float32)
    assert hip.m5_gemm(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y), lib.pf(wbuf)) == 0, lib.last_error()
    ref = np.zeros_like(Y)
    assert oracle.lib.or_gemm(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(ref)) == 0
    assert rel_err(Y, ref) <= TOL
    Y2 = np.zeros_like(Y)
    assert hip.m5_gemm_auto(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y2)) == 0
    assert np.array_equal(Y, Y2)


def test_gemm_equals_stacked_gemv(hip):
    from dracohip import lib
    W, X = _case(5, 24, 512, 2048, 3)
    Y = np.zeros((24, 512), np.float32)
    assert hip.m5_gemm_auto(5, lib.pf(X), lib.pu8(W), 24, 512, 2048, lib.pf(Y)) == 0
    G = np.stack([lib.gemv(5, X[t], W, 512, 2048) for t in range(24)])
    assert rel_err(Y, G) <= TOL


def test_gemm_unsupported_code_returns_minus_one(hip):
    from dracohip import lib
    X = np.zeros((2, 256), np.float32)
    W = np.zeros(4 * 110, np.uint8)
    Y = np.zeros((2, 4), np.float32)
    assert hip.m5_gemm_auto(2, lib.pf(X), lib.pu8(W), 2, 4, 256, lib.pf(Y)) == -1   # IQ3_S: caller falls back


@pytest.mark.parametrize("fname,code", [("q4k", 5), ("q6k", 4), ("q80", 0), ("q5k", 3)])
def test_fused_entries_equal_gemm_auto(hip, fname, code):
    """The per-format entries src/qwen35_prefill.py:76-80 looks up
    (src/m5/m5_gemm_fused.c:211-228) compute what m5_gemm_auto does."""
    from dracohip import lib
    T, n_out, n_in = 40, 96, 512
    W, X = _case(code, T, n_out, n_in, 77 + code)
    Y = np.full((T, n_out), np.nan, np.float32)
    getattr(hip, f"m5_gemm_{fname}")(lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y))
    Y2 = np.zeros_like(Y)
    assert hip.m5_gemm_auto(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y2)) == 0
    assert np.array_equal(Y, Y2)


@pytest.mark.parametrize("fname", ["iq4xs", "iq3s"])
def test_fused_entries_not_carried_leave_nan(hip, fname):
    from dracohip import lib
    X = np.ones((2, 256), np.float32)
    W = np.zeros(4 * 136, np.uint8)
    Y = np.zeros((2, 4), np.float32)
    getattr(hip, f"m5_gemm_{fname}")(lib.pf(X), lib.pu8(W), 2, 4, 256, lib.pf(Y))
    assert np.isnan(Y).all()



@pytest.mark.parametrize("T,n_out,n_in", [(1, 1, 32), (2, 33, 288), (31, 960, 960), (33, 17, 1056), (64, 320, 2528),
                                          (5, 16, 2080), (65, 2560, 736), (32, 31, 4064)])
def test_gemm_q8_ragged_rows_vs_oracle(hip, oracle, T, n_out, n_in):
    """Q8_0 rows that end inside a 256-value super-block (the last one padded
    with zero activations and zero scales), row counts off the 32-row tile.
    Bound: 1e-5 of the row dots' scale sum|w||x| (one-row and one-block
    products cancel)."""
    from dracohip import lib
    W, X = _case(0, T, n_out, n_in, T + n_out + n_in)
    Y = np.full((T, n_out), np.nan, np.float32)
    hip.m5_gemm_q80(lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y))
    ref = np.zeros_like(Y)
    assert oracle.lib.or_gemm(0, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(ref)) == 0
    blk = W.reshape(n_out, n_in // 32, 34)
    w = np.abs(blk[:, :, 2:].view(np.int8).astype(np.float64)) * np.abs(blk[:, :, :2].copy().view(np.float16).astype(np.float64))
    scale = np.abs(X.astype(np.float64)) @ w.reshape(n_out, n_in).T
    assert np.all(np.abs(Y.astype(np.float64) - ref) <= 1e-5 * scale + 1e-30)


def test_gemm_q8_nonfinite_tokens_stay_apart(hip, oracle):
    """An infinite or NaN activation makes its own token non-finite where the
    reference's fp32 dots are, and leaves every other token as it was."""
    from dracohip import lib
    T, n_out, n_in = 40, 70, 960
    W, X = _case(0, T, n_out, n_in, 9)
    X[3, 500], X[3, 17], X[36, 959] = np.inf, -np.inf, np.nan
    X[7, 11] = -np.inf
    Y = np.zeros((T, n_out), np.float32)
    hip.m5_gemm_q80(lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y))
    ref = np.zeros_like(Y)
    assert oracle.lib.or_gemm(0, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(ref)) == 0
    assert np.array_equal(np.isnan(Y), np.isnan(ref))
    assert np.array_equal(Y[np.isinf(ref)], ref[np.isinf(ref)])
    ok = np.isfinite(ref)
    assert ok.sum() >= (T - 3) * n_out and rel_err(Y[ok], ref[ok]) <= TOL


@pytest.mark.parametrize("code", [5, 4, 0, 3])
@pytest.mark.parametrize("T,n_out,n_in", [(33, 16, 256), (65, 100, 1024), (1, 33, 2304), (256, 4112, 1024)])
def test_gemm_slots_and_streams_vs_oracle(hip, oracle, code, T, n_out, n_in):
    """One, four and nine super-blocks a row (idle slots, a short second pass)
    and the two-stream form (short rows, many row tiles, an odd last tile)."""
    from dracohip import lib
    W, X = _case(code, T, n_out, n_in, 3 * T + n_out + code)
    Y = np.full((T, n_out), np.nan, np.float32)
    assert hip.m5_gemm_auto(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y)) == 0
    ref = np.zeros_like(Y)
    assert oracle.lib.or_gemm(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(ref)) == 0
    assert rel_err(Y, ref) <= TOL


@pytest.mark.parametrize("n_out,n_in", [(960, 960), (320, 2560), (64, 4064)])
def test_gemm_q8_errors_have_no_common_sign(hip, n_out, n_in):
    """The rounding errors of a Q8_0 product against 64 bits average out over
    tokens and rows.  Bound: 5e-9 of the result's rms, some three times the spread of
    the mean of 64 x 64 independent errors of 1.2e-7 (a GEMV per token: 3e-10
    over 256 x 960; a sum rounded downwards throughout: 3e-8 to 7e-8)."""
    from dracohip import lib
    T = 64
    rng = np.random.default_rng(n_out + n_in)
    W = lib.quantize(0, rng.standard_normal((n_out, n_in), dtype=np.float32) * np.float32(0.02))
    X = rng.standard_normal((T, n_in)).astype(np.float32)
    Y = np.zeros((T, n_out), np.float32)
    hip.m5_gemm_q80(lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y))
    blk = W.reshape(n_out, n_in // 32, 34)
    w = blk[:, :, 2:].view(np.int8).astype(np.float64) * blk[:, :, :2].copy().view(np.float16).astype(np.float64)
    ref = X.astype(np.float64) @ w.reshape(n_out, n_in).T
    assert abs(np.mean(Y - ref)) <= 5e-9 * np.sqrt(np.mean(ref ** 2))


@pytest.mark.parametrize("code", [5, 4, 0, 3])
@pytest.mark.parametrize("T,n_out,n_in", [(290, 4200, 256), (1100, 100, 512), (2050, 70, 512), (8200, 33, 256)])
def test_gemm_long_launches_vs_oracle(hip, oracle, code, T, n_out, n_in):
    """More than 256 tokens: row groups that do not divide by the eight XCDs,
    fewer than eight of them, one, and more token tiles than a round of blocks."""
    from dracohip import lib
    W, X = _case(code, T, n_out, n_in, T + n_out + code)
    Y = np.full((T, n_out), np.nan, np.float32)
    assert hip.m5_gemm_auto(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y)) == 0
    ref = np.zeros_like(Y)
    assert oracle.lib.or_gemm(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(ref)) == 0
    assert rel_err(Y, ref) <= TOL


@pytest.mark.parametrize("code", [5, 4, 0, 3])
@pytest.mark.parametrize("T,n_out,n_in", [(1, 129, 6400), (40, 511, 14336), (33, 2048, 4352), (256, 4100, 8192)])
def test_gemm_split_rows_vs_oracle(hip, oracle, code, T, n_out, n_in):
    """Rows of several passes whose passes run in blocks of their own: a last
    split with fewer super-blocks, results that are no multiple of four (the
    scalar sum), several row tiles a block."""
    from dracohip import lib
    W, X = _case(code, T, n_out, n_in, T + n_out + code)
    Y = np.full((T, n_out), np.nan, np.float32)
    assert hip.m5_gemm_auto(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y)) == 0
    ref = np.zeros_like(Y)
    assert oracle.lib.or_gemm(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(ref)) == 0
    assert rel_err(Y, ref) <= TOL


@pytest.mark.parametrize("code", [0, 3])
@pytest.mark.parametrize("T,n_out,n_in", [(1, 320, 1024), (2, 4096, 4096), (3, 512, 2048), (1, 33, 256)])
def test_short_gemm_is_stacked_gemvs(hip, code, T, n_out, n_in):
    """One and two tokens of Q8_0 and Q5_K, and three of a small matrix, take
    the GEMV per token (the operand image and the 32-token tile cost more):
    the same bits as m5_gemv's."""
    from dracohip import lib
    W, X = _case(code, T, n_out, n_in, T + n_out)
    Y = np.full((T, n_out), np.nan, np.float32)
    assert hip.m5_gemm_auto(code, lib.pf(X), lib.pu8(W), T, n_out, n_in, lib.pf(Y)) == 0
    assert np.array_equal(Y, np.stack([lib.gemv(code, X[t], W, n_out, n_in) for t in range(T)]))
