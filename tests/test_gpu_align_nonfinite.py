"""tcx_sbd_align on rows whose correlation is no number (a NaN, an infinity,
a norm that overflows) or has no norm: NumPy's argmax over them is index 0,
shift 1 - m, as tcx_assign gives it, for the row and for the one that shares
its transform, for every transform geometry, through the C ABI."""
import numpy as np
import pytest

import oracle_py as O
import timesc as T

pytestmark = pytest.mark.gpu

# every FFT length's group width, below, at and above one wave
LENGTHS = [3, 6, 12, 24, 50, 100, 200, 400, 900, 1500, 3000]


def _rows(m, n):
    X, _ = T.generate(17 * m, n + 1, m, 2, 0.3)
    Z = O.zscore(X.astype(np.float64)).astype(np.float32)
    return Z[:n].copy(), Z[n:].copy()


def _run(ctx, X, C, convention):
    d, dc = ctx.to_device(X), ctx.to_device(C)
    try:
        shift = ctx.assign(d, dc)[2]
        ctx.sbd_align(d, dc, convention)
        return d.numpy(), shift
    finally:
        d.free()
        dc.free()


@pytest.mark.parametrize("convention", [T.CONV_CPU, T.CONV_KSHAPE])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("m", LENGTHS)
def test_rows_that_are_no_numbers(ctx, m, bad, convention):
    X, C = _rows(m, 7)
    clean, _ = _run(ctx, X, C, convention)
    X[1, m // 2] = bad  # the second of a pair
    X[4, 0] = bad       # the first of a pair
    X[6, m // 3] = bad  # a row without a partner
    got, shift = _run(ctx, X, C, convention)
    for i in range(7):
        if i in (2, 3):
            assert np.array_equal(got[i], clean[i])
            continue
        want = np.zeros(m, np.float32)
        want[0] = X[i, m - 1]
        assert shift[i] == 1 - m and np.array_equal(got[i], want, equal_nan=True), i


@pytest.mark.parametrize("scale", [1e25, 1e-30])
@pytest.mark.parametrize("m", LENGTHS)
def test_norms_past_the_range(ctx, m, scale):
    """Pairs of rows whose squares overflow or vanish."""
    X, C = _rows(m, 5)
    X[2:] *= np.float32(scale)
    got, shift = _run(ctx, X, C, T.CONV_CPU)
    for i in range(5):
        assert np.array_equal(
            got[i], O.roll_zeropad(X[i].astype(np.float64), int(shift[i])).astype(np.float32)), i
