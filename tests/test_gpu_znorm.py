"""z-normalization at the edges of its forms (16 lanes or a wave per row, the
vectors a lane holds, the values after the last vector, rows longer than a
wave holds) and on rows of NaN, infinities, zeros and huge or tiny values,
against the FP64 oracle, through the C ABI."""
import numpy as np
import pytest

import oracle_py as O
import timesc as T

pytestmark = pytest.mark.gpu

# one float rounding of the FP64 value (relative 2^-24), the sums' order 1e-14
RTOL = 2.0 ** -23


def _check(ctx, X, ddof):
    d = ctx.to_device(X)
    try:
        ctx.znorm(d, ddof=ddof)
        got = d.numpy()
    finally:
        d.free()
    ref = O.zscore(X.astype(np.float64), ddof=ddof)
    assert np.all(np.abs(got - ref) <= RTOL * np.abs(ref) + 1e-12)


@pytest.mark.parametrize("ddof", [0, 1])
@pytest.mark.parametrize("m", [2, 3, 4, 5, 63, 127, 128, 129, 131, 509, 512, 513, 1023, 1025, 2047,
                               2052, 4095, 4096, 4097, 5000])
def test_forms(ctx, m, ddof):
    rng = np.random.default_rng(m)
    X = (rng.standard_normal((37, m)) * 3 + 1).astype(np.float32)
    X[5] = 2.0      # constant: zeros
    X[6] = 0.0
    X[7] *= 1e30    # sums of squares beyond float, not beyond double
    X[8] *= 1e-30
    _check(ctx, X, ddof)


@pytest.mark.parametrize("m", [6, 128, 365, 512, 4096])
def test_rows_that_are_not_numbers(ctx, m):
    """A row with a NaN or an infinity has no mean: zeros, and its
    neighbours in the same wave keep their values."""
    rng = np.random.default_rng(m)
    X = rng.standard_normal((21, m)).astype(np.float32)
    ref = O.zscore(X.astype(np.float64))
    for row, v in ((3, np.nan), (4, np.inf), (16, -np.inf), (20, np.nan)):
        X[row, m // 2] = v
        ref[row] = 0.0
    d = ctx.to_device(X)
    try:
        ctx.znorm(d)
        got = d.numpy()
    finally:
        d.free()
    assert np.all(np.abs(got - ref) <= RTOL * np.abs(ref) + 1e-12)


@pytest.mark.parametrize("m", [8, 128, 512])
def test_rows_off_a_vector_boundary(ctx, m):
    """A base pointer at 4 bytes past a 16-byte boundary."""
    X = np.random.default_rng(m).standard_normal(19 * m + 1).astype(np.float32)
    d = ctx.to_device(X)
    try:
        T.check(ctx.lib.tcx_znorm(ctx.h, d.ptr + 4, 19, m, 0))
        got = d.numpy()
    finally:
        d.free()
    assert got[0] == X[0]
    ref = O.zscore(X[1:].reshape(19, m).astype(np.float64))
    assert np.all(np.abs(got[1:].reshape(19, m) - ref) <= RTOL * np.abs(ref) + 1e-12)
