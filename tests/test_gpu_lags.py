"""The lag maximum where no lag reaches the circular wrap's values: positive
series against negative centroids, so that every correlation is below the
zeros between the positive and the negative lags and the maximum is the
smallest overlap, for every transform geometry, through the C ABI."""
import numpy as np
import pytest

import oracle_py as O
import timesc as T

pytestmark = pytest.mark.gpu

# every FFT length's group width; n odd, so the last series has no partner
LENGTHS = [3, 6, 12, 24, 50, 100, 200, 400, 900, 1500, 3000]


def _case(m):
    """x[0] = 0.5 against the last value of a centroid of about -1 is the one
    overlap below 0.75 in size, every other lag's sum is at least 0.9 below
    zero: a gap of 0.15 / (|x| |c|) >= 0.15 / (2 m) = 2.5e-5 in the NCC."""
    rng = np.random.default_rng(m)
    X = rng.uniform(1.0, 1.5, (7, m)).astype(np.float32)
    X[:, 0] = 0.5
    C = -rng.uniform(0.9, 1.1, (3, m)).astype(np.float32)
    return X, C


@pytest.mark.parametrize("dmat", [False, True])
@pytest.mark.parametrize("m", LENGTHS)
def test_all_correlations_negative(ctx, m, dmat):
    X, C = _case(m)
    d, dc = ctx.to_device(X), ctx.to_device(C)
    try:
        out = ctx.assign(d, dc, dmat=dmat)
    finally:
        d.free()
        dc.free()
    lab, dist, sh, odm = O.assign(X.astype(np.float64), C.astype(np.float64), dmat=True)
    got = odm[np.arange(len(X)), out[0]]
    assert np.abs(got - dist).max() <= 2e-6  # the oracle's label up to a tie
    assert np.abs(out[1] - dist).max() <= 2e-6
    assert np.array_equal(out[2], np.full(len(X), 1 - m))
    if dmat:
        assert np.abs(out[3] - odm).max() <= 2e-6


@pytest.mark.parametrize("convention", [T.CONV_CPU, T.CONV_KSHAPE])
@pytest.mark.parametrize("m", LENGTHS)
def test_align_all_correlations_negative(ctx, m, convention):
    X, C = _case(m)
    d, dc = ctx.to_device(X), ctx.to_device(C[:1])
    try:
        ctx.sbd_align(d, dc, convention)
        got = d.numpy()
    finally:
        d.free()
        dc.free()
    for i in range(len(X)):
        s = O.align_shift(X[i].astype(np.float64), C[0].astype(np.float64), convention)
        assert abs(s) == m - 1
        assert np.array_equal(got[i], O.roll_zeropad(X[i].astype(np.float64), s).astype(np.float32))
