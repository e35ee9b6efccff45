"""Assignments of few series in chunks of their centroids (tcx_assign) on
series and centroids that are no numbers, zero or past the range: the same
labels, distances and lags as the unsplit search (tcx_assign_noalloc), through
the C ABI."""
import numpy as np
import pytest

import oracle_py as O
import timesc as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("centroid", ["finite", "zero", "nan", "inf", "huge", "tiny"])
@pytest.mark.parametrize("m", [3, 17, 60, 128, 300, 700, 1500, 3000])
@pytest.mark.parametrize("n,k", [(9, 5), (40, 30)])
def test_chunked_equals_unsplit(ctx, m, n, k, centroid):
    X, _ = T.generate(m + n, n + k, m, 4, 0.3)
    Z = O.zscore(X.astype(np.float64)).astype(np.float32)
    X, C = Z[:n].copy(), Z[n:].copy()
    X[1, m // 2] = np.nan
    X[2, 1], X[3, 0] = np.inf, -np.inf
    X[4] = 0.0
    X[6:8] *= np.float32(1e25)  # a whole pair: its squares overflow
    X[8:10] *= np.float32(1e-30)
    j = k // 2
    if centroid == "zero":
        C[j] = 0.0
    elif centroid == "nan":
        C[j, 1] = np.nan
    elif centroid == "inf":
        C[j, 1] = np.inf
    elif centroid == "huge":
        C[j] *= np.float32(1e22)
    elif centroid == "tiny":
        C[j] *= np.float32(1e-30)
    d, dc = ctx.to_device(X), ctx.to_device(C)
    try:
        got = ctx.assign(d, dc)
        ref = ctx.assign(d, dc, noalloc=True)
    finally:
        d.free()
        dc.free()
    for a, b in zip(got, ref):
        assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f")
