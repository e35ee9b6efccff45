"""tcx_extract_shape without shifts on series without a correlation (a NaN or
an infinity in the row or in the row that shares its transform): such a series
has no lag, its shift lies past the row, and it adds nothing to its cluster.
The same centroids come out with those shifts given, through the C ABI."""
import numpy as np
import pytest

import oracle_py as O
import timesc as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("m", [12, 60, 200, 400, 900, 1500, 3000])
def test_rows_without_a_lag(ctx, m, bad):
    n, k = 41, 3
    X, _ = T.generate(m, n + k, m, k, 0.3)
    Z = O.zscore(X.astype(np.float64)).astype(np.float32)
    X, C = Z[:n].copy(), Z[n:].copy()
    labels = (np.arange(n) % k).astype(np.int32)
    lost = [6, 7, 20, 21, 40]  # pairs with one such row, and a row without a partner
    X[6, m // 2] = X[21, 0] = X[40, m - 1] = bad
    d, dl, dc = ctx.to_device(X), ctx.to_device(labels), ctx.to_device(C)
    finite = X.copy()
    finite[lost] = Z[lost]
    shift = np.empty(n, np.int32)
    for j in range(k):
        df, d1 = ctx.to_device(finite), ctx.to_device(C[j:j + 1])
        s = ctx.assign(df, d1)[2]
        shift[labels == j] = s[labels == j]
        df.free()
        d1.free()
    shift[lost] = 2 ** 31 - m
    ds = ctx.to_device(shift)
    out = []
    try:
        for given in (None, ds):
            dn = ctx.to_device(C)
            ctx.extract_shape(dl, d, given, dn)
            out.append(dn.numpy())
            dn.free()
    finally:
        for a in (d, dl, dc, ds):
            a.free()
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])
