"""tcx_ncc on series scaled by powers of two: the transforms, norms and
products scale exactly, so every value keeps its bits, whether it is divided
or multiplied by the reciprocal and corrected (the denominator's range from
2^-26 to 2^50, crossed here at both ends), through the C ABI."""
import numpy as np
import pytest

import timesc as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [5, 40, 250, 500, 1000, 3000])
def test_power_of_two_scales(ctx, m):
    X, _ = T.generate(3 * m, 7, m, 3, 0.3)
    X = (X - X.mean(1, keepdims=True)).astype(np.float32)
    X /= np.linalg.norm(X, axis=1, keepdims=True).astype(np.float32)
    C = X[4:]

    def ncc(ex, ec):
        d, dc = ctx.to_device(np.ldexp(X, ex)), ctx.to_device(np.ldexp(C, ec))
        try:
            return ctx.ncc(d, dc)
        finally:
            d.free()
            dc.free()

    ref = ncc(0, 0)  # denominators about 1
    assert np.abs(ref).max() <= 1.0 + 1e-5
    for ex, ec in ((-13, -12), (-13, -13), (-13, -14), (-20, -20), (-30, -19), (-30, -22),
                   (25, 24), (25, 25), (25, 26), (30, 28)):
        assert np.array_equal(ncc(ex, ec), ref), (ex, ec)
