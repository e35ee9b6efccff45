"""The refinement of a single fit: the plan of S made on the device or (when an
HBM budget has no room for the largest one) on the host, and the host's wait
for its results before the assignment (stop_on_collapse) or with it.  All of
them run the same kernels on the same plan, so the fits agree bit for bit, with
the clusters rerun through the eigenvector path too."""
import numpy as np
import pytest

import timesc as T

pytestmark = pytest.mark.gpu


def _fit(ctx, X, k, **kw):
    d = ctx.to_device(X)
    try:
        ctx.znorm(d, ddof=0)
        r = ctx.fit(d, k, max_iter=6, seed=3, labels_per_iter=True, **kw)
        r["workspace"] = ctx.workspace_bytes()
    finally:
        d.free()
    return r


# white noise of a few samples: small clusters of it now and then fail the
# power result's tests; k = 700 takes several tiles of the device's plan
@pytest.mark.parametrize("n,m,k,fallback", [
    (1, 5, 1, False), (40, 33, 3, False), (3000, 7, 700, True), (2500, 12, 300, True),
    (700, 300, 5, False), (20000, 130, 3, False), (300, 700, 260, False)])
def test_plans_and_waits_agree(ctx, n, m, k, fallback):
    rng = np.random.default_rng(n + m + k)
    X = rng.standard_normal((n, m)).astype(np.float32)
    ref = _fit(ctx, X, k)
    assert (ref["stats"]["fallbacks"] > 0) >= fallback
    need = ctx.fit_workspace_bound(n, m, k)
    with T.Context(0, need + X.nbytes + 4096) as small:
        host = _fit(small, X, k)
        assert host["workspace"] <= need
    # the collapse rule stops a fit with half of its clusters empty
    waits = _fit(ctx, X, k, stop_on_collapse=True)
    for name, got in (("host plan", host), ("waits", waits)):
        if got is waits and got["stats"]["collapsed"]:
            continue
        for f in ("labels", "centroids", "labels_per_iter"):
            assert np.array_equal(ref[f], got[f]), (name, f)
        for f in ("iterations", "sum_class", "power_steps_max", "fallbacks"):
            assert ref["stats"][f] == got["stats"][f], (name, f)
