"""The plan of S under an HBM budget: made on the device, with room for the
largest plan, wherever the budget is at least what tcx_fit_workspace_bound
says; made on the host, with what it needs, where only the largest plan does
not fit.  Which plan was made shows in the workspace held; the results are the
same bit for bit."""
import numpy as np
import pytest

import timesc as T

pytestmark = pytest.mark.gpu


def _fit(ctx, X, k, labels):
    d = ctx.to_device(X)
    try:
        ctx.znorm(d, ddof=0)
        r = ctx.fit(d, k, max_iter=4, seed=3, init_labels=labels, labels_per_iter=True)
        r["workspace"] = ctx.workspace_bytes()
    finally:
        d.free()
    return r


# every series in one cluster at first, so that the plan needed is far smaller
# than the largest; a resident, a multi-block and a two-launch power stage
@pytest.mark.parametrize("n,m,k", [(60, 130, 40), (90, 300, 40), (50, 1100, 12)])
def test_host_plan_only_without_room(ctx, n, m, k):
    X, _ = T.generate(n + m, n, m, 3, 0.3)
    labels = np.zeros(n, np.int32)
    with T.Context(0) as free:
        ref = _fit(free, X, k, labels)
        need = free.fit_workspace_bound(n, m, k)
    user = X.nbytes + 4096
    with T.Context(0, need + user) as bound:  # the documented budget
        dev = _fit(bound, X, k, labels)
    assert dev["workspace"] == ref["workspace"] <= need
    # partials of k clusters of ceil(m / 128)^2 upper blocks of 128 x 128 floats
    u = -(-m // 128)
    part = k * u * (u + 1) // 2 * 128 * 128 * 4
    with T.Context(0, ref["workspace"] - part // 2 + user) as tight:
        host = _fit(tight, X, k, labels)
    assert host["workspace"] <= ref["workspace"] - part // 2
    for got in (dev, host):
        for f in ("labels", "centroids", "labels_per_iter"):
            assert np.array_equal(ref[f], got[f]), f


def test_exchange_words_leave_room_for_later_refinements():
    """From the second iteration on the grouping takes more keys (distance
    bins, about 40 KB here).  A budget with room for that runs the fit, also
    where it has room for the exchange words of the many-block Lanczos (226 KB
    a launch), but not for both: the next form runs then."""
    n, m, k = 300, 700, 30
    X, _ = T.generate(3, n, m, 8, 0.4)

    def accepted(budget, iters):
        with T.Context(0, budget) as c:
            d = c.to_device(X)
            try:
                c.fit(d, k, max_iter=iters, seed=1)
            except T.TimescError:
                return False
            return c.workspace_bytes() + X.nbytes <= budget

    lo, hi = 0, 1 << 28
    while hi - lo > 256:  # the least budget of one iteration
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if accepted(mid, 1) else (mid, hi)
    for more in range(64 << 10, 400 << 10, 12 << 10):
        assert accepted(hi + more, 3), more
