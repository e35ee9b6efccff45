"""Every form of the Lanczos evaluation that a refinement can take above
order 256: many blocks per cluster with S in their registers (k_lz_multi), in
their LDS (k_lz_coop<true>, 512 < m <= 640 where the first would take several
launches) or in L2 (k_lz_coop<false>, m > 1024), and one block per cluster
(k_power_lanczos, many clusters), against the FP64 oracle; and what follows
when the blocks of a cluster give up waiting for each other."""
import numpy as np
import pytest

import oracle_py as O
import timesc as T
from parity import CENT_RTOL, assert_labels_match, centroid_errors, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(516, 16), (520, 16), (600, 16), (640, 17),   # S in LDS
                                 (1028, 3), (1100, 16),                        # S in L2
                                 (300, 200), (301, 150), (512, 150)])          # one block
def test_forms_against_the_oracle(ctx, m, k):
    X, y = T.generate(11 * m + k, 12 * k + 30, m, min(k, 24), 0.3)
    y = (np.arange(len(y)) % k).astype(np.int32) if k > 24 else y
    y[y == k // 2] = 0  # an empty cluster
    Z = O.zscore(X.astype(np.float64)).astype(np.float32)
    C0 = np.zeros((k, m), np.float32)
    d, dl, dc = ctx.to_device(Z), ctx.to_device(y), ctx.to_device(C0)
    try:
        ctx.extract_shape(dl, d, None, dc, it=1)
        got = dc.numpy()
    finally:
        for a in (d, dl, dc):
            a.free()
    ref, _, _ = O.refine(Z.astype(np.float64), y, C0.astype(np.float64), seed=0, it=1)
    assert max(centroid_errors(got, ref)) <= CENT_RTOL


@pytest.mark.parametrize("m,k", [(300, 24), (900, 8), (600, 16), (1500, 2)])
def test_forced_give_up_takes_the_power_iteration(ctx, monkeypatch, m, k):
    """A negative wait limit: every member gives up at its first wait, the
    clusters run the stepwise power iteration.  The next launch without the
    limit is not disturbed by what they left behind."""
    n = 150 * k
    X, _ = T.generate(m + k, n, m, k, 0.3)
    init = T.init_labels(m + k, n, k)

    def fit():
        d = ctx.to_device(X)
        try:
            ctx.znorm(d, ddof=0)
            r = ctx.fit(d, k, max_iter=1, seed=m + k)
            Z = d.numpy().astype(np.float64)
        finally:
            d.free()
        return r, Z

    ref, Z = fit()
    monkeypatch.setenv("TCX_LZ_COOP_TIMEOUT_US", "-1")
    forced, _ = fit()
    monkeypatch.delenv("TCX_LZ_COOP_TIMEOUT_US")
    again, _ = fit()
    assert ref["stats"]["power_steps_max"] < forced["stats"]["power_steps_max"] <= min(m, 1000)
    assert np.array_equal(again["centroids"], ref["centroids"])
    cent, _, _ = O.refine(Z, init, np.zeros((k, m)), seed=m + k, it=0)
    for r, what in ((forced, "forced"), (ref, "Lanczos")):
        errs = [rel_l2(a, b) for a, b in zip(r["centroids"], cent) if np.any(b)]
        assert max(errs) <= CENT_RTOL, (what, max(errs))
        olab, _, _, odm = O.assign(Z, r["centroids"].astype(np.float64), dmat=True)
        assert_labels_match(r["labels"], olab, odm, what=what)


def test_old_exchange_words_are_no_failure():
    """A launch of another shape leaves a tag (generation 1, a step) where the
    second cluster's failure word lies now; the generation reaches that value
    after 1024 launches and more, which must not make the cluster give up."""
    with T.Context(0) as c:
        steps = []
        # two exchange words per value and buffer; then two clusters of
        # 4 x 260 + 9 words each before the failure words
        for m, k, times in ((1000, 1, 1), (260, 2, 1400)):
            X, _ = T.generate(m + k, 20 * k, m, k, 0.3)
            d = c.to_device(O.zscore(X.astype(np.float64)).astype(np.float32))
            for _ in range(times):
                r = c.fit(d, k, max_iter=1, seed=5)
                steps.append(r["stats"]["power_steps_max"])
        assert set(steps[1:]) == {steps[1]}
