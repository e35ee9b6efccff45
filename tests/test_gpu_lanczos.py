"""The resident Lanczos (one block per cluster, matrix in registers, orders
up to 256) at the edges of its register splits, in both of its forms, and
past its basis rows in LDS, against the FP64 oracle, through the C ABI."""
import numpy as np
import pytest

import oracle_py as O
import timesc as T
from parity import CENT_RTOL, centroid_errors, rel_l2

pytestmark = pytest.mark.gpu


def _extract(ctx, X, labels, k):
    Z = O.zscore(X.astype(np.float64)).astype(np.float32)
    C0 = np.zeros((k, X.shape[1]), np.float32)
    d, dl, dc = ctx.to_device(Z), ctx.to_device(labels), ctx.to_device(C0)
    try:
        ctx.extract_shape(dl, d, None, dc, it=1)
        got = dc.numpy()
    finally:
        for a in (d, dl, dc):
            a.free()
    ref, _, _ = O.refine(Z.astype(np.float64), labels, C0.astype(np.float64), seed=0, it=1)
    return got, ref


@pytest.mark.parametrize("m", [2, 15, 16, 63, 64, 65, 127, 128, 129, 255, 256, 257])
def test_s_form_at_the_register_splits(ctx, m):
    X, y = T.generate(40 + m, 600, m, 3, 0.3)
    got, ref = _extract(ctx, X, y, 3)
    assert max(centroid_errors(got, ref)) <= CENT_RTOL


@pytest.mark.parametrize("n", [1, 3, 61, 64, 65, 125, 128, 129, 253, 256, 257])
def test_gram_form_at_the_register_splits(ctx, n):
    """One cluster of n members shorter than m: order n rounded up to 4."""
    m = 512
    X, _ = T.generate(90 + n, n, m, 1, 0.3)
    Z = O.zscore(X.astype(np.float64)).astype(np.float32)
    labels = np.zeros(n, np.int32)
    d = ctx.to_device(Z)
    try:
        with T.Batch(0, workers=1) as b:
            res = b.run([{"d": d, "k": 1, "max_iter": 1, "init_labels": labels, "seed": 3}],
                        grouped=True)[0]
    finally:
        d.free()
    ref, _, _ = O.refine(Z.astype(np.float64), labels, np.zeros((1, m)), seed=3, it=0)
    assert rel_l2(res["centroids"][0], ref[0]) <= CENT_RTOL


@pytest.mark.parametrize("m", [64, 128, 250])
def test_slow_convergence_uses_the_rows_past_lds(ctx, m):
    """White noise: a flat spectrum, so the check passes only after more
    steps than basis rows fit in LDS (or never, and the power steps take
    over).  The iterate M^I v0 then carries S's own rounding I-fold: FP32
    accumulation and split-BF16 products, each at most 2^-16 relative to the
    rows' norms, averaged over n members, about 2^-16 / sqrt(n) in S, so
    I 2^-16 / sqrt(n) at I = m <= 250, n = 4000: 6e-5; ten times that is
    allowed."""
    rng = np.random.default_rng(m)
    X = rng.standard_normal((4000, m)).astype(np.float32)
    labels = np.zeros(4000, np.int32)
    got, ref = _extract(ctx, X, labels, 1)
    assert rel_l2(got[0], ref[0]) <= 10 * m * 2.0 ** -16 / np.sqrt(4000.0)


@pytest.mark.parametrize("m,k", [(257, 1), (288, 3), (300, 24), (449, 5), (512, 16), (512, 17),
                                 (512, 33), (513, 2), (640, 8), (1023, 8), (1024, 8), (1024, 9)])
def test_blocks_of_one_cluster(ctx, m, k):
    """Orders above 256: 32 and 64 rows per block, 512 and 1024 columns, a
    last block with fewer rows, and the first sizes past what fits the device
    at once."""
    X, y = T.generate(7 * m + k, 40 * k + 3, m, k, 0.3)
    y[y == k // 2] = 0  # an empty cluster (k > 1)
    got, ref = _extract(ctx, X, y, k)
    assert max(centroid_errors(got, ref)) <= CENT_RTOL


@pytest.mark.parametrize("m,k", [(512, 17), (512, 65), (511, 40), (738, 22), (769, 31),
                                 (1024, 17)])
def test_blocks_in_several_launches(ctx, m, k):
    """More clusters than one launch holds (the first two take one, three; a
    device of 256 CUs), among them empty ones at the ends of launches: every
    cluster starts from its own vector."""
    X, y = T.generate(5 * m + k, 30 * k, m, k, 0.3)
    y[(y == 0) | (y == k - 1)] = k // 2
    got, ref = _extract(ctx, X, y, k)
    assert max(centroid_errors(got, ref)) <= CENT_RTOL


@pytest.mark.parametrize("m", [400, 900])
def test_blocks_slow_convergence(ctx, m):
    """White noise over many blocks: more steps than basis rows in LDS.  The
    tolerance is the one of the resident form above, at I = m."""
    X = np.random.default_rng(m).standard_normal((4000, m)).astype(np.float32)
    got, ref = _extract(ctx, X, np.zeros(4000, np.int32), 1)
    assert rel_l2(got[0], ref[0]) <= 10 * m * 2.0 ** -16 / np.sqrt(4000.0)
