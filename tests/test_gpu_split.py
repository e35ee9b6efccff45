"""Assignments of few series with their centroids split into chunks over the
grid, and the shift of each series against one given centroid, through the
C ABI.  The chunked search of tcx_assign and the unsplit pruned search of
tcx_assign_noalloc form each distance alike, so they agree bit for bit."""
import numpy as np
import pytest

import oracle_py as O
import timesc as T
from parity import CENT_RTOL, centroid_errors

pytestmark = pytest.mark.gpu


def _data(seed, n, m, k):
    X, _ = T.generate(seed, max(n, k), m, min(k, 6), 0.3)
    Z = O.zscore(X.astype(np.float64)).astype(np.float32)
    C = Z[np.random.default_rng(seed).permutation(len(Z))[:k]].copy()
    return Z[:n].copy(), C


@pytest.mark.parametrize("m", [2, 17, 60, 128, 500, 1000, 2000, 3000])
@pytest.mark.parametrize("n,k", [(1, 4), (1, 65), (2, 7), (3, 5), (33, 24), (130, 11)])
def test_chunked_equals_unsplit(ctx, m, n, k):
    k = min(k, (1 << 18) // O.fft_size(m))  # what tcx_assign_noalloc's scratch holds
    Z, C = _data(m + n + k, n, m, k)
    C[k // 2] = 0.0      # zero centroid: distance exactly 1
    C[k - 1] = C[0]      # equal to the first, in another chunk: the smaller index wins
    if n > 2:
        Z[2] = 0.0       # distance 1 to everything: label 0
    d, dc = ctx.to_device(Z), ctx.to_device(C)
    try:
        got = ctx.assign(d, dc)
        ref = ctx.assign(d, dc, noalloc=True)
        full = ctx.assign(d, dc, dmat=True)
    finally:
        d.free()
        dc.free()
    for a, b, c in zip(got, ref, full):
        assert np.array_equal(a, b) and np.array_equal(a, c)
    dm = full[3]
    assert np.array_equal(dm.argmin(1), got[0]) and np.array_equal(dm.min(1), got[1])
    assert np.all(dm[:, k // 2] == 1.0) and np.array_equal(dm[:, 0], dm[:, k - 1])


def test_budget_without_room_for_chunks_is_not_split():
    m, k, n = 128, 24, 40
    Z, C = _data(5, n, m, k)
    with T.Context(0) as big:
        many, dc = big.to_device(np.tile(Z, (3000, 1))), big.to_device(C)
        big.assign(many, dc)  # enough series: one chunk
        base = big.workspace_bytes()
        few = big.to_device(Z)
        ref = big.assign(few, dc)
        assert big.workspace_bytes() > base
    with T.Context(0, budget=base + 4 * (n * m + k * m + 3 * n) + 100) as ctx:
        d, dc = ctx.to_device(Z), ctx.to_device(C)
        got = ctx.assign(d, dc)
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("m", [16, 100, 512, 1000, 3000])
@pytest.mark.parametrize("n,k", [(1, 1), (7, 3), (90, 5)])
def test_extract_with_own_shifts(ctx, m, n, k):
    """tcx_extract_shape without shifts: pairs of equal and of different
    labels and a last series without a partner, against the oracle."""
    Z, C = _data(3 * m + n, n, m, k)
    labels = np.random.default_rng(n).integers(0, k, n).astype(np.int32)
    labels[: n // 2] = 0
    d, dl, dc = ctx.to_device(Z), ctx.to_device(labels), ctx.to_device(C)
    try:
        ctx.extract_shape(dl, d, None, dc)
        got = dc.numpy()
    finally:
        for a in (d, dl, dc):
            a.free()
    ref, _, _ = O.refine(Z.astype(np.float64), labels, C.astype(np.float64), seed=0, it=0)
    assert max(centroid_errors(got, ref)) <= CENT_RTOL


def test_extract_with_own_shifts_refuses_bad_labels(ctx):
    Z, C = _data(1, 9, 64, 3)
    for bad in (-1, 3, 1 << 30):
        labels = np.zeros(9, np.int32)
        labels[8] = bad
        d, dl, dc = ctx.to_device(Z), ctx.to_device(labels), ctx.to_device(C)
        try:
            with pytest.raises(T.TimescError) as e:
                ctx.extract_shape(dl, d, None, dc)
            assert e.value.code == T.ERR_ARG
        finally:
            for a in (d, dl, dc):
                a.free()
