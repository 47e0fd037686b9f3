"""The track queue's orders only change the order of work: every order gives
the results of the input order bit for bit, at the batch sizes where the sort
changes (one wavefront: none; up to 4 096 tracks: one workgroup; beyond:
tiles, and from ~17 000 tracks with ~1 000 keys more than one scan chunk)."""
import numpy as np
import pytest

import acts_amd as A
from acts_amd.fitter import DEFAULT_STATE_OUTPUTS, TRACK_ARRAYS

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def batch():
    return A.workload("endcap", n_tracks=25_000, seed=17)


@pytest.mark.parametrize("n", [64, 65, 4096, 4097, 25_000])
def test_orders_give_the_same_results(batch, n):
    det, field, ev = batch
    sub = ev.subset(np.arange(n))
    ref = None
    for order in (0, 1, 2, 3):
        print("queue order", order, "tracks", n, flush=True)
        fitter = A.KalmanFitter(det, field, A.KalmanFitterOptions(length_sorted=order))
        try:
            got = fitter.fit(sub)
        finally:
            fitter.close()
        if ref is None:
            ref = got
            assert np.all(got.n_steps > 0)
        for k in tuple(TRACK_ARRAYS) + DEFAULT_STATE_OUTPUTS:
            a, b = getattr(got, k), getattr(ref, k)
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (order, k)
