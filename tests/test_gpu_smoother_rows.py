"""The smoothed rows of large batches are written by a wavefront's lanes
together, those of small ones by each lane: a fit of 33 000 tracks (the last
wavefront partly filled) gives every track the rows it gets in batches of 16 500,
in either smoother, for failed tracks and tracks with empty slots, and with one of
the two outputs only."""
import numpy as np
import pytest

import acts_amd as A
from acts_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("smoother", [capi.SMOOTHER_GAIN_MATRIX, capi.SMOOTHER_MBF])
def test_shared_rows(smoother):
    n = 33_000
    det, field, ev = A.workload("ragged", n_tracks=n, seed=91)
    fitter = A.KalmanFitter(det, field, A.KalmanFitterOptions(smoother=smoother))
    try:
        parts = [fitter.fit(ev.subset(np.arange(a, a + n // 2)), outputs=("smoothed", "smoothed_cov"))
                 for a in (0, n // 2)]
        for outputs in (("smoothed", "smoothed_cov"), ("smoothed",), ("smoothed_cov",)):
            whole = fitter.fit(ev, outputs=outputs)
            for name in outputs + ("status", "n_states"):
                cut = np.concatenate([getattr(p, name) for p in parts])
                assert cut.tobytes() == getattr(whole, name).tobytes(), (outputs, name)
    finally:
        fitter.close()
    lengths = np.diff(ev.seq_offsets)
    assert np.any(parts[0].status != 0) and np.any(parts[0].n_states < lengths[:n // 2])
