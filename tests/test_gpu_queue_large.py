"""The queue places of large batches (acts_amd/csrc/kf_queue.hpp): with the
tracks that may become loopers spread wide and in one block (up to 4 batches of
the 65 536 resident lanes, and more), and with the layer navigator wide and
close together (up to 2 batches, and more), every track's results are those of
the input order."""
import numpy as np
import pytest

import acts_amd as A
from acts_amd import capi
from acts_amd.fitter import TRACK_ARRAYS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("navigator,sizes", [
    (capi.NAVIGATOR_DIRECT, (262_144, 262_145)),
    (capi.NAVIGATOR_LAYERS, (131_072, 131_073))])
def test_large_batches(navigator, sizes):
    det, field, events = A.workload("endcap", n_tracks=max(sizes), seed=23)
    for n in sizes:
        print("navigator", navigator, "tracks", n, flush=True)
        ev = events.subset(np.arange(n))
        if navigator == capi.NAVIGATOR_LAYERS:
            ev = A.with_state_slots(ev, np.diff(ev.seq_offsets) + 4)
        got = []
        for order in (0, 1):
            fitter = A.KalmanFitter(det, field, A.KalmanFitterOptions(
                length_sorted=order, navigator=navigator))
            try:
                got.append(fitter.fit(ev, outputs=("smoothed", "state_surface")))
            finally:
                fitter.close()
        assert np.all(got[0].n_steps > 0)
        for k in tuple(TRACK_ARRAYS) + ("smoothed", "state_surface"):
            assert getattr(got[0], k).tobytes() == getattr(got[1], k).tobytes(), (n, k)
