"""The search for a surface's measurement: expected first by position in the
track's list, ruled out by the set of the list's surfaces (indices below 128),
found by a search otherwise.  Fits do not depend on which: the measurements of
each track in sequence order, in the opposite order, and with a second, far
off measurement of the track's first surface after the others (the first one in
input order counts), with holes, on 24 and on 140 surfaces, smoothed and
filtered in reverse."""
import dataclasses

import numpy as np
import pytest

import acts_amd as A
from acts_amd.detector import barrel_detector, barrel_endcap_detector
from acts_amd.events import gen_config, generate
from acts_amd.fitter import ALL_STATE_OUTPUTS

pytestmark = pytest.mark.gpu


def _with_order(ev, order):
    """`ev` with measurement lists order(indices of the track's list)."""
    mo = ev.meas_offsets
    lists = [order(np.arange(mo[t], mo[t + 1])) for t in range(ev.n_tracks)]
    take = np.concatenate(lists)
    off = np.zeros_like(mo)
    off[1:] = np.cumsum([len(x) for x in lists])
    return dataclasses.replace(
        ev, meas_offsets=off,
        **{n: np.ascontiguousarray(getattr(ev, n)[take]) for n in (
            "meas_surfaces", "meas_values", "meas_cov", "truth_meas", "meas_is_outlier")})


def _with_duplicate(ev):
    out = _with_order(ev, lambda m: np.append(m, m[:1]))
    out.meas_values[out.meas_offsets[1:] - 1] += 50.0
    return out


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("surfaces", [24, 140])
def test_measurement_order(surfaces, reverse):
    det = (barrel_endcap_detector() if surfaces == 24
           else barrel_detector(radii=np.linspace(30.0, 1001.0, surfaces), thickness=0.02))
    assert len(det.surfaces) == surfaces
    field = A.ConstantField()
    ev = generate(det, field, gen_config(200, 5, pt=(1.0, 10.0), eta=(-0.9, 0.9),
                                         hole_probability=0.15, min_measurements=4))
    fitter = A.KalmanFitter(det, field, A.KalmanFitterOptions(reverse_filtering=reverse))
    try:
        ref, flipped, doubled = [fitter.fit(e, outputs=ALL_STATE_OUTPUTS) for e in (
            ev, _with_order(ev, lambda m: m[::-1]), _with_duplicate(ev))]
    finally:
        fitter.close()
    assert np.count_nonzero(ref.status == 0) > 190
    assert ref.n_holes.sum() > 100
    for other in (flipped, doubled):
        for name in ("status", "n_states", "chi2", "n_measurements", "n_holes", "n_steps",
                     "state_surface", "state_flags", "smoothed", "smoothed_cov", "filtered"):
            assert getattr(ref, name).tobytes() == getattr(other, name).tobytes(), name
