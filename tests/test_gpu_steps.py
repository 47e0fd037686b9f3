"""The Runge-Kutta step on every kind of field it is compiled for: a uniform
field, a cell-major map whose axes multiply by reciprocals, and a map whose
axes divide (bins that are not all of one width), with tracks that leave the
map.  Against the oracle at the FP64 bar (tests/parity.py), in either
stepper; in mixed precision the same statuses and, on states of converged
fits, the mixed fit's stated bounds (tests/test_gpu_mixed.py)."""
import numpy as np
import pytest

import acts_amd as A
from acts_amd import capi
from acts_amd.detector import FieldMap, barrel_endcap_detector
from acts_amd.events import gen_config, generate
from acts_amd.fitter import ALL_STATE_OUTPUTS

from parity import compare, error_report

pytestmark = pytest.mark.gpu

# points per axis; the solenoid map on 57 x 57 x 121 points has bins of more
# than one width (in the last bits), on 101 x 101 x 201 points it has not
MAPS = {"uniform": None, "reciprocals": (101, 101, 201), "divisions": (57, 57, 121)}


def _uniform_bins(n, lo, hi):
    step = (hi - lo) / (n - 1)
    w = ((hi + step) - lo) / n
    b = np.arange(1, n + 1)
    return len(set((lo + b * w) - (lo + (b - 1) * w))) == 1


@pytest.fixture(scope="module", params=list(MAPS))
def batch(request):
    points = MAPS[request.param]
    det = barrel_endcap_detector()
    if points is None:
        field = A.ConstantField()
    else:
        # the map ends inside the outermost discs: some tracks leave it
        field = FieldMap.solenoid(n=points, point_max=(2000.0, 2000.0, 2800.0),
                                  point_min=(-2000.0, -2000.0, -2800.0))
        assert all(_uniform_bins(n, lo, hi) for n, lo, hi in
                   zip(field.n, field.point_min, field.point_max)) == (
            request.param == "reciprocals")
    ev = generate(det, field, gen_config(1500, 77, pt=(0.5, 50.0), pt_log=True,
                                         eta=(-2.5, 2.5)))
    return det, field, ev


def _fit(det, field, ev, **kw):
    opts = A.KalmanFitterOptions(**kw)
    fitter = A.KalmanFitter(det, field, opts)
    try:
        return opts, fitter.fit(ev, outputs=ALL_STATE_OUTPUTS)
    finally:
        fitter.close()


@pytest.mark.parametrize("stepper", [capi.STEPPER_EIGEN, capi.STEPPER_SYMPY])
def test_field_kinds(oracle_mod, batch, stepper):
    det, field, ev = batch
    opts, got = _fit(det, field, ev, stepper=stepper)
    ref, _ = oracle_mod.fit(det, field, opts, ev, n_threads=0)
    # the SympyStepper's jacobian bar: tests/test_gpu_sympy.py
    rep = compare(got, ref, ev, max_chi2_ndf=100.0,
                  rel_jacobian=1e-8 if stepper == capi.STEPPER_SYMPY else None)
    print({k: v for k, v in rep.items()}, flush=True)
    assert rep["ok"], rep
    _, mixed = _fit(det, field, ev, stepper=stepper, precision=capi.PRECISION_MIXED)
    rep = error_report(mixed, ref, ev, max_chi2_ndf=100.0)
    assert rep["status_mismatch"] <= 0.005 * ev.n_tracks
    assert max(rep["smoothed_p999_rel"]) < 1e-5
