"""A step in a field map whose axes divide (bins that are not all of one width
in the last bits) costs a step in a map with reciprocals and the divisions: 18
of them, ~12 instructions more each, on a step of ~1 900.  That is 1.12 times
the step; more than 1.2 times means a lookup that branches or gathers where the
other does not.  One wavefront of tracks in short steps, the fastest of ten
forward kernels."""
import numpy as np
import pytest

import acts_amd as A
from acts_amd.detector import FieldMap, barrel_endcap_detector
from acts_amd.events import gen_config, generate

pytestmark = pytest.mark.gpu


def test_step_cost():
    det = barrel_endcap_detector()
    limits = dict(point_max=(2000.0, 2000.0, 2800.0), point_min=(-2000.0, -2000.0, -2800.0))
    ev = generate(det, A.ConstantField(), gen_config(64, 3, pt=(1.0, 10.0), eta=(-0.8, 0.8)))
    per_step = {}
    for name, points in (("reciprocals", (101, 101, 201)), ("divisions", (57, 57, 121))):
        fitter = A.KalmanFitter(det, FieldMap.solenoid(n=points, **limits),
                                A.KalmanFitterOptions(max_step_size=3.0, kernel_timing=True))
        try:
            times = []
            for _ in range(10):
                res = fitter.fit(ev)
                times.append(fitter.kernel_times()[0])
        finally:
            fitter.close()
        assert np.median(res.n_steps) > 300
        per_step[name] = min(times) / int(res.n_steps.max())
        print(name, per_step[name] * 1e3, "us a step,", int(res.n_steps.max()), "steps", flush=True)
    assert per_step["divisions"] < 1.2 * per_step["reciprocals"], per_step
