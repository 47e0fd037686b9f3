"""Transport skipping where the caller gives no number of steps: on in a
uniform field, and no result depends on it.  One context fits a batch smaller
than a wavefront, then larger ones (the checkpoints grow with the batch),
eagerly and under a replayed graph; tracks that end at the step limit, and
(low momenta between discs) tracks that come back to a surface."""
import numpy as np
import pytest

import acts_amd as A
from acts_amd import capi
from acts_amd.detector import barrel_endcap_detector
from acts_amd.events import gen_config, generate
from acts_amd.fitter import ALL_STATE_OUTPUTS

pytestmark = pytest.mark.gpu

SIZES = (50, 3000, 12000)


def _fits(det, field, batches, **kw):
    fitter = A.KalmanFitter(det, field, A.KalmanFitterOptions(**kw))
    try:
        return [fitter.fit(ev, outputs=ALL_STATE_OUTPUTS) for ev in batches]
    finally:
        fitter.close()


@pytest.mark.parametrize("kw", [
    {}, dict(precision=capi.PRECISION_MIXED), dict(stepper=capi.STEPPER_SYMPY),
    dict(use_graph=True), dict(reverse_filtering=True),
    dict(navigator=capi.NAVIGATOR_LAYERS)], ids=str)
def test_default_skip_does_not_change_results(kw):
    det, field = barrel_endcap_detector(), A.ConstantField()
    batches = [generate(det, field, gen_config(n, 7 + n, pt=(0.25, 10.0), pt_log=True,
                                               eta=(-2.5, 2.5))) for n in SIZES]
    if kw.get("navigator"):
        batches = [A.with_state_slots(ev, np.diff(ev.seq_offsets) + 4) for ev in batches]
    off = _fits(det, field, batches, sched_transport_skip_steps=-1, **kw)
    got = _fits(det, field, batches, **kw)
    # past the default of 200 steps since a surface: the branch is taken
    assert max(int(r.n_steps.max()) for r in off) > 400
    for n, a, b in zip(SIZES, off, got):
        for name in ("status", "n_states", "n_steps", "n_step_trials", "chi2") + ALL_STATE_OUTPUTS:
            x, y = getattr(a, name), getattr(b, name)
            assert x.tobytes() == y.tobytes(), (n, name)
