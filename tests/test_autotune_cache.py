"""The autotuner's cache: an entry stored when 0 meant "off" for the quarantine
and the transport skip is not taken for one in which it means the library's
default; no setting is in the search space twice.  No device."""
import json

import pytest
import torch

import acts_amd as A
from acts_amd import autotune as AT, device

# the library's default quarantine (acts_kf_options::sched_quarantine_steps 0)
QUARANTINE = 200


@pytest.fixture
def batch(monkeypatch):
    def timed(*_):
        raise RuntimeError("settings are timed")
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda *_: "gpu")
    monkeypatch.setattr(device, "DeviceEvents", timed)
    return A.workload("barrel", n_tracks=200, seed=2)


def _cache(path, sig, best):
    path.write_text(json.dumps({sig: {"best": best, "ms": {}}}))
    return str(path)


def test_entry_of_the_former_meaning_is_not_used(batch, tmp_path):
    det, field, ev = batch
    now = json.loads(AT.signature(ev, field, A.KalmanFitterOptions(), "gpu"))
    best = dict(AT.DEFAULTS)
    former = json.dumps({k: v for k, v in now.items() if k != "knobs"}, sort_keys=True)
    with pytest.raises(RuntimeError, match="settings are timed"):
        AT.autotune(det, field, ev, cache_path=_cache(tmp_path / "a.json", former, best))
    entry = json.dumps(now, sort_keys=True)
    assert AT.autotune(det, field, ev,
                       cache_path=_cache(tmp_path / "b.json", entry, best)) == (best, {})


def test_no_setting_twice():
    quarantine = [QUARANTINE if v == 0 else v for v in AT.SPACE["sched_quarantine_steps"]]
    for values in (quarantine, *AT.SPACE.values()):
        assert len(values) == len(set(values))
