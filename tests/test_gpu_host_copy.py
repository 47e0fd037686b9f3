"""The host-buffer entry point copies pageable arrays through pinned memory
of the context: one transfer for a small batch, chunks emptied by several
threads for a large one (acts_amd/csrc/kf_host_copy.hpp).  Every output
equals the device entry point's bit for bit: around the sizes where the way
changes, growing and shrinking on one context, and with some arrays in
pinned memory, which the device copies by itself."""
import ctypes as C

import numpy as np
import pytest

import acts_amd as A
from acts_amd import capi
from acts_amd.fitter import ALL_STATE_OUTPUTS, STATE_ARRAYS, TRACK_ARRAYS

pytestmark = pytest.mark.gpu

NAMES = tuple(TRACK_ARRAYS) + ALL_STATE_OUTPUTS
# all outputs of a barrel track: 10 states of 1 200 bytes; the block is one
# transfer up to 1 MiB (87 tracks) and chunks of 2 MiB from there
SIZES = (1, 87, 88, 175, 3000, 2)


def _device_fit(fitter, ev):
    import torch
    from acts_amd.device import DeviceEvents, DeviceResult
    din = DeviceEvents(ev)
    res = DeviceResult(din.n_tracks, din.n_slots, ALL_STATE_OUTPUTS)
    torch.cuda.synchronize()
    fitter.fit_device(din.batch_in(), res.batch_out())
    fitter.sync()
    return res


@pytest.mark.parametrize("workload", ["barrel", "telescope"])
def test_host_fit_equals_device_fit(workload):
    det, field, ev = A.workload(workload, n_tracks=max(SIZES), seed=5)
    fitter = A.KalmanFitter(det, field, A.KalmanFitterOptions())
    try:
        for n in SIZES:
            sub = ev.subset(np.arange(n))
            print("host copy:", workload, n, flush=True)
            got, want = fitter.fit(sub, outputs=ALL_STATE_OUTPUTS), _device_fit(fitter, sub)
            for k in NAMES:
                a, b = getattr(got, k), want.host(k)
                assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (n, k)
    finally:
        fitter.close()


def test_pinned_and_pageable_arrays_together():
    import torch
    n = 400
    det, field, ev = A.workload("barrel", n_tracks=n, seed=6)
    fitter = A.KalmanFitter(det, field, A.KalmanFitterOptions())
    try:
        want = _device_fit(fitter, ev)
        keep = []

        def pinned(a):
            t = torch.empty(max(a.nbytes, 1), dtype=torch.uint8, pin_memory=True)
            keep.append(t)
            p = t.numpy()[:a.nbytes].view(a.dtype).reshape(a.shape)
            p[...] = a
            return p

        bin_ = ev.batch_in()
        for name in ("start_cov", "seq_offsets", "meas_values"):
            setattr(bin_, name, pinned(getattr(ev, name)).ctypes.data)
        out, bout = {}, capi.BatchOut()
        slots = int(ev.seq_offsets[-1])
        for i, name in enumerate(NAMES):
            dt, w = STATE_ARRAYS.get(name, (TRACK_ARRAYS.get(name), 1))
            rows = slots if name in STATE_ARRAYS else n
            a = np.zeros((rows,) if w == 1 else (rows, w), dt)
            out[name] = pinned(a) if i % 3 == 0 else a
            setattr(bout, name, out[name].ctypes.data)
        capi.check(fitter.lib.acts_kf_fit_batch(fitter.ctx, C.byref(bin_), C.byref(bout), None),
                   "acts_kf_fit_batch")
        fitter.sync()
        for k in NAMES:
            b = want.host(k)
            assert np.array_equal(out[k].view(np.uint8), b.view(np.uint8)), k
    finally:
        fitter.close()
