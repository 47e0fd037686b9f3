"""The calls a user of this fitter makes, as cases to be timed.

A case is one fit of one batch (or, for "in_flight", of three batches, and
for "table", the track-state table of a fitted batch) through the public
entry points: ``KalmanFitter.fit`` on host buffers, ``KalmanFitter.fit_device``
on device buffers, ``track_states.device_table``.  The batches are the
repository's own workloads (acts_amd.events.WORKLOADS): the plane telescope
without a field, the barrel and the barrel with endcaps in 2 T, the same
detector in the solenoid's field map, and the ragged double-layer detector
with holes and outliers.

The fitter of a configuration (geometry, field, options) is kept between
batches, as a program that fits event after event keeps it.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import acts_amd as A
from acts_amd import capi, events as EV, track_states as TS
from acts_amd.device import DeviceEvents, DeviceResult
from acts_amd.fitter import ALL_STATE_OUTPUTS, DEFAULT_STATE_OUTPUTS, TRACK_ARRAYS

FITS_IN_FLIGHT = 3

# Largest batches, per workload, of the drawn cases.
RANGES = {"telescope": (16, 10_000), "barrel": (64, 20_000), "endcap": (500, 120_000),
          "solenoid": (500, 400_000), "ragged": (500, 200_000)}


def _case(name, workload, tracks, call="device", precision="fp64", examples=False,
          navigator="direct", reverse=False, outputs="default"):
    return dict(name=name, workload=workload, tracks=tracks, call=call, precision=precision,
                examples=examples, navigator=navigator, reverse=reverse, outputs=outputs)


def listed():
    return [
        # a test-beam event: a handful of tracks in host memory, 1D and 2D
        # measurements; launches, copies and the latency of one track count
        _case("telescope_100_host", "telescope", 100, call="host"),
        # the smallest benchmark configuration, with every output kept
        _case("barrel_1k_all", "barrel", 1_000, outputs="all"),
        # one event of the serving stream (median multiplicity) in the map
        _case("map_event_5k", "solenoid", 5_000),
        # the stream's largest event, from and to host memory, mixed precision
        _case("map_event_20k_host_mixed", "solenoid", 20_000, call="host", precision="mixed"),
        # the uniform-field benchmark batch, one fit at a time
        _case("endcap_100k", "endcap", 100_000),
        # the same batch as an event loop keeps it: three contexts at work
        _case("endcap_3x100k_in_flight", "endcap", 100_000, call="in_flight"),
        # the Examples' chain: SympyStepper, MbfSmoother, perigee parameters
        _case("map_examples_100k", "solenoid", 100_000, examples=True),
        # the headline batch in both precisions
        _case("map_500k", "solenoid", 500_000),
        _case("map_500k_mixed", "solenoid", 500_000, precision="mixed"),
        # 6-30 measurements per track, holes, rejected outliers
        _case("ragged_200k", "ragged", 200_000),
        # surfaces found from the geometry, each track filtered in reverse
        _case("endcap_layers_reverse_50k", "endcap", 50_000, navigator="layers", reverse=True),
        # the writer's columns of a fitted batch
        _case("endcap_table_100k", "endcap", 100_000, call="table", outputs="all"),
    ]


def draw(rng):
    workload = rng.choice(list(RANGES))
    lo, hi = RANGES[workload]
    tracks = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    call = rng.choice(["device", "device", "device", "host", "table", "in_flight"])
    if call in ("host", "table", "in_flight"):
        tracks = min(tracks, rng.randint(15_000, 60_000))
    outputs = rng.choice(["default", "default", "all"])
    outputs = {"table": "all", "in_flight": "default"}.get(call, outputs)
    examples = rng.random() < 0.3
    navigator, reverse = "direct", False
    # the variants that cost more per track stay below the largest case
    if workload != "ragged" and call == "device" and tracks < 100_000:
        navigator = rng.choice(["direct", "direct", "layers"])
        reverse = rng.random() < 0.25
    case = _case("", workload, tracks, call, rng.choice(["fp64", "fp64", "mixed"]), examples,
                 navigator, reverse, outputs)
    del case["name"]
    return case


# Mean surface-sequence length: what the buffers of a batch are made for.
SLOTS = {"telescope": 6.0, "barrel": 10.0, "endcap": 12.89, "solenoid": 12.89, "ragged": 21.49}


@functools.lru_cache(maxsize=None)
def _setup(workload):
    """(detector, field) of a workload."""
    det, field, _ = A.workload(workload, n_tracks=1, seed=1)
    return det, field


@functools.lru_cache(maxsize=2)
def _fitters(workload, precision, examples, navigator, reverse, count):
    det, field = _setup(workload)
    options = dict(precision=capi.PRECISION_MIXED if precision == "mixed"
                   else capi.PRECISION_FP64)
    if examples:
        options.update(stepper=capi.STEPPER_SYMPY, smoother=capi.SMOOTHER_MBF,
                       reference_surface=capi.REFERENCE_PERIGEE,
                       reference_strategy=capi.EXTRAPOLATE_FIRST)
    if navigator == "layers":
        options["navigator"] = capi.NAVIGATOR_LAYERS
    if reverse:
        options["reverse_filtering"] = True
    opts = EV.workload_options(workload, **options)
    return [A.KalmanFitter(det, field, opts) for _ in range(count)]


def _with_slots(lengths, tracks, slots):
    """The first `tracks` tracks, some exchanged for later ones of another
    sequence length, so that their lengths add up to `slots`."""
    take = np.arange(tracks)
    missing = slots - int(lengths[:tracks].sum())
    inside, spare = {}, {}
    for i in range(len(lengths) - 1, -1, -1):
        (inside if i < tracks else spare).setdefault(int(lengths[i]), []).append(i)
    while missing:
        sign = 1 if missing > 0 else -1
        a, b = max(((a, b) for a in inside if inside[a] for b in spare if spare[b]
                    if 0 < sign * (b - a) <= sign * missing),
                   key=lambda ab: sign * (ab[1] - ab[0]))
        take[inside[a].pop()] = spare[b].pop()
        missing -= b - a
    return take


def _events(workload, tracks, seed, navigator="direct"):
    det, field = _setup(workload)
    w = EV.WORKLOADS[workload]
    cfg = EV.gen_config(tracks, seed, pt=w["pt"], pt_log=w.get("pt_log", False), eta=w["eta"],
                        phi=w.get("phi", (-np.pi, np.pi)),
                        hole_probability=w.get("hole_probability", 0.0),
                        outlier_fraction=w.get("outlier_fraction", 0.0),
                        min_measurements=w.get("min_measurements", 1))
    # more tracks than the batch takes, so that it can have the number of
    # state slots that its fixed buffers were made for
    cfg.n_tracks = tracks + 64 + 4 * math.isqrt(tracks)
    ev = EV.generate(det, field, cfg)
    ev = ev.subset(_with_slots(np.diff(ev.seq_offsets), tracks, round(tracks * SLOTS[workload])))
    if det.kinds is not None:
        ev = EV.apply_measurement_kinds(ev, det, seed)
    if navigator == "layers":
        # room for a few surfaces more than the generated track crossed
        ev = A.with_state_slots(ev, np.diff(ev.seq_offsets) + 4)
    return ev


def _outputs(case):
    names = ALL_STATE_OUTPUTS if case["outputs"] == "all" else DEFAULT_STATE_OUTPUTS
    return names + (("reference_params", "reference_cov") if case["examples"] else ())


def prepare(case, seed):
    batches = FITS_IN_FLIGHT if case["call"] == "in_flight" else 1
    fitters = _fitters(case["workload"], case["precision"], case["examples"], case["navigator"],
                       case["reverse"], batches)
    events = [_events(case["workload"], case["tracks"], seed + 1_000_003 * b, case["navigator"])
              for b in range(batches)]
    state = dict(call=case["call"], fitters=fitters, events=events, outputs=_outputs(case))
    if case["call"] == "host":
        return state
    dev = [DeviceEvents(e) for e in events]
    res = [DeviceResult(d.n_tracks, d.n_slots, state["outputs"]) for d in dev]
    state.update(dev=dev, res=res, inputs=[d.batch_in() for d in dev],
                 results=[r.batch_out() for r in res])
    if case["call"] == "table":
        torch.cuda.synchronize()
        fitters[0].fit_device(state["inputs"][0], state["results"][0])
        fitters[0].sync()
        state["truth"] = torch.from_numpy(events[0].truth_meas).cuda()
    return state


def run(state):
    fitters = state["fitters"]
    if state["call"] == "host":
        r = fitters[0].fit(state["events"][0], outputs=state["outputs"])
        return {k: getattr(r, k) for k in tuple(TRACK_ARRAYS) + state["outputs"]}
    if state["call"] == "table":
        floats, ints = TS.device_table(fitters[0], state["dev"][0], state["res"][0],
                                       state["truth"])
        return {"floats": floats, "ints": ints}
    for f, i, o in zip(fitters, state["inputs"], state["results"]):
        f.fit_device(i, o)
    return [dict(r.t) for r in state["res"]] if len(fitters) > 1 else dict(state["res"][0].t)


# Mean track states, measurements, accepted steps and trials per track, as
# the fits of the workloads count them.
PER_TRACK = {"telescope": (6.0, 6.0, 6.0, 6.0), "barrel": (10.0, 10.0, 23.7, 23.7),
             "endcap": (12.9, 12.9, 25.3, 25.4), "solenoid": (12.9, 12.9, 36.4, 37.1),
             "ragged": (21.1, 19.8, 59.4, 59.6)}


def work(case):
    """Bytes: every input read once, every output written once.  Operations:
    the additions, multiplications, divisions, roots and transcendental calls
    of the algorithm (acts_amd.flops)."""
    from acts_amd import flops
    n = case["tracks"] * (FITS_IN_FLIGHT if case["call"] == "in_flight" else 1)
    states, meas, steps, trials = PER_TRACK[case["workload"]]
    slots = n * (SLOTS[case["workload"]] + (4 if case["navigator"] == "layers" else 0))
    widths = {name: np.dtype(dt).itemsize * w for name, (dt, w) in A.fitter.STATE_ARRAYS.items()}
    per_state = sum(widths[o] for o in _outputs(case) if o in widths)
    if case["call"] == "table":
        # three parameter vectors and covariance diagonals with the measured
        # block, the state's scalars, measurement and truth; one row out
        read = 3 * (48 + 48) + 32 + 36 + 48 + 48
        return {"bytes": slots * (read + 4.0 * (capi.TS_NFLOAT + capi.TS_NINT)),
                "flops": slots * 600.0}
    inputs = n * (8 * (6 + 36 + 12) + 16) + slots * 4 + n * meas * (4 + 16 + 32)
    outputs = n * (4 * len(TRACK_ARRAYS) + (336 if case["examples"] else 0)) + slots * per_state
    per_track = float(flops.flops_per_track(steps, trials, states, meas))
    return {"bytes": float(inputs + outputs),
            "flops": n * per_track * (1.8 if case["reverse"] else 1.0)}


# ---------------------------------------------------------------------------
# results in 64 bits, without the library
# ---------------------------------------------------------------------------
def exact(case, seed):
    """The track-state table, and the fit of the telescope (straight tracks
    through planes, so the whole filter and smoother are short closed forms).
    The other fits follow an adaptive Runge-Kutta integration step by step in
    64 bits already; there is no value beside it to compare with."""
    if case["call"] == "table":
        return _exact_table(case, seed)
    if (case["workload"] == "telescope" and case["call"] != "in_flight"
            and case["navigator"] == "direct" and not case["reverse"]):
        return _exact_telescope(case, _events("telescope", case["tracks"], seed))
    return None


def _directions(phi, theta):
    st = np.sin(theta)
    return np.stack([np.cos(phi) * st, np.sin(phi) * st, np.cos(theta)], -1)


def _wrap(phi):
    return phi - 2 * np.pi * np.floor((phi + np.pi) / (2 * np.pi))


def _slab(det, index):
    mat, thickness = det.materials[index]
    return dict(thickness=thickness, x0=mat.x0, ne=mat.z * mat.molar_rho,
                i=16e-9 * mat.z ** 0.9, vacuum=mat.ar <= 0)


def _material(slab, path, p, mass):
    """(energy loss, theta0^2, var(q/p)) of unit-charge particles of momentum
    p (RPP 2018, eqs. 33.5, 33.15 and the Landau width)."""
    me, k = 0.5109989461e-3, 0.0307075
    x = slab["thickness"] * path
    beta2 = p ** 2 / (p ** 2 + mass ** 2)
    bg, gamma = p / mass, np.sqrt(1 + (p / mass) ** 2)
    eps = 0.5 * k * slab["ne"] * x / beta2
    plasma = 28.816e-9 * np.sqrt(slab["ne"] * 1000.0)
    dhalf = np.where(bg >= 10, np.log(bg) + np.log(plasma / slab["i"]) - 0.5, 0.0)
    u = 2 * me * bg ** 2
    wmax = u / (1 + 2 * gamma * me / mass + (me / mass) ** 2)
    loss = eps * (np.log(u / slab["i"]) + np.log(wmax / slab["i"]) - 2 * beta2 - 2 * dhalf)
    t = np.sqrt(x / slab["x0"] / beta2)
    theta0 = 13.6e-3 / p * t * (1 + 0.076 * np.log(t))
    sigma = 4 * eps * 0.42466090014400953 / np.sqrt(beta2) / p ** 2
    return loss, theta0 ** 2, sigma ** 2


def _exact_telescope(case, ev):
    det, _ = _setup("telescope")
    n, mass, planes = ev.n_tracks, float(np.float32(A.fitter.MUON_MASS)), len(det.surfaces)
    if not np.all(np.diff(ev.seq_offsets) == planes):
        return None
    order = ev.seq_surfaces.reshape(n, planes)
    if not np.all(order == order[0]) or not np.array_equal(ev.meas_surfaces, ev.seq_surfaces):
        return None
    values = ev.meas_values.reshape(n, planes, 2)
    noise = ev.meas_cov.reshape(n, planes, 2, 2)
    x, cov = ev.start_params.copy(), ev.start_cov.reshape(n, 6, 6).copy()
    rot = ev.start_plane[:, :9].reshape(n, 3, 3)
    centre = ev.start_plane[:, 9:]
    path = np.zeros(n)
    keep = []
    swap = lambda a: np.swapaxes(a, -1, -2)  # noqa: E731
    for k, sid in enumerate(order[0]):
        desc = det.surfaces[sid]
        # the free state and its derivatives by the bound parameters
        d = _directions(x[:, 2], x[:, 3])
        pos = centre + rot[:, :, 0] * x[:, :1] + rot[:, :, 1] * x[:, 1:2]
        b2f = np.zeros((n, 8, 6))
        b2f[:, 0:3, 0], b2f[:, 0:3, 1] = rot[:, :, 0], rot[:, :, 1]
        b2f[:, 3, 5] = b2f[:, 7, 4] = 1
        b2f[:, 4:6, 2] = np.stack([-d[:, 1], d[:, 0]], -1)
        b2f[:, 4, 3] = d[:, 2] * np.cos(x[:, 2])
        b2f[:, 5, 3] = d[:, 2] * np.sin(x[:, 2])
        b2f[:, 6, 3] = -np.sin(x[:, 3])
        # along the line to the plane
        rot = np.broadcast_to(desc.rotation, (n, 3, 3))
        centre = np.broadcast_to(desc.translation, (n, 3))
        normal = rot[:, :, 2]
        dz = np.sum(normal * d, -1)
        s = np.sum(normal * (centre - pos), -1) / dz
        dtds = np.sqrt(1 + (mass * x[:, 4]) ** 2)
        pos = pos + s[:, None] * d
        path = path + s
        transport = np.zeros((n, 8, 8)) + np.eye(8)
        transport[:, 0, 4] = transport[:, 1, 5] = transport[:, 2, 6] = s
        transport[:, 3, 7] = s * mass ** 2 * x[:, 4] / dtds
        along = np.zeros((n, 8))
        along[:, :3], along[:, 3] = d, dtds
        back = np.zeros((n, 8))
        back[:, :3] = -normal / dz[:, None]
        f2b = np.zeros((n, 6, 8))
        sin_t, cos_t = np.hypot(d[:, 0], d[:, 1]), d[:, 2]
        cos_p, sin_p = d[:, 0] / sin_t, d[:, 1] / sin_t
        f2b[:, 0, :3], f2b[:, 1, :3] = rot[:, :, 0], rot[:, :, 1]
        f2b[:, 2, 4], f2b[:, 2, 5] = -sin_p / sin_t, cos_p / sin_t
        f2b[:, 3, 4], f2b[:, 3, 5], f2b[:, 3, 6] = cos_p * cos_t, sin_p * cos_t, -sin_t
        f2b[:, 4, 7] = f2b[:, 5, 3] = 1
        free = np.eye(8) + along[:, :, None] * back[:, None, :]
        jac = f2b @ free @ transport @ b2f
        rel = pos - centre
        x = np.stack([np.sum(rel * rot[:, :, 0], -1), np.sum(rel * rot[:, :, 1], -1),
                      np.arctan2(d[:, 1], d[:, 0]), np.arctan2(sin_t, cos_t), x[:, 4],
                      x[:, 5] + s * dtds], -1)
        cov = jac @ cov @ swap(jac)
        predicted = (x, cov)
        # the gain-matrix update
        dim, index, _ = det.kinds[sid]
        h = np.zeros((dim, 6))
        h[range(dim), index[:dim]] = 1
        v, m = noise[:, k, :dim, :dim], values[:, k, :dim]
        gain = cov @ h.T @ np.linalg.inv(h @ cov @ h.T + v)
        x = x + (gain @ (m - x @ h.T)[:, :, None])[:, :, 0]
        x[:, 2] = _wrap(x[:, 2])
        cov = cov - gain @ h @ cov
        res = (m - x @ h.T)[:, :, None]
        chi2 = (swap(res) @ np.linalg.inv((np.eye(dim) - h @ gain) @ v) @ res)[:, 0, 0]
        keep.append((predicted, (x, cov), jac, path, chi2))
        # the plane's material
        x, cov = x.copy(), cov.copy()
        d = _directions(x[:, 2], x[:, 3])
        p = 1 / np.abs(x[:, 4])
        loss, var_t, var_q = _material(_slab(det, desc.material),
                                       1 / np.abs(np.sum(normal * d, -1)), p, mass)
        energy = np.sqrt(mass ** 2 + p ** 2) - loss
        new_p = np.maximum(0.01, np.sqrt(np.maximum(energy ** 2 - mass ** 2, 0)))
        x[:, 4] = np.sign(x[:, 4]) / new_p
        cov[:, 2, 2] += var_t / (d[:, 0] ** 2 + d[:, 1] ** 2)
        cov[:, 3, 3] += var_t
        cov[:, 4, 4] += var_q
    # the smoother, from the last plane back (both smoothers give this)
    smoothed = [keep[-1][1]]
    for k in range(planes - 2, -1, -1):
        (xf, cf), ((xp, cp), _, jac, _, _) = keep[k][1], keep[k + 1]
        xs, cs = smoothed[0]
        g = cf @ swap(jac) @ np.linalg.inv(cp)
        dx = xs - xp
        dx[:, 2:4] = _wrap(dx[:, 2:4])
        x = xf + (g @ dx[:, :, None])[:, :, 0]
        x[:, 2] = _wrap(x[:, 2])
        smoothed.insert(0, (x, cf + g @ (cs - cp) @ swap(g)))
    per_state = lambda a: np.ascontiguousarray(  # noqa: E731
        np.stack(a, 1).reshape((n * planes,) + a[0].shape[1:]))
    flat = lambda a: a.reshape(len(a), 36)  # noqa: E731
    out = {"state_path": per_state([k[3] for k in keep]),
           "state_chi2": per_state([k[4] for k in keep]),
           "chi2": np.sum([k[4] for k in keep], 0)}
    if case["outputs"] == "all":
        out["predicted"] = per_state([k[0][0] for k in keep])
        out["predicted_cov"] = flat(per_state([k[0][1] for k in keep]))
        out["filtered"] = per_state([k[1][0] for k in keep])
        out["filtered_cov"] = flat(per_state([k[1][1] for k in keep]))
        out["jacobian"] = flat(per_state([k[2] for k in keep]))
    out["smoothed"] = per_state([s[0] for s in smoothed])
    out["smoothed_cov"] = flat(per_state([s[1] for s in smoothed]))
    names = tuple(TRACK_ARRAYS) + _outputs(case)
    return {name: out.get(name) for name in names}


def _local_to_global(det, sid, l0, l1):
    out = np.full((len(sid), 3), np.nan)
    for i, s in enumerate(det.surfaces):
        at = sid == i
        a, b = l0[at], l1[at]
        if s.type == capi.SURFACE_CYLINDER:
            r = s.bounds[0]
            loc = np.stack([r * np.cos(a / r), r * np.sin(a / r), b], -1)
        elif s.type == capi.SURFACE_DISC:
            loc = np.stack([a * np.cos(b), a * np.sin(b), 0 * a], -1)
        else:
            loc = np.stack([a, b, 0 * a], -1)
        out[at] = loc @ np.asarray(s.rotation).T + s.translation
    return out


def _exact_table(case, seed):
    state = prepare(case, seed)
    det, _ = _setup(case["workload"])
    ev = state["events"][0]
    fit = {k: v.cpu().numpy() for k, v in state["res"][0].t.items()}
    slots = len(fit["state_surface"])
    track = np.repeat(np.arange(ev.n_tracks), np.diff(ev.seq_offsets))
    k = np.arange(slots) - ev.seq_offsets[track]
    rows = np.flatnonzero((fit["status"][track] == 0) & (k < fit["n_states"][track]))
    col = {name: np.full(slots, np.nan) for name in TS.FLOAT_COLUMNS}
    sid, mi = fit["state_surface"][rows], fit["state_measurement"][rows]
    link = mi >= 0
    col["chi2"][rows], col["pathLength"][rows] = fit["state_chi2"][rows], fit["state_path"][rows]
    nan = np.where(link, 0.0, np.nan)
    at = np.where(link, mi, 0)
    truth = ev.truth_meas[at] + nan[:, None]
    dims = np.full(len(rows), 2) if ev.meas_dims is None else ev.meas_dims[at].astype(int)
    index = (np.broadcast_to([0, 1], (len(rows), 2)) if ev.meas_indices is None
             else ev.meas_indices[at].astype(int))
    two = dims == 2
    ia, ib = index[:, 0], np.where(two, index[:, 1], index[:, 0])
    m = ev.meas_values[at] + nan[:, None]
    v = ev.meas_cov[at].reshape(-1, 2, 2)
    t_pos, t_dir = (_local_to_global(det, sid, truth[:, 0], truth[:, 1]),
                    _directions(truth[:, 2], truth[:, 3]))
    for i, a in enumerate("xyz"):
        col["t_" + a][rows], col["t_d" + a][rows] = t_pos[:, i], t_dir[:, i]
    col["t_r"][rows] = np.hypot(t_pos[:, 0], t_pos[:, 1])
    for i, name in enumerate(TS.PARAMS):
        col["t_" + name][rows] = truth[:, i]
    local = [np.where(ia == j, m[:, 0], np.where(two & (ib == j), m[:, 1], 0 * m[:, 0]))
             for j in (0, 1)]
    hit = _local_to_global(det, sid, *local)
    col["l_x_hit"][rows], col["l_y_hit"][rows] = local
    for i, a in enumerate("xyz"):
        col[f"g_{a}_hit"][rows] = hit[:, i]
    pick = lambda a, i: np.take_along_axis(a, i[:, None], 1)[:, 0]  # noqa: E731
    sets = []
    for name in ("predicted", "filtered", "smoothed"):
        c = fit[name + "_cov"][rows].reshape(-1, 6, 6)
        sets.append((fit[name][rows], np.einsum("nii->ni", c).copy(), c))
    with np.errstate(all="ignore"):
        x, diag, _ = sets[0]
        for j, (axis, i) in enumerate((("x", ia), ("y", ib))):
            used = np.where(link & (two | (j == 0)), 0.0, np.nan)
            res = m[:, j] - pick(x, i) + used
            rc = v[:, j, j] + pick(diag, i)
            col[f"res_{axis}_hit"][rows] = res
            col[f"err_{axis}_hit"][rows] = np.sqrt(v[:, j, j]) + used
            col[f"pull_{axis}_hit"][rows] = np.where(rc > 0, res / np.sqrt(rc), np.nan)
        # the smoothed state without its measurement
        x, diag, c = sets[2]
        r = np.arange(len(rows))
        s00, s11 = c[r, ia, ia] - v[:, 0, 0], np.where(two, c[r, ib, ib] - v[:, 1, 1], 1.0)
        s01 = np.where(two, c[r, ia, ib] - v[:, 0, 1], 0.0)
        det2 = s00 * s11 - s01 * s01
        pa, pb = c[r, :, ia], np.where(two[:, None], c[r, :, ib], 0.0)
        k0 = (pa * s11[:, None] - pb * s01[:, None]) / det2[:, None]
        k1 = np.where(two[:, None], (pb * s00[:, None] - pa * s01[:, None]) / det2[:, None], 0)
        r0, r1 = m[:, 0] - pick(x, ia), np.where(two, m[:, 1] - pick(x, ib), 0.0)
        sets.append((x + k0 * r0[:, None] + k1 * r1[:, None],
                     diag - k0 * pa - k1 * pb + nan[:, None], None))
        for name, (x, diag, _) in zip(TS.PARAM_SETS, sets):
            err = np.sqrt(diag)
            res = x - truth
            res[:, 2] = _wrap(res[:, 2])
            pull = np.where(err > 0, res / err, np.nan)
            for i, p in enumerate(TS.PARAMS):
                col[f"{p}_{name}"][rows] = x[:, i]
                col[f"res_{p}_{name}"][rows] = res[:, i]
                col[f"err_{p}_{name}"][rows] = err[:, i]
                col[f"pull_{p}_{name}"][rows] = pull[:, i]
            pos = _local_to_global(det, sid, x[:, 0], x[:, 1])
            d = _directions(x[:, 2], x[:, 3])
            p = np.abs(1 / x[:, 4])
            perp = np.hypot(d[:, 0], d[:, 1])
            for i, a in enumerate("xyz"):
                col[f"g_{a}_{name}"][rows] = pos[:, i]
                col[f"p{a}_{name}"][rows] = p * d[:, i]
            col[f"eta_{name}"][rows] = np.arcsinh(d[:, 2] / perp)
            col[f"pT_{name}"][rows] = p * perp
    return {"floats": np.stack([col[c] for c in TS.FLOAT_COLUMNS]), "ints": None}
