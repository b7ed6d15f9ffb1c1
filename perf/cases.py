"""Measured cases: the stages of a correlation run through the package's entry points.

A user of this package turns day-long traces into window spectra (S2sPlan), correlates the
station pairs of a day (XcPlan, or XcBatch for segments of uneven shape), and stacks the
correlations of many days (linear_stack, pws, tfpws).  The listed cases are those calls at the
sizes of the package's own configurations and benchmark; draw() spreads over the same ranges.

Every case is one call (two for the stack case) on tensors that are already on the GPU, with the
plan a program keeps between the days it processes.
"""
import math
import random

import numpy as np
import torch

from fastxc_amd import ops

DEV = "cuda:0"
WINDOW_S = 3600.0  # every configuration correlates one-hour windows


# ------------------------------------------------------------------ shapes
def _even_smooth(n):
    """Smallest even number >= n whose prime factors are 2, 3, 5 and 7."""
    n += n % 2
    while True:
        m = n
        for p in (2, 3, 5, 7):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n += 2


def _lengths(case):
    """(window, filter FFT, output FFT) in samples: the window rounded up to a smooth length, the
    filter's ringing (20 s) and the kept lags padded on."""
    dt = case["delta"]
    seg = _even_smooth(round(WINDOW_S / dt))
    keep = round(case["lag_s"] / dt)
    return seg, _even_smooth(seg + round(20.0 / dt)), _even_smooth(seg + keep)


def _s2s_shape(case):
    dt = case["delta"]
    seg, nff, nfo = _lengths(case)
    shift = round(case["shift_s"] / dt)
    return seg, nff, nfo, shift, seg + (case["windows"] - 1) * shift


def _bands(case):
    """Broad band first, then (for the multi-band running mean) its two halves."""
    lo, hi = 0.1, min(2.0, 0.4 / case["delta"])
    if case["normalize"] != 1:
        return [(lo, hi)]
    mid = math.sqrt(lo * hi)
    return [(lo, hi), (lo, mid), (mid, hi)]


def _power_response(nfft, dt, lo, hi):
    """|H|^2 of a second-order Butterworth band-pass (bilinear transform), bins 0..nfft/2."""
    w = np.tan(np.pi * np.minimum(np.arange(nfft // 2 + 1) / nfft, 0.4999999))
    a, b = math.tan(math.pi * lo * dt), math.tan(math.pi * hi * dt)
    x = np.zeros_like(w)
    x[1:] = (w[1:] ** 2 - a * b) / (w[1:] * (b - a))
    p = 1.0 / (1.0 + x ** 4)
    p[0] = 0.0
    return p.astype(np.float32)


def _taper_bins(case, seg):
    lo, hi = _bands(case)[0]
    df = 1.0 / (seg * case["delta"])
    return [int(lo * 0.667 / df), int(lo / df), int(hi / df), int(hi * 1.333 / df)]


def _batch_sizes(case):
    r = random.Random(case["layout"])
    k = case["segments"]
    sta = [r.randint(case["min_stations"], case["max_stations"]) for _ in range(k)]
    win = [r.randint(case["min_windows"], case["max_windows"]) for _ in range(k)]
    return sta, win


def _groups(case):
    """Group counts of the pairs: most pairs have the full count, some fewer (stations that
    recorded on part of the days).  A time-frequency stack of one group is zero but for rounding,
    so there every pair has two."""
    r = np.random.RandomState(case["pairs"] * 7 + case["groups"])
    g = np.full(case["pairs"], case["groups"], np.int64)
    if case["ragged"]:
        some = r.rand(case["pairs"]) < 0.4
        g[some] = r.randint(2 if case["stage"] == "tfpws" else 1, case["groups"] + 1, int(some.sum()))
    return np.concatenate([[0], np.cumsum(g)])


def _pairs(n):
    return np.triu_indices(n, k=1)


# ------------------------------------------------------------------- cases
def listed():
    s2s = {"stage": "s2s", "lag_s": 100.0, "shift_s": 3600.0, "windows": 24, "whiten": 2, "normalize": 3}
    xc = {"stage": "xc", "lag_s": 100.0, "windows": 24}
    return [
        # one three-component station, one day at 1 Hz, multi-band running mean: the smallest call
        dict(s2s, name="s2s_station_1hz", channels=3, num_ch=3, delta=1.0, normalize=1),
        # a day of a 1000-station vertical array at 10 Hz, the benchmark's workload
        dict(s2s, name="s2s_array_10hz", channels=1000, num_ch=1, delta=0.1),
        # three components with half-overlapping windows: the shared running mean of a station
        dict(s2s, name="s2s_three_component", channels=300, num_ch=3, delta=0.1, shift_s=1800.0, windows=47),
        # 20 Hz: windows whose transforms are longer than one compute unit's memory
        dict(s2s, name="s2s_array_20hz", channels=60, num_ch=1, delta=0.05),
        # eight stations, one day: launches and latency
        dict(xc, name="xc_8_stations", stations=8, delta=0.1, precision="fp32"),
        # the channels of a 200-station three-component network, one day with overlap, in the
        # arithmetic that the executables use unless told otherwise
        dict(xc, name="xc_network_fp32", stations=600, windows=47, delta=0.1, precision="fp32"),
        # the benchmark's headline: 1000 stations, one day, split-bf16
        dict(xc, name="xc_array_bf16x3", stations=1000, delta=0.1, precision="bf16x3"),
        # 20 Hz: the long lag transform
        dict(xc, name="xc_20hz", stations=120, delta=0.05, precision="bf16x3"),
        # one window of a subnetwork, as the streaming engine correlates each segment
        dict(xc, name="xc_one_window", stations=300, windows=1, delta=0.1, precision="bf16x3"),
        # independent segments of uneven shape with gaps, in one set of launches
        {"name": "xc_uneven_batch", "stage": "batch", "segments": 24, "min_stations": 20, "max_stations": 200,
         "min_windows": 6, "max_windows": 48, "layout": 13, "delta": 0.1, "lag_s": 100.0, "gaps": "exclude"},
        # a month of daily correlations: linear and phase-weighted stack of each pair
        {"name": "stack_month", "stage": "stack", "pairs": 6000, "groups": 30, "ragged": True, "n": 2001},
        # time-frequency phase-weighted stack over three sub-stacks
        {"name": "tfpws_three_groups", "stage": "tfpws", "pairs": 400, "groups": 3, "ragged": False, "n": 2001,
         "delta": 0.1, "fmin": 0.0, "fmax": 0.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    stage = rng.choice(("s2s", "xc", "xc", "batch", "stack", "tfpws"))
    delta = rng.choice((1.0, 0.2, 0.1, 0.1, 0.05))
    if stage == "s2s":
        num_ch = rng.choice((1, 3))
        half = rng.random() < 0.4
        return {"stage": "s2s", "lag_s": float(rng.randint(40, 110)), "shift_s": 1800.0 if half else 3600.0,
                "windows": rng.randint(2, 47 if half else 24), "whiten": rng.choice((2, 2, 1, 3, 0)),
                "normalize": rng.choice((3, 3, 1, 2, 0)), "channels": num_ch * _log(rng, 1, 180 // num_ch),
                "num_ch": num_ch, "delta": delta}
    if stage == "xc":
        most = {1.0: 600, 0.2: 400, 0.1: 400, 0.05: 150}[delta]
        return {"stage": "xc", "lag_s": float(rng.randint(20, 110)), "windows": _log(rng, 1, 64),
                "stations": _log(rng, 4, most), "delta": delta,
                "precision": rng.choice(("fp32", "fp32", "bf16x3", "bf16x3", "fp16x3", "fp16"))}
    if stage == "batch":
        return {"stage": "batch", "segments": _log(rng, 2, 32), "min_stations": rng.randint(2, 30),
                "max_stations": rng.randint(31, 180), "min_windows": rng.randint(1, 8),
                "max_windows": rng.randint(9, 48), "layout": rng.randint(1, 10 ** 6),
                "delta": rng.choice((1.0, 0.2, 0.1)), "lag_s": float(rng.randint(40, 110)),
                "gaps": rng.choice(("keep", "exclude"))}
    n = 2 * _log(rng, 100, 2000) + 1
    if stage == "stack":
        return {"stage": "stack", "pairs": _log(rng, 1, 6000), "groups": _log(rng, 1, 40),
                "ragged": rng.random() < 0.7, "n": n}
    band = rng.random() < 0.4
    most = max(2, int(400 * (2001 / n) ** 2 / (3 if n > 1000 else 1)))
    return {"stage": "tfpws", "pairs": _log(rng, 1, most), "groups": _log(rng, 2, 9), "ragged": rng.random() < 0.5,
            "n": n, "delta": 0.1, "fmin": 0.1 if band else 0.0, "fmax": 2.0 if band else 0.0}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEV, dtype=dtype)


def _traces(case, seed, npts):
    """Raw counts: a common wavefield and each channel's own noise, an offset and a drift."""
    g, n = _gen(seed), case["channels"]
    x = _randn(g, n, npts)
    x += 0.7 * _randn(g, 1, npts)
    x *= 800.0
    x += 300.0 * _randn(g, n, 1)
    x += (200.0 * _randn(g, n, 1)) * torch.linspace(0.0, 1.0, npts, device=DEV)
    return x


def _spectra(g, windows, stations, nspec, delta):
    """Whitened window spectra: a common wavefield delayed per station and each station's noise,
    inside the band's taper (a thousandth of it remains outside)."""
    f = torch.arange(nspec, device=DEV) / (2.0 * (nspec - 1) * delta)
    hi = min(2.0, 0.4 / delta)
    shape = torch.where((f > 0.067) & (f < 1.333 * hi), 1.0, 1e-3)
    delay = 20.0 * torch.rand((stations, 1), generator=g, device=DEV)
    ramp = torch.polar(torch.ones_like(delay * f), -2.0 * math.pi * f * delay)
    out = torch.empty((windows, stations, nspec), dtype=torch.complex64, device=DEV)
    for w in range(windows):
        z = _randn(g, stations, nspec, dtype=torch.complex64)
        z += 0.5 * _randn(g, 1, nspec, dtype=torch.complex64) * ramp
        out[w] = z * shape
    return out


def _records(case, seed):
    """Correlations of the pairs' days: an arrival that recurs, under noise."""
    g, n = _gen(seed), case["n"]
    off = _groups(case)
    t = torch.arange(n, device=DEV) - n // 2
    at = (torch.rand((case["pairs"], 1), generator=g, device=DEV) - 0.5) * 0.8 * n
    arrival = torch.exp(-((t - at) / 30.0) ** 2) * torch.cos(0.4 * (t - at))
    of = torch.from_numpy(np.repeat(np.arange(case["pairs"]), np.diff(off))).to(DEV)
    return (0.05 * (_randn(g, int(off[-1]), n) + 1.5 * arrival[of])).contiguous(), off, of


def prepare(case, seed):
    stage = case["stage"]
    if stage == "s2s":
        seg, nff, nfo, shift, npts = _s2s_shape(case)
        bands = _bands(case)
        resp = np.stack([_power_response(nff, case["delta"], lo, hi) for lo, hi in bands])
        plan = ops.S2sPlan(npts, seg, shift, nff, nfo, case["num_ch"], case["delta"], bands[0][0],
                           _taper_bins(case, seg), resp, [lo for lo, _ in bands], whiten=case["whiten"],
                           normalize=case["normalize"])
        return {"stage": stage, "plan": plan, "x": _traces(case, seed, npts),
                "steps": np.arange(case["windows"], dtype=np.int32)}
    if stage == "xc":
        nspec = _lengths(case)[2] // 2 + 1
        spec = _spectra(_gen(seed), case["windows"], case["stations"], nspec, case["delta"])
        plan = ops.XcPlan(nspec, case["windows"], case["delta"], round(case["lag_s"] / case["delta"]),
                          case["precision"])
        src, rec = _pairs(case["stations"])
        plan.set_pairs(case["stations"], src, rec)
        return {"stage": stage, "plan": plan, "spec": spec}
    if stage == "batch":
        nspec = _lengths(case)[2] // 2 + 1
        sta, win = _batch_sizes(case)
        g = _gen(seed)
        spec = torch.cat([_spectra(g, w, n, nspec, case["delta"]).reshape(-1) for n, w in zip(sta, win)])
        valid = torch.cat([(torch.rand((w * n,), generator=g, device=DEV) > 0.1).to(torch.uint8)
                           for n, w in zip(sta, win)])
        plan = ops.XcBatch(nspec, case["delta"], round(case["lag_s"] / case["delta"]), sta, win,
                           gaps=case["gaps"], max_rows=131072)
        plan.set_grouping(1)
        return {"stage": stage, "plan": plan, "spec": spec, "valid": valid}
    rows, off, of = _records(case, seed)
    count = torch.from_numpy(np.diff(off).astype(np.float32)).to(DEV)
    weights = (1.0 / count)[of].contiguous()
    state = {"stage": stage, "rows": rows, "weights": weights, "off": off}
    if stage == "tfpws":  # rows are sums of ten days each, the linear stack their mean
        lin = torch.zeros((case["pairs"], case["n"]), dtype=torch.float64, device=DEV)
        lin.index_add_(0, of, rows.double())
        state["linear"] = (lin / (10.0 * count.double()[:, None])).float()
        state["band"] = (case["fmin"], case["fmax"], 0.1) if case["fmax"] > 0 else None
        state["delta"] = case["delta"]
    return state


def run(state):
    stage = state["stage"]
    if stage == "s2s":
        return state["plan"].process(state["x"], state["steps"])
    if stage == "xc":
        return state["plan"].correlate(state["spec"])
    if stage == "batch":
        return state["plan"].correlate(state["spec"], state["valid"])
    if stage == "stack":
        lin = ops.linear_stack(state["rows"], state["off"])
        return {"linear": lin, "pws": ops.pws(state["rows"], state["weights"], state["off"], lin)}
    return ops.tfpws(state["rows"], state["weights"], state["off"], state["linear"], band=state["band"],
                     delta=state["delta"])


# -------------------------------------------------------------------- work
def _real_fft(n):
    return 2.5 * n * math.log2(n)


def work(case):
    stage = case["stage"]
    if stage == "s2s":
        seg, nff, nfo, _, npts = _s2s_shape(case)
        rows = case["channels"] * case["windows"]
        ffts = 2 * _real_fft(nff) + _real_fft(nfo)
        ffts += 2 * _real_fft(seg) * {0: 0, 1: 1, 2: 1, 3: 2}[case["whiten"]]
        if case["normalize"] == 1:
            ffts += (1 + len(_bands(case)) - 1) * _real_fft(nff)
        return {"bytes": 4.0 * case["channels"] * npts + 8.0 * rows * (nfo // 2 + 1), "flops": rows * ffts}
    if stage in ("xc", "batch"):
        nfft = _lengths(case)[2]
        nspec, ncc = nfft // 2 + 1, 2 * round(case["lag_s"] / case["delta"]) + 1
        sizes = zip(*_batch_sizes(case)) if stage == "batch" else [(case["stations"], case["windows"])]
        b = f = 0.0
        for n, w in sizes:
            pairs = n * (n - 1) / 2
            b += 8.0 * n * w * nspec + 4.0 * pairs * ncc
            f += pairs * (8.0 * nspec * w + _real_fft(nfft))
        return {"bytes": b, "flops": f}
    n, groups = case["n"], int(_groups(case)[-1])
    if stage == "stack":
        return {"bytes": 4.0 * n * (groups + 2 * case["pairs"]), "flops": groups * (3 * _real_fft(n) + 8.0 * n)}
    voices = n // 2 + 1
    return {"bytes": 4.0 * n * (groups + 2 * case["pairs"]), "flops": (groups + case["pairs"]) * voices * 2 * _real_fft(n)}


# Relative errors between two correct forms, about four times what the present code and the 64-bit
# evaluation below differ by over the ranges of draw().
def tolerance(case):
    stage = case["stage"]
    if stage == "s2s":
        # the sign of samples within rounding of zero decides one-bit outputs
        return {"rel": 4e-3, "max": 0.9} if case["normalize"] == 2 else {"rel": 1e-5, "max": 1e-3}
    if stage in ("xc", "batch"):
        form = case.get("precision", "bf16x3")
        if case.get("windows", 2) == 1:
            form = "fp32"
        return {"fp32": {"rel": 1e-6, "max": 1e-4}, "fp16x3": {"rel": 2e-6, "max": 1e-4},
                "bf16x3": {"rel": 1.5e-5, "max": 1e-3}, "fp16": {"rel": 6e-4, "max": 2e-2}}[form]
    return {"rel": 3e-6, "max": 1e-2} if stage == "stack" else {"rel": 1e-5, "max": 1e-2}


# ----------------------------------------------------------- 64-bit results
def _running_mean(x, win):
    """Centred window sums over the last axis, cut off at its ends, / win."""
    n = x.shape[-1]
    c = torch.nn.functional.pad(torch.cumsum(x, -1), (1, 0))
    start = torch.arange(n, device=x.device) - win // 2
    return (c[..., (start + win).clamp(0, n)] - c[..., start.clamp(0, n)]) / win


def _cos_taper(n, width):
    f = torch.ones(n, dtype=torch.float64, device=DEV)
    i = torch.arange(n, dtype=torch.float64, device=DEV)
    if width > 0:
        f = torch.where(i < width, 0.5 * (1 - torch.cos(math.pi * i / width)), f)
        f = torch.where((i >= width) & (i >= n - width), 0.5 * (1 - torch.cos(math.pi * (n - i) / width)), f)
    return f


def _exact_s2s(case, seed):
    seg, nff, nfo, shift, npts = _s2s_shape(case)
    dt, nch = case["delta"], case["num_ch"]
    x = _traces(case, seed, npts)
    bands = _bands(case)
    resp = [torch.from_numpy(_power_response(nff, dt, lo, hi)).to(DEV).double() for lo, hi in bands]
    dt32, lo32 = float(np.float32(dt)), np.float32(bands[0][0])
    i1, i2, i3, i4 = _taper_bins(case, seg)
    nbin = seg // 2 + 1
    i4 = min(i4, nbin)
    k = torch.arange(nbin, dtype=torch.float64, device=DEV)
    taper = torch.ones(nbin, dtype=torch.float64, device=DEV)
    taper = torch.where((k >= i1) & (k < i2), (1 - torch.cos(math.pi * (k - i1) / max(i2 - i1, 1))) / 2, taper)
    taper = torch.where((k >= i3) & (k < i4), (1 + torch.cos(math.pi * (k - i3) / max(i4 - i3, 1))) / 2, taper)
    taper = torch.where((k < i1) | (k >= i4), 0.0, taper)
    ramp = torch.arange(seg, dtype=torch.float64, device=DEV)
    ramp -= ramp.mean()
    edge = _cos_taper(seg, int(np.float32(np.float32(2.0) * (np.float32(1.0) / lo32)) / np.float32(dt)))

    def band(v, r):
        return torch.fft.irfft(torch.fft.rfft(v, n=nff) * r, n=nff)[..., :seg]

    def whiten(v):
        X = torch.fft.rfft(v)
        win = max(int(0.02 * seg * dt32), 1)
        w = _running_mean(X.abs() * dt32, win).sum(-2, keepdim=True)
        return torch.fft.irfft(X * dt32 / w * taper, n=seg) / dt32

    def running(v, low):
        win = max(2 * int(1.0 / float(np.float32(low) * np.float32(dt))) + 1, 1)
        w = _running_mean(v.abs(), win).sum(-2, keepdim=True)
        return (v / w).clamp(-20.0, 20.0)

    out = torch.empty((case["windows"], case["channels"], nfo // 2 + 1), dtype=torch.complex128, device=DEV)
    block = nch * max(1, 240000000 // (nff * 16 * nch * 4))
    for s in range(case["windows"]):
        for c in range(0, case["channels"], block):
            v = x[c:c + block, s * shift:s * shift + seg].double()
            v = v - v.mean(-1, keepdim=True)
            v = v - (v * ramp).sum(-1, keepdim=True) / (ramp * ramp).sum() * ramp
            v = band((v * edge).reshape(-1, nch, seg), resp[0])
            if case["whiten"] in (1, 3):
                v = whiten(v)
            if case["normalize"] == 1:
                v = sum(running(band(v, r), lo) for r, (lo, _) in zip(resp[1:], bands[1:]))
            elif case["normalize"] == 2:
                v = torch.sign(v)
            elif case["normalize"] == 3:
                v = running(v, lo32 * np.float32(0.667))
            if case["whiten"] in (2, 3):
                v = whiten(v)
            out[s, c:c + block] = torch.fft.rfft(v, n=nfo).reshape(-1, nfo // 2 + 1) * dt32
    return out


def _exact_xc(spec, nfft, half, delta, valid=None):
    """spec [windows, stations, bins]; rows of the pairs i < j, row-major."""
    w, n, nspec = spec.shape
    z = spec.to(torch.complex128).permute(2, 1, 0).contiguous()  # [bin][station][window]
    out = torch.empty((n * (n - 1) // 2, 2 * half + 1), dtype=torch.float64, device=DEV)
    lag = torch.arange(-half, half + 1, device=DEV) % nfft
    step = max(1, min(32, 300000000 // (n * nspec)))
    done = 0
    for a in range(0, n - 1, step):
        b = min(a + step, n - 1)
        x = torch.bmm(z[:, a:b].conj().resolve_conj(), z[:, a + 1:].transpose(1, 2).contiguous())
        i, j = (t.to(DEV) for t in torch.triu_indices(b - a, n - a - 1))
        for c in range(0, len(i), 2048):
            rows = x[:, i[c:c + 2048], j[c:c + 2048]].T.contiguous()
            y = torch.fft.irfft(rows, n=nfft)[:, lag] / delta
            if valid is None:
                y /= w
            else:
                v = valid.double()
                y /= (v[:, a + i[c:c + 2048]] * v[:, a + 1 + j[c:c + 2048]]).sum(0).clamp(min=1.0)[:, None]
            out[done:done + len(y)] = y
            done += len(y)
    return out


def _analytic(x):
    n = x.shape[-1]
    A = 2.0 * torch.fft.fft(x.double())
    A[..., 0] = 0
    A[..., (n + 1) // 2:] = 0
    return A


def exact(case, seed):
    stage = case["stage"]
    if stage == "s2s":
        return _exact_s2s(case, seed)
    state = prepare(case, seed)
    if stage == "xc":
        half = round(case["lag_s"] / case["delta"])
        return _exact_xc(state["spec"], _lengths(case)[2], half, float(np.float32(case["delta"])))
    if stage == "batch":
        nfft, half = _lengths(case)[2], round(case["lag_s"] / case["delta"])
        nspec, parts, at, vat = nfft // 2 + 1, [], 0, 0
        for n, w in zip(*_batch_sizes(case)):
            z = state["spec"][at:at + n * w * nspec].reshape(w, n, nspec)
            v = state["valid"][vat:vat + n * w].reshape(w, n)
            at, vat = at + n * w * nspec, vat + n * w
            parts.append(_exact_xc(z * v[:, :, None], nfft, half, float(np.float32(case["delta"])),
                                   v if case["gaps"] == "exclude" else None))
        return torch.cat(parts)
    n, off = case["n"], state["off"]
    of = torch.from_numpy(np.repeat(np.arange(case["pairs"]), np.diff(off))).to(DEV)
    if stage == "stack":
        total = torch.zeros((case["pairs"], n), dtype=torch.float64, device=DEV)
        total.index_add_(0, of, state["rows"].double())
        lin = total / torch.from_numpy(np.diff(off)).to(DEV).double()[:, None]
        W = torch.zeros((case["pairs"], n), dtype=torch.complex128, device=DEV)
        for a in range(0, len(of), 16384):
            z = torch.fft.ifft(_analytic(state["rows"][a:a + 16384]))
            z /= z.abs().clamp(min=1e-7)
            W.index_add_(0, of[a:a + 16384], z * state["weights"][a:a + 16384].double()[:, None])
        return {"linear": lin, "pws": lin * W.abs()}
    half, voices = (n + 1) // 2, n // 2 + 1
    Ag, Al = _analytic(state["rows"]), _analytic(state["linear"])
    c = torch.arange(n, dtype=torch.float64, device=DEV)
    c = torch.where(c < half, c, n - c)
    wg = state["weights"].double()
    v = torch.zeros((case["pairs"], n), dtype=torch.complex128, device=DEV)
    for f in range(voices):
        g = torch.ones_like(c) if f == 0 else torch.exp(-0.2 * math.pi ** 2 * c * c / (f * f)) * (c > 0) * (c < half)
        W = torch.zeros((case["pairs"], n), dtype=torch.complex128, device=DEV)
        z = torch.fft.ifft(torch.roll(Ag, -f, -1) * g, norm="forward")
        m = z.abs()
        W.index_add_(0, of, z * (wg[:, None] / (torch.where(m <= 1e-7, 1.0, m) * n)))
        v[:, f] = (torch.fft.ifft(torch.roll(Al, -f, -1) * g, norm="forward") * W.abs()).sum(-1)
    if state["band"] is not None:
        fmin, fmax, taper = state["band"]
        taper = min(taper, 0.5 * (fmax - fmin))
        fr = torch.arange(voices, dtype=torch.float64, device=DEV) / (n * case["delta"])
        inside = (fr >= fmin) & (fr <= fmax)
        edge = torch.minimum(fr - fmin, fmax - fr).clamp(0.0, taper)
        alpha = torch.where(inside, 0.5 - 0.5 * torch.cos(math.pi * edge / taper), 0.0)
        mixed = Al.clone()
        mixed[:, :voices] = Al[:, :voices] * (1 - alpha) + v[:, :voices] * alpha
        v = mixed
    return torch.fft.ifft(v).real
