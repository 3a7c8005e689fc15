"""Timed workloads of the engine, through its public Python entry points.

Each case stands for one thing that a user has the engine do: a request for
one short trace, a minute pushed into a stream, a whole day of a network, an
uneven batch, short templates on every path that takes them, the Detector
steps on computed rows, and requests served from a resident library.  The
sizes are those of bench.py's workloads and of the tests, from the smallest
calls to the largest.

Inputs are made on the GPU from the seed: band-passed Gaussian noise with a
DC offset, Hann-tapered band-limited template bursts, injected events, and
(short templates) gaps that hold a constant.
"""
import math
import random

import numpy as np
import torch

from mflib_amd import capi

FS = 100.0
DTYPES = {"f32": (np.float32, torch.float32), "f64": (np.float64, torch.float64)}


# ---- the cases ------------------------------------------------------------
def listed():
    return [
        # One hour of one channel against one template in FP64, the plain
        # request: hand the trace over, correlate, find the peaks.
        {"name": "hour_single_f64", "kind": "net", "dtype": "f64", "events": 1, "channels": 1, "n": 360_000,
         "lt": 400, "load": True},
        # A multi-channel event on two and a half hours of a network in FP64,
        # the precision of the Python API.
        {"name": "network_hours_f64", "kind": "net", "dtype": "f64", "events": 1, "channels": 24, "n": 900_001,
         "lt": 700, "load": True},
        # A minute of 24 channels pushed into a live stream of 16 events.
        {"name": "push_minute_f32", "kind": "push", "dtype": "f32", "events": 16, "channels": 24, "n": 6_000, "lt": 512},
        # A day of 24 channels against 16 events, the largest batch.
        {"name": "network_day_f32", "kind": "net", "dtype": "f32", "events": 16, "channels": 24, "n": 8_640_000,
         "lt": 512, "load": False},
        # Templates of 200-3000 samples on channels of 1-8 hours, every
        # template with its own length and channels.
        {"name": "uneven_f32", "kind": "uneven", "dtype": "f32", "events": 28, "channels": 28, "n": 2_880_000,
         "lt": 3_000, "mix": 4},
        # 256 templates of 128-256 samples on gappy channels with a large DC
        # offset: the FFT path ...
        {"name": "short_fft_f32", "kind": "short", "variant": 0, "templates": 256, "channels": 4, "n": 2_000_000,
         "lt": 256, "mix": 3},
        # ... and the matrix-core paths, at odd sizes.
        {"name": "short_fp16_f32", "kind": "short", "variant": 3, "templates": 256, "channels": 4, "n": 1_000_003,
         "lt": 256, "mix": 3},
        {"name": "short_bf16_f32", "kind": "short", "variant": 4, "templates": 150, "channels": 3, "n": 500_001,
         "lt": 200, "mix": 5},
        # The Detector on computed rows: maximum over the templates, its
        # peaks, and their refined times and amplitudes.
        {"name": "detector_reduced_f32", "kind": "detector", "dtype": "f32", "policy": "reduced", "templates": 128,
         "n": 1_000_000, "lt": 256},
        # The Detector's other policy, one peak list per template.
        {"name": "detector_single_f64", "kind": "detector", "dtype": "f64", "policy": "single", "templates": 40,
         "n": 720_000, "lt": 300},
        # One small request to a server, waited for.
        {"name": "serve_one_f32", "kind": "serve", "dtype": "f32", "requests": 1, "channels": 3, "templates": 5,
         "n": 6_000, "mix": 1},
        # Requests of every size, batched.
        {"name": "serve_mix_f32", "kind": "serve", "dtype": "f32", "requests": 24, "channels": 48, "templates": 100,
         "n": 360_000, "mix": 7},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["net", "net", "push", "uneven", "short", "short", "detector", "serve"])
    if kind == "net":
        dtype = rng.choice(["f32", "f64"])
        n = _log(rng, 20_000, 8_640_000 if dtype == "f32" else 2_000_000)
        rows = max(1, min(384, int(3.0e9 / n) if dtype == "f32" else int(1.0e8 / n)))
        events = _log(rng, 1, min(16, rows))
        return {"kind": "net", "dtype": dtype, "events": events,
                "channels": _log(rng, 1, max(1, min(24, rows // events))), "n": n,
                "lt": _log(rng, 100, 2_500 if dtype == "f32" else 1_500), "load": rng.random() < 0.5}
    if kind == "push":
        return {"kind": "push", "dtype": rng.choice(["f32", "f32", "f64"]), "events": _log(rng, 1, 16),
                "channels": _log(rng, 1, 24), "n": _log(rng, 500, 30_000), "lt": _log(rng, 100, 1_000)}
    if kind == "uneven":
        return {"kind": "uneven", "dtype": "f32", "events": _log(rng, 4, 28), "channels": _log(rng, 4, 28),
                "n": _log(rng, 400_000, 2_880_000), "lt": _log(rng, 800, 3_000), "mix": rng.randrange(1 << 20)}
    if kind == "short":
        return {"kind": "short", "variant": rng.choice([0, 3, 4]), "templates": _log(rng, 8, 256),
                "channels": rng.randint(1, 4), "n": _log(rng, 50_000, 2_000_000), "lt": _log(rng, 40, 256),
                "mix": rng.randrange(1 << 20)}
    if kind == "detector":
        dtype = rng.choice(["f32", "f64"])
        return {"kind": "detector", "dtype": dtype, "policy": rng.choice(["reduced", "single"]),
                "templates": _log(rng, 4, 128 if dtype == "f32" else 40), "n": _log(rng, 60_000, 1_000_000),
                "lt": _log(rng, 100, 600)}
    return {"kind": "serve", "dtype": "f32", "requests": _log(rng, 1, 24), "channels": _log(rng, 1, 48),
            "templates": _log(rng, 1, 100), "n": _log(rng, 6_000, 360_000), "mix": rng.randrange(1 << 20)}


# ---- sizes that follow from a case (not from the seed) -----------------------
def _uneven_shape(case):
    r = random.Random(case["mix"])
    ns = [r.randint(case["n"] // 8, case["n"]) for _ in range(case["channels"])]
    lts = [r.randint(200, case["lt"]) for _ in range(case["events"])]
    chans = [sorted(r.sample(range(case["channels"]), r.randint(1, case["channels"]))) for _ in lts]
    return ns, lts, chans


def _moveouts(case):
    """Moveout of every channel for every event, in samples."""
    r = random.Random(1000 * case["events"] + case["channels"])
    most = min(200, max(1, case["n"] // 20))
    return [[r.randint(0, most) for _ in range(case["channels"])] for _ in range(case["events"])]


def _uneven_moveouts(case):
    r = random.Random(case["mix"] + 1)
    return [r.randint(0, 500) for cs in _uneven_shape(case)[2] for _ in cs]


def _short_lengths(case):
    r = random.Random(case["mix"])
    return [r.randint(max(8, case["lt"] // 2), case["lt"]) for _ in range(case["templates"])]


def _detector_lengths(case):
    return [case["lt"] - (i % 8) * (case["lt"] // 16) for i in range(case["templates"])]


def _serve_library(case):
    r = random.Random(case["mix"] + 1)
    return [r.randint(200, 2_000) for _ in range(120)]


def _serve_shapes(case):
    """(channels, window, template ids) of every request of a pass."""
    r = random.Random(case["mix"])
    lib = _serve_library(case)
    if case["requests"] == 1:
        ids = sorted(r.sample(range(len(lib)), case["templates"]))
        return [(case["channels"], max(case["n"], 2_600), ids)]
    out = []
    for _ in range(case["requests"]):
        n = max(_log(r, 6_000, max(case["n"], 6_000)), 2_600)
        ids = sorted(r.sample(range(len(lib)), r.randint(1, case["templates"])))
        out.append((r.randint(1, case["channels"]), n, ids))
    return out


# ---- inputs -----------------------------------------------------------------
def _smooth(n):
    """The smallest length >= n of the form 2^a 3^b 5^c with a >= 4."""
    best = None
    for b in range(3):
        for c in range(3):
            m = 16 * 3 ** b * 5 ** c
            while m < n:
                m *= 2
            best = m if best is None or m < best else best
    return best


def _noise(g, rows, n, lo=1.0, hi=10.0):
    """Band-passed Gaussian noise of unit RMS, [rows, n] FP32."""
    m = _smooth(n)
    x = torch.fft.rfft(torch.randn(rows, m, generator=g, device="cuda"))
    f = torch.arange(m // 2 + 1, device="cuda", dtype=torch.float32) * (FS / m)
    resp = 1.0 / torch.sqrt(1.0 + ((f * f - lo * hi) / ((hi - lo) * f.clamp_min(1e-6))) ** 4)
    x = torch.fft.irfft(x * resp, n=m)[:, :n]
    return x / x.square().mean().sqrt()


def _bursts(g, lengths, lo=1.0, hi=10.0):
    """Unit-energy Hann-tapered bursts on the GPU, FP64, [rows, longest] with
    zeros past each row's length."""
    most = max(lengths)
    x = torch.cat([_noise(g, min(256, len(lengths) - k), most, lo, hi) for k in range(0, len(lengths), 256)]).double()
    L = torch.tensor(lengths, device="cuda", dtype=torch.float64)[:, None]
    k = torch.arange(most, device="cuda", dtype=torch.float64)[None, :]
    x = x * torch.where(k < L, 0.5 - 0.5 * torch.cos(2 * math.pi * k / (L - 1)), torch.zeros_like(x))
    return x / x.square().sum(1, keepdim=True).sqrt()


def _origins(r, n, span, count):
    """Injection origins, one in each of `count` equal cells, `span` samples apart at least."""
    count = max(1, min(count, n // (2 * span)))
    cell = n // count
    room = max(1, cell - span)
    return [k * cell + r.randrange(room) for k in range(count)]


def _place(x, chans, starts, waves):
    """x[chans[i], starts[i] + k] += waves[i, k]; the places are distinct."""
    at = starts[:, None] + torch.arange(waves.shape[1], device="cuda")[None, :]
    ok = at < x.shape[1]
    at = at.clamp_max(x.shape[1] - 1)
    c = chans[:, None].expand_as(at)
    x[c[ok], at[ok]] = x[c[ok], at[ok]] + waves[ok].to(x.dtype)


def _net_inputs(case, seed):
    """Signals [channels][n], templates [event, channel] and moveouts."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = random.Random(seed)
    E, C, n, lt = case["events"], case["channels"], case["n"], case["lt"]
    x = torch.cat([_noise(g, min(8, C - k), n) for k in range(0, C, 8)])
    t = _bursts(g, [lt] * (E * C)).view(E, C, lt)
    shifts = _moveouts(case)
    most = max(max(v) for v in shifts)
    cs = torch.arange(C, device="cuda")
    for e in range(E):
        sh = torch.tensor(shifts[e], device="cuda")
        for o in _origins(r, n - lt - most - 1, lt + most, 50):
            amp = 0.6 + 0.9 * torch.rand(C, 1, generator=g, device="cuda")
            _place(x, cs, sh + o, amp * math.sqrt(lt) * t[e])
    x = x + (200.0 * torch.rand(C, 1, generator=g, device="cuda") - 100.0)
    return x.to(DTYPES[case["dtype"]][1]), t, shifts


def _uneven_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = random.Random(seed)
    ns, lts, chans = _uneven_shape(case)
    x = [_noise(g, 1, n)[0] for n in ns]
    pairs = [(e, c) for e in range(len(lts)) for c in chans[e]]
    t = _bursts(g, [lts[e] for e, _ in pairs])
    shifts = _uneven_moveouts(case)
    for e in range(len(lts)):
        mine = [k for k, p in enumerate(pairs) if p[0] == e]
        span = min(ns[c] for c in chans[e]) - lts[e] - 501
        for o in _origins(r, span, lts[e] + 500, 6):
            for k in mine:
                c = pairs[k][1]
                w = t[k, :lts[e]] / t[k].abs().max()
                x[c][o + shifts[k]:o + shifts[k] + lts[e]] += (r.uniform(2.0, 6.0) * w).float()
    return [v + r.uniform(-100.0, 100.0) for v in x], t, pairs, shifts


def _short_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = random.Random(seed)
    C, n, lts = case["channels"], case["n"], _short_lengths(case)
    x = _noise(g, C, n, 2.0, 20.0).double()
    t = _bursts(g, lts, 2.0, 20.0)
    for c in range(C):
        for o in _origins(r, n - case["lt"], case["lt"], 30):
            k = r.randrange(len(lts))
            x[c, o:o + lts[k]] += 5.0 * t[k, :lts[k]] / t[k].abs().max()
        x[c] += 1.0e4
        for _ in range(max(1, min(20, n // 50_000))):
            m = r.randint(500, 5_000)
            o = r.randrange(n - m)
            x[c, o:o + m] = 1.0e4 + r.uniform(-50.0, 50.0) + 1e-6 * torch.randn(m, generator=g, device="cuda").double()
    return x.float(), t, lts


def _detector_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = random.Random(seed)
    lts, n = _detector_lengths(case), case["n"]
    x = _noise(g, 1, n)[0].double()
    t = _bursts(g, lts)
    for o in _origins(r, n - case["lt"], case["lt"], 400):
        k = r.randrange(len(lts))
        x[o:o + lts[k]] += r.uniform(1.5, 4.0) * math.sqrt(lts[k]) * t[k, :lts[k]]
    return (x + 30.0).to(DTYPES[case["dtype"]][1]), t, lts


def _serve_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    lib = _serve_library(case)
    t = _bursts(g, lib)
    windows = []
    for nc, n, ids in _serve_shapes(case):
        x = _noise(g, nc, n) + (200.0 * torch.rand(nc, 1, generator=g, device="cuda") - 100.0)
        for k, i in enumerate(ids[:4]):  # a few of its templates are in the window
            o = (n - lib[i]) * k // 4
            x[:, o:o + lib[i]] += (3.0 * math.sqrt(lib[i]) * t[i, :lib[i]]).float()
        windows.append(x.contiguous())
    return windows, t, lib


# ---- device memory of the engine as torch tensors ------------------------------
class _Memory:
    """Device memory of `owner` (a Handle or Server), which lives as long as
    any tensor over it."""

    def __init__(self, owner, ptr, shape, strides, dtype):
        d = np.dtype(dtype)
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": d.str, "data": (int(ptr), False),
                                         "strides": tuple(int(s) * d.itemsize for s in strides), "version": 3}


def _view(owner, ptr, shape, strides, dtype):
    return torch.as_tensor(_Memory(owner, ptr, shape, strides, dtype), device="cuda")


def _rows_view(handle, rows):
    """The correlation rows `rows` (consecutive, of one length) as one tensor."""
    n = handle.filtered_length(rows[0])
    p0 = handle.rho_device_ptr(rows[0])
    item = handle.dtype.itemsize
    ld = (handle.rho_device_ptr(rows[1]) - p0) // item if len(rows) > 1 else n
    return _view(handle, p0, (len(rows), n), (ld, 1), handle.dtype)


def _stack_views(handle):
    got = []
    for k in range(handle.number_of_groups()):
        p, n = handle.stack_device(k)
        got.append(_view(handle, p, (n,), (1,), handle.dtype))
    return got


def _host(t, lengths):
    t = t.cpu().numpy()
    return [np.ascontiguousarray(t[i, :m]) for i, m in enumerate(lengths)]


def _listed(values, dtype, room=8_192):
    """A list of peaks or products with room for more of them, as the C
    interface fills it."""
    out = np.zeros(room, dtype=dtype)
    out[:len(values)] = values
    return out


# ---- prepare and run ----------------------------------------------------------
def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, seed)
    torch.cuda.synchronize()  # the engine reads the inputs from its own streams
    return state


def run(state):
    return state["pass"](state)


def _net_handle(case, t, shifts, streaming=False):
    E, C, n, lt = case["events"], case["channels"], case["n"], case["lt"]
    h = capi.Handle(DTYPES[case["dtype"]][0], "batched")
    h.set_templates(_host(t.reshape(E * C, lt), [lt] * (E * C)), shifts=sum(shifts, []), weights=[1.0] * (E * C))
    h.set_batch_layout([n] * C, list(range(C)) * E, np.repeat(np.arange(E), C), E)
    if streaming:
        h.set_streaming(True)
    h.initialize()
    return h


def _prepare_net(case, seed):
    x, t, shifts = _net_inputs(case, seed)
    h = _net_handle(case, t, shifts)
    if not case["load"]:
        for c in range(case["channels"]):
            h.set_signal_device(c, x[c].data_ptr(), case["n"])
    return {"pass": _run_net, "case": case, "h": h, "x": x, "stacks": None,
            "rho": _rows_view(h, range(case["events"] * case["channels"]))}


def _run_net(s):
    h, x = s["h"], s["x"]
    if s["case"]["load"]:
        for c in range(x.shape[0]):
            h.set_signal_device(c, x[c].data_ptr(), x.shape[1])
    h.apply()
    peaks = h.detect(0.5, s["case"]["lt"])
    if s["stacks"] is None:
        s["stacks"] = _stack_views(h)
    return {"rho": s["rho"], "stacks": s["stacks"], "peaks": _listed(np.concatenate(peaks), np.int64)}


def _prepare_push(case, seed):
    x, t, shifts = _net_inputs(case, seed)
    h = _net_handle(case, t, shifts, streaming=True)
    return {"pass": _run_push, "case": case, "h": h, "x": x, "stacks": None,
            "rho": _rows_view(h, range(case["events"] * case["channels"]))}


def _run_push(s):
    h, x = s["h"], s["x"]
    h.push_chunks_device([x[c].data_ptr() for c in range(x.shape[0])], x.shape[1])
    h.apply()
    peaks = h.stream_peaks_all(0.5, s["case"]["lt"])
    if s["stacks"] is None:
        s["stacks"] = _stack_views(h)
    return {"rho": s["rho"], "stacks": s["stacks"], "peaks": _listed(np.concatenate(peaks), np.int64)}


def _prepare_uneven(case, seed):
    x, t, pairs, shifts = _uneven_inputs(case, seed)
    ns, lts, _ = _uneven_shape(case)
    h = capi.Handle(np.float32, "batched")
    h.set_templates(_host(t, [lts[e] for e, _ in pairs]), shifts=shifts, weights=[1.0] * len(pairs))
    h.set_batch_layout(ns, [c for _, c in pairs], [e for e, _ in pairs], len(lts))
    h.set_graph_launch(True)
    h.initialize()
    for c in range(len(ns)):
        h.set_signal_device(c, x[c].data_ptr(), ns[c])
    groups = [[k for k, p in enumerate(pairs) if p[0] == e] for e in range(len(lts))]
    return {"pass": _run_uneven, "h": h, "stacks": None, "rho": [_rows_view(h, rows) for rows in groups]}


def _run_uneven(s):
    h = s["h"]
    h.apply()
    peaks = h.detect(0.6, 500)
    if s["stacks"] is None:
        s["stacks"] = _stack_views(h)
    return {"rho": s["rho"], "stacks": s["stacks"], "peaks": _listed(np.concatenate(peaks), np.int64)}


def _prepare_short(case, seed):
    x, t, lts = _short_inputs(case, seed)
    C, T = case["channels"], len(lts)
    h = capi.Handle(np.float32, "batched")
    h.set_templates(_host(t, lts) * C)
    h.set_batch_layout([case["n"]] * C, np.repeat(np.arange(C), T), np.repeat(np.arange(C), T), C)
    if case["variant"]:
        h.set_kernel_variant(case["variant"])
    h.initialize()
    for c in range(C):
        h.set_signal_device(c, x[c].data_ptr(), case["n"])
    return {"pass": _run_short, "h": h, "rho": _rows_view(h, range(C * T))}


def _run_short(s):
    s["h"].apply()
    return s["rho"]


def _prepare_detector(case, seed):
    x, t, lts = _detector_inputs(case, seed)
    dtype, ttype = DTYPES[case["dtype"]]
    h = capi.Handle(dtype, "single")
    h.set_templates(_host(t, lts))
    h.set_signal_size(case["n"])
    h.initialize()
    h.set_signal_device(0, x.data_ptr(), case["n"])
    h.apply()
    h.synchronize()
    n = h.filtered_length(0)
    return {"pass": _run_reduced if case["policy"] == "reduced" else _run_single, "case": case, "h": h, "n": n,
            "det": torch.empty(n, dtype=ttype, device="cuda"), "ids": torch.empty(n, dtype=torch.int32, device="cuda")}


def _run_reduced(s):
    h, n, case = s["h"], s["n"], s["case"]
    h.reduce_device(0, False, s["det"].data_ptr(), s["ids"].data_ptr(), n)
    peaks = capi.peaks_device(s["det"].data_ptr(), n, h.dtype, 0.6, case["lt"], cap=65_536)
    ids = s["ids"][torch.from_numpy(peaks).to("cuda", torch.int64)].cpu().numpy()
    products = h.detection_products(peaks, ids, [1.0 / FS] * case["templates"], interpolation=capi.INTERP_QUADRATIC)
    return {"det": s["det"], "ids": s["ids"], "peaks": _listed(peaks, np.int64), "count": len(peaks),
            "products": {k: _listed(v, v.dtype) for k, v in products.items()}}


def _run_single(s):
    h, case = s["h"], s["case"]
    lists = h.detect_templates(0.6, case["lt"], cap=1 << 20)
    peaks = np.concatenate(lists)
    ids = np.repeat(np.arange(case["templates"], dtype=np.int32), [len(v) for v in lists])
    products = h.detection_products(peaks, ids, [1.0 / FS] * case["templates"],
                                    interpolation=capi.INTERP_LANCZOS)
    return {"peaks": _listed(peaks, np.int64), "ids": _listed(ids, np.int32), "count": len(peaks),
            "products": {k: _listed(v, v.dtype) for k, v in products.items()}}


def _prepare_serve(case, seed):
    windows, t, lib = _serve_inputs(case, seed)
    shapes = _serve_shapes(case)
    need = sum(4 * (nc * len(ids) * (n + 256) + 64) for nc, n, ids in shapes)
    s = capi.Server(np.float32, budget_bytes=float(2 * need + (64 << 20)), max_batch=64, max_inflight=2)
    s.add_templates(_host(t, lib))
    return {"pass": _run_serve, "server": s, "windows": windows, "shapes": shapes, "held": []}


def _run_serve(s):
    srv = s["server"]
    for rid in s["held"]:  # the last pass's rows go back before new requests come
        srv.release(rid)
    s["held"] = [srv.submit([w[c].data_ptr() for c in range(nc)], ids, on_device=True, lengths=[n] * nc)
                 for w, (nc, n, ids) in zip(s["windows"], s["shapes"])]
    rows = []
    for rid, (nc, _, ids) in zip(s["held"], s["shapes"]):
        srv.wait(rid)
        count = nc * len(ids)
        p, n = srv.rho_device(rid, 0, 0)
        last = srv.rho_device(rid, len(ids) - 1, nc - 1)[0]
        ld = (last - p) // 4 // (count - 1) if count > 1 else n
        rows.append(_view(srv, p, (count, n), (ld, 1), np.float32))
    return rows


# ---- what a pass cannot do without -------------------------------------------
def _fft_flops(outputs, nb):
    """Operations of `outputs` correlation outputs by blocks of four template lengths."""
    return outputs * (5.0 * math.log2(4 * nb) + 6.0)


def work(case):
    kind = case["kind"]
    if kind in ("net", "push"):
        size = 4 if case["dtype"] == "f32" else 8
        E, C, n, lt = case["events"], case["channels"], case["n"], case["lt"]
        outs = float(E * C) * (n - lt + 1 if kind == "net" else n)
        return {"bytes": size * (C * n + outs + E * n) + 8.0 * E * C * lt, "flops": _fft_flops(outs, lt) + 2 * outs}
    if kind == "uneven":
        ns, lts, chans = _uneven_shape(case)
        outs = flops = stacks = 0.0
        for lt, cs in zip(lts, chans):
            m = min(ns[c] for c in cs) - lt + 1
            outs += m * len(cs)
            stacks += m
            flops += _fft_flops(m * len(cs), lt)
        return {"bytes": 4.0 * (sum(ns) + outs + stacks), "flops": flops + 2 * outs}
    if kind == "short":
        lts = _short_lengths(case)
        outs = float(case["channels"]) * len(lts) * (case["n"] - max(lts) + 1)
        return {"bytes": 4.0 * (case["channels"] * case["n"] + outs), "flops": _fft_flops(outs, max(lts))}
    if kind == "detector":
        size = 4 if case["dtype"] == "f32" else 8
        outs = float(case["templates"]) * (case["n"] - case["lt"] + 1)
        back = (size + 4) * (case["n"] - case["lt"] + 1) if case["policy"] == "reduced" else 0
        return {"bytes": size * outs + back, "flops": 2 * outs}
    lib = _serve_library(case)
    outs = flops = ins = 0.0
    for nc, n, ids in _serve_shapes(case):
        nb = max(lib[i] for i in ids)
        outs += float(nc) * len(ids) * (n - nb + 1)
        flops += nc * sum(_fft_flops(n - nb + 1, lib[i]) for i in ids)
        ins += nc * n + 2 * sum(lib[i] for i in ids)
    return {"bytes": 4.0 * (ins + outs), "flops": flops}


def tolerance(case):
    # four times the error against 64 bits that the paths show
    if case.get("dtype") == "f64":
        return {"rel": 1e-12, "max": 1e-10}
    if case["kind"] == "detector":
        # a refined time is a small difference of neighbouring lags, and the
        # maximum over rows may fall on another row where two agree to
        # rounding
        return {"rel": 2e-5, "max": 5e-4, "differ": 1e-4}
    # "max": the correlations' contract, 1e-5 absolute, over their RMS
    return {"rel": 1.5e-6, "max": 1e-4}


# ---- the values in 64 bits, by plain torch -------------------------------------
def _pearson(x, templates, lengths, n_out):
    """Pearson correlation rows [len(templates)][n_out] of one FP64 signal."""
    n = x.numel()
    m = _smooth(n)
    x = x - x.mean()
    X = torch.fft.rfft(x, n=m)
    zero = x.new_zeros(1)
    p1, p2 = torch.cat([zero, x.cumsum(0)]), torch.cat([zero, x.square().cumsum(0)])
    same = torch.cat([zero.long(), (x[1:] == x[:-1]).long().cumsum(0)])
    out = x.new_empty(len(templates), n_out)
    for k, (t, lt) in enumerate(zip(templates, lengths)):
        t = t[:lt] - t[:lt].mean()
        t = t / t.square().sum().sqrt()
        num = torch.fft.irfft(X * torch.fft.rfft(t, n=m).conj(), n=m)[:n_out]
        s1 = p1[lt:lt + n_out] - p1[:n_out]
        var = p2[lt:lt + n_out] - p2[:n_out] - s1 * s1 / lt
        flat = same[lt - 1:lt - 1 + n_out] - same[:n_out] == lt - 1
        out[k] = torch.where(flat, torch.zeros_like(num), num / var.clamp_min(1e-300).sqrt())
    return out


def _stack(rho, shifts):
    n = rho.shape[1] - max(shifts)
    return sum(rho[k, s:s + n].abs() for k, s in enumerate(shifts)) / len(shifts)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("net", "push"):
        x, t, shifts = _net_inputs(case, seed)
        E, C, n, lt = case["events"], case["channels"], case["n"], case["lt"]
        if kind == "push":  # the first push of a stream: the carry before it is zeros
            carry = lt - 1 + max(max(s) for s in shifts)
            x = torch.cat([x.new_zeros(C, carry), x], 1)
            n = n + carry
        m = n - lt + 1
        rho = torch.empty(E * C, m, dtype=torch.float64, device="cuda")
        for c in range(C):
            rho[c::C] = _pearson(x[c].double(), list(t[:, c]), [lt] * E, m)
        return {"rho": rho, "stacks": [_stack(rho[e * C:(e + 1) * C], shifts[e]) for e in range(E)], "peaks": None}
    if kind == "uneven":
        x, t, pairs, shifts = _uneven_inputs(case, seed)
        ns, lts, chans = _uneven_shape(case)
        rows, stacks = [], []
        for e, lt in enumerate(lts):
            mine = [k for k, p in enumerate(pairs) if p[0] == e]
            m = min(ns[c] for c in chans[e]) - lt + 1
            rho = torch.cat([_pearson(x[pairs[k][1]].double(), [t[k]], [lt], m) for k in mine])
            rows.append(rho)
            stacks.append(_stack(rho, [shifts[k] for k in mine]))
        return {"rho": rows, "stacks": stacks, "peaks": None}
    if kind == "short":
        x, t, lts = _short_inputs(case, seed)
        m = case["n"] - max(lts) + 1
        rho = torch.empty(case["channels"] * len(lts), m, dtype=torch.float64, device="cuda")
        for c in range(case["channels"]):
            rho[c * len(lts):(c + 1) * len(lts)] = _pearson(x[c].double(), list(t), lts, m)
        return rho
    if kind == "detector":
        if case["policy"] != "reduced":
            return None
        x, t, lts = _detector_inputs(case, seed)
        det = _pearson(x.double(), list(t), lts, case["n"] - max(lts) + 1).amax(0).clamp(-1.0, 1.0)
        return {"det": det, "ids": None, "peaks": None, "count": None, "products": None}
    windows, t, lib = _serve_inputs(case, seed)
    rows = []
    for x, (nc, n, ids) in zip(windows, _serve_shapes(case)):
        m = n - max(lib[i] for i in ids) + 1
        rho = torch.empty(len(ids), nc, m, dtype=torch.float64, device="cuda")
        for c in range(nc):
            rho[:, c] = _pearson(x[c].double(), [t[i] for i in ids], [lib[i] for i in ids], m)
        rows.append(rho.view(len(ids) * nc, m))
    return rows
