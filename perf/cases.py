"""Cases for measuring the compositing paths through the package's public entry points.

Each case is a plain dict; prepare() builds what a program holds before the call (a resident
stack generated from the seed, output buffers, a planned batch, a running server) and run() makes
one pass.  Outputs are whole numbers (image samples, mask bytes, pixel offsets), so there is no
64-bit value to compare them with: they have to stay equal.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "chrono-photo_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "chrono-photo_amd"))
import chrono_photo_amd as cpa  # noqa: E402

_state = {}


def _context():
    """One context for the process, as a program has it."""
    if "ctx" not in _state:
        torch.cuda.init()
        _state["ctx"] = cpa.Context(0)
    return _state["ctx"]


# ------------------------------------------------------------------------------ the cases

def _outlier(name, width, height, channels, bps, frames, threshold, background, outlier, **more):
    c = {"name": name, "kind": "outlier", "width": width, "height": height, "channels": channels, "bps": bps,
         "frames": frames, "threshold": threshold, "background": background, "outlier": outlier, "crop": 0,
         "sample": 0, "weights": "", "fade": ""}
    c.update(more)
    return c


def listed():
    return [
        # a short hand-held burst at VGA size: the smallest ordinary call, bound by its latency
        _outlier("burst_vga_16f", 640, 480, 3, 1, 16, "abs/0.05/0.2", "first", "extreme"),
        # one photo from a full-HD burst, thresholds relative to each pixel's own spread
        _outlier("hd_64f_relative", 1920, 1080, 3, 1, 64, "rel/2.0/4.0", "first", "average"),
        # star trails and light painting: the lighter mode over the same burst
        {"name": "hd_64f_lighter", "kind": "simple", "width": 1920, "height": 1080, "channels": 3, "bps": 1,
         "frames": 64, "darker": False, "crop": 0, "fade": ""},
        # 4K frames developed to 16 bits, stabilised by per-frame crops: the headline composite
        _outlier("uhd_rgb16_256f", 3840, 2160, 3, 2, 256, "abs/0.05/0.2", "first", "forward", crop=8),
        # the stabilisation of that stack: 5 anchors, radius 32, search radius 12
        {"name": "uhd_rgb16_256f_shake", "kind": "shake", "width": 3840, "height": 2160, "channels": 3, "bps": 2,
         "frames": 256, "anchors": 5, "radius": 32, "search": 12},
        # a night's queue: 48 stacks of uneven sizes, thresholds and modes in one planned batch
        {"name": "batch_48_stacks", "kind": "batch", "jobs": 48, "min_frames": 8, "max_frames": 200,
         "min_width": 640, "max_width": 1920},
        # a chrono-video: windows of 60 frames at stride 1 over a resident full-HD stream, served
        {"name": "video_hd_60f_windows", "kind": "video", "width": 1920, "height": 1080, "channels": 3,
         "window": 60, "windows": 24, "threshold": "abs/0.05/0.2", "outlier": "extreme"},
        # a gallery photo: 1200 full-HD frames of a longer time lapse
        _outlier("gallery_1200f", 1920, 1080, 3, 1, 1200, "abs/0.05/0.2", "first", "extreme"),
        # the same with the medians taken from 64 of the frames (--sample)
        _outlier("gallery_1200f_sample64", 1920, 1080, 3, 1, 1200, "abs/0.05/0.2", "first", "extreme", sample=64),
        # a long time lapse with relative thresholds, outliers fading out over the last frames
        _outlier("lapse_700f_relative", 1280, 720, 3, 1, 700, "rel/2.5/5.0", "average", "backward",
                 fade="clamp/rel/0,1.0/300,0.25"),
        # a monochrome 16-bit camera at an odd size
        _outlier("mono16_100f", 1937, 1091, 1, 2, 100, "abs/0.05/0.2", "median", "extreme"),
        # 16-bit colour frames with --sample
        _outlier("rgb16_300f_sample48", 960, 541, 3, 2, 300, "abs/0.05/0.2", "first", "last", sample=48),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, frames, px_bytes, most):
    """Width and height of any parity, at most `most` bytes of stack."""
    w = _log_uniform(rng, 160, 3840)
    h = max(90, int(w * rng.choice((9 / 16, 2 / 3, 3 / 4))) + rng.randrange(-3, 4))
    while w * h * frames * px_bytes > most and w > 64:
        w, h = max(64, int(w * 0.83)), max(40, int(h * 0.83))
    return w, h


def draw(rng):
    kind = rng.choices(("outlier", "simple", "shake", "batch", "video"), (12, 3, 2, 1, 2))[0]
    if kind == "outlier":
        bps = rng.choice((1, 1, 1, 2))
        channels = rng.choice((1, 2, 3, 3, 3, 3, 4, 4))
        frames = _log_uniform(rng, 5, 1200 if bps == 1 else 480)
        # bytes bounded so that no drawn composite costs more than the largest listed ones
        w, h = _size(rng, frames, channels * bps, 3.0e9 if bps == 1 else 4.0e8)
        relative = frames >= 8 and rng.random() < 0.4
        sample = rng.randrange(5, min(frames, 96)) if frames > 40 and rng.random() < 0.25 else 0
        return {"kind": kind, "width": w, "height": h, "channels": channels, "bps": bps, "frames": frames,
                "threshold": rng.choice(("rel/2.0/4.0", "rel/3.0", "rel/1.5/6.0")) if relative
                else rng.choice(("abs/0.05/0.2", "abs/0.03/0.1", "abs/0.1")),
                "background": rng.choice(("first", "first", "random", "average", "median")),
                "outlier": rng.choice(("first", "last", "extreme", "average", "forward", "backward")),
                "crop": rng.choice((0, 0, 0, 3, 8)), "sample": sample,
                "weights": rng.choice(("", "", "", "", "0.5,1.0,0.25,1.0")),
                "fade": rng.choice(("", "", "", "clamp/abs/0,0.2/40,1.0", "repeat/rel/0,1.0/12,0.0"))}
    if kind == "simple":
        bps = rng.choice((1, 1, 2))
        channels = rng.choice((1, 3, 3, 4))
        frames = _log_uniform(rng, 4, 400)
        w, h = _size(rng, frames, channels * bps, 4.0e9)
        return {"kind": kind, "width": w, "height": h, "channels": channels, "bps": bps, "frames": frames,
                "darker": rng.random() < 0.5, "crop": rng.choice((0, 0, 5)),
                "fade": rng.choice(("", "", "clamp/abs/0,0.2/40,1.0"))}
    if kind == "shake":
        bps = rng.choice((1, 2))
        channels = rng.choice((1, 3, 3, 4))
        frames = _log_uniform(rng, 8, 256)
        w, h = _size(rng, frames, channels * bps, 4.0e9)
        radius = rng.randrange(6, 33) if min(w, h) >= 200 else rng.randrange(3, 9)
        return {"kind": kind, "width": w, "height": h, "channels": channels, "bps": bps, "frames": frames,
                "anchors": rng.randrange(1, 6), "radius": radius,
                "search": rng.randrange(2, 13) if min(w, h) >= 200 else rng.randrange(2, 6)}
    if kind == "batch":
        lo = rng.choice((160, 320, 640))
        return {"kind": kind, "jobs": rng.randrange(8, 49), "min_frames": rng.randrange(5, 20),
                "max_frames": rng.choice((48, 64, 120)), "min_width": lo, "max_width": 2 * lo}
    w = rng.choice((640, 1280, 1366, 1920))
    return {"kind": kind, "width": w, "height": w * 9 // 16, "channels": 3, "window": rng.randrange(12, 100),
            "windows": rng.randrange(6, 24), "threshold": rng.choice(("abs/0.05/0.2", "rel/2.0/4.0")),
            "outlier": rng.choice(("extreme", "forward", "average"))}


# ------------------------------------------------------------------------------ inputs

def _scene(seed, width, height, channels, bps, frames, shake=0):
    """Frames as the path meets them: a gradient with sensor noise, a few things that move
    through it and, in 8 bits, a bright flash now and then; stabilised stacks carry texture."""
    small = max(2, min(width, height) // 30)
    more = dict(shake_max=shake, texture_amp=12 if bps == 1 else 3000) if shake else {}
    if bps == 1:
        return cpa.Scene(seed=seed, width=width, height=height, channels=channels, bytes_per_sample=1, n_frames=frames,
                         base_lo=40, base_hi=200, sigma=3.0, n_disks=3, disk_r_min=max(2, small // 3),
                         disk_r_max=small, blob_permille=50, blob_r=max(2, small), blob_val=230, **more)
    return cpa.Scene(seed=seed, width=width, height=height, channels=channels, bytes_per_sample=2, n_frames=frames,
                     base_lo=8000, base_hi=50000, sigma=200.0, n_disks=3, disk_r_min=max(2, small // 3),
                     disk_r_max=small, disk_val_lo=2000, disk_val_hi=4000, **more)


def _resident(scene):
    ctx = _context()
    st = cpa.Stack(ctx, scene.width, scene.height, scene.channels, scene.bytes_per_sample, capacity=scene.n_frames)
    scene.generate_device(st.device_ptr, 0, scene.n_frames, stream=ctx.stream)
    ctx.synchronize()
    st.commit(scene.n_frames)
    return st


def _crop(case, scene):
    if not case["crop"]:
        return None
    return cpa.Crop.create(scene.shake_truth(case["frames"]), case["width"], case["height"])


def _fade(case):
    return cpa.Fade.from_str(case["fade"]) if case["fade"] else None


def _image(h, w, c, bps):
    return torch.empty((h, w, c), dtype=torch.uint8 if bps == 1 else torch.int16, device="cuda")


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _prepare_outlier(case, seed):
    scene = _scene(seed, case["width"], case["height"], case["channels"], case["bps"], case["frames"], case["crop"])
    st = _resident(scene)
    sample = None
    if case["sample"]:
        sample = np.sort(np.random.default_rng(seed).choice(case["frames"], case["sample"], replace=False))
    weights = [float(v) for v in case["weights"].split(",")] if case["weights"] else (1.0, 1.0, 1.0, 1.0)
    proc = cpa.OutlierProcessor(cpa.Threshold.from_str(case["threshold"]),
                                cpa.BackgroundMode.from_str(case["background"]),
                                cpa.OutlierSelectionMode.from_str(case["outlier"]), weights=weights,
                                fade=_fade(case), sample_indices=sample, seed=seed)
    sel = cpa._FrameSel(st, None, _crop(case, scene))
    h, w, c = sel.out_shape(st)
    px, mask = _image(h, w, c, case["bps"]), _image(h, w, c, 1)
    outs = cpa.cp_outputs(px.data_ptr(), mask.data_ptr(), None, None)
    torch.cuda.synchronize()
    return {"kind": "outlier", "stack": st, "proc": proc, "sel": sel, "params": proc.params(case["bps"]), "px": px,
            "mask": mask, "outs": outs}


def _prepare_simple(case, seed):
    scene = _scene(seed, case["width"], case["height"], case["channels"], case["bps"], case["frames"], case["crop"])
    st = _resident(scene)
    proc = cpa.SimpleProcessor(fade=_fade(case), darker=case["darker"])
    sel = cpa._FrameSel(st, None, _crop(case, scene))
    h, w, c = sel.out_shape(st)
    px = _image(h, w, c, case["bps"])
    torch.cuda.synchronize()
    return {"kind": "simple", "stack": st, "proc": proc, "sel": sel, "fade": proc.fade.native(), "px": px}


def _prepare_shake(case, seed):
    scene = _scene(seed, case["width"], case["height"], case["channels"], case["bps"], case["frames"],
                   max(1, case["search"] // 2))
    rng = np.random.default_rng(seed)
    m = case["radius"] + case["search"]
    anchors = [(int(rng.integers(m, case["width"] - m)), int(rng.integers(m, case["height"] - m)))
               for _ in range(case["anchors"])]
    return {"kind": "shake", "stack": _resident(scene), "anchors": anchors, "radius": case["radius"],
            "search": case["search"]}


def _batch_jobs(case):
    """Frames, size and options of each job: fixed by the case, so that its work does not depend on the seed."""
    rng = np.random.default_rng(3)
    for i in range(case["jobs"]):
        yield (i, int(rng.integers(case["min_frames"], case["max_frames"] + 1)),
               int(rng.integers(case["min_width"], case["max_width"] + 1)),
               int(rng.integers(case["min_width"] * 3 // 4, case["max_width"] * 9 // 16 + case["min_width"] // 4)))


def _prepare_batch(case, seed):
    ctx = _context()
    stacks, outs, jobs = [], [], []
    modes = list(cpa.OutlierSelectionMode)
    for i, n, w, h in _batch_jobs(case):
        sc = cpa.Scene(seed=seed * 1000 + i, width=w, height=h, n_frames=n, n_disks=2, disk_r_min=10, disk_r_max=30,
                       blob_permille=100)
        st = _resident(sc)
        thr = cpa.Threshold.abs(0.05, 0.2) if i % 2 == 0 else cpa.Threshold.rel(2.0, 4.0)
        px = _image(h, w, 3, 1)
        proc = cpa.OutlierProcessor(thr, cpa.BackgroundMode.FIRST, modes[i % 6])
        jobs.append(cpa.Job(cpa.CP_MODE_OUTLIER, st, px.data_ptr(), None, processor=proc))
        stacks.append(st)
        outs.append(px)
    torch.cuda.synchronize()
    return {"kind": "batch", "stacks": stacks, "outs": outs, "batch": cpa.Batch(ctx, jobs)}


def _server():
    if "server" not in _state:
        _state["server"] = cpa.Server(_context(), max_inflight=8)
    return _state["server"]


def _prepare_video(case, seed):
    n = case["window"] + case["windows"] - 1
    st = _resident(_scene(seed, case["width"], case["height"], case["channels"], 1, n))
    proc = cpa.OutlierProcessor(cpa.Threshold.from_str(case["threshold"]), cpa.BackgroundMode.FIRST,
                                cpa.OutlierSelectionMode.from_str(case["outlier"]))
    shape = (case["height"], case["width"], case["channels"])
    outs = [torch.empty(shape, dtype=torch.uint8, pin_memory=True) for _ in range(case["windows"])]
    return {"kind": "video", "server": _server(), "stack": st, "proc": proc, "window": case["window"], "outs": outs,
            "views": [o.numpy() for o in outs]}


# ------------------------------------------------------------------------------ one pass

def run(state):
    kind = state["kind"]
    if kind == "outlier":
        st = state["stack"]
        cpa._check(st.lib.cp_outlier(st.ctx.handle, st.handle, ctypes.byref(state["sel"].c),
                                     ctypes.byref(state["params"]), ctypes.byref(state["outs"]),
                                     cpa.CP_FLAG_DEVICE_OUT))
        return [state["px"], state["mask"]]
    if kind == "simple":
        st, proc = state["stack"], state["proc"]
        cpa._check(st.lib.cp_simple(st.ctx.handle, st.handle, ctypes.byref(state["sel"].c),
                                    proc.weights.ctypes.data_as(ctypes.POINTER(ctypes.c_float)),
                                    ctypes.byref(state["fade"]), int(proc.darker),
                                    ctypes.c_void_p(state["px"].data_ptr()), cpa.CP_FLAG_DEVICE_OUT))
        return state["px"]
    if kind == "shake":
        return cpa.ShakeAnalyzer().analyze(state["stack"], state["anchors"], state["radius"], state["search"])
    if kind == "batch":
        state["batch"].launch()
        return state["outs"]
    srv, tickets = state["server"], []
    for k, view in enumerate(state["views"]):
        job = cpa.Job(cpa.CP_MODE_OUTLIER, state["stack"], None, processor=state["proc"],
                      image_indices=range(k, k + state["window"]))
        tickets.append(srv.submit(job, host_out=view))
    for t in tickets:
        srv.wait(t)
    return state["outs"]


def work(case):
    """Bytes: every input sample and every output byte once.  Operations only where the path is
    arithmetic on pairs of samples (the search's products); the composites select and compare."""
    kind = case["kind"]
    if kind == "batch":
        return {"bytes": sum((n + 1) * w * h * 3 for _, n, w, h in _batch_jobs(case)), "flops": 0}
    if kind == "video":
        px = case["width"] * case["height"] * case["channels"]
        return {"bytes": px * (case["window"] + case["windows"] - 1 + case["windows"]), "flops": 0}
    if kind == "shake":
        side = 2 * (case["radius"] + case["search"]) + 1
        per = case["anchors"] * case["channels"]
        return {"bytes": case["frames"] * per * side * side * case["bps"] + 8 * case["frames"],
                "flops": 2 * (case["frames"] - 1) * per * (2 * case["search"] + 1) ** 2 * (2 * case["radius"] + 1) ** 2}
    px = case["width"] * case["height"] * case["channels"]
    return {"bytes": px * case["bps"] * (case["frames"] + 1) + (px if kind == "outlier" else 0), "flops": 0}
