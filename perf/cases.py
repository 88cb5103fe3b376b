"""The work a program gives this decoder, as cases to be timed.

A case is a dict of plain values; `kind` says which public entry point it goes
through:

  frame      one frame from a plan already resident on the device
             (HipDecoder.decode_planned with the NV12 pack in the same launch
             sequence): what a player or transcoder whose parser threads plan
             ahead calls for every frame. The output is the packed picture on
             the device.
  batch      one frame of each of several streams decoded as one batch
             (decode_planned_batch): a multi-stream server's round.
  wire       one frame from its syntax in host memory, flattened, uploaded,
             decoded and handed back to the host (decode_wire with read back,
             or followed by to_rgb / to_nv12): the plain per-frame call.
  pipe       the frames of one stream through the ingest pipeline (Pipe):
             planner threads ahead of an in-order decode worker.
  costmodel  the superblock cost model: `op` predict (one call per planned
             frame), train (Adam over recorded superblocks) or gradients.

Syntax comes from the seeded generator of this package with the statistics of
its named workloads: "c1" (8 x 8 and larger DCT/ADST, single reference, Wiener
restoration), "c2" (full tool set: compound, 64-point and rectangular
transforms, superres 3/4, self-guided restoration, film grain) and
"tools_mini" (warp, masks, OBMC, inter-intra, intra block copy, palette, CFL,
filter intra). Decoded pictures are whole numbers and must match to the bit.
"""
import math

import numpy as np
import torch

import av1ongpu_amd as pkg

H, IN = 64, pkg.CM_FEATURES

# streams of a batch, smallest first: (width, height, bit depth), cycled through
STREAMS = [(426, 240, 8), (854, 480, 10), (1280, 720, 8), (1920, 1080, 10)]


def listed():
    return [
        # the smallest call: a thumbnail or tiny fixture stream, launches and latency only
        {"name": "inter_160x96", "kind": "frame", "clip": "c1", "width": 160, "height": 96, "depth": 8,
         "key": False, "levels": False},
        # a low-resolution stream's key frame (scene cut, seek)
        {"name": "key_426x240", "kind": "frame", "clip": "c1", "width": 426, "height": 240, "depth": 8,
         "key": True, "levels": False},
        # the ordinary inter frame of a 720p 8-bit stream
        {"name": "inter_1280x720", "kind": "frame", "clip": "c1", "width": 1280, "height": 720, "depth": 8,
         "key": False, "levels": False},
        # the benchmark's frame: 1080p 10 bit with every tool of its workload
        {"name": "inter_1080p10", "kind": "frame", "clip": "c2", "width": 1920, "height": 1080, "depth": 10,
         "key": False, "levels": False},
        # that stream's key frame: every block intra, a long dependency chain
        {"name": "key_1080p10", "kind": "frame", "clip": "c2", "width": 1920, "height": 1080, "depth": 10,
         "key": True, "levels": False},
        # the largest stream served: 4K 10 bit with superres and grain
        {"name": "inter_2160p10", "kind": "frame", "clip": "c2", "width": 3840, "height": 2160, "depth": 10,
         "key": False, "levels": False},
        # odd size, rare tools, coded levels dequantised on the device
        {"name": "tools_853x479", "kind": "frame", "clip": "tools_mini", "width": 853, "height": 479, "depth": 10,
         "key": False, "levels": True},
        # a server's round: eight streams of four sizes
        {"name": "batch8_mix", "kind": "batch", "clip": "c1", "streams": 8, "first": 0, "scale": 1.0, "key": False},
        # the plain per-frame call of a program without planner threads
        {"name": "wire_1280x720", "kind": "wire", "clip": "c1", "width": 1280, "height": 720, "depth": 8,
         "key": False, "out": "planes"},
        # a stream from syntax as fast as it goes: the start of the benchmark's clip
        {"name": "pipe_1080p10", "kind": "pipe", "clip": "c2", "width": 1920, "height": 1080, "depth": 10,
         "frames": 12, "planners": 10},
        # refitting the cost model on a few recorded frames
        {"name": "costmodel_train", "kind": "costmodel", "op": "train", "n": 8192, "epochs": 2},
        # the superblocks of one 4K frame (60 x 34) predicted before it is queued
        {"name": "costmodel_predict", "kind": "costmodel", "op": "predict", "n": 2040, "epochs": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, max_width):
    """A picture size: widths over their logarithm, common and odd shapes."""
    w = _log(rng, 64, max_width)
    h = max(34, min(int(w * rng.choice((0.5, 0.5625, 0.5625, 0.75))), max_width * 9 // 16))
    if rng.random() < 0.5:  # decoders mostly see even sizes, but must take any
        w, h = (w + 1) & ~1, (h + 1) & ~1
    return w, h


def draw(rng):
    kind = rng.choice(("frame", "frame", "frame", "frame", "batch", "wire", "pipe", "costmodel"))
    if kind == "frame":
        clip = rng.choice(("c1", "c2", "c2", "tools_mini"))
        key = rng.random() < 0.3
        w, h = _size(rng, 1280 if clip == "tools_mini" else 1920 if key else 3840)
        return {"kind": kind, "clip": clip, "width": w, "height": h, "depth": rng.choice((8, 10)), "key": key,
                "levels": rng.random() < 0.3}
    if kind == "batch":
        return {"kind": kind, "clip": rng.choice(("c1", "c2")), "streams": rng.randint(2, 12), "first": rng.randint(0, 3),
                "scale": round(rng.uniform(0.3, 1.0), 3), "key": rng.random() < 0.25}
    if kind == "wire":
        w, h = _size(rng, 1920)
        return {"kind": kind, "clip": rng.choice(("c1", "c2")), "width": w, "height": h, "depth": rng.choice((8, 10)),
                "key": rng.random() < 0.3, "out": rng.choice(("planes", "planes", "rgb", "nv12"))}
    if kind == "pipe":
        w, h = _size(rng, 1920)
        return {"kind": kind, "clip": rng.choice(("c1", "c2")), "width": w, "height": h, "depth": rng.choice((8, 10)),
                "frames": rng.randint(3, 12), "planners": rng.randint(2, 10)}
    op = rng.choice(("predict", "train", "gradients"))
    return {"kind": kind, "op": op, "n": _log(rng, 40, 8192), "epochs": rng.randint(1, 2) if op == "train" else 0}


def _pitch(width):
    return (width + 255) & ~255


def _clip(name, seed, width, height, depth, frames, levels=False):
    """A seeded clip of a named workload at this size."""
    over = {"width": width, "height": height, "bit_depth": depth, "frames": frames, "levels": 1 if levels else 0}
    if name == "c2":
        over["coded_width"] = (width * 3 // 4 + 1) & ~1
    return pkg.Clip(name, seed & 0x7FFFFFFF, **over)


def _frames_before(name, key):
    """Frames to decode before the one timed: an inter frame's references."""
    return 0 if key else 1 if name == "c1" else 3


class _Stream:
    """One stream's decoder, its references decoded, its next frame's wire."""

    def __init__(self, name, seed, width, height, depth, key, levels=False, nv12=True):
        before = _frames_before(name, key)
        clip = _clip(name, seed, width, height, depth, before + 1, levels)
        self.width, self.height = width, height
        self.dec = pkg.HipDecoder(0)
        self.dec.set_pool_slots(8)
        if nv12:
            self.dec.set_decode_nv12(_pitch(width))
        slots = {}
        for f in range(before):
            wire = pkg.wire_set_slots(clip.wire(f), [slots[r] for r in clip.refs[f]])
            slots[f], _ = self.dec.decode_wire(wire, keep=True, read_back=False)
        self.wire = pkg.wire_set_slots(clip.wire(before), [slots[r] for r in clip.refs[before]])
        self.plan = None

    def plan_it(self):
        self.plan = self.dec.plan_wire(self.wire)
        return self

    def nv12(self):
        """The decoder's packed picture, a view of its device buffer."""
        rows = self.height + (self.height + 1) // 2
        return _device_view(self, pkg.hip_lib().av1h_nv12_device_buffer(self.dec.handle), (rows, _pitch(self.width)))

    def __del__(self):
        if getattr(self, "dec", None) is not None:
            if getattr(self, "plan", None) is not None:
                self.dec.discard_plan(self.plan)
            self.dec.close()


class _DeviceArray:
    def __init__(self, owner, address, shape):
        self.owner = owner  # the buffer lives as long as the view
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "|u1", "data": (address, False), "version": 2,
                                         "strides": None}


def _device_view(owner, address, shape):
    return torch.as_tensor(_DeviceArray(owner, address, shape), device="cuda")


class _PipeState:
    def __init__(self, case, seed):
        self.clip = _clip(case["clip"], seed, case["width"], case["height"], case["depth"], case["frames"])
        self.keep, self.release, refs = pkg.slot_schedule(self.clip)
        self.wires = [pkg.wire_set_slots(self.clip.wire(f), refs[f]) for f in range(self.clip.frames)]
        self.width, self.height = case["width"], case["height"]
        self.dec = pkg.HipDecoder(0)
        self.dec.set_pool_slots(16)
        self.dec.set_decode_nv12(_pitch(self.width))
        self.pipe = pkg.Pipe(self.dec, planner_threads=case["planners"], depth=64)

    nv12 = _Stream.nv12

    def __del__(self):
        if getattr(self, "pipe", None) is not None:
            self.pipe.close()
        if getattr(self, "dec", None) is not None:
            self.dec.close()


def _samples(case, seed):
    """Recorded superblocks: counts and fractions of their syntax, and the
    microseconds of queue work they took."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    x = rng.gamma(1.5, 8.0, (n, IN)).astype(np.float32)
    x[:, 10:14] = rng.random((n, 4), np.float32)
    x[:, 14:18] = rng.integers(0, 2, (n, 4))
    y = (2.0 + 1.3 * x[:, 0] + 0.4 * x[:, 1] * x[:, 11] + 3.0 * x[:, 14] * x[:, 2]
         + rng.gamma(2.0, 1.0, n)).astype(np.float32)
    w = rng.standard_normal(pkg.CM_PARAMS).astype(np.float32)
    for lo, hi, dev in ((0, H * IN, (2 / IN) ** 0.5), (H * IN, H * IN + H, 0.1),
                        (H * IN + H, H * IN + H + H * H, (2 / H) ** 0.5),
                        (H * IN + H + H * H, H * IN + 2 * H + H * H, 0.1), (H * IN + 2 * H + H * H, w.size, 0.2)):
        w[lo:hi] *= np.float32(dev)
    mean = x.mean(0, dtype=np.float64).astype(np.float32)
    dev = np.maximum(x.std(0, dtype=np.float64), 1e-3).astype(np.float32)
    return {"x": x, "y": y, "w": w, "mean": mean, "dev": dev, "y_mean": np.float32(y.mean(dtype=np.float64)),
            "y_dev": np.float32(y.std(dtype=np.float64))}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("frame", "wire"):
        st = _Stream(case["clip"], seed, case["width"], case["height"], case["depth"], case["key"],
                     case.get("levels", False), nv12=kind == "frame")
        return {"case": case, "streams": [st.plan_it() if kind == "frame" else st]}
    if kind == "batch":
        streams = []
        for i in range(case["streams"]):
            w, h, depth = STREAMS[(case["first"] + i) % len(STREAMS)]
            w, h = (max(64, int(v * case["scale"])) & ~1 for v in (w, h))
            streams.append(_Stream(case["clip"], seed * 64 + i, w, h, depth, case["key"]).plan_it())
        return {"case": case, "streams": streams, "decoders": [s.dec for s in streams],
                "plans": [s.plan for s in streams]}
    if kind == "pipe":
        return {"case": case, "pipe": _PipeState(case, seed)}
    s = _samples(case, seed)
    s["case"], s["model"] = case, pkg.CostModel(0, seed=1)
    s["model"].set_params(s["w"])
    s["model"].set_norm(s["mean"], s["dev"], s["y_mean"], s["y_dev"])
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "frame":
        st = state["streams"][0]
        st.dec.release(st.dec.decode_planned(st.plan, keep=True))
        return st.nv12()
    if kind == "batch":
        slots = pkg.decode_planned_batch(state["decoders"], state["plans"])
        for dec, slot in zip(state["decoders"], slots):
            dec.release(slot)
        return [st.nv12() for st in state["streams"]]
    if kind == "wire":
        st = state["streams"][0]
        slot, planes = st.dec.decode_wire(st.wire, keep=True, read_back=case["out"] == "planes")
        if case["out"] == "rgb":
            planes = st.dec.to_rgb(slot, 1, 0, st.width, st.height)
        elif case["out"] == "nv12":
            planes = st.dec.to_nv12(slot, _pitch(st.width), st.width, st.height)
        st.dec.release(slot)
        return planes
    if kind == "pipe":
        p = state["pipe"]
        for f, wire in enumerate(p.wires):
            p.pipe.submit(wire, keep=p.keep[f] >= 0, reserved=p.keep[f], release=p.release[f])
        p.pipe.wait()
        return p.nv12()
    model = state["model"]
    if case["op"] == "predict":
        return model.predict(state["x"])
    if case["op"] == "gradients":
        g, loss = model.gradients(state["x"], state["y"])
        return {"grad": g, "loss": loss}
    model.set_params(state["w"])  # a fit starts from the same weights each time
    losses = model.train(state["x"], state["y"], epochs=case["epochs"], lr=1e-3, seed=1)
    return {"params": model.params(), "losses": losses}


def _frame_bytes(clip, width, height, key, out):
    """One frame: its coefficients (16 bit, four transforms in five coded)
    and the reference samples it predicts from read once, the kept picture and
    the output written once."""
    coded = width * 3 // 4 if clip == "c2" else width
    px, cpx = width * height, coded * height
    refs = 0 if key else (3 if clip == "c1" else 4.5) * px
    return 3 * 0.8 * cpx + refs + 3 * px + out * px


def work(case):
    kind = case["kind"]
    if kind == "frame":
        return {"bytes": _frame_bytes(case["clip"], case["width"], case["height"], case["key"], 1.5), "flops": 0}
    if kind == "wire":
        out = {"planes": 3, "rgb": 3, "nv12": 1.5}[case["out"]]
        return {"bytes": _frame_bytes(case["clip"], case["width"], case["height"], case["key"], out), "flops": 0}
    if kind == "batch":
        total = 0
        for i in range(case["streams"]):
            w, h, _ = STREAMS[(case["first"] + i) % len(STREAMS)]
            total += _frame_bytes(case["clip"], w * case["scale"], h * case["scale"], case["key"], 1.5)
        return {"bytes": total, "flops": 0}
    if kind == "pipe":
        w, h, n = case["width"], case["height"], case["frames"]
        return {"bytes": _frame_bytes(case["clip"], w, h, True, 1.5)
                + (n - 1) * _frame_bytes(case["clip"], w, h, False, 1.5), "flops": 0}
    n = case["n"]
    forward = 2 * (IN * H + H * H + H)
    if case["op"] == "predict":
        return {"bytes": 4 * (n * (IN + 1) + pkg.CM_PARAMS), "flops": n * forward}
    passes = max(1, case["epochs"])
    return {"bytes": 4 * (n * (IN + 1) + 2 * pkg.CM_PARAMS), "flops": passes * n * 3 * forward}


def tolerance(case):
    if case["kind"] != "costmodel":
        return "exact"
    # 32-bit sums in two orders against 64 bits over 40..8192 samples, times four:
    # gradients were up to 1.0e-6 off (largest value 4.7e-6), weights after two
    # epochs 4.1e-7 (6.1e-6), predictions 2.2e-7
    if case["op"] == "predict":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 4e-6, "max": 3e-5}


def exact(case, seed):
    if case["kind"] != "costmodel" or case["op"] == "train":
        return None  # whole numbers; or the order samples are drawn in is the library's
    s = _samples(case, seed)
    w, at = s["w"].astype(np.float64), 0
    part = []
    for shape in ((H, IN), (H,), (H, H), (H,), (H,), (1,)):
        n = int(np.prod(shape))
        part.append(w[at:at + n].reshape(shape))
        at += n
    w1, b1, w2, b2, w3, b3 = part
    x = (s["x"].astype(np.float64) - s["mean"]) / s["dev"]
    h1 = np.maximum(x @ w1.T + b1, 0)
    h2 = np.maximum(h1 @ w2.T + b2, 0)
    out = h2 @ w3 + b3[0]
    if case["op"] == "predict":
        return out * np.float64(s["y_dev"]) + np.float64(s["y_mean"])
    y = (s["y"].astype(np.float64) - np.float64(s["y_mean"])) / np.float64(s["y_dev"])
    e = out - y
    d3 = 2 * e / len(e)
    d2 = (d3[:, None] * w3) * (h2 > 0)
    d1 = (d2 @ w2) * (h1 > 0)
    grad = np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), d3 @ h2, [d3.sum()]])
    return {"grad": grad, "loss": float(np.mean(e * e))}
