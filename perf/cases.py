"""Measured workloads of gjxl_amd: what a program that uses it has it do.

Whole encodes of the plain path over the range of image sizes that its tests
and benchmark use (a thumbnail, 512x512, an odd HD frame, the 12 megapixel
frame), the learned form, a batch of mixed small images, and the stage entry
points that a caller with its own pipeline drives one by one (front end,
candidate costs and strategy search, one adaptive-quantization evaluation, a
Butteraugli comparison, AC tokenization, one training step of the proposal
network).

Everything but the training step is a fixed sequence of binary32, binary64
and integer operations that the library reproduces bit for bit, so its
outputs are compared exactly.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import gjxl_amd
from gjxl_amd import proposal

_device = None


def _dev() -> gjxl_amd.Device:
    """The program's one device handle."""
    global _device
    if _device is None:
        _device = gjxl_amd.Device(0)
    return _device


# ---- cases ---------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # a thumbnail: launches and waits
        {"name": "encode 77x45", "kind": "encode", "w": 77, "h": 45, "distance": 1.0,
         "source": "pinned", "texture": False},
        # the small benchmark image, pixels in pinned host memory
        {"name": "encode 512x512", "kind": "encode", "w": 512, "h": 512, "distance": 1.0,
         "source": "pinned", "texture": False},
        # a video-sized frame with ragged edges at a lower quality
        {"name": "encode 1921x1083", "kind": "encode", "w": 1921, "h": 1083, "distance": 2.0,
         "source": "pinned", "texture": True},
        # the headline image: pixels in device memory, tokens read back
        {"name": "encode 4032x3024", "kind": "encode", "w": 4032, "h": 3024, "distance": 1.0,
         "source": "resident", "texture": True},
        # the learned form at its defaults on the images its network was trained on
        {"name": "learned 2048x1536", "kind": "learned", "w": 2048, "h": 1536, "distance": 1.0,
         "texture": True},
        # a folder of small images through the batch driver
        {"name": "batch of 16", "kind": "batch", "count": 16, "low": 256, "high": 1024,
         "lanes": 3},
        # RGBA pixels to the quant field, its masks and the chroma-from-luma maps
        {"name": "front end 4032x3024", "kind": "front", "w": 4032, "h": 3024, "bpp": 4,
         "distance": 1.0, "texture": True},
        # the encoder's transform choice
        {"name": "strategy 1288x968", "kind": "strategy", "w": 1288, "h": 968, "distance": 1.0,
         "texture": True},
        # one trial quantization: code, predict DC, reconstruct, filter
        {"name": "evaluate 2048x1536", "kind": "evaluate", "w": 2048, "h": 1536,
         "distance": 1.0, "texture": True},
        # a quality metric's use: one image against a distorted copy
        {"name": "butteraugli 1537x1153", "kind": "butteraugli", "w": 1537, "h": 1153,
         "texture": True},
        # a quantized frame's coefficient orders, contexts and tokens
        {"name": "tokens 2048x1536", "kind": "tokens", "w": 2048, "h": 1536, "distance": 1.0,
         "texture": True},
        # one optimizer step of the network at the trainer's batch of crops
        {"name": "train 32x32x32", "kind": "train", "n": 32, "h": 32, "w": 32},
    ]


def _log_uniform(rng, low: float, high: float) -> float:
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _extent(rng, low: int, high: int) -> tuple[int, int]:
    """A width and a height: the area over its logarithm, aspect 1:2 to 2:1."""
    area = _log_uniform(rng, low, high)
    aspect = _log_uniform(rng, 0.5, 2.0)
    w = max(16, int(math.sqrt(area * aspect)))
    return w, max(16, int(area / w))


def draw(rng) -> dict:
    kind = rng.choice(["encode", "encode", "encode", "learned", "batch", "front", "strategy",
                       "evaluate", "butteraugli", "tokens", "train"])
    distance = round(_log_uniform(rng, 0.5, 4.0), 2)
    texture = rng.random() < 0.7
    if kind == "train":
        return {"kind": kind, "n": rng.randint(1, 48), "h": rng.randint(8, 32),
                "w": rng.randint(8, 32)}
    if kind == "batch":
        low = rng.randint(64, 512)
        return {"kind": kind, "count": rng.randint(2, 20), "low": low,
                "high": low + rng.randint(8, 512), "lanes": rng.randint(1, 4)}
    w, h = _extent(rng, 2_000, 12_000_000)
    if kind == "encode":
        return {"kind": kind, "w": w, "h": h, "distance": distance,
                "source": rng.choice(["pinned", "resident"]), "texture": texture}
    if kind == "learned":
        return {"kind": kind, "w": w, "h": h, "distance": distance, "texture": texture}
    if kind == "front":
        return {"kind": kind, "w": w, "h": h, "bpp": rng.choice([3, 4]), "distance": distance,
                "texture": texture}
    if kind == "butteraugli":
        return {"kind": kind, "w": w, "h": h, "texture": texture}
    return {"kind": kind, "w": w, "h": h, "distance": distance, "texture": texture}


# ---- inputs ----------------------------------------------------------------------

def _image(w: int, h: int, seed: int, texture: bool) -> torch.Tensor:
    """An (h, w, 3) uint8 image on the GPU: smooth colour gradients, band-limited
    noise, filled rectangles and thin strokes; with texture also patches of
    periodic patterns and flat regions (the recipes of gjxl_amd.synthetic)."""
    rng = np.random.default_rng(seed)
    g = torch.Generator("cuda").manual_seed(seed)
    y = torch.linspace(0.0, 1.0, h, device="cuda")[:, None]
    x = torch.linspace(0.0, 1.0, w, device="cuda")[None, :]
    image = torch.empty((3, h, w), device="cuda")
    for c in range(3):
        a, b, d = rng.uniform(-1.0, 1.0, 3)
        fx, fy = rng.uniform(0.5, 2.5, 2)
        image[c] = 128.0 + 60.0 * (a * x + b * y) + 40.0 * d * torch.sin(
            2 * math.pi * (fx * x + fy * y) + rng.uniform(0, 2 * math.pi))
    noise = torch.randn((3, h, w), device="cuda", generator=g)
    taps = [math.exp(-0.5 * (i / 2.0) ** 2) for i in range(-6, 7)]
    for dim in (1, 2):
        noise = sum(t * torch.roll(noise, i - 6, dim) for i, t in enumerate(taps))
    image += 6.0 * noise / noise.std()

    def box(low, divisor):
        bw = int(rng.integers(min(low, w), max(min(low, w) + 1, w // divisor)))
        bh = int(rng.integers(min(low, h), max(min(low, h) + 1, h // divisor)))
        x0, y0 = int(rng.integers(0, w - bw + 1)), int(rng.integers(0, h - bh + 1))
        return slice(y0, y0 + bh), slice(x0, x0 + bw)

    def colour():
        return torch.tensor(rng.uniform(0, 255, 3), device="cuda",
                            dtype=torch.float32)[:, None, None]

    if texture:
        for period in (2, 4, 8, 16):
            for _ in range(max(2, w * h // 400_000)):
                ys, xs = box(4 * period, 8)
                yy = torch.arange(ys.stop - ys.start, device="cuda")[:, None]
                xx = torch.arange(xs.stop - xs.start, device="cuda")[None, :]
                kind = int(rng.integers(0, 3))
                if kind == 0:
                    p = ((xx // period + yy // period) % 2).float()
                else:
                    p = 0.5 + 0.5 * torch.sin(2 * math.pi * (xx + (kind - 1) * yy) / period)
                low, high = colour(), colour()
                image[:, ys, xs] = low + (high - low) * p
        covered = 0
        while covered < 0.1 * w * h:
            ys, xs = box(16, 5)
            image[:, ys, xs] = colour()
            covered += (ys.stop - ys.start) * (xs.stop - xs.start)
    for _ in range(40):
        ys, xs = box(4, 6)
        image[:, ys, xs] = colour()
    for k in range(200):
        thick = int(rng.integers(1, 4))
        ys, xs = box(8, 8)
        if k % 2:
            ys = slice(ys.start, ys.start + thick)
        else:
            xs = slice(xs.start, xs.start + thick)
        image[:, ys, xs] = float(rng.integers(0, 2) * 255)
    return image.round_().clamp_(0, 255).to(torch.uint8).permute(1, 2, 0).contiguous()


class _Span:
    """A library buffer as torch sees it; keeps its owner alive."""

    def __init__(self, array, owner, typestr=None):
        kind = typestr or np.dtype(array.dtype).str
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": kind, "version": 2,
                                         "data": (array.ptr, False)}


def _tensor(array, owner, typestr=None) -> torch.Tensor:
    return torch.as_tensor(_Span(array, owner, typestr), device="cuda")


def _array(dev, tensor: torch.Tensor, dtype=None):
    """A torch tensor's memory as a library array."""
    names = {torch.float32: np.float32, torch.uint8: np.uint8, torch.int8: np.int8,
             torch.int16: np.uint16, torch.int32: np.int32}
    a = gjxl_amd.DeviceArray(dev, tensor.shape, dtype or names[tensor.dtype],
                             pointer=tensor.data_ptr())
    a.tensor = tensor
    return a


def _new(dev, shape, dtype=torch.float32):
    return _array(dev, torch.empty(tuple(int(s) for s in shape), dtype=dtype, device="cuda"))


def _host(array: np.ndarray, owner) -> torch.Tensor:
    t = torch.from_numpy(array)
    t.owner = owner  # the memory belongs to it
    return t


def _extent_of(case) -> tuple[int, int, int, int]:
    w, h = case["w"], case["h"]
    return w, h, gjxl_amd.pad8(w), gjxl_amd.pad8(h)


def _front_arrays(dev, w, h, pw, ph) -> dict:
    bw, bh = pw // 8, ph // 8
    tiles = ((ph + 63) // 64, (pw + 63) // 64)
    scratch = gjxl_amd.library().gjxl_amd_initial_quant_field_scratch_bytes(pw, ph)
    return {"linear": _new(dev, (3, h, w)), "opsin": _new(dev, (3, ph, pw)),
            "preprocessed": _new(dev, (3, ph, pw)),
            "aq": {"quant_field": _new(dev, (bh, bw)), "strategy_mask": _new(dev, (bh, bw)),
                   "pixel_mask": _new(dev, (ph, pw))},
            "cfl": {"y_to_x": _new(dev, tiles, torch.int8), "y_to_b": _new(dev, tiles, torch.int8)},
            "scratch": _new(dev, (scratch,), torch.uint8),
            "costs": _new(dev, (7, bh, bw)), "cells": _new(dev, (bh, bw), torch.uint8)}


def _run_front(dev, s, w, h, bpp, distance):
    dev.srgb8_to_linear_and_opsin(s["pixels"], w, h, bytes_per_pixel=bpp, linear=s["linear"],
                                  opsin=s["opsin"])
    dev.gaborish_inverse(s["opsin"], out=s["preprocessed"])
    dev.initial_quant_field(s["opsin"], distance, 1.0, out=s["aq"], scratch=s["scratch"])
    dev.initial_cfl(s["preprocessed"], out=s["cfl"])


def _run_strategy(dev, s, distance):
    dev.ac_strategy_costs(s["preprocessed"], s["aq"]["quant_field"], s["aq"]["pixel_mask"],
                          s["cfl"]["y_to_x"], s["cfl"]["y_to_b"], distance, costs=s["costs"])
    dev.ac_strategy_search(s["costs"], distance, cells=s["cells"])


def prepare(case: dict, seed: int):
    dev, kind = _dev(), case["kind"]
    s = {"case": case}
    if kind == "train":
        return _prepare_train(dev, s, case, seed)
    if kind == "batch":
        rng = np.random.default_rng(case["count"])
        s["images"], capacity = [], 0
        for i in range(case["count"]):
            w, h = (int(v) for v in rng.integers(case["low"], case["high"] + 1, 2))
            s["images"].append(_image(w, h, seed + 1000 * i, i % 2 == 0).cpu().numpy())
            capacity += 3 * 65 * (gjxl_amd.pad8(w) // 8) * (gjxl_amd.pad8(h) // 8)
        # where the program gathers the images' streams, one after another
        s["values"], s["contexts"] = np.zeros(capacity, np.int32), np.zeros(capacity, np.int16)
        s["options"] = [{"distance": 1.0} for _ in s["images"]]
        s["batch"] = gjxl_amd.Batch(0, case["lanes"])
        return s
    w, h, pw, ph = _extent_of(case)
    pixels = _image(w, h, seed, case["texture"])
    if kind in ("encode", "learned"):
        path = s["path"] = gjxl_amd.NativePlainPath(dev, w, h, case["distance"])
        # the streams' buffers hold the longest stream: the rest stays zero
        path.values.array[:] = 0
        path.contexts.array[:] = 0
        if kind == "learned":
            s["net"] = proposal.ProposalNet(dev, path.bw * path.bh,
                                            proposal.load_parameters())
            path.set_proposal(s["net"])
        if case.get("source") == "pinned":
            path.pixels.array[:] = pixels.cpu().numpy().reshape(-1)
        else:
            s["pixels"] = _array(dev, pixels)
        return s
    if kind == "butteraugli":
        s["metric"] = gjxl_amd.Butteraugli(dev, w, h)
        linear = torch.empty((2, 3, h, w), device="cuda")
        encoded = pixels.permute(2, 0, 1).float()
        g = torch.Generator("cuda").manual_seed(seed + 7)
        noise = torch.randn((3, h, w), device="cuda", generator=g)
        for i, v in enumerate((encoded, (encoded + 3.0 * noise).clamp(0, 255))):
            v = v / 255.0
            linear[i] = torch.where(v <= 0.04045, v / 12.92, ((v + 0.055) / 1.055) ** 2.4)
        s["reference"], s["distorted"] = _array(dev, linear[0]), _array(dev, linear[1])
        s["map"] = _new(dev, (h, w))
        return s
    bpp = case.get("bpp", 3)
    if bpp == 4:
        pixels = torch.cat([pixels, torch.full_like(pixels[:, :, :1], 255)], dim=2)
    s["pixels"] = _array(dev, pixels.contiguous())
    s.update(_front_arrays(dev, w, h, pw, ph))
    if kind == "front":
        return s
    torch.cuda.synchronize()  # the library's stream reads what torch's wrote
    _run_front(dev, s, w, h, bpp, case["distance"])
    if kind == "strategy":
        return s
    _run_strategy(dev, s, case["distance"])
    session = s["session"] = gjxl_amd.AqSession(dev, w, h)
    session.prepare(s["opsin"], s["preprocessed"], s["cells"], s["aq"]["quant_field"],
                    case["distance"])
    store = ((session.bw + 31) // 32) * ((session.bh + 31) // 32) * 65536
    blocks = (session.bh, session.bw)
    s["field"] = session.buffer("adjusted_field", blocks)
    s["coded"] = {"quantized": session.buffer("quantized", (3, store), np.int32),
                  "raw_quant": session.buffer("raw_quant", blocks, np.int32),
                  "dc_quantized": session.buffer("dc_quantized", (3,) + blocks, np.int32),
                  "y_to_x": session.buffer("y_to_x", s["cfl"]["y_to_x"].shape, np.int8),
                  "y_to_b": session.buffer("y_to_b", s["cfl"]["y_to_b"].shape, np.int8),
                  "linear": session.buffer("linear", (3, h, w))}
    if kind == "tokens":
        session.evaluate(s["field"])
        dev.synchronize()
        tok = s["tokenizer"] = gjxl_amd.Tokenizer(dev, w, h)
        s["stream"] = {"values": _tensor(tok.buffer("values"), tok, "<i4"),
                       "contexts": _tensor(tok.buffer("contexts"), tok, "<i2"),
                       "group_offsets": _tensor(tok.buffer("group_offsets"), tok, "<i4")}
        # the buffers hold the longest stream: the rest stays zero
        for t in s["stream"].values():
            t.zero_()
    return s


def _train_inputs(case: dict, seed: int):
    """Features, strategy labels, field targets and parameters as the trainer has
    them: standardised-looking features, the searched strategies' codes."""
    n, h, w = case["n"], case["h"], case["w"]
    g = torch.Generator("cuda").manual_seed(seed)
    x = torch.randn((n, h, w, proposal.FEATURES), device="cuda", generator=g)
    x[..., 13:] = 0.0
    codes = torch.tensor(proposal.STRATEGIES, dtype=torch.uint8, device="cuda")
    pick = torch.randint(0, len(proposal.STRATEGIES), (n, h, w), device="cuda", generator=g)
    targets = 0.18 * torch.randn((n, h, w), device="cuda", generator=g)
    return x.to(torch.bfloat16), codes[pick], targets, proposal.init_parameters(seed)


_TRAIN = {"lr": 2e-3, "beta1": 0.9, "beta2": 0.999, "eps": 1e-8}


def _prepare_train(dev, s, case, seed):
    x, labels, targets, params = _train_inputs(case, seed)
    positions = labels.numel()
    s["net"] = proposal.ProposalNet(dev, positions, params)
    s["features"] = _array(dev, x.view(torch.int16))
    s["labels"], s["targets"] = _array(dev, labels), _array(dev, targets)
    s["head"] = s["net"].head(positions)
    count = proposal.parameter_count()
    # the network's device buffers (1: master parameters, 2: gradients)
    s["parameters"] = s["net"].buffer(1, (count,), np.float32)
    s["gradients"] = s["net"].buffer(2, (count,), np.float32)
    return s


# ---- one pass ----------------------------------------------------------------------

def run(s):
    case, kind, dev = s["case"], s["case"]["kind"], _dev()
    if kind in ("encode", "learned"):
        path = s["path"]
        path.run(resident=s.get("pixels"))
        if "views" not in s:
            s["views"] = {k: _tensor(path.view(k), path) for k in
                          ("cells", "quant_field", "block_distance", "raw_quant",
                           "dc_quantized", "y_to_x", "y_to_b")}
        return {"values": _host(path.values.array.view(np.int32), path),
                "contexts": _host(path.contexts.array.view(np.int16), path),
                "group_offsets": _host(path.group_offsets.array.view(np.int32), path),
                "scores": path.scores(), **s["views"]}
    if kind == "batch":
        count = len(s["images"])
        results = s["batch"].encode(s["images"], s["options"])
        at, counts, scores = 0, [], []
        for r in results:
            if r.status != 0:
                raise RuntimeError(r.message.decode())
            n = int(r.token_count)
            ctypes.memmove(s["values"].ctypes.data + 4 * at, r.token_values, 4 * n)
            ctypes.memmove(s["contexts"].ctypes.data + 2 * at, r.token_contexts, 2 * n)
            at += n
            counts.append(n)
            scores.append(r.scores_list())
        gjxl_amd.Batch.free_results(results, count)
        return {"values": s["values"], "contexts": s["contexts"],
                "counts": np.array(counts), "scores": np.array(scores)}
    if kind == "train":
        net = s["net"]
        net.forward(s["features"], case["n"], case["h"], case["w"])
        sums = net.backward(s["labels"], s["targets"], 1.0)
        net.adam(_TRAIN["lr"], _TRAIN["beta1"], _TRAIN["beta2"], _TRAIN["eps"],
                 grad_scale=1.0 / s["labels"].tensor.numel())
        return {"head": _tensor(s["head"], net), "gradients": _tensor(s["gradients"], net),
                "parameters": _tensor(s["parameters"], net),
                "cross_entropy": sums[0], "squared_error": sums[1]}
    if kind == "butteraugli":
        s["metric"].prepare(s["reference"])
        s["metric"].compare(s["distorted"], s["map"])
        return {"map": s["map"].tensor, "score": s["metric"].score()}
    if kind == "front":
        _run_front(dev, s, case["w"], case["h"], case["bpp"], case["distance"])
        out = {k: s[k].tensor for k in ("linear", "opsin", "preprocessed")}
        out.update({k: v.tensor for k, v in {**s["aq"], **s["cfl"]}.items()})
        return out
    if kind == "strategy":
        _run_strategy(dev, s, case["distance"])
        return {"costs": s["costs"].tensor, "cells": s["cells"].tensor}
    if kind == "evaluate":
        s["session"].evaluate(s["field"])
        return {k: _tensor(v, s["session"]) for k, v in s["coded"].items()}
    tok, coded = s["tokenizer"], s["coded"]
    inputs = (coded["quantized"], s["cells"], coded["raw_quant"])
    tok.set_entropy_inputs(gjxl_amd.entropy_inputs(tok.frame_statistics(*inputs)))
    tok.tokenize(*inputs)
    return s["stream"]


# ---- what a pass cannot do without -----------------------------------------------------

# Operations per pixel.  The candidate costs transform each candidate forward and
# back in three channels: 12 (W + H) per covered pixel and candidate, over the
# searched positions of a 64x64 tile.  An evaluation transforms the frame back (and
# the encode once forward) at about 8x8 to 32x32: 6 (W + H) per pixel, about 200.  A
# Butteraugli image blurs three planes at radius 16 and 7, two at 3 and one at 6 (3 per
# tap pair, two passes) at two scales; a comparison adds six Malta maps of about 16 lines
# of 5 to 9 taps.
_COSTS = sum(positions * w * h * 12 * (w + h) for positions, w, h in
             ((64, 8, 8), (56, 8, 16), (56, 16, 8), (49, 16, 16), (12, 16, 32), (12, 32, 16),
              (9, 32, 32))) / 4096
_EVALUATION = 200
_BLURS = 1.25 * 2 * 3 * (3 * 16 + 3 * 7 + 2 * 3 + 6)
_MALTA = 1.25 * 6 * 16 * 8


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "train":
        positions = case["n"] * case["h"] * case["w"]
        macs = 9 * 32 * (16 + 5 * 32)
        params = proposal.parameter_count()
        return {"bytes": positions * (2 * 16 + 1 + 4 + 4 * 32) + 4 * 7 * params,
                "flops": positions * 2 * (3 * macs - 9 * 32 * 16)}
    loop = 3 * (_EVALUATION + _MALTA) + 4 * _BLURS
    if kind == "batch":
        side = (case["low"] + case["high"]) / 2
        px = case["count"] * side * side
        return {"bytes": px * (3 + 4), "flops": px * (_COSTS + _EVALUATION + loop)}
    w, h, pw, ph = _extent_of(case)
    px, padded = w * h, pw * ph
    if kind == "encode":
        return {"bytes": px * (3 + 4), "flops": px * (_COSTS + _EVALUATION + loop)}
    if kind == "learned":
        return {"bytes": px * (3 + 4), "flops": px * (0.4 * _COSTS + 2.0 / 3.0 * loop)}
    if kind == "front":
        return {"bytes": px * (case["bpp"] + 12) + padded * (24 + 4 + 8 / 64), "flops": px * 400}
    if kind == "strategy":
        return {"bytes": padded * (12 + 4 + (4 + 28 + 1) / 64), "flops": padded * _COSTS}
    if kind == "evaluate":
        return {"bytes": padded * (12 + 12 + (4 + 4 + 12) / 64) + 12 * px,
                "flops": padded * _EVALUATION}
    if kind == "butteraugli":
        return {"bytes": px * (24 + 4), "flops": px * (2 * _BLURS + _MALTA)}
    return {"bytes": padded * (12 + 5 / 64) + px * 4, "flops": px * 10}


def tolerance(case: dict):
    if case["kind"] == "train":
        # bfloat16 activations and gradients: a product summed in another order
        # moves some of them by one step of 2^-8
        return {"rel": 1e-2, "max": 0.5}
    return "exact"


# ---- results in 64 bits ------------------------------------------------------------------

def exact(case: dict, seed: int):
    if case["kind"] == "front":
        return _exact_front(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, seed)
    # The others are defined by their operations' order and roundings (decisions
    # and integers follow from them); they are compared bit for bit instead.
    return None


def _exact_front(case, seed):
    """The linear image, XYB and its Gaborish inverse; the quant field and its
    masks rest on binary32 approximations and the maps are whole numbers."""
    w, h, pw, ph = _extent_of(case)
    v = _image(w, h, seed, case["texture"]).permute(2, 0, 1).double() / 255.0
    linear = torch.where(v <= 0.04045, v / 12.92, ((v + 0.055) / 1.055) ** 2.4)
    matrix = torch.tensor([[0.30, 0.622, 0.078], [0.23, 0.692, 0.078],
                           [0.24342268924547819, 0.20476744424496821, 0.55180986650955360]],
                          dtype=torch.float64, device="cuda")
    bias = 0.0037930732552754493
    ys = torch.arange(ph, device="cuda").clamp(max=h - 1)
    xs = torch.arange(pw, device="cuda").clamp(max=w - 1)
    padded = linear[:, ys][:, :, xs].reshape(3, -1)
    gamma = (matrix @ padded + bias) ** (1.0 / 3.0) - bias ** (1.0 / 3.0)
    opsin = torch.stack([0.5 * (gamma[0] - gamma[1]), 0.5 * (gamma[0] + gamma[1]),
                         gamma[2]]).reshape(3, ph, pw)
    side, diagonal, side2, corner, knight = (-0.09495815671340026, -0.041031725066768575,
                                             0.013710004822696948, -0.0014789063378272242,
                                             0.006510206083837737)
    weights = {(0, 0): 1.0, (0, 1): side, (1, 1): diagonal, (0, 2): side2, (2, 2): corner,
               (1, 2): knight}
    total = 1.0 + 4.0 * (side + diagonal + side2 + corner + 2.0 * knight)

    def mirrored(n):
        i = torch.arange(-2, n + 2, device="cuda")
        return torch.where(i < 0, -i - 1, torch.where(i >= n, 2 * n - 1 - i, i))

    wide = opsin[:, mirrored(ph)][:, :, mirrored(pw)]
    inverse = torch.zeros_like(opsin)
    for dy in range(-2, 3):
        for dx in range(-2, 3):
            k = weights[tuple(sorted((abs(dy), abs(dx))))] / total
            inverse += k * wide[:, 2 + dy:2 + dy + ph, 2 + dx:2 + dx + pw]
    return {"linear": linear, "opsin": opsin, "preprocessed": inverse, "quant_field": None,
            "strategy_mask": None, "pixel_mask": None, "y_to_x": None, "y_to_b": None}


def _exact_train(case, seed):
    """The step without any rounding between layers, but from the bfloat16
    weights that the products take."""
    x, labels, targets, flat = _train_inputs(case, seed)
    n, h, w = case["n"], case["h"], case["w"]
    master = torch.tensor(flat, device="cuda").double()
    layers, at = [], 0
    for layer in range(proposal.LAYERS):
        cin = proposal.layer_inputs(layer)
        size = 9 * 32 * cin
        layers.append((at, at + size, cin))
        at += size + 32
    rounded = torch.tensor(flat, device="cuda").to(torch.bfloat16).double()

    def shifted(a, dy, dx):
        a = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1))
        return a[:, 1 + dy:1 + dy + h, 1 + dx:1 + dx + w].reshape(n * h * w, -1)

    taps = [(t, t // 3 - 1, t % 3 - 1) for t in range(9)]
    a, inputs = x.double(), []
    for i, (lo, hi, cin) in enumerate(layers):
        inputs.append(a)
        k = rounded[lo:hi].view(9, 32, cin)
        z = sum(shifted(a, dy, dx) @ k[t].T for t, dy, dx in taps) + master[hi:hi + 32]
        a = (z if i == len(layers) - 1 else z.clamp(min=0)).view(n, h, w, 32)
    head = a.view(-1, 32)
    logits, label = head[:, :27], labels.view(-1).long()[:, None]
    logp = torch.log_softmax(logits, dim=1)
    error = head[:, 27] - targets.view(-1).double()
    d = torch.zeros_like(head)
    d[:, :27] = logp.exp()
    d[:, :27] = d[:, :27].scatter_add(1, label, torch.full_like(logp[:, :1], -1.0))
    d[:, 27] = 2.0 * error
    gradients = torch.zeros_like(master)
    for i in range(len(layers) - 1, -1, -1):
        lo, hi, cin = layers[i]
        gradients[lo:hi] = torch.stack([d.T @ shifted(inputs[i], dy, dx)
                                        for _, dy, dx in taps]).reshape(-1)
        gradients[hi:hi + 32] = d.sum(0)
        if i:
            k = rounded[lo:hi].view(9, 32, cin)
            image = d.view(n, h, w, 32)
            d = sum(shifted(image, -dy, -dx) @ k[t] for t, dy, dx in taps)
            d = d * (inputs[i].reshape(-1, 32) > 0)
    g = gradients / (n * h * w)
    # the first step of Adam: both moments' bias corrections cancel
    parameters = master - _TRAIN["lr"] * g / (g.abs() + _TRAIN["eps"])
    return {"head": head, "gradients": gradients, "parameters": parameters,
            "cross_entropy": float(-logp.gather(1, label).sum()),
            "squared_error": float((error ** 2).sum())}
