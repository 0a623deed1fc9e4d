"""Performance cases of the OCR backend: what a serving program has it do.

A program keeps one context and one loaded model per input shape, uploads a
page once and calls the detector on quads of it, then the recognizer on the
crops it found, or hands over batches that are already preprocessed.  Every
case is one such call through the public Python binding: a detector or a
recognizer call (image or host batch in, host result out), or the database of
boxes (DB postprocess) of probability maps.

The OCR engine's page call is made of these calls; with seeded weights its
number of detections is decided by pixels at the threshold, so the engine is
not a case of its own.

Sizes are the repository's: 416x736 pages and 832x1472 large pages, 48-pixel
lines, batches 1, 6 (the engine's recognizer batch), 8, 64 and 256.

``exact`` restates the networks in float64 torch, written here so that the
figures do not lean on the code they measure.
"""

import atexit
import math
import pathlib
import random
import shutil
import sys
import tempfile

import numpy as np
import torch
import torch.nn.functional as F

ROOT = pathlib.Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "ppocr-rs_amd"))

import ppocr_hip  # noqa: E402
import seeded  # noqa: E402

MIB = float(1 << 20)


# ------------------------------------------------------------------- cases

def _case(name, kind, tier, batch, height, width, precision="f32", source="image", greedy=False):
    return {"name": name, "kind": kind, "tier": tier, "batch": batch, "height": height, "width": width,
            "precision": precision, "source": source, "greedy": greedy}


def listed():
    return [
        # One line, already preprocessed by the caller, class probabilities
        # back: the smallest model call, bound by launches and host work.
        _case("rec_tiny_line", "rec", "tiny", 1, 48, 320, source="host"),
        # The lines of a busy page on the edge tier, decoded on the device.
        _case("rec_tiny_b64", "rec", "tiny", 64, 48, 320, greedy=True),
        # One engine batch: six crops of one page with a shared ragged canvas.
        _case("rec_small_ragged", "rec", "small", 6, 48, 500, greedy=True),
        # A full-accuracy batch of lines.
        _case("rec_medium_b64", "rec", "medium", 64, 48, 320, greedy=True),
        # Bulk serving of the accurate recognizer in bf16: the largest call.
        _case("rec_medium_b256_bf16", "rec", "medium", 256, 48, 320, precision="bf16", greedy=True),
        # One page on the edge tier, its 1920x1080 image resident.
        _case("det_tiny_page", "det", "tiny", 1, 416, 736),
        # A thumbnail handed over as planes by the caller, bf16.
        _case("det_tiny_thumb_bf16", "det", "tiny", 1, 96, 160, precision="bf16", source="host"),
        # A large page at full input size.
        _case("det_small_large", "det", "small", 1, 832, 1472),
        # One page on the accurate tier, handed over as planes.
        _case("det_medium_page", "det", "medium", 1, 416, 736, source="host"),
        # Batched serving of the accurate detector: the benchmark's workload.
        _case("det_medium_b8", "det", "medium", 8, 416, 736),
        # The same in bf16.
        _case("det_medium_b8_bf16", "det", "medium", 8, 416, 736, precision="bf16"),
        # Boxes from a page's probability map held by the host.
        _case("db_page", "db", "none", 1, 416, 736, source="host"),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        kind = rng.choices(("det", "rec", "db"), (5, 5, 1))[0]
        tier = rng.choice(("tiny", "small", "medium"))
        precision = rng.choices(("f32", "bf16"), (7, 3))[0]
        source = rng.choice(("image", "host"))
        if kind == "db":
            c = _case("", "db", "none", log_int(1, 4), 32 * log_int(3, 26), 32 * log_int(5, 46), source="host")
        elif kind == "det":
            c = _case("", "det", tier, log_int(1, 8), 32 * log_int(2, 26), 32 * log_int(3, 46), precision, source)
        else:
            batch, width = log_int(1, 256), 4 * log_int(10, 400)
            steps = -(-width // 8)
            wide = batch * steps * CLASSES[tier] * 4 > 16 * MIB
            c = _case("", "rec", tier, batch, 48, width, precision, source, wide or rng.random() < 0.5)
        flops = work(c)["flops"]
        if flops > (2.9e12 if precision == "bf16" else 4.0e11):
            continue
        if c["batch"] * c["height"] * c["width"] > 8 * 416 * 736 * 1.6:
            continue
        del c["name"]
        return c


# ------------------------------------------------------------------- inputs

CLASSES = {"tiny": 6906, "small": 18710, "medium": 18710}

_kept = {"gpu": None, "models": {}, "files": {}, "dir": None}


def _weights_file(kind, tier):
    if _kept["dir"] is None:
        _kept["dir"] = tempfile.mkdtemp(prefix="ppocr_cases_")
        atexit.register(shutil.rmtree, _kept["dir"], ignore_errors=True)
    if (kind, tier) not in _kept["files"]:
        path = pathlib.Path(_kept["dir"]) / f"{kind}_{tier}.safetensors"
        _kept["files"][(kind, tier)] = seeded.write_weights(path, kind, tier, seed=1)
    return _kept["files"][(kind, tier)]


def _gpu():
    if _kept["gpu"] is None:
        _kept["gpu"] = ppocr_hip.Gpu(0)
    return _kept["gpu"]


def _model(case):
    """The loaded model a program keeps for its input shape."""
    key = tuple(case[k] for k in ("kind", "tier", "batch", "height", "width", "precision", "greedy"))
    if key not in _kept["models"]:
        shape = (case["batch"], 3, case["height"], case["width"])
        path = _weights_file(case["kind"], case["tier"])
        if case["kind"] == "det":
            m = ppocr_hip.Detector.load(_gpu(), path, case["tier"], shape, case["precision"])
        else:
            m = ppocr_hip.Recognizer.load(_gpu(), path, case["tier"], shape, case["precision"],
                                          greedy=case["greedy"])
        _kept["models"][key] = m
    return _kept["models"][key]


def _page(rng, height, width):
    """A light page with dark text-like strokes, RGB8."""
    img = rng.integers(190, 256, size=(height, width, 3), dtype=np.uint8)
    line = max(8, height // 30)
    for y in range(line // 2, height - line, line + line // 2):
        x = int(rng.integers(4, 40))
        while x < width - 8:
            w = int(rng.integers(2, max(3, line)))
            h = int(rng.integers(max(2, line // 2), line + 1))
            shade = int(rng.integers(0, 80))
            img[y:y + h, x:x + w] = shade + rng.integers(0, 30, size=img[y:y + h, x:x + w].shape, dtype=np.uint8)
            x += w + int(rng.integers(2, max(3, line // 2)))
    return img


def _quads(case, rng, height, width):
    """Detector: overlapping tiles of the page; recognizer: slightly turned
    line crops with their content widths."""
    n = case["batch"]
    if case["kind"] == "det":
        if n == 1:
            boxes = [(0.0, 0.0, float(width), float(height))]
        else:
            boxes = []
            for _ in range(n):
                w, h = width * rng.uniform(0.5, 0.8), height * rng.uniform(0.5, 0.8)
                x, y = rng.uniform(0, width - w), rng.uniform(0, height - h)
                boxes.append((x, y, x + w, y + h))
        quads = [[(a, b), (c, b), (c, d), (a, d)] for a, b, c, d in boxes]
        return np.array(quads, np.float32), None
    quads, widths = [], []
    for _ in range(n):
        content = int(rng.integers(max(1, case["width"] // 2), case["width"] + 1))
        h = rng.uniform(24.0, 48.0)
        w = min(content * h / 48.0, width * 0.9)
        turn = rng.uniform(-0.05, 0.05)
        cx, cy = rng.uniform(w / 2, width - w / 2), rng.uniform(h, height - h)
        c, s = math.cos(turn), math.sin(turn)
        quads.append([(cx + c * dx - s * dy, cy + s * dx + c * dy)
                      for dx, dy in ((-w / 2, -h / 2), (w / 2, -h / 2), (w / 2, h / 2), (-w / 2, h / 2))])
        widths.append(content)
    return np.array(quads, np.float32), widths


def _inputs(case, seed):
    """Host data of a case, from the seed alone."""
    rng = np.random.Generator(np.random.PCG64([seed, 77]))
    if case["kind"] == "db":
        return {"maps": _text_maps(rng, case["batch"], case["height"], case["width"])}
    if case["source"] == "host":
        det = case["kind"] == "det"
        pages = [_page(rng, case["height"], case["width"]) for _ in range(min(case["batch"], 8))]
        planes = [seeded.normalize_identity(p, det) for p in pages]
        x = np.empty((case["batch"], 3, case["height"], case["width"]), np.float32)
        for i in range(case["batch"]):  # a few pages, each shifted sideways anew
            x[i] = np.roll(planes[i % len(planes)], 13 * i, axis=2)
        return {"planes": x}
    page = _page(rng, 1080, 1920)
    quads, widths = _quads(case, rng, 1080, 1920)
    return {"page": page, "quads": quads, "widths": widths}


def _text_maps(rng, n, height, width):
    """Probability maps with separate line-shaped components above a faint
    background, none of them square or at a threshold."""
    maps = rng.uniform(0.0, 0.1, size=(n, height, width)).astype(np.float32)
    for m in maps:
        y = 4
        while y + 12 < height:
            x = 4
            while x + 44 < width:
                w, h = int(rng.integers(24, 41)), int(rng.integers(4, 9))
                slope = rng.uniform(-0.08, 0.08)
                for dx in range(w):
                    top = y + 2 + int(slope * dx)
                    m[max(0, top):top + h, x + dx] = rng.uniform(0.55, 0.98)
                x += 56
            y += 18
    return maps


def prepare(case, seed):
    data = _inputs(case, seed)
    if case["kind"] == "db":
        transforms = [(case["width"], case["height"], case["width"], case["height"])] * case["batch"]
        return {"case": case, "gpu": _gpu(), "maps": data["maps"], "transforms": transforms}
    state = {"case": case, "model": _model(case)}
    if case["source"] == "host":
        state["planes"] = data["planes"]
    else:
        state["image"] = _gpu().upload_rgb(data["page"])
        state["quads"], state["widths"] = data["quads"], data["widths"]
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "db":
        found = state["gpu"].db_postprocess(state["maps"], state["transforms"])
        return [{"polygons": np.array([d.polygon for d in dets], np.float32).reshape(-1, 4, 2),
                 "scores": np.array([d.score for d in dets], np.float32)} for dets in found]
    if case["source"] == "host":
        out = state["model"].forward(state["planes"])
    else:
        out = state["model"].forward_image(state["image"], state["quads"], state["widths"])
    values = out.array()
    if case["greedy"]:
        # Class index and probability of each step.
        return {"classes": values[..., 0].astype(np.int32), "probabilities": values[..., 1]}
    return values


# -------------------------------------------------------------------- work

# GFLOP of the reference's algorithm per image at 416x736 and per line at
# 48x320 (two per multiply-add), and the weights in MB.
_DET_GFLOP = {"tiny": 1.973, "small": 6.467, "medium": 48.73}
_REC_GFLOP = {"tiny": 0.369, "small": 2.183, "medium": 11.36}
_WEIGHT_MB = {("det", "tiny"): 1.79, ("det", "small"): 9.94, ("det", "medium"): 44.0,
              ("rec", "tiny"): 4.47, ("rec", "small"): 21.2, ("rec", "medium"): 76.7}


def work(case):
    n, h, w = case["batch"], case["height"], case["width"]
    if case["kind"] == "db":
        return {"bytes": float(n * h * w * 4), "flops": 0.0}
    weights = _WEIGHT_MB[(case["kind"], case["tier"])] * 1e6 * (0.5 if case["precision"] == "bf16" else 1.0)
    read = n * 3 * h * w * 4 if case["source"] == "host" else 1080 * 1920 * 3
    if case["kind"] == "det":
        flops = n * _DET_GFLOP[case["tier"]] * 1e9 * (h * w) / (416 * 736)
        written = n * h * w * 4
    else:
        flops = n * _REC_GFLOP[case["tier"]] * 1e9 * w / 320
        written = n * -(-w // 8) * (2 if case["greedy"] else CLASSES[case["tier"]]) * 4
    return {"bytes": float(weights + read + written), "flops": float(flops)}


def tolerance(case):
    if case["kind"] == "db":
        # Moments are summed in 64 bits in any order; corners are 32-bit.
        return {"rel": 1e-6, "max": 1e-4}
    det = case["kind"] == "det"
    if case["precision"] == "bf16":
        # Storage rounding travels through the whole network: another order
        # of the sums moves an output by as much as bf16 itself does (4e-3 to
        # 6e-3 of a detector map, 1.6e-2 of the recognizer's probabilities),
        # and near-tied classes change sides.
        return {"rel": 0.02 if det else 0.03, "max": 0.9, "differ": 0.01}
    # 32-bit sums in another order, through the whole network (errors of 3e-7
    # to 6e-7 of a map, 2e-6 to 5e-6 of probabilities at batch 1 to 64); the
    # share is that of steps whose two best classes are nearly tied.
    return {"rel": 4e-6 if det else 4e-5, "max": 4e-4 if det else 4e-3, "differ": 0.005}


# ------------------------------------------------------------------- exact

class _Net:
    """The networks in float64 on the GPU, from the weight file alone.
    Batch norm, the 9x9 layers and the intraclass branches run as stored."""

    def __init__(self, path):
        from safetensors.numpy import load_file

        self.t = {k: torch.from_numpy(v).double().cuda() for k, v in load_file(str(path)).items()}

    def conv(self, p, x, stride=(1, 1), pads=(0, 0, 0, 0), bias=False):
        """Convolution as one product per tap; x is [N, H, W, C]."""
        w = self.t[f"{p}.weight"]
        kh, kw = w.shape[2], w.shape[3]
        top, left, bottom, right = pads
        x = F.pad(x, (0, 0, left, right, top, bottom))
        h, v = (x.shape[1] - kh) // stride[0] + 1, (x.shape[2] - kw) // stride[1] + 1
        depthwise = w.shape[1] == 1 and x.shape[3] > 1
        y = None
        for ky in range(kh):
            for kx in range(kw):
                s = x[:, ky:ky + (h - 1) * stride[0] + 1:stride[0], kx:kx + (v - 1) * stride[1] + 1:stride[1]]
                if depthwise:
                    part = s * w[:, 0, ky, kx]
                else:
                    part = (s.reshape(-1, s.shape[3]) @ w[:, :, ky, kx].t().contiguous()).reshape(s.shape[:3] + (-1,))
                y = part if y is None else y.add_(part)
        return y + self.t[f"{p}.bias"] if bias else y

    def bn(self, p, x):
        t = self.t
        return (x - t[f"{p}.running_mean"]) / torch.sqrt(t[f"{p}.running_var"] + 1e-5) * t[f"{p}.weight"] + t[f"{p}.bias"]

    def cba(self, p, x, stride=(1, 1), pads=(0, 0, 0, 0), bias=False, norm="normalization", act=None):
        y = self.bn(f"{p}.{norm}", self.conv(f"{p}.convolution", x, stride, pads, bias))
        return act(y) if act else y

    def gate(self, p, x, slope, a, b):
        g = F.relu(self.conv(f"{p}.{a}", x.mean(dim=(1, 2), keepdim=True), bias=True))
        return (self.conv(f"{p}.{b}", g, bias=True) * slope + 0.5).clamp(0.0, 1.0)

    def block(self, p, x, ci, co, stride):
        plain = ci == co and stride == (1, 1)
        one = (1, 1, 1, 1)
        t = self.conv(f"{p}.token_conv", x, stride, one, True) if plain else self.cba(f"{p}.token_conv", x, stride, one)
        se = f"{p}.token_squeeze_excitation"
        if f"{se}.convolutions.0.weight" in self.t:
            t = t * self.gate(se, t, 1 / 6, "convolutions.0", "convolutions.2")
        o = self.cba(f"{p}.channel_conv2", self.cba(f"{p}.channel_conv1", t, act=F.gelu))
        return t + o if plain else o

    def backbone(self, x, stages, small):
        p, one, two = "model.backbone.encoder.convolution", (1, 1, 1, 1), (2, 2)
        if small:
            x = self.cba(f"{p}.conv2", self.cba(f"{p}.conv1", x, two, one, act=F.gelu), two, one)
        else:
            e = self.cba(f"{p}.stem1", x, two, one, act=F.relu)
            br = self.cba(f"{p}.stem2a", e, pads=(0, 0, 1, 1), act=F.relu)
            br = self.cba(f"{p}.stem2b", br, pads=(0, 0, 1, 1), act=F.relu)
            q = F.pad(e, (0, 0, 0, 1, 0, 1), value=-math.inf)
            q = torch.maximum(torch.maximum(q[:, :-1, :-1], q[:, 1:, :-1]), torch.maximum(q[:, :-1, 1:], q[:, 1:, 1:]))
            x = self.cba(f"{p}.stem3", torch.cat([q, br], 3), two, one, act=F.relu)
            x = self.cba(f"{p}.stem4", x, act=F.relu)
        outs = []
        for s, blocks in enumerate(stages):
            for b, (ci, co, stride) in enumerate(blocks):
                x = self.block(f"model.backbone.encoder.blocks.{s}.blocks.{b}", x, ci, co, stride)
            outs.append(x)
        return outs

    @staticmethod
    def up(x, k):
        return x.repeat_interleave(k, 1).repeat_interleave(k, 2) if k > 1 else x

    def detector(self, tier, x):
        c = {"medium": (128, 256, 512, 896), "small": (48, 96, 192, 384), "tiny": (32, 48, 64, 160)}[tier]
        depth = (1, 3, 5, 3)
        stages = [[(c[max(0, s - 1)] if b == 0 else c[s], c[s], (2, 2) if s and b == 0 else (1, 1))
                   for b in range(depth[s] + (s == 0))] for s in range(4)]
        f = self.backbone(x, stages, False)
        x = self.medium_neck(f) if tier == "medium" else self.fpn(f, 7 if tier == "small" else 5)
        d = self.cba("head.conv_down", x, pads=(1, 1, 1, 1), norm="norm", act=F.relu)
        u = F.relu(self.bn("head.conv_up.norm", self.deconv("head.conv_up.convolution", d)))
        return torch.sigmoid(self.deconv("head.conv_final", u)).permute(0, 3, 1, 2)

    def deconv(self, p, x):
        """2x2 transposed convolution of stride 2; the weight is [I, O, 2, 2]."""
        w = self.t[f"{p}.weight"]
        n, h, v, ci = x.shape
        y = (x.reshape(-1, ci) @ w.permute(0, 2, 3, 1).reshape(ci, -1)).reshape(n, h, v, 2, 2, w.shape[1])
        return y.permute(0, 1, 3, 2, 4, 5).reshape(n, 2 * h, 2 * v, -1) + self.t[f"{p}.bias"]

    def fpn(self, stages, k):
        g = ("conv1", "conv2")
        f = []
        for i, x in enumerate(stages):
            h = self.conv(f"model.neck.insert_conv.{i}.in_conv", x)
            f.append(h + h * self.gate(f"model.neck.insert_conv.{i}.squeeze_excitation_block", h, 0.2, *g))
        for i in (2, 1, 0):
            f[i] = f[i] + self.up(f[i + 1], 2)
        out = []
        for i, x in enumerate(f):
            p = f"model.neck.input_conv.{i}"
            h = self.conv(f"{p}.depthwise_convolution", x, pads=(k // 2,) * 4, bias=True)
            h = self.conv(f"{p}.pointwise_convolution", h)
            out.append(h + h * self.gate(f"{p}.squeeze_excitation_module", h, 0.2, *g))
        return torch.cat([self.up(x, s) for x, s in zip(out[::-1], (8, 4, 2, 1))], 3)

    def medium_neck(self, stages):
        n, four = "model.neck", (4, 4, 4, 4)
        f = [self.conv(f"{n}.input_channel_adjustment_convolution.{i}", x) for i, x in enumerate(stages)]
        for i in (2, 1, 0):
            f[i] = f[i] + self.up(f[i + 1], 2)
        f = [self.conv(f"{n}.input_feature_projection_convolution.{i}", x, pads=four, bias=True) for i, x in enumerate(f)]
        for i in (1, 2, 3):
            f[i] = f[i] + self.conv(f"{n}.path_aggregation_head_convolution.{i - 1}", f[i - 1], (2, 2), (1, 1, 1, 1))
        f = [self.conv(f"{n}.path_aggregation_lateral_convolution.{i}", x, pads=four, bias=True) for i, x in enumerate(f)]
        out = []
        for i, x in enumerate(f):
            p = f"{n}.intraclass_blocks.{i}"
            r = self.conv(f"{p}.conv_reduce_channel", x, bias=True)
            for ratio, q in (("longratio", 3), ("midratio", 2), ("shortratio", 1)):
                r = (self.conv(f"{p}.symmetric_conv_long_{ratio}", r, pads=(q, q, q, q), bias=True)
                     + self.conv(f"{p}.vertical_long_to_small_conv_{ratio}", r, pads=(q, 0, q, 0), bias=True)
                     + self.conv(f"{p}.horizontal_small_to_long_conv_{ratio}", r, pads=(0, q, 0, q), bias=True))
            out.append(x + self.cba(f"{p}.conv_final", r, bias=True, norm="norm", act=F.relu))
        return torch.cat([self.up(x, s) for x, s in zip(out[::-1], (8, 4, 2, 1))], 3)

    def linear(self, p, x):
        w, b = self.t[f"{p}.weight"], self.t[f"{p}.bias"]
        return (x.reshape(-1, x.shape[-1]) @ w.t().contiguous()).reshape(x.shape[:-1] + (-1,)) + b

    def norm(self, p, x):
        x = x - x.mean(-1, keepdim=True)
        return x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-6) * self.t[f"{p}.weight"] + self.t[f"{p}.bias"]

    def attention(self, p, x):
        n, t, c = x.shape
        q, k, v = self.linear(f"{p}.qkv", x).reshape(n, t, 3, 8, c // 8).permute(2, 0, 3, 1, 4).contiguous()
        a = torch.softmax((q @ k.transpose(2, 3).contiguous()) * (c // 8) ** -0.5, -1)
        return self.linear(f"{p}.projection", (a @ v).transpose(1, 2).reshape(n, t, c))

    def recognizer(self, tier, x):
        one, two = (1, 1), (2, 1)
        c, depth = {"medium": ((128, 128, 256, 512, 768), (1, 3, 7, 3)), "small": ((96, 96, 96, 192, 384), (1, 2, 7, 3)),
                    "tiny": ((48, 48, 48, 96, 160), (1, 1, 3, 4))}[tier]
        stages = [[(c[s] if b == 0 else c[s + 1], c[s + 1], two if s > 1 and b == 0 else one) for b in range(depth[s])]
                  for s in range(4)]
        x = self.backbone(x, stages, tier == "tiny")[-1]
        n, h, w, c = x.shape
        h, w = h // 3, w // 2
        x = x[:, :3 * h, :2 * w].reshape(n, h, 3, w, 2, c).mean(dim=(2, 4))
        if tier == "tiny":
            self.t.setdefault("head.conv1_2d.weight", self.t["head.conv1.weight"].unsqueeze(2))
            self.t.setdefault("head.conv2_2d.weight", self.t["head.conv2.weight"].unsqueeze(2))
            s = F.hardswish(self.bn("head.norm1", self.conv("head.conv1_2d", x, pads=(0, 2, 0, 2))))
            s = F.hardswish(self.bn("head.norm2", self.conv("head.conv2_2d", s)))
            return torch.softmax(self.linear("head.fc2", self.linear("head.fc1", s[:, 0])), -1)
        e = "head.encoder"
        skip = self.cba(f"{e}.conv_block.0", x, act=F.silu)
        x = self.cba(f"{e}.conv_block.1", x, act=F.silu)
        x = x + self.cba(f"{e}.conv_block.2", x, pads=(0, 3, 0, 3), act=F.silu)
        s = x.reshape(n, -1, x.shape[3])
        for i in range(2):
            p = f"{e}.svtr_block.{i}"
            s = s + self.attention(f"{p}.self_attn", self.norm(f"{p}.layer_norm1", s))
            s = s + self.linear(f"{p}.mlp.fc2", F.silu(self.linear(f"{p}.mlp.fc1", self.norm(f"{p}.layer_norm2", s))))
        s = self.norm(f"{e}.norm", s) + skip.reshape(n, -1, skip.shape[3])
        return torch.softmax(self.linear("head.head", s), -1)


def _sample(page, quad, content, height, width, detector):
    """The reference's quad-bilinear sampling of a page.  The sample is
    rounded to a whole pixel value, so it is computed in the same 32-bit steps;
    its normalisation is not."""
    one, half = np.float32(1), np.float32(0.5)
    q = quad.astype(np.float32)
    v = ((np.arange(height, dtype=np.float32) + half) / np.float32(height))[:, None]
    u = ((np.arange(content, dtype=np.float32) + half) / np.float32(content))[None, :]
    ou, ov = one - u, one - v
    at = []
    for a, most in ((0, page.shape[1] - 1), (1, page.shape[0] - 1)):
        s = (q[0, a] * ou + q[1, a] * u) * ov + (q[3, a] * ou + q[2, a] * u) * v - half
        at.append(np.minimum(np.maximum(s, np.float32(0)), np.float32(most)))
    x0, y0 = (np.floor(s).astype(np.int64) for s in at)
    tx, ty = ((s - i.astype(np.float32))[..., None] for s, i in zip(at, (x0, y0)))
    x1, y1 = np.minimum(x0 + 1, page.shape[1] - 1), np.minimum(y0 + 1, page.shape[0] - 1)
    p = page.astype(np.float32)
    top = p[y0, x0] * (one - tx) + p[y0, x1] * tx
    bottom = p[y1, x0] * (one - tx) + p[y1, x1] * tx
    s = top * (one - ty) + bottom * ty
    whole = np.trunc(s)
    whole = np.clip(whole + (s - whole >= half), 0, 255)[..., ::-1].astype(np.float64)
    mean, std = ((0.485, 0.456, 0.406), (0.229, 0.224, 0.225)) if detector else ((0.5,) * 3, (0.5,) * 3)
    out = np.zeros((height, width, 3))
    out[:, :content] = (whole / 255.0 - mean) / std
    return out


def exact(case, seed):
    if case["kind"] == "db":
        # Corners come from a component's axis and extents; there is no
        # rounding of a sum to compare.
        return None
    if work(case)["flops"] * (2.7 if case["kind"] == "det" and case["tier"] == "medium" else 1.0) > 8e12:
        return None
    data = _inputs(case, seed)
    n, h, w = case["batch"], case["height"], case["width"]
    if case["source"] == "host":
        x = data["planes"].transpose(0, 2, 3, 1).astype(np.float64)
    else:
        widths = data["widths"] or [w] * n
        x = np.stack([_sample(data["page"], q, c, h, w, case["kind"] == "det") for q, c in zip(data["quads"], widths)])
    net = _Net(_weights_file(case["kind"], case["tier"]))
    call = net.detector if case["kind"] == "det" else net.recognizer
    step = max(1, int(4e6 // (h * w)))
    parts = []
    with torch.no_grad():
        for i in range(0, n, step):
            y = call(case["tier"], torch.from_numpy(np.ascontiguousarray(x[i:i + step])).cuda())
            parts.append(y.amax(-1) if case["greedy"] else y)
        y = torch.cat(parts)
    return {"classes": None, "probabilities": y} if case["greedy"] else y


if __name__ == "__main__":
    for c in listed() + [draw(random.Random(7)) for _ in range(3)]:
        print(c, work(c))
