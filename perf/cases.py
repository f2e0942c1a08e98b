"""What a user of this backend has it do, as cases to be measured.

The work of the framework is a page's: its detector input and the detector
(`det`), the crops of its boxes as recogniser inputs (`crops`), the
recogniser over a batch of lines (`rec`), and under those the layers a
program can also call alone: a transformer block (`encoder`), the CTC head
(`ctc`), and the layer kernels on device memory (`mean`, `argmax`). Sizes are
those of the page pipeline, the page worker, the benchmark and the tests; all
numbers are f32, the only type the framework computes in.

The networks are the synthetic PP-OCR detector and recogniser of the
benchmark, written here once (`detector`, `recogniser`, ...) against a small
builder interface: `PlanBuilder` makes the plan file of it, `Float64` runs it
in 64 bits on plain torch.
"""
from __future__ import annotations

import ctypes as C
import importlib.util
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent


def _package():
    if "ppocr_native_amd" not in sys.modules:
        d = ROOT / "ppocr-native_amd"
        spec = importlib.util.spec_from_file_location("ppocr_native_amd", d / "__init__.py",
                                                      submodule_search_locations=[str(d)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["ppocr_native_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["ppocr_native_amd"]


P = _package()
from ppocr_native_amd import images  # noqa: E402
from ppocr_native_amd.planfile import PlanBuilder  # noqa: E402

DEV = "cuda"


# ---------------------------------------------------------------- the cases

def listed() -> list[dict]:
    return [
        # One line read alone: the worker's re-read of a turned line. The
        # smallest call of a network; launches and latency count.
        {"name": "rec 1 line", "kind": "rec", "lines": 1, "narrow": 320, "wide": 320, "mix": 0},
        # A full batch of a page's lines, each squeezed to 320 columns: the
        # page pipeline's and the benchmark's batch.
        {"name": "rec 16 lines", "kind": "rec", "lines": 16, "narrow": 320, "wide": 320, "mix": 0},
        # A full batch with each line at its own width, as the reference's
        # worker (and this one's, uncapped) reads long lines.
        {"name": "rec 16 ragged", "kind": "rec", "lines": 16, "narrow": 320, "wide": 1100, "mix": 7},
        # A snippet of a page.
        {"name": "det 224x320", "kind": "det", "page_w": 331, "page_h": 223, "w": 320, "h": 224},
        # A letter page at 300 dpi, its long side limited to 960: the page
        # pipeline's detector.
        {"name": "det 736x960", "kind": "det", "page_w": 2550, "page_h": 3300, "w": 736, "h": 960},
        # The same page at the size the reference's worker detects it at.
        {"name": "det 1536x1984", "kind": "det", "page_w": 2550, "page_h": 3300, "w": 1536, "h": 1984},
        # The 16 tilted line boxes of a batch to recogniser inputs, uncapped.
        {"name": "crops 16", "kind": "crops", "lines": 16, "long": 900, "page_w": 2550, "page_h": 3300, "mix": 3},
        # One transformer block over a batch of 80-step lines.
        {"name": "encoder 16x80", "kind": "encoder", "lines": 16, "steps": 80},
        # The CTC head over the benchmark's 18385 classes.
        {"name": "ctc 16x80", "kind": "ctc", "lines": 16, "steps": 80, "classes": 18385},
        # A squeeze-and-excite mean of the benchmark's size, as a layer call.
        {"name": "mean 3600x480", "kind": "mean", "pixels": 3600, "channels": 480},
        # The CTC choice over a batch's logits, as a layer call.
        {"name": "argmax 1280x18385", "kind": "argmax", "rows": 1280, "cols": 18385},
    ]


def _log(rng: random.Random, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["rec", "rec", "det", "det", "crops", "encoder", "ctc", "mean", "argmax"])
    mix = rng.randrange(1 << 20)
    if kind == "rec":
        # Any number of lines up to a batch; capped (all 320 wide) or each
        # line as wide as it is.
        wide = 320 if rng.random() < 0.4 else rng.randrange(330, 1100)
        return {"kind": kind, "lines": rng.randint(1, 16), "narrow": 320, "wide": wide, "mix": mix}
    if kind == "det":
        # Both sides snapped to 32, from a snippet to the largest page.
        w, h = 32 * _log(rng, 3, 48), 32 * _log(rng, 3, 62)
        return {"kind": kind, "page_w": int(w * rng.uniform(0.9, 2.2)), "page_h": int(h * rng.uniform(0.9, 2.2)),
                "w": w, "h": h}
    if kind == "crops":
        return {"kind": kind, "lines": rng.randint(1, 16), "long": rng.randint(200, 900),
                "page_w": rng.randint(1100, 2550), "page_h": rng.randint(1500, 3300), "mix": mix}
    if kind == "encoder":
        return {"kind": kind, "lines": rng.randint(1, 16), "steps": _log(rng, 20, 160)}
    if kind == "ctc":
        return {"kind": kind, "lines": rng.randint(1, 16), "steps": _log(rng, 20, 160),
                "classes": rng.choice([6625, 18385, 18710, rng.randint(96, 18710)])}
    if kind == "mean":
        return {"kind": kind, "pixels": _log(rng, 60, 25600), "channels": 4 * rng.randint(6, 120)}
    return {"kind": kind, "rows": _log(rng, 20, 1280), "cols": _log(rng, 96, 18710)}


# ---------------------------------------------------------------- networks

class Weights:
    """Seeded weights: N(0, gain / sqrt(fan in)), biases N(0, 0.05), which
    keep the signal's scale through the depth."""

    def __init__(self, seed: int, gain: float):
        self.rng = np.random.default_rng(seed)
        self.gain = gain

    def w(self, shape, fan_in: int, gain: float | None = None) -> np.ndarray:
        std = (self.gain if gain is None else gain) / math.sqrt(fan_in)
        return self.rng.normal(0.0, std, size=shape).astype(np.float32)

    def b(self, n: int) -> np.ndarray:
        return self.rng.normal(0.0, 0.05, size=n).astype(np.float32)

    def conv(self, b, x, oc: int, k: int, s=(1, 1), pad=None, fused="none", x2=None):
        ci = x.c + (x2.c if x2 is not None else 0)
        p = (k - 1) // 2
        return b.conv(x, self.w((k, k, ci, oc), k * k * ci), self.b(oc), k=(k, k), s=s,
                      pad=(p, p, p, p) if pad is None else pad, fused=fused, x2=x2)

    def gate(self, b, x, fused: str):
        h = self.conv(b, b.mean(x), max(1, x.c // 4), 1, fused="relu")
        return self.conv(b, h, x.c, 1, fused=fused)

    def dw_block(self, b, x, oc: int, k: int, s=(1, 1), se: bool = False):
        p = (k - 1) // 2
        d = b.dwconv(x, self.w((k, k, x.c), k * k), self.b(x.c), k=(k, k), s=s, pad=(p, p, p, p),
                     fused="hardswish")
        if se:
            d = b.channelmul(d, self.gate(b, d, "hardsigmoid"))
        residual = tuple(s) == (1, 1) and oc == x.c
        y = self.conv(b, d, oc, 1, fused="none" if residual else "hardswish")
        return b.add(y, x) if residual else y

    def rse(self, b, x, oc: int, k: int):
        y = self.conv(b, x, oc, k)
        return b.add(y, b.channelmul(y, self.gate(b, y, "hardsigmoidfifth")))


def detector(b, r: Weights):
    act = "hardswish"
    after = (0, 1, 0, 1)
    s1 = r.conv(b, b.input, 24, 3, s=(2, 2), fused=act)
    s2 = r.conv(b, s1, 12, 2, pad=after, fused=act)
    s2 = r.conv(b, s2, 24, 2, pad=after, fused=act)
    z = r.conv(b, b.maxpool(s1), 32, 3, s=(2, 2), fused=act, x2=s2)
    z = r.conv(b, z, 32, 1, fused=act)
    c2 = r.dw_block(b, z, 48, 3)
    z = r.dw_block(b, c2, 96, 3, s=(2, 2))
    c3 = r.dw_block(b, z, 96, 3)
    z = r.dw_block(b, c3, 192, 5, s=(2, 2))
    z = r.dw_block(b, z, 192, 5)
    c4 = r.dw_block(b, z, 192, 7, se=True)
    z = r.dw_block(b, c4, 384, 5, s=(2, 2), se=True)
    c5 = r.dw_block(b, z, 384, 7, se=True)
    in5 = r.rse(b, c5, 96, 1)
    out4 = b.upsampleadd(in5, r.rse(b, c4, 96, 1), 2)
    out3 = b.upsampleadd(out4, r.rse(b, c3, 96, 1), 2)
    out2 = b.upsampleadd(out3, r.rse(b, c2, 96, 1), 2)
    p5, p4, p3, p2 = (r.rse(b, t, 24, 3) for t in (in5, out4, out3, out2))
    cat = b.concat(b.concat(b.upsample(p5, 8), b.upsample(p4, 4)), b.upsample(p3, 2))
    hd = r.conv(b, cat, 24, 3, fused="relu", x2=p2)
    hd = b.convtranspose(hd, r.w((24, 2, 2, 24), 24), r.b(24), k=(2, 2), fused="relu")
    return b.convtranspose(hd, r.w((24, 2, 2, 1), 24), r.b(1), k=(2, 2), fused="sigmoid")


def layernorm(b, r: Weights, x):
    return b.layernorm(x, r.rng.normal(1.0, 0.1, x.c), r.rng.normal(0.0, 0.1, x.c), 1e-6)


def transformer(b, r: Weights, z, heads: int = 8):
    d = z.c
    qkv = b.conv(layernorm(b, r, z), r.w((1, 1, d, 3 * d), d, 1.0), r.b(3 * d))
    a = b.attention(qkv, heads, float(np.float32((d // heads) ** -0.5)))
    z = b.add(z, b.conv(a, r.w((1, 1, d, d), d, 1.0), r.b(d)))
    f = b.conv(layernorm(b, r, z), r.w((1, 1, d, 2 * d), d), r.b(2 * d), fused="swish")
    return b.add(z, b.conv(f, r.w((1, 1, 2 * d, d), 2 * d, 1.0), r.b(d)))


def recogniser(b, r: Weights, classes: int = 18385, dim: int = 120):
    z = r.conv(b, b.input, 48, 3, s=(2, 2), fused="hardswish")
    z = r.dw_block(b, z, 64, 3)
    z = r.dw_block(b, z, 128, 3, s=(2, 2))
    z = r.dw_block(b, z, 128, 3)
    z = r.dw_block(b, z, 256, 3, s=(2, 1))
    z = r.dw_block(b, z, 256, 5)
    z = r.dw_block(b, z, 256, 5)
    z = r.dw_block(b, z, 480, 5, s=(2, 1), se=True)
    z = r.dw_block(b, z, 480, 5, se=True)
    z = b.avgpool(z, (z.h, 1), (z.h, 1))
    z = b.conv(z, r.w((1, 1, 480, dim), 480), r.b(dim), fused="swish")
    for _ in range(2):
        z = transformer(b, r, z)
    return ctc_head(b, r, layernorm(b, r, z), classes)


def ctc_head(b, r: Weights, x, classes: int):
    # Logits with a spread of about 3: a trained head's steps are mostly sure.
    return b.ctcargmax(x, r.w((x.c, classes), x.c, 3.0), r.b(classes))


def encoder(b, r: Weights):
    return layernorm(b, r, transformer(b, r, b.input))


def _plan(h: int, w: int, c: int, net) -> bytes:
    b = PlanBuilder(h, w, c)
    return b.to_bytes([net(b)])


# ---------------------------------------------------------------- 64 bits

class Map:
    """A [lanes, h, w, c] map in 64 bits."""

    def __init__(self, t: torch.Tensor):
        self.t = t
        self.h, self.w, self.c = t.shape[1:]


def _t64(a) -> torch.Tensor:
    return torch.from_numpy(np.asarray(a, np.float32)).to(DEV).double()


def _act64(t: torch.Tensor, fused: str) -> torch.Tensor:
    if fused == "relu":
        return t.clamp(min=0)
    if fused == "sigmoid":
        return torch.sigmoid(t)
    if fused == "swish":
        return t * torch.sigmoid(t)
    if fused == "hardsigmoid":
        return (t / 6 + 0.5).clamp(0, 1)
    if fused == "hardsigmoidfifth":
        return (t * 0.2 + 0.5).clamp(0, 1)
    if fused == "hardswish":
        return t * (t / 6 + 0.5).clamp(0, 1)
    assert fused == "none", fused
    return t


class Float64:
    """The builder's operations, run at once on plain torch in 64 bits."""

    def __init__(self, x: torch.Tensor):
        self.input = Map(x)

    @staticmethod
    def _taps(t, k, s, pad):
        pt, pb, pl, pr = pad
        t = torch.nn.functional.pad(t, (0, 0, pl, pr, pt, pb))
        oh, ow = (t.shape[1] - k[0]) // s[0] + 1, (t.shape[2] - k[1]) // s[1] + 1
        for y in range(k[0]):
            for x in range(k[1]):
                yield y, x, t[:, y:y + (oh - 1) * s[0] + 1:s[0], x:x + (ow - 1) * s[1] + 1:s[1]]

    def conv(self, x, weight, bias, *, k=(1, 1), s=(1, 1), pad=(0, 0, 0, 0), fused="none", x2=None):
        t = x.t if x2 is None else torch.cat([x.t, x2.t], 3)
        w = _t64(weight)
        y = sum(torch.matmul(v.reshape(-1, t.shape[3]), w[i, j]).reshape(*v.shape[:3], -1)
                for i, j, v in self._taps(t, k, s, pad))
        return Map(_act64(y + _t64(bias), fused))

    def dwconv(self, x, weight, bias, *, k, s=(1, 1), pad, fused="none"):
        w = _t64(weight)
        return Map(_act64(sum(v * w[i, j] for i, j, v in self._taps(x.t, k, s, pad)) + _t64(bias), fused))

    def add(self, a, b):
        return Map(a.t + b.t)

    def channelmul(self, x, gate):
        return Map(x.t * gate.t)

    def mean(self, x):
        return Map(x.t.mean((1, 2), keepdim=True))

    def maxpool(self, x):
        t = torch.nn.functional.pad(x.t, (0, 0, 0, 1, 0, 1), value=-math.inf)
        return Map(torch.maximum(torch.maximum(t[:, :-1, :-1], t[:, :-1, 1:]),
                                 torch.maximum(t[:, 1:, :-1], t[:, 1:, 1:])))

    def avgpool(self, x, k, s):
        return Map(x.t.mean(1, keepdim=True))  # the whole height, one column

    def concat(self, a, b):
        return Map(torch.cat([a.t, b.t], 3))

    def upsample(self, x, f):
        return Map(x.t.repeat_interleave(f, 1).repeat_interleave(f, 2))

    def upsampleadd(self, x, addend, f):
        return Map(self.upsample(x, f).t + addend.t)

    def convtranspose(self, x, weight, bias, *, k, fused="none"):
        w = _t64(weight)
        L, h, wd, ic = x.t.shape
        y = torch.matmul(x.t.reshape(-1, ic), w.reshape(ic, -1)).reshape(L, h, wd, k[0], k[1], -1)
        y = y.permute(0, 1, 3, 2, 4, 5).reshape(L, h * k[0], wd * k[1], -1)
        return Map(_act64(y + _t64(bias), fused))

    def layernorm(self, x, gamma, beta, eps):
        m = x.t.mean(3, keepdim=True)
        v = (x.t - m).square().mean(3, keepdim=True)
        return Map((x.t - m) / torch.sqrt(v + eps) * _t64(gamma) + _t64(beta))

    def attention(self, qkv, heads, scale):
        L, _, T, c3 = qkv.t.shape
        c = c3 // 3
        q, k, v = (qkv.t.reshape(L, T, 3, heads, c // heads).permute(2, 0, 3, 1, 4)[i] for i in range(3))
        s = torch.softmax(torch.matmul(q * scale, k.transpose(2, 3).contiguous()), 3)
        return Map(torch.matmul(s, v.contiguous()).permute(0, 2, 1, 3).reshape(L, 1, T, c))

    def ctcargmax(self, x, weight, bias):
        y = torch.matmul(x.t.reshape(-1, x.c), _t64(weight)) + _t64(bias)
        return torch.softmax(y, 1).amax(1).reshape(x.t.shape[0], -1)  # each step's best probability


# ---------------------------------------------------------------- inputs

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _page(w: int, h: int, seed: int, pitch: int = 40) -> torch.Tensor:
    """A page on the GPU, h x w x 3 bytes: dark strokes in text-like bands on
    light paper."""
    g = _gen(seed)
    paper = torch.randint(236, 256, (h, w, 3), generator=g, device=DEV, dtype=torch.uint8)
    ink = torch.randint(0, 90, (h, w, 1), generator=g, device=DEV, dtype=torch.uint8)
    yy = torch.arange(h, device=DEV)[:, None]
    xx = torch.arange(w, device=DEV)[None, :]
    words = torch.rand((h // pitch + 1, w // 24 + 1), generator=g, device=DEV) < 0.8
    mask = (yy % pitch >= 8) & (yy % pitch < pitch - 6) & words[yy // pitch, xx // 24]
    mask &= torch.rand((h, w), generator=g, device=DEV) < 0.4
    return torch.where(mask[..., None], ink, paper).contiguous()


def _line_boxes(case: dict) -> tuple[int, int, list[tuple[int, int, int, int]], list[tuple[int, int]]]:
    """The page of a `rec` case: its size, each line's box (x, y, w, h), and
    the tensor and resized widths a box gives (48 rows; at least 320 wide)."""
    rng = random.Random(case["mix"])
    boxes, widths, y = [], [], 16
    for _ in range(case["lines"]):
        want = rng.randint(case["narrow"], case["wide"])
        if case["wide"] == 320:
            want = rng.randint(150, 320)  # short lines pad to 320
        h = rng.randint(28, 60)
        w = max(8, want * h // 48)
        x = rng.randint(0, 60)
        boxes.append((x, y, w, h))
        y += h + rng.randint(4, 12)
        width = int(48.0 * max(320.0 / 48.0, w / h))
        widths.append((width, min(width, math.ceil(48.0 * (w / h)))))
    return max(x + w for x, _, w, _ in boxes) + 40, y + 16, boxes, widths


def _tilted(case: dict) -> np.ndarray:
    """The tilted boxes of a `crops` case, n x 4 corners."""
    rng = random.Random(case["mix"])
    out = []
    for i in range(case["lines"]):
        w, h, t = rng.uniform(0.3, 1.0) * case["long"], rng.uniform(24, 60), rng.uniform(-0.04, 0.04)
        x = rng.uniform(20, case["page_w"] - w - 80)
        y = rng.uniform(80, case["page_h"] - 160)
        c, s = math.cos(t), math.sin(t)
        out.append([[x, y], [x + w * c, y + w * s], [x + w * c - h * s, y + w * s + h * c], [x - h * s, y + h * c]])
    return np.asarray(out, np.float32)


def _crop_widths(quads: np.ndarray) -> list[int]:
    return [images.rec_width_fit(*images.crop_size(q), 0)[0] for q in quads]


def _dims(case: dict) -> list[tuple[int, int]]:
    return [(1, case["steps"])] * case["lines"]


def _queries(case: dict, seed: int) -> np.ndarray:
    """What reaches the encoder or the CTC head: normalised rows of 120."""
    return np.random.default_rng(seed).normal(0, 1, (case["lines"], case["steps"], 120)).astype(np.float32)


def _layer_model(case: dict, seed: int, net) -> dict:
    """A layer as a plan, its lanes' inputs in the model's host memory."""
    g = P.GpuModel.load(_plan(1, case["steps"], 120, net))
    g.set_sizes(_dims(case))
    for i, x in enumerate(_queries(case, seed)):
        g.lane_input_mut(i)[:] = x.reshape(-1)
    return {"model": g, "outs": _outs(g, case["lines"])}


class _Held:
    """Host memory of a model's, which stays while an array of it does."""

    def __init__(self, g, address: int, count: int, kind: str):
        self.g = g
        self.__array_interface__ = {"shape": (count,), "typestr": kind, "data": (address, False), "version": 3}


def _outs(g, lanes: int, index: int = 0) -> list[np.ndarray]:
    """Every lane's output, as the model's own host buffers."""
    L, n = P.lib(), C.c_size_t()
    got = []
    for i in range(lanes):
        p = L.ppocr_gpu_lane_output(g._h, i, index, C.byref(n))
        got.append(np.asarray(_Held(g, C.cast(p, C.c_void_p).value, n.value, "<f4")))
    return got


NET_SEED = 21  # a program's weights stay while its inputs change


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    s: dict = {"kind": kind}
    if kind == "rec":
        w, h, boxes, widths = _line_boxes(case)
        g = P.GpuModel.load(_plan(48, 320, 3, lambda b: recogniser(b, Weights(NET_SEED, 1.6))))
        g.set_sizes([(48, tw) for tw, _ in widths])
        n = len(boxes)
        quads = np.asarray([[[x, y], [x + bw, y], [x + bw, y + bh], [x, y + bh]] for x, y, bw, bh in boxes], np.float32)
        s.update(model=g, page=_page(w, h, seed), w=w, h=h, n=n, quads=quads, sizes=[(48, tw) for tw, _ in widths],
                 flat=quads.ctypes.data_as(C.POINTER(C.c_float)), outs=_outs(g, n),
                 at=(C.c_void_p * n)(*[g.lane_input_device(i)[0] for i in range(n)]),
                 caps=(C.c_size_t * n)(*[g.lane_input_device(i)[1] for i in range(n)]), got=(C.c_size_t * n)(),
                 abi=images._sig())
    elif kind == "det":
        g = P.GpuModel.load(_plan(case["h"], case["w"], 3, lambda b: detector(b, Weights(NET_SEED, 1.3))))
        g.set_db_mask(0, 0.3)
        s.update(model=g, page=_page(case["page_w"], case["page_h"], seed, 44), w=case["w"], h=case["h"],
                 mean=(C.c_double * 3)(*images.MEAN), std=(C.c_double * 3)(*images.STD), abi=images._sig(),
                 at=g.lane_input_device(0)[0])
        wpr, rows = C.c_size_t(), C.c_size_t()
        p = P.lib().ppocr_gpu_lane_db_mask(g._h, 0, C.byref(wpr), C.byref(rows))
        s["outs"] = {"map": _outs(g, 1)[0],
                     "bits": np.asarray(_Held(g, p, wpr.value * rows.value, "<i8"))}
    elif kind == "crops":
        quads = _tilted(case)
        widths = _crop_widths(quads)
        outs = [torch.empty(48 * w * 3, device=DEV) for w in widths]
        n = len(outs)
        s.update(page=_page(case["page_w"], case["page_h"], seed), w=case["page_w"], h=case["page_h"], n=n, quads=quads,
                 flat=quads.ctypes.data_as(C.POINTER(C.c_float)), outs=outs,
                 at=(C.c_void_p * n)(*[o.data_ptr() for o in outs]), caps=(C.c_size_t * n)(*[o.numel() for o in outs]),
                 got=(C.c_size_t * n)(), abi=images._sig())
    elif kind == "encoder":
        s.update(_layer_model(case, seed, lambda b: encoder(b, Weights(NET_SEED, 1.6))))
    elif kind == "ctc":
        s.update(_layer_model(case, seed, lambda b: ctc_head(b, Weights(NET_SEED, 1.6), b.input, case["classes"])))
    elif kind == "mean":
        # What a hard swish leaves: mostly small, some channels large.
        x = torch.randn(case["pixels"], case["channels"], generator=_gen(seed), device=DEV)
        s.update(x=torch.nn.functional.hardswish(x), y=torch.empty(case["channels"], device=DEV), case=case)
    else:
        x = torch.randn(case["rows"], case["cols"], generator=_gen(seed), device=DEV) * 3
        s.update(x=x, y=torch.empty(case["rows"], 2, device=DEV), case=case)
    return s


def _pairs(outs: list[np.ndarray]) -> dict:
    """The recogniser's [T][2] results as a decoder takes them."""
    pairs = [o.reshape(-1, 2) for o in outs]
    return {"best": [p[:, 0].astype(np.int64) for p in pairs], "prob": [p[:, 1] for p in pairs]}


def run(s: dict):
    kind = s["kind"]
    if kind == "rec":
        # The worker's batch: lane sizes, every line's input from the page,
        # the network, the results to the host.
        g = s["model"]
        g.set_sizes(s["sizes"])
        images._check(s["abi"].ppocr_hip_crop_rec_inputs(s["page"].data_ptr(), s["w"], s["h"], s["flat"], s["n"], 0,
                                                         s["at"], s["caps"], s["got"], g.stream() or None), "crops")
        g.run_device()
        return _pairs(s["outs"])
    if kind == "det":
        # The worker's detector: the input from the page, the network, the
        # map and its threshold to the host.
        g, p = s["model"], s["page"]
        images._check(s["abi"].ppocr_hip_det_input(p.data_ptr(), p.shape[1], p.shape[0], s["at"], s["w"], s["h"],
                                                   s["mean"], s["std"], g.stream() or None), "det_input")
        g.run_device()
        return s["outs"]
    if kind == "crops":
        stream = torch.cuda.current_stream().cuda_stream
        images._check(s["abi"].ppocr_hip_crop_rec_inputs(s["page"].data_ptr(), s["w"], s["h"], s["flat"], s["n"], 0,
                                                         s["at"], s["caps"], s["got"], stream or None), "crops")
        return s["outs"]
    if kind == "encoder":
        s["model"].run()
        return s["outs"]
    if kind == "ctc":
        s["model"].run()
        return _pairs(s["outs"])
    c, stream = s["case"], torch.cuda.current_stream().cuda_stream
    if kind == "mean":
        P.hip_channel_mean(s["x"].data_ptr(), s["y"].data_ptr(), c["pixels"], c["channels"], stream)
        return s["y"]
    P.hip_row_argmax(s["x"].data_ptr(), s["y"].data_ptr(), c["rows"], c["cols"], stream)
    return {"best": s["y"][:, 0], "prob": s["y"][:, 1]}


# ---------------------------------------------------------------- work

class Count:
    """The builder's operations, counted: floating-point operations, and the
    floats of the weights."""

    def __init__(self, h: int, w: int, c: int):
        self.b = PlanBuilder(h, w, c)
        self.input = self.b.input
        self.flops = 0.0
        self.weights = 0

    def __getattr__(self, name):
        op = getattr(self.b, name)

        def call(x, *a, **k):
            y = op(x, *a, **k)
            for v in a[:2]:
                if isinstance(v, np.ndarray):
                    self.weights += v.size
            out = y.h * y.w
            if name == "conv":
                self.flops += 2.0 * out * a[0].size
            elif name in ("dwconv", "ctcargmax"):
                self.flops += 2.0 * out * a[0].size
            elif name == "convtranspose":
                self.flops += 2.0 * x.h * x.w * a[0].size
            elif name == "attention":
                self.flops += 4.0 * x.w * x.w * y.c
            else:
                self.flops += float(max(out * y.c, x.h * x.w * x.c))
            return y
        return call


class Zeros(Weights):
    """Weights for counting: their shapes alone."""

    def w(self, shape, fan_in, gain=None):
        return np.broadcast_to(np.float32(0), shape)

    def b(self, n):
        return np.broadcast_to(np.float32(0), (n,))


def _counted(h: int, w: int, c: int, net) -> tuple[float, int]:
    k = Count(h, w, c)
    net(k, Zeros(0, 1.0))
    return k.flops, k.weights


def work(case: dict) -> dict:
    """Inputs and weights read once, outputs written once; every layer's
    floating-point operations."""
    kind = case["kind"]
    if kind == "rec":
        _, _, boxes, widths = _line_boxes(case)
        per = {}
        for tw, _ in widths:
            if tw not in per:
                per[tw] = _counted(48, tw, 3, recogniser)
        flops = sum(per[tw][0] for tw, _ in widths)
        weights = next(iter(per.values()))[1]
        return {"flops": flops, "bytes": 4.0 * weights + sum(3.0 * w * h for _, _, w, h in boxes) +
                sum(8.0 * (tw // 4) for tw, _ in widths)}
    if kind == "det":
        flops, weights = _counted(case["h"], case["w"], 3, detector)
        px = case["w"] * case["h"]
        # The page's bytes that the resize's taps touch, at most.
        page = 3.0 * min(case["page_w"], 2 * case["w"]) * min(case["page_h"], 2 * case["h"])
        return {"flops": flops, "bytes": 4.0 * weights + page + px * 4.0 + px / 8.0}
    if kind == "crops":
        quads = _tilted(case)
        px = sum(48.0 * 3 * w for w in _crop_widths(quads))
        src = sum(3.0 * w * h for w, h in map(images.crop_size, quads))
        # A resized value: two taps a side of 16-tap bicubic pixels.
        return {"flops": px * 4 * 2 * 16, "bytes": 4.0 * px + src}
    if kind in ("encoder", "ctc"):
        net = encoder if kind == "encoder" else (lambda b, r: ctc_head(b, r, b.input, case["classes"]))
        flops, weights = _counted(1, case["steps"], 120, net)
        rows = case["lines"] * case["steps"]
        return {"flops": case["lines"] * flops,
                "bytes": 4.0 * (weights + rows * 120 + rows * (120 if kind == "encoder" else 2))}
    if kind == "mean":
        n = case["pixels"] * case["channels"]
        return {"flops": float(n), "bytes": 4.0 * (n + case["channels"])}
    n = case["rows"] * case["cols"]
    return {"flops": 3.0 * n, "bytes": 4.0 * n + 8.0 * case["rows"]}


# ---------------------------------------------------------------- tolerances

def tolerance(case: dict):
    """About four times what these measured against 64 bits (rec up to 6.8e-6,
    det 5.5e-7, encoder 3e-7, ctc 1.7e-6, mean 2.5e-8, argmax 2.2e-7): f32
    throughout. A step's class may differ where two logits tie to within
    rounding, a map's bit where a probability does with the threshold. The
    crops are the reference's own arithmetic on bytes."""
    return {"rec": {"rel": 3e-5, "max": 5e-4, "differ": 0.005},
            "det": {"rel": 2.5e-6, "max": 1e-4, "differ": 0.005},
            "crops": "exact",
            "encoder": {"rel": 1.5e-6, "max": 3e-5},
            "ctc": {"rel": 8e-6, "max": 1e-4, "differ": 0.005},
            "mean": {"rel": 1.5e-7, "max": 1e-6},
            "argmax": {"rel": 1e-6, "max": 1e-5}}[case["kind"]]


# ---------------------------------------------------------------- exact

def _taps(src: int, dst: int):
    """OpenCV's 8-bit bilinear taps: source indices and 1/2048 weights."""
    d = np.arange(dst, dtype=np.float64)
    f = ((d + 0.5) * (1.0 / (dst / src)) - 0.5).astype(np.float32)
    fl = np.floor(f)
    a = (f - fl).astype(np.float32)
    s = fl.astype(np.int64)
    one = np.float32(1)
    return [torch.from_numpy(v).to(DEV) for v in (
        np.clip(s, 0, src - 1), np.clip(s + 1, 0, src - 1),
        np.rint((one - a) * np.float32(2048)).astype(np.int64), np.rint(a * np.float32(2048)).astype(np.int64))]


def _resize(img: torch.Tensor, w: int, h: int) -> torch.Tensor:
    """cv2.resize INTER_LINEAR on 8 bits, as whole numbers."""
    x = img.long()
    n, f, nw, fw = _taps(x.shape[1], w)
    x = x[:, n] * nw[None, :, None] + x[:, f] * fw[None, :, None]
    n, f, nw, fw = _taps(img.shape[0], h)
    v = (((x[n] >> 4) * nw[:, None, None]) >> 16) + (((x[f] >> 4) * fw[:, None, None]) >> 16)
    return ((v + 2) >> 2).clamp(0, 255)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "rec":
        w, h, boxes, widths = _line_boxes(case)
        page = _page(w, h, seed)
        probs: list = [None] * len(boxes)
        for tw in {t for t, _ in widths}:
            mine = [i for i, (t, _) in enumerate(widths) if t == tw]
            x = torch.zeros(len(mine), 48, tw, 3, device=DEV, dtype=torch.float64)
            for k, i in enumerate(mine):
                bx, by, bw, bh = boxes[i]
                rw = widths[i][1]
                x[k, :, :rw] = _resize(page[by:by + bh, bx:bx + bw], rw, 48).double() / 127.5 - 1.0
            for i, p in zip(mine, recogniser(Float64(x), Weights(NET_SEED, 1.6))):
                probs[i] = p
        return {"best": None, "prob": probs}
    if kind == "det":
        page = _page(case["page_w"], case["page_h"], seed, 44)
        x = _resize(page, case["w"], case["h"]).double() / 255.0
        mean, std = (torch.tensor(v, device=DEV, dtype=torch.float64) for v in (images.MEAN, images.STD))
        y = detector(Float64(((x - mean) / std)[None]), Weights(NET_SEED, 1.3))
        return {"map": y.t.reshape(-1), "bits": None}
    if kind == "encoder":
        x = _t64(_queries(case, seed))[:, None]
        return list(encoder(Float64(x), Weights(NET_SEED, 1.6)).t.reshape(case["lines"], -1))
    if kind == "ctc":
        b = Float64(_t64(_queries(case, seed))[:, None])
        return {"best": None, "prob": list(ctc_head(b, Weights(NET_SEED, 1.6), b.input, case["classes"]))}
    if kind == "mean":
        return prepare(case, seed)["x"].double().mean(0)
    if kind == "argmax":
        x = prepare(case, seed)["x"].double()
        return {"best": x.argmax(1).double(), "prob": torch.softmax(x, 1).amax(1)}
    return None  # the crops round to bytes on the way
