"""What the speed of this library is measured on: the calls that programs which read pages with it
make, through its public entry points, on the two model families that it has synthetic models for
(the ocrs architecture and the PP-OCRv6 architecture, `ocrhip.synth` and `ocrhip.synth_pp`).

Every call of the device path is queued on the context's stream: inputs and outputs are device
memory of the caller's (torch tensors here). `run` waits for nothing itself. The one host-memory
case is the page pipeline, whose pages a program has in host memory.

`exact` evaluates the same ONNX files in float64 with torch, from this file's own reader.
"""
from __future__ import annotations

import ctypes
import functools
import math
import os
import struct
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "wgpu-ocr_amd"))
import ocrhip  # noqa: E402
from ocrhip import synth, synth_pp  # noqa: E402

GPU = "cuda"
LINE_H, PAGE_W, PAGE_H = 64, 2550, 3300
TEXT_LINES, TEXT_CHARS = 256, 256  # of a page, kept by the page pipeline's case


def listed():
    return [
        # One text line, as an interactive program reads a field: latency.
        {"name": "rec_1_line", "kind": "rec", "lines": 1, "wmin": 200, "wmax": 200, "round": 50, "f32": False},
        # The recogniser configuration of this repository's benchmark: 36 lines, widths in
        # [200, 800], in batches of like width (rounded up to 50, at most 20 lines a batch).
        {"name": "rec_36_lines", "kind": "rec", "lines": 36, "wmin": 200, "wmax": 800, "round": 50, "f32": False},
        # The same lines on a trained model's weights, float32 values that are not float16 ones.
        {"name": "rec_36_lines_f32", "kind": "rec", "lines": 36, "wmin": 200, "wmax": 800, "round": 50, "f32": True},
        # A recognition pass over six pages' lines: the largest pass of the page pipeline.
        {"name": "rec_540_lines", "kind": "rec", "lines": 540, "wmin": 200, "wmax": 800, "round": 50, "f32": False},
        # The detector on one prepared 800 x 600 image in host memory (its own input size).
        {"name": "det_map", "kind": "map", "h": 800, "w": 600},
        # One scanned page (US Letter at 300 dpi) to its mask, the bytes resident on the GPU.
        {"name": "det_page", "kind": "mask", "sizes": "2550x3300"},
        # A detection pass over six pages of the sizes that scanners and screens give: Letter and
        # A4 at 300 dpi, Letter at 150 dpi, a screenshot, a page narrower than the model's input.
        {"name": "det_pages_mixed", "kind": "mask",
         "sizes": "2550x3300 2480x3508 1275x1650 1921x1079 577x911 2550x3301"},
        # The benchmark: 12 Letter pages from host memory to text.
        {"name": "pages_12", "kind": "pages", "pages": 12, "w": PAGE_W, "h": PAGE_H, "merge": 6},
        # The PP-OCR recogniser: one line, and a batch of 16 (its batch size) at a width among the
        # widest of a page. The arg-max is the text, the logits its confidences.
        {"name": "pp_rec_1_line", "kind": "pp_rec", "lines": 1, "w": 320},
        {"name": "pp_rec_16_lines", "kind": "pp_rec", "lines": 16, "w": 872},
        # The SVTR neck alone on a batch's sequence (2 transformer blocks, dim 120, 8 heads).
        {"name": "pp_svtr_16", "kind": "pp_svtr", "lines": 16, "steps": 109},
        # PP-OCR detection of four pages (the pipeline's group): model input, DB map, threshold.
        {"name": "pp_det_4_pages", "kind": "pp_det", "pages": 4, "w": PAGE_W, "h": PAGE_H},
    ]


def draw(rng):
    """A case of the same ranges: every kind, sizes spread over their logarithm, odd ones among
    them, none above the largest listed case of its kind."""
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["rec", "rec", "rec", "map", "mask", "mask", "pages", "pp_rec", "pp_rec", "pp_svtr", "pp_det"])
    if kind == "rec":
        wmin = log(100, 700)
        wmax, f32, rounding = rng.randint(wmin, 800), rng.random() < 0.3, rng.choice([50, 50, 1])
        most = 60 if rounding == 1 else 120 if f32 else 540 * 1000 // max(1000, wmin + wmax)
        return {"kind": kind, "lines": log(1, most), "wmin": wmin, "wmax": wmax, "round": rounding, "f32": f32}
    if kind == "map":  # 2 x 3 upsampling at the coarsest level: the width is an odd multiple of 8
        return {"kind": kind, "h": 16 * rng.randint(8, 50), "w": 8 * (2 * rng.randint(8, 37) + 1)}
    if kind == "mask":
        return {"kind": kind, "sizes": " ".join(f"{log(300, 2550)}x{log(300, 3508)}" for _ in range(rng.randint(1, 6)))}
    if kind == "pages":
        return {"kind": kind, "pages": log(1, 12), "w": rng.randint(1200, PAGE_W), "h": rng.randint(1500, PAGE_H),
                "merge": rng.choice([2, 4, 6])}
    if kind == "pp_rec":
        return {"kind": kind, "lines": log(1, 16), "w": 8 * log(15, 109)}
    if kind == "pp_svtr":
        return {"kind": kind, "lines": log(1, 16), "steps": log(10, 109)}
    return {"kind": kind, "pages": rng.randint(1, 4), "w": rng.randint(900, PAGE_W), "h": rng.randint(900, PAGE_H)}


# ---- models and handles a program keeps --------------------------------------------------------
def _fields(buf):
    """The fields of a protobuf message: (number, value), a value an int or bytes."""
    at, end = 0, len(buf)

    def varint():
        nonlocal at
        v = s = 0
        while True:
            b = buf[at]
            at += 1
            v |= (b & 127) << s
            s += 7
            if b < 128:
                return v

    while at < end:
        key = varint()
        if key & 7 == 0:
            yield key >> 3, varint()
        else:
            n = varint() if key & 7 == 2 else {1: 8, 5: 4}[key & 7]
            yield key >> 3, buf[at: at + n]
            at += n


def _ints(buf):
    out, v, s = [], 0, 0
    for b in buf:
        v |= (b & 127) << s
        s += 7
        if b < 128:
            out.append(v - (1 << 64) if v >> 63 else v)
            v = s = 0
    return out


class Model:
    """An ONNX file's graph: nodes [(op, inputs, outputs, attributes)], float and integer
    constants, input and output names."""

    def __init__(self, data):
        self.nodes, self.weights, self.ints = [], {}, {}
        graph = next(bytes(v) for k, v in _fields(memoryview(data)) if k == 7)
        for k, v in _fields(memoryview(graph)):
            if k == 1:
                f = list(_fields(v))
                attrs = dict(self._attr(a) for n, a in f if n == 5)
                self.nodes.append((next(bytes(a).decode() for n, a in f if n == 4), [bytes(a).decode() for n, a in f if n == 1],
                                   [bytes(a).decode() for n, a in f if n == 2], attrs))
            elif k == 5:
                f = list(_fields(v))
                d = dict(f)
                shape = [a for n, a in f if n == 1]
                (self.weights if d[2] == 1 else self.ints)[bytes(d[8]).decode()] = np.frombuffer(
                    bytes(d[9]), "<f4" if d[2] == 1 else "<i8").reshape(shape)
            elif k in (11, 12):
                setattr(self, "input" if k == 11 else "output", bytes(dict(_fields(v))[1]).decode())

    @staticmethod
    def _attr(buf):
        d = dict(_fields(buf))
        name, kind = bytes(d[1]).decode(), d[20]
        return name, {1: lambda: struct.unpack("<f", d[2])[0], 2: lambda: _ints_one(d[3]), 3: lambda: bytes(d[4]).decode(),
                      6: lambda: list(np.frombuffer(bytes(d[7]), "<f4")), 7: lambda: _ints(bytes(d[8]))}[kind]()

    def parsed(self):
        return ocrhip.ParsedGraph(self.nodes, self.weights, self.ints, self.input, self.output)

    def part(self, first, last):
        """The nodes from the one that reads value `first` to the one that writes `last`."""
        m = object.__new__(Model)
        need, keep = {last}, []
        for n in reversed(self.nodes):
            if any(o in need and o != first for o in n[2]):
                keep.append(n)
                need |= set(n[1])
        m.nodes, m.input, m.output = keep[::-1], first, last
        m.weights = {k: v for k, v in self.weights.items() if k in need}
        m.ints = {k: v for k, v in self.ints.items() if k in need}
        return m


def _ints_one(v):
    return v - (1 << 64) if v >> 63 else v


@functools.lru_cache(None)
def model(kind):
    if kind == "rec":
        return Model(synth.rec_model(0))
    if kind == "rec_f32":
        return Model(synth.rec_model(0, exact=False))
    if kind == "det":
        return Model(synth.det_model(0))
    if kind == "pp_det":
        return Model(synth_pp.det_model(0))
    m = Model(synth_pp.rec_model(0))
    if kind == "pp_svtr":  # from the neck's first Transpose to the second one's input
        turns = [n for n in m.nodes if n[0] == "Transpose" and n[3]["perm"] == [0, 2, 1]]
        return m.part(turns[0][2][0], turns[1][1][0])
    return m


@functools.lru_cache(None)
def context():
    return ocrhip.Context()


@functools.lru_cache(None)
def handle(kind):
    m = model(kind).parsed()
    if kind in ("rec", "rec_f32"):
        return ocrhip.Recognizer(context(), m)
    if kind == "det":
        return ocrhip.Detector(context(), m)
    return ocrhip.NdGraph(context(), m, stop_before_softmax=True)


@functools.lru_cache(None)
def pipeline(merge):
    return ocrhip.Pipeline(handle("det"), handle("rec"), merge=merge, det_batch=3)


class Held(ocrhip.DeviceBuffer):
    """A torch tensor's memory as the device buffer that the entry points take."""

    def __init__(self, tensor):
        self.ctx, self.tensor, self.ptr = context(), tensor, tensor.data_ptr()
        self.nbytes = tensor.numel() * tensor.element_size()

    def free(self):
        self.ptr = None


# ---- inputs ------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(GPU).manual_seed(int(seed))


def _line_images(rng, gen, widths, w):
    """Grey line images [n][64][w] as the pipeline's batches hold them: background 1.0, dark
    strokes of 0 to 0.3 over about 30 % of the pixels, -0.5 right of each line's own width."""
    n = len(widths)
    img = torch.ones(n, LINE_H, w, device=GPU)
    ys, xs = torch.arange(LINE_H, device=GPU)[None, :, None], torch.arange(w, device=GPU)[None, None, :]
    count = max(1, int(0.36 * LINE_H * w / 350))
    box = np.stack([rng.integers(0, 60, (count, n)), rng.integers(3, 41, (count, n)), rng.integers(-10, w, (count, n)),
                    rng.integers(2, 31, (count, n))], 1)
    box = torch.from_numpy(box).to(GPU)
    ink = torch.rand(count, n, 1, 1, generator=gen, device=GPU) * 0.3
    for k in range(count):
        y0, bh, x0, bw = (box[k, i][:, None, None] for i in range(4))
        img = torch.where((ys >= y0) & (ys < y0 + bh) & (xs >= x0) & (xs < x0 + bw), ink[k], img)
    own = torch.tensor(widths, device=GPU)[:, None, None]
    return torch.where(xs < own, img, torch.full_like(img, -0.5)).contiguous()


def _batches(case, seed):
    """[(images [n][64][w], n, w)]: the lines grouped by width rounded up, 20 a batch at most."""
    rng, gen = np.random.default_rng(seed), _generator(seed)
    groups = {}
    for w in sorted(int(v) for v in rng.integers(case["wmin"], case["wmax"] + 1, case["lines"])):
        groups.setdefault(-(-w // case["round"]) * case["round"], []).append(w)
    out = []
    for wr, ws in sorted(groups.items()):
        imgs = _line_images(rng, gen, ws, wr)
        out += [(imgs[k: k + 20].contiguous(), len(ws[k: k + 20]), wr) for k in range(0, len(ws), 20)]
    return out


def _page(seed, w, h):
    """A synthetic page [h][w][3] bytes: white, a text line every 80 pixels made of word blocks of
    dark vertical strokes, Gaussian noise (sigma 4)."""
    rng = np.random.default_rng(seed)
    grey = torch.full((h, w), 255.0, device=GPU)
    pitch = 80
    for i in range(max(1, (h - 60) // pitch)):
        row = np.full(w, 255.0, np.float32)
        x, end = int(rng.integers(w // 20, w // 12 + 2)), w - int(rng.integers(w // 20, w // 3))
        while x < end:
            x1, ink = min(x + int(rng.integers(40, 320)), end), float(rng.uniform(0, 60))
            while x < x1:
                s = int(rng.integers(4, 10))
                row[x: min(x + s, x1)] = ink
                x += s + int(rng.integers(1, 3))
            x = x1 + int(rng.integers(22, 40))
        y0, lh = 30 + i * pitch + int(rng.integers(0, 40)), int(rng.integers(24, 37))
        grey[y0: y0 + lh] = torch.from_numpy(row).to(GPU)
    noise = torch.randn(h, w, 3, generator=_generator(seed), device=GPU) * 4
    return (grey[:, :, None] + noise).round().clamp(0, 255).to(torch.uint8)


def _sizes(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["sizes"].split()]


def _sequence(case, seed):
    """What the neck reads: activations after a ReLU, about half of them zero."""
    return torch.relu(torch.randn(case["lines"], case["steps"], synth_pp.DIM, generator=_generator(seed), device=GPU))


def _pp_lines(case, seed):
    out = torch.zeros(case["lines"], 3, synth_pp.REC_H, case["w"])
    for i, img in enumerate(synth_pp.rec_lines(case["lines"], seed, max(16, case["w"] // 2), case["w"])):
        out[i, :, :, : img.shape[2]] = torch.from_numpy(img)
    return out.to(GPU)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "rec":
        s["rec"] = handle("rec_f32" if case["f32"] else "rec")
        s["batches"] = [(Held(d), n, w) for d, n, w in _batches(case, seed)]
        tmax, ntot, classes = s["rec"].dims(s["batches"])
        # Rows past a line's own steps are not written: they keep these zeros.
        s["logits"] = torch.zeros(tmax, ntot, classes, device=GPU)
        s["best"] = torch.zeros(tmax, ntot, dtype=torch.int32, device=GPU)
    elif kind == "map":
        s["det"] = handle("det")
        s["image"] = _map_image(case, seed).cpu().numpy()
    elif kind == "mask":
        s["det"] = handle("det")
        s["sizes"] = _sizes(case)
        s["pages"] = [Held(_page(seed * 16 + k, w, h)) for k, (w, h) in enumerate(s["sizes"])]
        s["bits"] = [Held(torch.zeros(h, (w + 31) // 32, dtype=torch.int32, device=GPU)) for w, h in s["sizes"]]
    elif kind == "pages":
        s["pipe"] = pipeline(case["merge"])
        s["pages"] = [_page(seed * 16 + k, case["w"], case["h"]).cpu().numpy() for k in range(case["pages"])]
        s["text"] = np.zeros((case["pages"], TEXT_LINES, TEXT_CHARS), np.uint8)
        s["counts"] = np.zeros((case["pages"], 2), np.int32)
    elif kind == "pp_rec":
        s["x"] = _pp_lines(case, seed)
        shape = handle("pp_rec").dims(s["x"].shape)
        s["logits"] = torch.zeros(shape, device=GPU)
        s["best"] = torch.zeros(shape[:2], dtype=torch.int32, device=GPU)
    elif kind == "pp_svtr":
        s["x"] = _sequence(case, seed)
        s["y"] = torch.zeros(handle("pp_svtr").dims(s["x"].shape), device=GPU)
    elif kind == "pp_det":
        s["pages"] = [_page(seed * 16 + k, case["w"], case["h"]) for k in range(case["pages"])]
        ow, oh, _ = ocrhip.det_input_dims(case["w"], case["h"], synth_pp.DET_MAX_SIDE)
        s["x"] = torch.zeros(case["pages"], 3, oh, ow, device=GPU)
        s["map"] = torch.zeros(case["pages"], 1, oh, ow, device=GPU)
        s["bits"] = torch.zeros(case["pages"], oh, (ow + 31) // 32, dtype=torch.int32, device=GPU)
    if kind.startswith("pp_"):
        s["graph"] = handle(kind)
    return s


def _map_image(case, seed):
    """A detector input: background 1.0 and dark text-like bands 8 to 20 pixels tall."""
    rng = np.random.default_rng(seed)
    h, w = case["h"], case["w"]
    img = np.ones((h, w), np.float32)
    for _ in range(max(2, h // 20)):
        bh = int(rng.integers(8, 21))
        y0, x, end = int(rng.integers(0, h - bh)), int(rng.integers(0, w // 6)), int(rng.integers(w // 2, w + 1))
        while x < end:
            ww = int(rng.integers(10, 70))
            img[y0: y0 + bh, x: min(x + ww, end)] = rng.uniform(0.0, 0.3)
            x += ww + int(rng.integers(4, 12))
    return torch.from_numpy(img)


# ---- one pass ----------------------------------------------------------------------------------
def _ok(rc):
    if rc != 0:
        raise ocrhip.OcrError(ocrhip.lib().ocr_last_error().decode())


def _shape(t):
    return (ctypes.c_int64 * t.dim())(*t.shape)


def _nd_run(graph, x, y):
    _ok(ocrhip.lib().ocr_nd_run_device(graph.handle, x.data_ptr(), _shape(x), x.dim(), y.data_ptr()))


def run(s):
    kind = s["kind"]
    if kind == "rec":
        lens = s["rec"].recognize_device(s["batches"], Held(s["logits"]), Held(s["best"]))
        return {"logits": s["logits"], "best": s["best"], "lens": lens.astype(np.int64)}
    if kind == "map":
        return s["det"].detect(s["image"])
    if kind == "mask":
        s["det"].detect_pages_device(s["pages"], [w for w, _ in s["sizes"]], [h for _, h in s["sizes"]], 0.5, s["bits"])
        return [b.tensor for b in s["bits"]]
    if kind == "pages":
        return _read_pages(s)
    if kind == "pp_rec":
        s["graph"].argmax_device(_Ptr(s["x"]), s["x"].shape, _Ptr(s["best"]))
        _nd_run(s["graph"], s["x"], s["logits"])
        return {"best": s["best"], "logits": s["logits"]}
    if kind == "pp_svtr":
        _nd_run(s["graph"], s["x"], s["y"])
        return s["y"]
    L, ctx = ocrhip.lib(), context().handle
    for page, x in zip(s["pages"], s["x"]):
        h, w = page.shape[:2]
        _ok(L.ocr_nd_det_input_device(ctx, page.data_ptr(), w, h, synth_pp.DET_MAX_SIDE, x.data_ptr()))
    _nd_run(s["graph"], s["x"], s["map"])
    for m, b in zip(s["map"], s["bits"]):
        _ok(L.ocr_db_threshold_device(ctx, m.data_ptr(), m.shape[2], m.shape[1], 0.3, b.data_ptr()))
    return {"input": s["x"], "map": s["map"], "bits": s["bits"]}


class _Ptr:
    def __init__(self, tensor):
        self.ptr = tensor.data_ptr()


def _read_pages(s):
    """The pipeline over the pages, then every line's text (its bytes, zero-filled rows)."""
    pipe, text, counts, L = s["pipe"], s["text"], s["counts"], ocrhip.lib()
    pipe.run(s["pages"])
    text[:] = 0
    lines, words, n = ctypes.c_uint32(), ctypes.c_uint32(), ctypes.c_uint32()
    for p in range(len(text)):
        _ok(L.ocr_pipeline_page(pipe.handle, p, ctypes.byref(lines), ctypes.byref(words)))
        counts[p] = lines.value, words.value
        row = text[p].ctypes.data
        for i in range(min(lines.value, TEXT_LINES)):
            _ok(L.ocr_pipeline_line_text(pipe.handle, p, i, ctypes.cast(row + i * TEXT_CHARS, ctypes.c_char_p), TEXT_CHARS,
                                         ctypes.byref(n)))
    return {"text": text, "counts": counts}


# ---- the work and the tolerance ----------------------------------------------------------------
def _weights(kind):
    return sum(v.size for v in model(kind).weights.values())


def _flops(kind, shape):
    """2 x the multiply-adds of a model on an input of this shape (shapes only, no data)."""
    count = [0]
    x = torch.empty(shape, device="meta", dtype=torch.float64)
    evaluate(model(kind), x, count)
    return count[0]


def work(case):
    kind = case["kind"]
    if kind == "rec":
        rng = np.random.default_rng(0)
        groups = {}
        for w in rng.integers(case["wmin"], case["wmax"] + 1, case["lines"]):
            wr = -(-int(w) // case["round"]) * case["round"]
            groups[wr] = groups.get(wr, 0) + 1
        px = sum(LINE_H * w * n for w, n in groups.items())
        rows = sum(w // 4 * n for w, n in groups.items())
        return {"bytes": 4 * px + rows * (4 * synth.CLASSES + 4) + 2 * _weights("rec"),
                "flops": sum(n * _flops("rec", (1, 1, LINE_H, w)) for w, n in groups.items())}
    if kind == "map":
        return {"bytes": 8 * case["h"] * case["w"] + 2 * _weights("det"), "flops": _flops("det", (1, 1, case["h"], case["w"]))}
    if kind == "mask":
        # Two source rows of the page for each of the model's 800 rows, the mask's words.
        sizes = _sizes(case)
        return {"bytes": sum(3 * w * min(h, 2 * synth.DET_H) + (w + 31) // 32 * 4 * h for w, h in sizes) + 2 * _weights("det"),
                "flops": len(sizes) * _flops("det", (1, 1, synth.DET_H, synth.DET_W))}
    if kind == "pages":
        # The pages, and their text lines (one every 80 rows) at about 700 pixels of line image.
        lines = case["pages"] * ((case["h"] - 60) // 80)
        return {"bytes": case["pages"] * 3 * case["w"] * case["h"] + 4 * lines * LINE_H * 700,
                "flops": case["pages"] * _flops("det", (1, 1, synth.DET_H, synth.DET_W))
                + lines * _flops("rec", (1, 1, LINE_H, 700))}
    if kind == "pp_rec":
        n, w = case["lines"], case["w"]
        return {"bytes": 4 * n * (3 * synth_pp.REC_H * w + w // 8 * (synth_pp.PP_CLASSES + 1)) + 2 * _weights("pp_rec"),
                "flops": _flops("pp_rec", (n, 3, synth_pp.REC_H, w))}
    if kind == "pp_svtr":
        shape = (case["lines"], case["steps"], synth_pp.DIM)
        return {"bytes": 8 * math.prod(shape) + 2 * _weights("pp_svtr"), "flops": _flops("pp_svtr", shape)}
    ow, oh, _ = ocrhip.det_input_dims(case["w"], case["h"], synth_pp.DET_MAX_SIDE)
    n = case["pages"]
    return {"bytes": n * (3 * case["w"] * min(case["h"], 2 * oh) + 4 * 4 * ow * oh + ow // 8 * oh) + 2 * _weights("pp_det"),
            "flops": _flops("pp_det", (n, 3, oh, ow))}


def tolerance(case):
    """Float32-class arithmetic throughout (float16 hi + lo operands, float32 sums): against
    float64 the logits and maps are 3e-7 to 1.1e-6 off (measured; the largest with float32
    weights and in the detectors), and four times that is stated. Bits, arg-maxes and text
    differ only where a sum's rounding meets a threshold or a tie."""
    return {"rec": {"rel": 4.5e-6, "max": 2e-4, "differ": 1e-4},
            "map": {"rel": 3.5e-6, "max": 2e-4},
            "mask": {"rel": 0.0, "differ": 2e-4},
            "pages": {"rel": 0.0, "differ": 2e-3},
            "pp_rec": {"rel": 1.2e-6, "max": 5e-5, "differ": 1e-3},
            "pp_svtr": {"rel": 2e-6, "max": 8e-5},
            "pp_det": {"rel": 4e-6, "max": 2e-4, "differ": 2e-4}}[case["kind"]]


# ---- the same results in 64 bits ---------------------------------------------------------------
def _conv(x, w, b, at, count):
    pt, pl, pb, pr = at.get("pads", [0, 0, 0, 0])
    sy, sx = at.get("strides", [1, 1])
    group, (cout, cg, kh, kw) = at.get("group", 1), w.shape
    x = torch.nn.functional.pad(x, (pl, pr, pt, pb))
    n, c, h, wd = x.shape
    oh, ow = (h - kh) // sy + 1, (wd - kw) // sx + 1
    y = 0
    for ky in range(kh):
        for kx in range(kw):
            t = x[:, :, ky: ky + sy * (oh - 1) + 1: sy, kx: kx + sx * (ow - 1) + 1: sx]
            if group == 1:
                y = y + torch.matmul(w[:, :, ky, kx], t.reshape(n, c, oh * ow)).view(n, cout, oh, ow)
            else:  # depthwise
                y = y + t * w[:, 0, ky, kx][None, :, None, None]
    count[0] += 2 * n * oh * ow * cout * cg * kh * kw
    return y if b is None else y + b[None, :, None, None]


def _conv_t(x, w, b, at, count):
    sy, sx = at["strides"]
    n, c, h, wd = x.shape
    _, cout, kh, kw = w.shape
    y = torch.zeros(n, cout, (h - 1) * sy + kh, (wd - 1) * sx + kw, dtype=x.dtype, device=x.device)
    for ky in range(kh):
        for kx in range(kw):
            t = torch.matmul(w[:, :, ky, kx].t().contiguous(), x.reshape(n, c, h * wd)).view(n, cout, h, wd)
            y[:, :, ky: ky + sy * (h - 1) + 1: sy, kx: kx + sx * (wd - 1) + 1: sx] += t
    count[0] += 2 * n * h * wd * c * cout * kh * kw
    return y if b is None else y + b[None, :, None, None]


def _gru(x, w, r, b, count):
    """ONNX GRU, bidirectional, linear_before_reset: [T, N, C] -> [T, 2, N, H]. The recurrent
    weights as float16 values, as the library (and its reference by default) holds them."""
    steps, n, c = x.shape
    hid = r.shape[2]
    count[0] += 2 * 2 * steps * n * 3 * hid * (c + hid)
    if x.device.type == "meta":
        return torch.empty(steps, 2, n, hid, dtype=x.dtype, device=x.device)
    r = r.half().to(x.dtype)
    out = torch.empty(steps, 2, n, hid, dtype=x.dtype, device=x.device)
    for d in range(2):
        g = torch.matmul(x, w[d].t()) + b[d, : 3 * hid]
        rt, rb, h = r[d].t().contiguous(), b[d, 3 * hid:], torch.zeros(n, hid, dtype=x.dtype, device=x.device)
        for t in range(steps) if d == 0 else range(steps - 1, -1, -1):
            u = torch.addmm(rb, h, rt)
            z = torch.sigmoid(g[t, :, :hid] + u[:, :hid])
            q = torch.sigmoid(g[t, :, hid: 2 * hid] + u[:, hid: 2 * hid])
            a = torch.tanh(g[t, :, 2 * hid:] + q * u[:, 2 * hid:])
            h = (1 - z) * a + z * h
            out[t, d] = h
    return out


def evaluate(m, x, count=None, stop=("Softmax", "LogSoftmax")):
    """The graph on x in x's type, up to a final (log-)softmax."""
    count = count if count is not None else [0]
    dev, F = x.device, torch.nn.functional
    val = {k: torch.from_numpy(np.array(v)).to(x.dtype).to(dev) for k, v in m.weights.items()}
    val.update({k: [int(i) for i in np.asarray(v).reshape(-1)] for k, v in m.ints.items()})
    val[m.input] = x
    for op, ins, outs, at in m.nodes:
        if op in stop and outs[0] == m.output:
            return val[ins[0]]
        a = [val[i] if i else None for i in ins]
        if op == "Conv":
            y = _conv(a[0], a[1], a[2] if len(a) > 2 else None, at, count)
        elif op == "ConvTranspose":
            y = _conv_t(a[0], a[1], a[2] if len(a) > 2 else None, at, count)
        elif op == "GRU":
            y = _gru(a[0], a[1], a[2], a[3], count)
        elif op == "MatMul":
            count[0] += 2 * a[0].numel() * a[1].shape[-1]
            y = torch.matmul(a[0], a[1])
        elif op == "Relu":
            y = torch.relu(a[0])
        elif op == "Sigmoid":
            y = torch.sigmoid(a[0])
        elif op == "HardSigmoid":
            y = torch.clamp(at["alpha"] * a[0] + at["beta"], 0, 1)
        elif op == "Erf":
            y = torch.erf(a[0])
        elif op == "Sqrt":
            y = torch.sqrt(a[0])
        elif op in ("Add", "Sub", "Mul", "Div"):
            y = getattr(torch, op.lower())(a[0], a[1])
        elif op == "Pow":
            y = a[0] ** a[1]
        elif op == "Softmax":
            y = torch.softmax(a[0], at["axis"])
        elif op == "BatchNormalization":
            g, b, mean, var = (v[None, :, None, None] for v in a[1:5])
            y = (a[0] - mean) / torch.sqrt(var + at["epsilon"]) * g + b
        elif op in ("MaxPool", "AveragePool"):
            pool = F.max_pool2d if op == "MaxPool" else F.avg_pool2d
            y = pool(a[0], tuple(at["kernel_shape"]), tuple(at["strides"]))
        elif op == "GlobalAveragePool":
            y = a[0].mean((2, 3), keepdim=True)
        elif op == "ReduceMean":
            y = a[0].mean(at["axes"], keepdim=bool(at["keepdims"]))
        elif op == "Concat":
            y = sum(a, []) if isinstance(a[0], list) else torch.cat(a, at["axis"])
        elif op == "Resize":
            f = int(m.weights[ins[2]][2])
            y = a[0].repeat_interleave(f, 2).repeat_interleave(f, 3)
        elif op == "Shape":
            y = list(a[0].shape)
        elif op == "Gather":
            y = [a[0][i] for i in a[1]]
        elif op == "Reshape":
            y = a[0].reshape([a[0].shape[i] if d == 0 else d for i, d in enumerate(a[1])])
        elif op == "Transpose":
            y = a[0].permute(at["perm"])
        elif op == "Squeeze":
            y = a[0].squeeze(a[1][0])
        elif op == "Unsqueeze":
            y = a[0].unsqueeze(a[1][0])
        elif op == "Slice":
            y = a[0].narrow(a[3][0], a[1][0], a[2][0] - a[1][0])
        else:
            raise ValueError(op)
        for o in outs:
            val[o] = y
    return val[m.output]


def _det_input(page, ow, oh):
    """[3][oh][ow] of a page: bilinear at half-pixel positions, BGR, ImageNet mean and deviation."""
    h, w = page.shape[:2]

    def taps(n, out):
        pos = (torch.arange(out, device=GPU).float() + 0.5) * np.float32(n / out) - 0.5
        pos = pos.clamp(0, n - 1)
        lo = pos.long()
        return lo, (lo + 1).clamp(max=n - 1), (pos - lo).double()

    (x1, x2, fx), (y1, y2, fy) = taps(w, ow), taps(h, oh)
    p = page.double()
    top, low = (p[y][:, x1] * (1 - fx)[None, :, None] + p[y][:, x2] * fx[None, :, None] for y in (y1, y2))
    v = (top * (1 - fy)[:, None, None] + low * fy[:, None, None]) / 255
    mean, dev = (torch.tensor(t, dtype=torch.float64, device=GPU) for t in ((0.485, 0.456, 0.406), (0.229, 0.224, 0.225)))
    return ((v.flip(2) - mean) / dev).permute(2, 0, 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "rec":
        name = "rec_f32" if case["f32"] else "rec"
        parts = [evaluate(model(name), d[:, None].double()) for d, _, _ in _batches(case, seed)]
        logits = torch.zeros(max(p.shape[0] for p in parts), case["lines"], synth.CLASSES, dtype=torch.float64, device=GPU)
        at = 0
        for p in parts:
            logits[: p.shape[0], at: at + p.shape[1]] = p
            at += p.shape[1]
        return {"logits": logits, "best": None, "lens": None}
    if kind == "map":
        return evaluate(model("det"), _map_image(case, seed).to(GPU).double()[None, None])[0, 0]
    if kind == "pp_rec":
        return {"best": None, "logits": evaluate(model("pp_rec"), _pp_lines(case, seed).double())}
    if kind == "pp_svtr":
        return evaluate(model("pp_svtr"), _sequence(case, seed).double())
    if kind == "pp_det":
        ow, oh, _ = ocrhip.det_input_dims(case["w"], case["h"], synth_pp.DET_MAX_SIDE)
        x = torch.stack([_det_input(_page(seed * 16 + k, case["w"], case["h"]), ow, oh) for k in range(case["pages"])])
        return {"input": x, "map": evaluate(model("pp_det"), x), "bits": None}
    return None
