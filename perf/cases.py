"""What a program that runs on this framework has it do, as cases that can be
measured: the feed-forward block and single projections at every lane count
from one decode step to a whole prompt, the attention of a step and of a
prompt, and a whole session on the engine.

Every case goes through the entry points a program calls: `Backend` and the C
ABI behind it on device buffers (here torch tensors), and `Engine`.  Kinds:

  mlp      gate and up projections, the gelu gate, the down projection, int4
           with a gain for every 32 codes; recorded once and replayed where a
           decode loop would, else enqueued
  project  one projection: int4 group-32, 2/4/8-bit with one gain a row, or
           float rows; bf16 in and out, fp32, or between activation grids
  attend   queries over a byte key/value ring, one lane or a prompt's lanes
  engine   a session: a prompt, forced decode steps, one speculative block
"""
import ctypes
import json
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from igllm_amd import native
from igllm_amd.backend import Backend, CodePlane
from igllm_amd.engine import Engine, prompt_ids, write_gemma
from igllm_amd.native import Plane

ENTER, LEAVE = 0.04, 0.1  # activation grids of a calibrated projection
REAL_TYPES = {"bf16": (native.IGL_STORE_BF16, torch.bfloat16), "f16": (native.IGL_STORE_F16, torch.float16),
              "f32": (native.IGL_STORE_F32, torch.float32)}


# ---- the cases ----------------------------------------------------------------

def listed():
    return [
        # one token's feed-forward block, as a decode loop replays it
        {"name": "mlp_1_lane", "kind": "mlp", "lanes": 1, "hidden": 1536, "inner": 6144, "replay": True},
        # the same for a speculative block of four, on a double-wide layer
        {"name": "mlp_4_lanes", "kind": "mlp", "lanes": 4, "hidden": 1536, "inner": 12288, "replay": True},
        # a short prompt, or a batch of sessions: fewer lanes than a matrix tile
        {"name": "mlp_37_lanes", "kind": "mlp", "lanes": 37, "hidden": 1536, "inner": 6144, "replay": False},
        # a prompt of a thousand ids
        {"name": "mlp_1000_lanes", "kind": "mlp", "lanes": 1000, "hidden": 1536, "inner": 6144, "replay": False},
        # bf16 prefill products, the shortest and the longest prompt chunk
        {"name": "bf16_64_lanes", "kind": "project", "form": "q4", "rows": 2048, "cols": 8192, "lanes": 64,
         "act": "bf16", "grid": False},
        {"name": "bf16_2048_lanes", "kind": "project", "form": "q4", "rows": 8192, "cols": 2048, "lanes": 2048,
         "act": "bf16", "grid": False},
        # a calibrated projection of the shipped export over a whole prompt
        {"name": "grid_2047_lanes", "kind": "project", "form": "c4", "rows": 6144, "cols": 1536, "lanes": 2047,
         "act": "f32", "grid": True},
        # the export's output head, 2-bit codes, one token
        {"name": "head_1_lane", "kind": "project", "form": "c2", "rows": 262144, "cols": 1536, "lanes": 1,
         "act": "f32", "grid": False},
        # the export's float projection into the per-layer inputs, a prompt chunk
        {"name": "real_500_lanes", "kind": "project", "form": "bf16", "rows": 8960, "cols": 1536, "lanes": 500,
         "act": "f32", "grid": False},
        # one decode step's attention over a long context
        {"name": "attend_16384", "kind": "attend", "lanes": 1, "head": 256, "place": 16383, "window": 0,
         "format": "int8", "kv": 1},
        # a prompt's attention on a global layer
        {"name": "attend_2047_lanes", "kind": "attend", "lanes": 2047, "head": 512, "place": 0, "window": 0,
         "format": "e4m3", "kv": 1},
        # a session: a prompt in one pass, forced decode steps, one speculative block
        {"name": "session", "kind": "engine", "layers": 10, "shared": 4, "vocab": 8192, "prompt": 512, "steps": 16,
         "block": 4},
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over the logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _times(rng, low, high, unit):
    return unit * _spread(rng, (low + unit - 1) // unit, high // unit)


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "project", "project", "project", "attend", "attend", "engine"])
    if kind == "mlp":
        lanes = _spread(rng, 1, 2048)
        return {"kind": kind, "lanes": lanes, "hidden": rng.choice([512, 1024, 1536, 2048, 2048 + 96]),
                "inner": _times(rng, 1024, 12288 if lanes <= 1024 else 6144, 32), "replay": lanes <= 16}
    if kind == "project":
        form = rng.choice(["q4", "q4", "q4", "c4", "c2", "c8", "bf16", "f16"])
        if form == "q4":
            act = rng.choice(["f32", "bf16"])
            lanes = _spread(rng, 64, 2048) if act == "bf16" else _spread(rng, 1, 2048)
            return {"kind": kind, "form": form, "rows": _spread(rng, 256, 8192), "cols": _times(rng, 256, 8192, 32),
                    "lanes": lanes, "act": act, "grid": False}
        if form[0] == "c":
            return {"kind": kind, "form": form, "rows": _times(rng, 256, 12288, 16),
                    "cols": _times(rng, 256, 6144, 128), "lanes": _spread(rng, 1, 2048), "act": "f32", "grid": True}
        return {"kind": kind, "form": form, "rows": _times(rng, 256, 8960, 16), "cols": _times(rng, 256, 2048, 32),
                "lanes": _spread(rng, 1, 512), "act": "f32", "grid": False}
    if kind == "attend":
        lanes = rng.choice([1, 1, _spread(rng, 2, 63), _spread(rng, 64, 2047)])
        place = _spread(rng, 1, 16384) - 1 if lanes < 64 else rng.choice([0, 0, _spread(rng, 1, 2048)])
        return {"kind": kind, "lanes": lanes, "head": rng.choice([256, 512]), "place": place,
                "window": rng.choice([0, 512]), "format": rng.choice(["int8", "e4m3"]),
                "kv": rng.choice([1, 1, 2])}
    return {"kind": kind, "layers": 10, "shared": 4, "vocab": 4096, "prompt": _spread(rng, 8, 512),
            "steps": rng.randint(1, 16), "block": rng.choice([1, 2, 3, 4, 6, 8, 12])}


# ---- what a program holds -------------------------------------------------------

_BACKEND = None


def backend():
    """The process's one desk."""
    global _BACKEND
    if _BACKEND is None:
        _BACKEND = Backend()
    return _BACKEND


class Buffer:
    """A torch tensor as the backend's device buffer."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()


class State(dict):
    """What a pass needs; gives planes, replays and sessions back when dropped."""

    def __del__(self):
        be = backend()
        if self.get("replay"):
            be.replay_free(self["replay"])
        if self.get("engine") is not None:
            self["engine"].close()
        for cp in self.get("planes", ()):
            be.detach(cp)


def _random(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _codes(g, form, rows, cols):
    """Packed code rows and their gains, on the device: int4 with a gain for
    every 32 codes ("q4"), or 2, 4 or 8 bits with one gain a row."""
    if form == "q4":
        codes = torch.randint(0, 256, (rows, cols // 2), dtype=torch.uint8, device="cuda", generator=g)
        return codes, (torch.randn((rows, cols // 32), device="cuda", generator=g) * 0.02).abs()
    bits = int(form[1])
    spread = torch.rand((rows, 1), device="cuda", generator=g) * 0.5 + 0.75
    if bits == 2:  # codes whose values average zero: 2/16, 3/16, 4/16, 7/16
        pick = torch.randint(0, 16, (rows, cols // 4, 4), dtype=torch.uint8, device="cuda", generator=g)
        code = (pick >= 2).to(torch.uint8) + (pick >= 5) + (pick >= 9)
        weight = torch.tensor([1, 4, 16, 64], dtype=torch.uint8, device="cuda")
        return (code * weight).sum(-1, dtype=torch.uint8), spread * 0.05
    codes = torch.randint(0, 256, (rows, cols * bits // 8), dtype=torch.uint8, device="cuda", generator=g)
    return codes, spread * (0.02 if bits == 4 else 0.0012)


def _weight(codes, gains, form, cols):
    """The plane's weights in 64 bits."""
    bits = 4 if form == "q4" else int(form[1])
    shifts = torch.arange(0, 8, bits, device="cuda", dtype=torch.uint8)
    code = (codes.unsqueeze(-1) >> shifts) & ((1 << bits) - 1)
    value = code.reshape(codes.shape[0], cols).double() - (1 << (bits - 1))
    return value * gains.double().repeat_interleave(cols // gains.shape[1], 1)


def _bind(codes, gains, form, cols, grid=False):
    be = backend()
    p = Plane()
    p.row_count, p.col_count = codes.shape[0], cols
    if form in REAL_TYPES:
        p.form, p.real_type = native.IGL_PLANE_REAL, REAL_TYPES[form][0]
        cp = CodePlane(p, codes, None)
        return be.bind_dev(cp, Buffer(codes), Buffer(codes))
    bits = 4 if form == "q4" else int(form[1])
    p.form, p.gain_type = native.IGL_PLANE_CODE, native.IGL_STORE_F32
    p.row_stride = codes.shape[1]
    p.bit_count, p.code_bias = bits, 1 << (bits - 1)
    p.group_count = gains.shape[1]
    p.group_size = cols // gains.shape[1]
    if grid:
        p.enter_gain, p.leave_gain = ENTER, LEAVE
    return be.bind_dev(CodePlane(p, codes, gains), Buffer(codes), Buffer(gains))


def _mlp_inputs(case, seed):
    g = _random(seed)
    h, i, lanes = case["hidden"], case["inner"], case["lanes"]
    sheets = [_codes(g, "q4", i, h), _codes(g, "q4", i, h), _codes(g, "q4", h, i)]
    return sheets, torch.randn((lanes, h), device="cuda", generator=g)


def _mlp_pass(s):
    be, lanes, h, i = backend(), s["lanes"], s["hidden"], s["inner"]
    gate, up, down = s["planes"]
    be.mat_mat_dev(gate, s["act"], h, lanes, s["gate"], i)
    be.mat_mat_dev(up, s["act"], h, lanes, s["rise"], i)
    be._check(be.lib.igl_gelu_gate_dev(ctypes.byref(be.desk), s["gate"].ptr, s["rise"].ptr, lanes * i), "gelu_gate")
    be.mat_mat_dev(down, s["gate"], i, lanes, s["out"], h)


def _project_inputs(case, seed):
    g = _random(seed)
    rows, cols, lanes, form = case["rows"], case["cols"], case["lanes"], case["form"]
    if form in REAL_TYPES:
        sheet = (torch.randn((rows, cols), device="cuda", generator=g) * 0.02).to(REAL_TYPES[form][1]), None
    else:
        sheet = _codes(g, form, rows, cols)
    act = torch.randn((lanes, cols), device="cuda", generator=g)
    return sheet, act.to(torch.bfloat16) if case["act"] == "bf16" else act


def _attend_shape(case):
    """Positions the lanes see, and the ring that holds them."""
    last = case["place"] + case["lanes"]
    span = min(last, case["window"] + case["lanes"]) if case["window"] else last
    return last, span


def _attend_inputs(case, seed):
    """Byte rings and their scales, and queries: keys normed and turned as a
    model's are (unit variance), clipped to the calibrated range."""
    g = _random(seed)
    _, span = _attend_shape(case)
    width = case["kv"] * case["head"]
    scale = 4.0 / 127.0 if case["format"] == "int8" else 6.0 / 448.0
    rings = []
    for _ in range(2):
        v = torch.randn((span, width), device="cuda", generator=g).clamp_(-4, 4) / scale
        if case["format"] == "int8":
            rings.append(v.round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8))
        else:
            rings.append(v.clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))
    query = torch.randn((case["lanes"], 8 * width), device="cuda", generator=g)
    return rings, scale, query


ENGINE_HIDDEN, ENGINE_INNER, ENGINE_WINDOW = 1536, 6144, 512


def _engine_files(case, seed, folder):
    return write_gemma(folder, seed=seed, layers=case["layers"], shared_layers=case["shared"], vocab=case["vocab"])


def _engine_ids(case, seed):
    return prompt_ids(case["prompt"] + case["steps"] + case["block"], case["vocab"], seed=seed)


def prepare(case, seed):
    be = backend()
    s = State(kind=case["kind"])
    if case["kind"] == "mlp":
        sheets, act = _mlp_inputs(case, seed)
        lanes, h, i = case["lanes"], case["hidden"], case["inner"]
        s.update(lanes=lanes, hidden=h, inner=i, act=Buffer(act))
        for name, width in (("gate", i), ("rise", i), ("out", h)):
            s[name] = Buffer(torch.empty((lanes, width), device="cuda"))
        torch.cuda.synchronize()
        s["planes"] = [_bind(c, gain, "q4", w) for (c, gain), w in zip(sheets, (h, h, i))]
        if case["replay"]:
            _mlp_pass(s)  # each entry once before it is recorded
            be.sync()
            be.record_begin()
            _mlp_pass(s)
            s["replay"] = be.record_end()
    elif case["kind"] == "project":
        (codes, gains), act = _project_inputs(case, seed)
        s.update(case=dict(case), act=Buffer(act),
                 out=Buffer(torch.empty((case["lanes"], case["rows"]), device="cuda", dtype=act.dtype)))
        torch.cuda.synchronize()
        s["planes"] = [_bind(codes, gains, case["form"], case["cols"], case["grid"])]
    elif case["kind"] == "attend":
        rings, scale, query = _attend_inputs(case, seed)
        s.update(case=dict(case), rings=[Buffer(r) for r in rings], scale=scale, query=Buffer(query),
                 span=rings[0].shape[0], out=Buffer(torch.empty_like(query)))
        torch.cuda.synchronize()
    else:
        folder = tempfile.mkdtemp(prefix="igl_case_")
        try:
            _engine_files(case, seed, folder)
            s["engine"] = Engine(be, folder, window_limit=4096, lane_limit=2048, precise=False)
        finally:
            shutil.rmtree(folder, ignore_errors=True)
        s.update(ids=_engine_ids(case, seed), prompt=case["prompt"], steps=case["steps"], block=case["block"])
    return s


def run(s):
    be = backend()
    if s["kind"] == "mlp":
        if s.get("replay"):
            be.replay_run(s["replay"])
        else:
            _mlp_pass(s)
        return s["out"].tensor
    if s["kind"] == "project":
        c, plane = s["case"], s["planes"][0]
        entry = be.plane_lift_dev if c["grid"] else be.gemm_bf16_dev if c["act"] == "bf16" else be.mat_mat_dev
        entry(plane, s["act"], c["cols"], c["lanes"], s["out"], c["rows"])
        return s["out"].tensor
    if s["kind"] == "attend":
        c = s["case"]
        fmt = native.IGL_CACHE_INT8 if c["format"] == "int8" else native.IGL_CACHE_E4M3
        key, value = s["rings"]
        # queries of unit variance: the score scale stands for the model's own norms
        be._check(be.lib.igl_attend_lanes_dev(
            ctypes.byref(be.desk), key.ptr, value.ptr, fmt, s["scale"], s["scale"], s["span"], c["kv"], 8, c["head"],
            s["query"].ptr, c["kv"] * 8 * c["head"], c["place"], c["window"], c["lanes"], 1.0 / math.sqrt(c["head"]),
            s["out"].ptr), "attend_lanes")
        return s["out"].tensor
    e, ids, at = s["engine"], s["ids"], s["prompt"]
    e.reset()
    e.prime(ids[:at])  # all but the last id; the first step takes that one
    for t in ids[at - 1:at - 1 + s["steps"]]:
        e.step(t)
    step = e.logits()
    e.guess(ids[at - 1 + s["steps"]:at - 1 + s["steps"] + s["block"]])
    block = np.stack([e.logits(lane) for lane in range(s["block"])])
    e.keep(0)
    return {"step": step, "block": block}


# ---- what a pass cannot do without ----------------------------------------------

def _plane_bytes(form, rows, cols):
    if form in REAL_TYPES:
        return rows * cols * (4 if form == "f32" else 2)
    bits = 4 if form == "q4" else int(form[1])
    return rows * (cols * bits // 8 + 4 * (cols // 32 if form == "q4" else 1))


def work(case):
    lanes = case.get("lanes", 1)
    if case["kind"] == "mlp":
        h, i = case["hidden"], case["inner"]
        return {"bytes": 2 * _plane_bytes("q4", i, h) + _plane_bytes("q4", h, i) + 8 * lanes * h,
                "flops": 6 * lanes * h * i}
    if case["kind"] == "project":
        rows, cols = case["rows"], case["cols"]
        size = 2 if case["act"] == "bf16" else 4
        return {"bytes": _plane_bytes(case["form"], rows, cols) + size * lanes * (rows + cols),
                "flops": 2 * lanes * rows * cols}
    if case["kind"] == "attend":
        last, _ = _attend_shape(case)
        seen = [min(p + 1, case["window"] or p + 1) for p in range(case["place"], last)]
        rows = last - max(0, case["place"] + 1 - seen[0])
        width = case["kv"] * case["head"]
        return {"bytes": 2 * rows * width + 2 * 4 * lanes * 8 * width, "flops": 4 * 8 * width * sum(seen)}
    codes, macs = _engine_weights(case)
    passes = 2 + case["steps"]
    return {"bytes": codes * passes, "flops": 2 * macs * (case["prompt"] + case["steps"] + case["block"])}


def _engine_layers(case):
    """(head size, full, shares a ring, feed-forward width) of every layer."""
    n, first = case["layers"], case["layers"] - case["shared"]
    full = [(i + 1) % 5 == 0 or i == n - 1 for i in range(n)]
    return [(512 if full[i] else 256, full[i], i >= first, ENGINE_INNER * (2 if i >= first else 1)) for i in range(n)]


def _engine_weights(case):
    """Bytes and multiply-adds of one token through every projection."""
    planes = [(case["vocab"], ENGINE_HIDDEN), (256 * case["layers"], ENGINE_HIDDEN)]
    for head, _, shared, inner in _engine_layers(case):
        planes += [(8 * head, ENGINE_HIDDEN), (ENGINE_HIDDEN, 8 * head)]
        planes += [] if shared else [(head, ENGINE_HIDDEN)] * 2
        planes += [(inner, ENGINE_HIDDEN)] * 2 + [(ENGINE_HIDDEN, inner), (256, ENGINE_HIDDEN), (ENGINE_HIDDEN, 256)]
    return sum(_plane_bytes("q4", r, c) for r, c in planes), sum(r * c for r, c in planes)


def tolerance(case):
    """Sums in 32 bits measured up to 8e-7 off the 64-bit result and bf16 outputs
    1.7e-3 (their own rounding); another order of the sums stays within these."""
    if case["kind"] == "mlp":
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "project":
        if case["act"] == "bf16":
            return {"rel": 7e-3, "max": 0.02}
        if case["grid"]:  # on the leave grid: a near-tie moves one step
            return {"rel": 1e-3, "max": 0.1}
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "attend":
        return {"rel": 1e-5, "max": 1e-4}
    # 1e-7 off at the start; a byte of the key/value cache can round the other way
    return {"rel": 1e-5, "max": 1e-4}


# ---- the same in 64 bits, in plain torch ----------------------------------------

def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _rms(x, gain=None, eps=1e-6):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if gain is None else y * gain


def exact(case, seed):
    if case["kind"] == "mlp":
        sheets, act = _mlp_inputs(case, seed)
        widths = (case["hidden"], case["hidden"], case["inner"])
        gate, up, down = (_weight(c, gain, "q4", w) for (c, gain), w in zip(sheets, widths))
        x = act.double()
        return (_gelu(x @ gate.T) * (x @ up.T)) @ down.T
    if case["kind"] == "project":
        (codes, gains), act = _project_inputs(case, seed)
        x = act.double()
        if case["grid"]:
            x = (act / ENTER).round().clamp(-128, 127).double() * float(np.float32(ENTER))
        out = torch.empty((case["lanes"], case["rows"]), device="cuda", dtype=torch.float64)
        for r in range(0, case["rows"], 16384):
            w = codes[r:r + 16384]
            w = w.double() if gains is None else _weight(w, gains[r:r + 16384], case["form"], case["cols"])
            out[:, r:r + 16384] = x @ w.T
        if case["grid"]:
            leave = float(np.float32(LEAVE))
            out = (out / leave).round().clamp(-128, 127) * leave
        return out
    if case["kind"] == "attend":
        return _exact_attend(case, seed)
    return _exact_engine(case, seed)


def _exact_attend(case, seed):
    rings, scale, query = _attend_inputs(case, seed)
    last, span = _attend_shape(case)
    first = max(0, case["place"] + 1 - case["window"]) if case["window"] else 0
    places = torch.arange(first, last, device="cuda")
    kind = torch.int8 if case["format"] == "int8" else torch.float8_e4m3fn
    key, value = (r.view(kind)[places % span].to(torch.float32).double() * scale for r in rings)
    out = torch.empty(query.shape, device="cuda", dtype=torch.float64)
    head, q = case["head"], query.double()
    lane = case["place"] + torch.arange(case["lanes"], device="cuda")[:, None]
    hide = places[None] > lane
    if case["window"]:
        hide = hide | (places[None] <= lane - case["window"])
    for h in range(8 * case["kv"]):
        at, kv = slice(h * head, (h + 1) * head), slice(h // 8 * head, (h // 8 + 1) * head)
        score = (q[:, at] @ key[:, kv].T / math.sqrt(head)).masked_fill(hide, -math.inf)
        out[:, at] = torch.softmax(score, -1) @ value[:, kv]
    return out


def _exact_engine(case, seed):
    folder = tempfile.mkdtemp(prefix="igl_case_")
    try:
        _engine_files(case, seed, folder)
        with open(os.path.join(folder, "model.safetensors"), "rb") as f:
            head = json.loads(f.read(int.from_bytes(f.read(8), "little")))
            at, t = f.tell(), {}
            for name, said in head.items():
                if name == "__metadata__":
                    continue
                begin, end = said["data_offsets"]
                f.seek(at + begin)
                raw = torch.frombuffer(bytearray(f.read(end - begin)), dtype=torch.uint8).cuda()
                raw = raw.view(torch.float32) if said["dtype"] == "F32" else raw
                t[name.replace("model.language_model.", "")] = raw.view(said["shape"])
    finally:
        shutil.rmtree(folder, ignore_errors=True)
    ids = torch.from_numpy(_engine_ids(case, seed)).cuda().long()[:case["prompt"] - 1 + case["steps"] + case["block"]]

    def sheet(stem, rows=None):
        kind = "embedding_quantized" if stem + ".embedding_quantized" in t else "weight"
        codes, gains = t[stem + "." + kind], t[stem + (".embedding_scale" if kind != "weight" else ".weight_scale")]
        codes, gains = (codes, gains) if rows is None else (codes[rows], gains[rows])
        return _weight(codes, gains, "q4", 2 * codes.shape[1])

    def vec(stem):
        return t[stem + ".weight"].double()

    def lin(x, stem):
        return x @ sheet(stem).T

    n, width, ple = len(ids), ENGINE_HIDDEN, 256
    place = torch.arange(n, device="cuda")
    x = sheet("embed_tokens", ids) * math.sqrt(width)
    seeds = sheet("embed_tokens_per_layer", ids).view(n, case["layers"], ple) * math.sqrt(ple)
    rooms = lin(x, "per_layer_model_projection").view(n, case["layers"], ple) / math.sqrt(width)
    rooms = (_rms(rooms, vec("per_layer_projection_norm")) + seeds) / math.sqrt(2)

    def turn(v, head, full):
        half = head // 2
        live = head // 8 if full else half  # a quarter of a global head's pairs turn
        j = torch.arange(half, device="cuda").double()
        step = torch.where(j < live, (1e6 if full else 1e4) ** (-2 * j / head), torch.zeros_like(j)).float().double()
        angle = place.double()[:, None, None] * step
        lo, hi = v[..., :half], v[..., half:]
        return torch.cat([lo * angle.cos() - hi * angle.sin(), hi * angle.cos() + lo * angle.sin()], -1)

    def byte(v, scale):
        return (v / scale).float().clamp(-448, 448).to(torch.float8_e4m3fn).float().double() * scale

    rings = {}
    for i, (head, full, shared, _) in enumerate(_engine_layers(case)):
        p = "layers.%d." % i
        h = _rms(x, vec(p + "input_layernorm"))
        q = turn(_rms(lin(h, p + "self_attn.q_proj").view(n, 8, head), vec(p + "self_attn.q_norm")), head, full)
        if not shared:
            k = turn(_rms(lin(h, p + "self_attn.k_proj").view(n, 1, head), vec(p + "self_attn.k_norm")), head, full)
            v = _rms(lin(h, p + "self_attn.v_proj"))
            rings[full] = (byte(k[:, 0], t[p + "self_attn.k_cache_scale"].double()),
                           byte(v, t[p + "self_attn.v_cache_scale"].double()))
        key, value = rings[full]
        hide = place[None] > place[:, None]
        if not full:
            hide = hide | (place[None] <= place[:, None] - ENGINE_WINDOW)
        score = (q.transpose(0, 1).reshape(8 * n, head) @ key.T).view(8, n, n).masked_fill(hide, -math.inf)
        blend = (torch.softmax(score, -1).view(8 * n, n) @ value).view(8, n, head).transpose(0, 1).reshape(n, -1)
        x = x + _rms(lin(blend, p + "self_attn.o_proj"), vec(p + "post_attention_layernorm"))
        h = _rms(x, vec(p + "pre_feedforward_layernorm"))
        h = lin(_gelu(lin(h, p + "mlp.gate_proj")) * lin(h, p + "mlp.up_proj"), p + "mlp.down_proj")
        x = x + _rms(h, vec(p + "post_feedforward_layernorm"))
        h = lin(_gelu(lin(x, p + "per_layer_input_gate")) * rooms[:, i], p + "per_layer_projection")
        x = (x + _rms(h, vec(p + "post_per_layer_input_norm"))) * t[p + "layer_scalar"].double()
    rows = x[-1 - case["block"]:]
    logits = 30.0 * torch.tanh(lin(_rms(rows, vec("norm")), "lm_head") / 30.0)
    logits = logits.cpu().numpy()
    return {"step": logits[0], "block": logits[1:]}
