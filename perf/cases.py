"""The measured cases: what a program that uses this framework has it do, through its public entry points.

`listed()` names them, `draw()` gives more of the same ranges, `prepare()` makes a case's inputs on the
device, `run()` is one pass, `exact()` the same pass in 64-bit torch.  The shapes are those of the
synthetic models in `wavo_amd.synth` (Parakeet, GigaAM and Whisper), which the benchmark and the tests
use.  A program opens the device and loads its model once and keeps a buffer per input and output, so
the models here are shared by the states and every state has its own buffers.
"""

import functools
import math
import os
import struct

import numpy as np
import torch

import wavo_amd as wa
from wavo_amd import synth

DEV = "cuda:0"
TYPES = {"q8_0": wa.Q8_0, "q4_0": wa.Q4_0, "f16": wa.F16}
BYTES = {"q8_0": 34 / 32, "q4_0": 18 / 32, "f16": 2.0}
EPILOGUES = {"bias": wa.BIAS, "silu": wa.SILU, "relu": wa.RELU, "gelu": wa.GELU}
# (heads, head size) of the three attention forms: Parakeet's relative one, GigaAM's rotary one (q and k
# beside v), Whisper's plain one.
ATTENTION = {"relative": (8, 128), "rotary": (16, 48), "plain": (20, 64)}
VOCAB = 51904  # Whisper's 51866 logits in whole groups of 64, as the head writes them


def listed():
    return [
        # The feed-forward of a Whisper decoder layer for one token, two one-row calls: the smallest work.
        {"name": "token_ffn", "kind": "ffn", "d": 1280, "ff": 5120, "type": "q8_0"},
        # The decoder's vocabulary head, the largest call with one row.
        {"name": "token_head", "kind": "gemv", "rows": 51866, "k": 1280, "type": "q8_0", "epi": "bias"},
        # A feed-forward layer's first projection over one 60 s window, f16 in and out as between layers.
        {"name": "ffn_up_60s", "kind": "gemm", "m": 750, "rows": 4096, "k": 1024, "type": "q8_0", "epi": "silu",
         "half": True},
        # A second projection over a 30 s Whisper window, 4-bit weights, f32 activations at the boundary.
        {"name": "ffn_down_30s", "kind": "gemm", "m": 1500, "rows": 1280, "k": 5120, "type": "q4_0", "epi": "bias",
         "half": False},
        # The same first projection over a batch of windows of long audio (an uneven number of rows).
        {"name": "ffn_up_batch", "kind": "gemm", "m": 11616, "rows": 4096, "k": 1024, "type": "q8_0", "epi": "silu",
         "half": True},
        # An attention layer with relative positions over one 60 s window.
        {"name": "attention_60s", "kind": "attention", "form": "relative", "t": 750, "valid": 750},
        # A whole encoder call over 60 s of audio, the benchmark's step.
        {"name": "encode_60s", "kind": "parakeet", "batch": 1, "mel": 6001, "shortest": 6001},
        # Long audio: 16 windows of different lengths in one padded call.
        {"name": "encode_batch", "kind": "parakeet", "batch": 16, "mel": 5801, "shortest": 4401},
        # A short utterance from its samples to its text: features, encoder, CTC decoding.
        {"name": "transcribe_11s", "kind": "gigaam", "samples": 176000},
        # Whisper's encoder over its 30 s window, four of its equal layers.
        {"name": "whisper_window", "kind": "whisper", "tokens": 0, "frames": 1500},
        # Whisper's decoder: the window's cross keys and values, then 32 tokens one after the other.
        {"name": "whisper_tokens", "kind": "whisper", "tokens": 32, "frames": 1500},
        # The greedy transducer decoding of 60 s of encoder output, one decision after the other.
        {"name": "tdt_60s", "kind": "tdt", "frames": 750},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ffn", "gemv", "gemm", "gemm", "attention", "parakeet", "parakeet", "gigaam", "whisper", "tdt"])
    wtype = rng.choice(["q8_0", "q8_0", "q4_0", "f16"])
    if kind == "ffn":
        d = 64 * _spread(rng, 4, 20)
        return {"kind": kind, "d": d, "ff": 4 * d, "type": wtype}
    if kind == "gemv":
        return {"kind": kind, "rows": _spread(rng, 640, 51866), "k": 64 * _spread(rng, 8, 80), "type": wtype,
                "epi": rng.choice(["bias", "gelu"])}
    if kind == "gemm":
        return {"kind": kind, "m": _spread(rng, 12, 12000), "rows": 64 * _spread(rng, 8, 80), "k": 64 * _spread(rng, 8, 80),
                "type": wtype, "epi": rng.choice(["bias", "silu", "relu", "gelu"]), "half": rng.random() < 0.7}
    if kind == "attention":
        t = _spread(rng, 25, 1500)
        return {"kind": kind, "form": rng.choice(sorted(ATTENTION)), "t": t, "valid": t if rng.random() < 0.6 else rng.randint(t // 2, t)}
    if kind == "parakeet":
        batch = rng.choice([1, 1, 1, 2, 4, 9, 16])
        mel = _spread(rng, 101, 5800)
        return {"kind": kind, "batch": batch, "mel": mel, "shortest": mel if batch == 1 else rng.randint(mel // 2, mel)}
    if kind == "gigaam":
        return {"kind": kind, "samples": _spread(rng, 8000, 480000)}
    if kind == "whisper":
        return {"kind": kind, "tokens": _spread(rng, 4, 48), "frames": rng.choice([1500, rng.randint(50, 1500)])}
    return {"kind": kind, "frames": _spread(rng, 25, 750)}


# ------------------------------------------------------------------------------- device and models


@functools.lru_cache(None)
def _gpu():
    return wa.Gpu(0)


@functools.lru_cache(None)
def _path(family):
    """A family's model file.  Whisper's encoder has 4 of its 32 equal layers here, to be written quickly;
    the transducer decoder's file has one encoder layer and a blank likely enough for 60 s of frames to
    give about 250 tokens, as speech does."""
    if family == "whisper":
        name, config = "whisper-4-encoder-layers", dict(synth.CONFIGS["whisper"], layers=4)
    elif family == "tdt":
        name, config = "parakeet-tdt-decoder", dict(synth.CONFIGS["parakeet"], layers=1, blank_bias=0.7)
    else:
        return synth.model_path(family)
    where = os.environ.get("WAVO_MODELS", "/tmp/wavo_models")
    os.makedirs(where, exist_ok=True)
    path = os.path.join(where, name + ".gguf")
    if not os.path.exists(path):
        synth.write_model(path, config)
    return path


@functools.lru_cache(None)
def _model(family):
    return wa.Model(_gpu(), _path(family))


def _rand(seed, what, *shape, scale=1.0):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000 * seed + what)
    return scale * torch.randn(*shape, generator=g, device=DEV)


def _features(seed, frames, mels):
    """Log-mel features as the frontends make them: near N(0, 1) per bin, neighbouring frames alike."""
    x = _rand(seed, 1, frames + 4, mels)
    return sum(w * x[i:i + frames] for i, w in enumerate((0.3, 0.6, 0.8, 0.6, 0.3))).div(math.sqrt(1.54)).contiguous()


def _speech(seed, samples):
    """Noise and three tones that come and go, in [-1, 1]."""
    t = torch.arange(samples, device=DEV, dtype=torch.float64) / synth.SR
    x = _rand(seed, 2, samples, scale=0.05).double()
    for f, r in _rand(seed, 3, 3, 2).tolist():
        x += 0.1 * torch.sin(2 * math.pi * (400 + 300 * abs(f)) * t) * torch.sin(3 * r * t)
    return x.float().contiguous()


# ---------------------------------------------------------------------------------------- weights


def _encode(w, wtype):
    """[rows][k] f32 weights in a GGUF type's bytes (a uint8 tensor) and their exact values."""
    if wtype == "f16":
        h = w.half()
        return h.view(torch.uint8).reshape(-1), h.double()
    b = w.reshape(-1, 32)
    if wtype == "q8_0":
        d = (b.abs().amax(1, keepdim=True) / 127).half()
        q = (b / d.float()).round().clamp(-127, 127).to(torch.int8)
        raw = torch.cat([d.view(torch.uint8), q.view(torch.uint8)], 1)
        return raw.reshape(-1), (q.double() * d.double()).reshape(w.shape)
    far = b.gather(1, b.abs().argmax(1, keepdim=True))
    d = (far / -8).half()
    q = (b / d.float() + 8).round().clamp(0, 15).to(torch.uint8)
    raw = torch.cat([d.view(torch.uint8), q[:, :16] | (q[:, 16:] << 4)], 1)
    return raw.reshape(-1), ((q.double() - 8) * d.double()).reshape(w.shape)


def _layer(seed, rows, k, wtype):
    """A layer's weights as stored, their values and its bias."""
    raw, values = _encode(_rand(seed, 4 + rows, rows, k, scale=0.02), wtype)
    return raw, values, _rand(seed, 5 + rows, rows, scale=0.02)


def _linear_of(seed, rows, k, wtype):
    raw, _, bias = _layer(seed, rows, k, wtype)
    return _gpu().linear([(raw.cpu().numpy().tobytes(), TYPES[wtype], k, rows)], bias.cpu().numpy())


def _width(rows):
    return rows if rows % 32 == 0 else -(-rows // 64) * 64


# ------------------------------------------------------------------------------------- one pass


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "ffn":
        d, ff = case["d"], case["ff"]
        s["up"], s["down"] = _linear_of(seed, ff, d, case["type"]), _linear_of(seed, d, ff, case["type"])
        s["x"], s["h"], s["y"] = _rand(seed, 6, d), torch.empty(ff, device=DEV), torch.empty(d, device=DEV)
    elif kind in ("gemv", "gemm"):
        s["layer"] = _linear_of(seed, case["rows"], case["k"], case["type"])
        m, half = case.get("m", 1), case.get("half", False)
        a = _rand(seed, 6, m, case["k"])
        s["a"] = a.half() if half else a
        s["c"] = torch.empty(m, s["layer"].width, dtype=torch.float16 if half else torch.float32, device=DEV)
    elif kind == "attention":
        heads, hd = ATTENTION[case["form"]]
        t, d = case["t"], heads * hd
        s["qk"] = _rand(seed, 7, t, d * {"relative": 4, "rotary": 2, "plain": 3}[case["form"]])
        s["v"] = _rand(seed, 8, t, d) if case["form"] == "rotary" else None
        s["pos"] = _rand(seed, 9, 2 * t + 15, d, scale=0.5) if case["form"] == "relative" else None
        s["o"] = torch.empty(t, d, device=DEV)
    else:
        model = s["model"] = _model(kind)
        if kind == "parakeet":
            s["valid"] = _lengths(case, seed)
            mel = torch.zeros(case["batch"], case["mel"], model.mels, device=DEV)
            for b, v in enumerate(s["valid"]):
                mel[b, :v] = _features(100 * seed + b, v, model.mels)
            s["mel"] = mel
            frames, width = model.frames(case["mel"])
            s["out"] = torch.empty(case["batch"], frames, width, device=DEV)
        elif kind == "gigaam":
            s["pcm"] = _speech(seed, case["samples"])
            mel_frames = model.mel_frames(case["samples"])
            s["mel"] = torch.empty(mel_frames, model.mels, device=DEV)
            s["out"] = torch.empty(*model.frames(mel_frames), device=DEV)
        elif kind == "whisper" and not case["tokens"]:
            s["mel"] = (0.25 * _features(seed, 2 * case["frames"], model.mels)).clamp(-1.0, 1.0)
            s["out"] = torch.empty(case["frames"], model.d, device=DEV)
        elif kind == "whisper":
            s["enc"] = _rand(seed, 10, case["frames"], model.d)
            s["tokens"] = np.random.default_rng(seed).integers(0, 50000, case["tokens"]).tolist()
            s["out"] = torch.empty(VOCAB, device=DEV)
        else:
            # Far below zero on average: the joint's rectifier leaves few of its units on, other ones in
            # every frame, so that tokens, blanks and durations vary.
            s["enc"] = _rand(seed, 11, case["frames"], model.width, scale=2.0) - 3.0
    torch.cuda.synchronize()
    return s


def _lengths(case, seed):
    """The windows' real lengths: the longest first, the others anywhere down to the shortest."""
    rng = np.random.default_rng(seed)
    return [case["mel"]] + rng.integers(case["shortest"], case["mel"] + 1, case["batch"] - 1).tolist()


def run(s):
    gpu, kind, case = _gpu(), s["kind"], s["case"]
    if kind == "ffn":
        gpu.gemv(s["x"].data_ptr(), s["up"], s["h"].data_ptr(), wa.GELU)
        gpu.gemv(s["h"].data_ptr(), s["down"], s["y"].data_ptr(), wa.BIAS)
        return s["h"], s["y"]
    if kind == "gemv":
        gpu.gemv(s["a"].data_ptr(), s["layer"], s["c"].data_ptr(), EPILOGUES[case["epi"]])
        return s["c"]
    if kind == "gemm":
        call = functools.partial(gpu.gemm_h, out16=True) if case["half"] else gpu.gemm
        call(s["a"].data_ptr(), s["layer"], s["c"].data_ptr(), case["m"], EPILOGUES[case["epi"]])
        return s["c"]
    if kind == "attention":
        heads, hd = ATTENTION[case["form"]]
        at = lambda x: None if x is None else x.data_ptr()  # noqa: E731
        gpu.attention(at(s["qk"]), at(s["v"]), at(s["pos"]), at(s["o"]), case["t"], heads, hd, case["valid"])
        return s["o"]
    model = s["model"]
    if kind == "parakeet":
        if case["batch"] == 1:
            model.encode_device(s["mel"].data_ptr(), case["mel"], s["out"].data_ptr())
        else:
            model.encode_batch_device(s["mel"].data_ptr(), case["batch"], case["mel"], s["valid"], s["out"].data_ptr())
        return s["out"]
    if kind == "gigaam":
        mel_frames = model.mel_device(s["pcm"].data_ptr(), case["samples"], s["mel"].data_ptr())
        model.encode_device(s["mel"].data_ptr(), mel_frames, s["out"].data_ptr())
        frames, width = s["out"].shape
        return {"mel": s["mel"], "logits": s["out"], "ids": _by_frame(model.greedy_device(s["out"].data_ptr(), frames, width), frames)}
    if kind == "whisper" and not case["tokens"]:
        model.encode_device(s["mel"].data_ptr(), 2 * case["frames"], s["out"].data_ptr())
        return s["out"]
    if kind == "whisper":
        model.whisper_begin(s["enc"].data_ptr(), case["frames"])
        for pos, token in enumerate(s["tokens"]):
            model.whisper_step(token, pos, s["out"].data_ptr())
        return s["out"]
    return _by_frame(model.greedy_device(s["enc"].data_ptr(), case["frames"], model.width), case["frames"])


def _by_frame(pairs, frames):
    """The (token, frame) pairs as a row per frame: how many tokens it has, the first and the last of them."""
    out = np.full((frames, 3), -1, np.int64)
    out[:, 0] = 0
    for token, frame in pairs:
        if out[frame, 0] == 0:
            out[frame, 1] = token
        out[frame, 0] += 1
        out[frame, 2] = token
    return out


# ------------------------------------------------------------------------- work and tolerances


def work(case):
    kind = case["kind"]
    if kind == "ffn":
        n, ff = case["d"] * case["ff"], case["ff"]
        return {"bytes": 2 * n * BYTES[case["type"]] + 12.0 * (ff + case["d"]), "flops": 4.0 * n}
    if kind in ("gemv", "gemm"):
        m, n, k = case.get("m", 1), case["rows"], case["k"]
        size = 2 if case.get("half") else 4
        return {"bytes": n * k * BYTES[case["type"]] + 4 * n + size * m * (k + n), "flops": 2.0 * m * n * k}
    if kind == "attention":
        heads, hd = ATTENTION[case["form"]]
        t, v, d = case["t"], case["valid"], heads * hd
        rel = case["form"] == "relative"
        return {"bytes": 4.0 * d * ((5 if rel else 4) * t + (2 * t + 15 if rel else 0)), "flops": 2.0 * d * t * v * (3 if rel else 2)}
    c = synth.CONFIGS["parakeet" if kind == "tdt" else kind]
    d = c.get("d")
    if kind in ("parakeet", "gigaam"):
        # Per frame and layer: two feed-forwards, q, k, v and out, the conv module's 3 d² and its taps.
        weights = 4 * d * c["d_ff"] + 7 * d * d
        if kind == "parakeet":
            mel, batch = case["mel"], case["batch"]
            t = _half(_half(_half(mel - 1)))
            ch, cells = c["ch"], _half(_half(mel)) * (c["mels"] // 4)
            stem = cells * (2.0 * 9 * 4 * ch + 2.0 * 9 * ch + 2.0 * ch * ch) + t * (c["mels"] // 8) * (18.0 * ch + 2.0 * ch * ch)
            stem += 2.0 * t * ch * (c["mels"] // 8) * d + 2.0 * t * d * c["joint"]
            rest = ch * (c["mels"] // 8) * d + d * c["joint"]
            io = 4.0 * (mel * c["mels"] + t * c["joint"])
        else:
            batch, mel = 1, (case["samples"] - 320) // 160 + 1
            t = _half(_half(mel))
            stem = 2.0 * _half(mel) * 5 * c["mels"] * d + 2.0 * t * 5 * d * d + 2.0 * t * d * c["classes"]
            rest = 5 * c["mels"] * d + 5 * d * d + d * c["classes"]
            io = 4.0 * (case["samples"] + 2 * mel * c["mels"] + t * 320)
        attention = 2.0 * t * t * d * (3 if kind == "parakeet" else 2)
        flops = batch * (stem + c["layers"] * (t * (2.0 * weights + 2 * c["kernel"] * d) + attention))
        return {"bytes": (c["layers"] * weights + rest) * BYTES["q8_0"] + batch * io, "flops": flops}
    if kind == "whisper":
        t, ff, layers = case["frames"], c["d_ff"], 4
        weights = layers * (4 * d * d + 2 * d * ff)
        if not case["tokens"]:
            conv = 3 * c["mels"] * d + 3 * d * d
            return {"bytes": (weights + conv) * BYTES["q8_0"] + 4.0 * t * (2 * c["mels"] + d),
                    "flops": 2.0 * t * (weights + 2 * 3 * c["mels"] * d + 3 * d * d) + layers * 4.0 * t * t * d}
        # Per token every weight (the cross keys' and values' once per window) and the cross cache in f16.
        n, token = case["tokens"], layers * (6 * d * d + 2 * d * ff) + c["vocab"] * d
        return {"bytes": n * (token * BYTES["q8_0"] + layers * 4.0 * t * d + 4.0 * c["vocab"]) + layers * 2 * d * d * BYTES["q8_0"] + 4.0 * t * d,
                "flops": 2.0 * n * (token + layers * 2 * t * d) + 2.0 * t * layers * 2 * d * d}
    # About two decisions per three frames; each needs the joint, the LSTM and the predictor's projection.
    hidden, joint = c["hidden"], c["joint"]
    decision = (c["vocab"] + 5) * joint + 8 * hidden * hidden + hidden * joint
    return {"bytes": decision * BYTES["q8_0"] + 4.0 * case["frames"] * joint, "flops": 2.0 * decision * max(1, 2 * case["frames"] // 3)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("ffn", "gemv"):
        return {"rel": 4e-6}  # f32 sums in another order: about 5e-7 off 64 bits
    if kind == "gemm":
        # f32 sums in another order; an f16 output also rounds the other way now and then (one ulp, 1e-3).
        return {"rel": 1e-4, "max": 2e-3} if case["half"] else {"rel": 1e-5}
    if kind == "attention":
        return {"rel": 2e-3, "max": 2e-2}  # f16 queries, keys, probabilities and values
    if kind == "tdt":
        return {"rel": 0.0, "differ": 0.01}  # 32-bit logits: another token only at a tie of two
    if kind == "whisper" and case["tokens"]:
        return {"rel": 1e-3, "max": 1e-2}  # keys and values kept in f16
    # Whole encoders: f16 products through every layer; ids beside logits differ at ties.
    return {"rel": 4e-3, "max": 5e-2, "differ": 0.01}


# -------------------------------------------------------------------------------- 64-bit passes


class _File:
    """The tensors of a GGUF file by name, as 64-bit values on the device."""

    SIZES = {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}

    def __init__(self, path):
        self.raw = np.memmap(path, np.uint8, "r")
        self.at = 8
        tensors, values = self._n("<Q"), self._n("<Q")
        for _ in range(values):
            self._text()
            self._skip(self._n("<I"))
        infos = {}
        for _ in range(tensors):
            name = self._text()
            dims = [self._n("<Q") for _ in range(self._n("<I"))]
            infos[name] = (dims, self._n("<I"), self._n("<Q"))
        data = -(-self.at // 32) * 32
        self.infos = {n: (dims, ty, data + off) for n, (dims, ty, off) in infos.items()}
        self.values = {}

    def _n(self, fmt):
        size = struct.calcsize(fmt)
        self.at += size
        return struct.unpack(fmt, self.raw[self.at - size:self.at].tobytes())[0]

    def _text(self):
        n = self._n("<Q")
        self.at += n
        return self.raw[self.at - n:self.at].tobytes().decode()

    def _skip(self, ty):
        if ty == 8:
            self._text()
        elif ty == 9:
            item, n = self._n("<I"), self._n("<Q")
            if item == 8:
                for _ in range(n):
                    self._text()
            else:
                self.at += n * self.SIZES[item]
        else:
            self.at += self.SIZES[ty]

    def has(self, name):
        return name in self.infos

    def __call__(self, name):
        """A tensor as [last dimension][the others], kept for the layers' next window."""
        if name not in self.values:
            self.values[name] = self._read(*self.infos[name])
        return self.values[name]

    def _read(self, dims, ty, at):
        n = math.prod(dims)
        size = n * 4 if ty == 0 else n * 2 if ty == 1 else n // 32 * 34
        raw = torch.from_numpy(np.array(self.raw[at:at + size])).to(DEV)
        if ty in (0, 1):
            x = raw.view(torch.float32 if ty == 0 else torch.float16).double()
        else:
            b = raw.reshape(-1, 34)
            x = b[:, 2:].contiguous().view(torch.int8).double() * b[:, :2].contiguous().view(torch.float16).double()
        return x.reshape(dims[-1], -1)

    def vector(self, name):
        return self(name).reshape(-1)


@functools.lru_cache(None)
def _file(family):
    return _File(_path(family))


def _half(n):
    return (n - 1) // 2 + 1


def _apply(epi, x):
    return {"bias": lambda v: v, "silu": torch.nn.functional.silu, "relu": torch.relu, "gelu": torch.nn.functional.gelu}[epi](x)


def _norm(F, name, x):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], F.vector(name + ".weight"), F.vector(name + ".bias"), 1e-5)


def _linear(F, name, x):
    b = F.vector(name + ".bias") if F.has(name + ".bias") else None
    return torch.nn.functional.linear(x, F(name + ".weight"), b)


def _attend(q, k, v, heads, valid, more=None):
    """softmax((q·kᵀ + more) / √hd)·v per head over the first `valid` keys; rows of heads·hd."""
    hd = q.shape[1] // heads
    out = torch.empty_like(q)
    for h in range(heads):
        at = slice(h * hd, (h + 1) * hd)
        score = q[:, at] @ k[:valid, at].T
        if more is not None:
            score += more(h, at)[:, :valid]
        out[:, at] = torch.softmax(score / math.sqrt(hd), 1) @ v[:valid, at]
    return out


def _relative(q, pos, t):
    """The position scores of head rows `at`: (i, j) takes row j − i + t + 15 of the positions."""
    row = torch.arange(t, device=DEV)
    index = row[None, :] - row[:, None] + t + 15
    return lambda h, at: torch.gather(q[:, at] @ pos[:, at].T, 1, index)


def _conformer_block(F, c, i, x, valid):
    relative = c["arch"] == "parakeet"
    p, t, d, heads = f"enc.blocks.{i}.", x.shape[0], c["d"], c["heads"]
    ffn = lambda y, n: _linear(F, p + n + ".linear2", _apply("silu", _linear(F, p + n + ".linear1", y)))  # noqa: E731
    x = x + 0.5 * ffn(_norm(F, p + "norm_ff1", x), "ff1")
    y = _norm(F, p + "norm_attn", x)
    if relative:
        q, k, v = (_linear(F, p + "attn.linear_" + n, y) for n in "qkv")
        angle = (t + 15 - torch.arange(2 * t + 15, device=DEV))[:, None].double()
        angle = angle * torch.exp(torch.arange(0, d, 2, device=DEV).double() * (-math.log(10000.0) / d))
        pos = torch.stack([angle.sin(), angle.cos()], 2).reshape(2 * t + 15, d)
        pos = _linear(F, p + "attn.linear_pos", pos)
        o = _attend(q + F.vector(p + "attn.pos_bias_u"), k, v, heads, valid, _relative(q + F.vector(p + "attn.pos_bias_v"), pos, t))
    else:
        angle = torch.arange(t, device=DEV)[:, None].double() * 5000.0 ** (-2.0 * torch.arange(d // heads // 2, device=DEV).double() * heads / d)
        first, second = y.reshape(t, heads, 2, -1).unbind(2)
        cos, sin = angle.cos()[:, None], angle.sin()[:, None]
        turned = torch.stack([first * cos - second * sin, second * cos + first * sin], 2).reshape(t, d)
        q, k = (_linear(F, p + "attn.linear_" + n, turned) for n in "qk")
        o = _attend(q, k, _linear(F, p + "attn.linear_v", y), heads, valid)
    x = x + _linear(F, p + "attn.linear_out", o)
    gated = torch.nn.functional.glu(_linear(F, p + "conv.pointwise1", _norm(F, p + "norm_conv", x)), 1)
    gated[valid:] = 0.0
    bias = None if relative else F.vector(p + "conv.depthwise.bias")
    taps = F(p + "conv.depthwise.weight").reshape(d, 1, c["kernel"])
    y = torch.nn.functional.conv1d(gated.T[None], taps, bias, padding=c["kernel"] // 2, groups=d)[0].T
    if relative:
        n = p + "conv.bn."
        y = (y - F.vector(n + "running_mean")) / torch.sqrt(F.vector(n + "running_var") + 1e-5) * F.vector(n + "weight") + F.vector(n + "bias")
    else:
        y = _norm(F, p + "conv.ln", y)
    x = x + _linear(F, p + "conv.pointwise2", _apply("silu", y))
    x = x + 0.5 * ffn(_norm(F, p + "norm_ff2", x), "ff2")
    return _norm(F, p + "norm_out", x)


def _parakeet(F, c, mel, valid, alone):
    """One window [mel frames][mels] whose first `valid` frames are real; alone: not in a batch."""
    ch, frames = c["ch"], mel.shape[0]
    t = _half(_half(_half(frames - 1)))
    conv = torch.nn.functional.conv2d
    taps = lambda i: (F(f"enc.pre_encode.conv.{i}.weight").reshape(ch, 1, 3, 3), F.vector(f"enc.pre_encode.conv.{i}.bias"))  # noqa: E731
    point = lambda i, x: torch.relu(_linear(F, f"enc.pre_encode.conv.{i}", x.permute(1, 2, 0)))  # noqa: E731
    x = torch.relu(conv(mel[None, None, :valid].double(), *taps(0), stride=2, padding=1))
    x = conv(x, *taps(2), stride=2, padding=1, groups=ch)[0]  # [ch][⌈valid / 4⌉][mels / 4]
    rows = _half(_half(frames)) if alone else x.shape[1]
    x = torch.nn.functional.pad(x, (0, 0, 0, rows - x.shape[1]))
    x = point(3, x).permute(2, 0, 1)
    x = torch.nn.functional.pad(x, (0, 0, 0, max(0, 2 * t + 1 - rows)))
    x = conv(x[None], *taps(5), stride=2, padding=1, groups=ch)[0][:, :t]
    x = point(6, x).permute(0, 2, 1).reshape(t, -1)
    x = _linear(F, "enc.pre_encode.out", x)
    keys = t if alone else min(t, _half(_half(_half(max(valid, 3) - 1))))
    for i in range(c["layers"]):
        x = _conformer_block(F, c, i, x, keys)
    return _linear(F, "joint.enc", x)


def _gigaam(F, c, pcm):
    frames = pcm.double().unfold(0, 320, 160)
    power = torch.fft.rfft(frames * F.vector("frontend.window")).abs().square()
    mel = torch.log((power @ F("frontend.mel_filterbank").T).clamp(1e-9, 1e9))
    x = mel
    for i in (0, 2):
        n = f"enc.pre_encode.conv.{i}"
        w = F(n + ".weight").reshape(c["d"], -1, 5)
        x = torch.relu(torch.nn.functional.conv1d(x.T[None], w, F.vector(n + ".bias"), stride=2, padding=2))[0].T
    for i in range(c["layers"]):
        x = _conformer_block(F, c, i, x, x.shape[0])
    return mel, torch.nn.functional.pad(_linear(F, "head.ctc", x), (0, _width(c["classes"]) - c["classes"]))


def _whisper_window(F, c, mel):
    x = mel.double()
    for i in (0, 1):
        n = f"enc.conv.{i}"
        w = F(n + ".weight").reshape(c["d"], -1, 3)
        x = _apply("gelu", torch.nn.functional.conv1d(x.T[None], w, F.vector(n + ".bias"), stride=1 + i, padding=1))[0].T
    x = x + F("enc.pos_emb.weight")[:x.shape[0]]
    for i in range(4):
        p = f"enc.blocks.{i}."
        y = _norm(F, p + "norm_attn", x)
        o = _attend(*(_linear(F, p + "attn." + n, y) for n in "qkv"), c["heads"], x.shape[0])
        x = x + _linear(F, p + "attn.out", o)
        x = x + _linear(F, p + "ffn.fc2", _apply("gelu", _linear(F, p + "ffn.fc1", _norm(F, p + "norm_ffn", x))))
    return _norm(F, "enc.final_norm", x)


def _whisper_tokens(F, c, enc, tokens):
    heads, n = c["dec_heads"], len(tokens)
    words = F("dec.token_embd.weight")
    x = words[tokens] + F("dec.pos_emb.weight")[:n]
    later = torch.full((n, n), -math.inf, device=DEV, dtype=torch.float64).triu(1)
    for i in range(c["dec_layers"]):
        p = f"dec.blocks.{i}."
        y = _norm(F, p + "norm_self", x)
        o = _attend(*(_linear(F, p + "self_attn." + m, y) for m in "qkv"), heads, n, lambda h, at: later)
        x = x + _linear(F, p + "self_attn.out", o)
        q = _linear(F, p + "cross_attn.q", _norm(F, p + "norm_cross", x))
        k, v = (_linear(F, p + "cross_attn." + m, enc.double()) for m in "kv")
        x = x + _linear(F, p + "cross_attn.out", _attend(q, k, v, heads, enc.shape[0]))
        x = x + _linear(F, p + "ffn.fc2", _apply("gelu", _linear(F, p + "ffn.fc1", _norm(F, p + "norm_ffn", x))))
    return torch.nn.functional.pad(words @ _norm(F, "dec.final_norm", x)[-1], (0, VOCAB - c["vocab"]))


def exact(case, seed):
    kind = case["kind"]
    if kind == "ffn":
        (_, up, b0), (_, down, b1) = (_layer(seed, *n, case["type"]) for n in ((case["ff"], case["d"]), (case["d"], case["ff"])))
        h = _apply("gelu", torch.nn.functional.linear(_rand(seed, 6, case["d"]).double(), up, b0.double()))
        return h, torch.nn.functional.linear(h, down, b1.double())
    if kind in ("gemv", "gemm"):
        _, w, bias = _layer(seed, case["rows"], case["k"], case["type"])
        a = _rand(seed, 6, case.get("m", 1), case["k"])
        a = (a.half() if case.get("half") else a).double()
        c = _apply(case["epi"], torch.nn.functional.linear(a, w, bias.double()))
        return torch.nn.functional.pad(c, (0, _width(case["rows"]) - case["rows"]))
    if kind == "tdt":
        return None  # whole numbers
    s = prepare(case, seed)
    if kind == "attention":
        heads, hd = ATTENTION[case["form"]]
        d, t = heads * hd, case["t"]
        part = lambda i: s["qk"][:, i * d:(i + 1) * d].double()  # noqa: E731
        more = _relative(part(3), s["pos"].double(), t) if case["form"] == "relative" else None
        return _attend(part(0), part(1), s["v"].double() if case["form"] == "rotary" else part(2), heads, case["valid"], more)
    F, c = _file(kind), synth.CONFIGS["parakeet" if kind == "tdt" else kind]
    if kind == "parakeet":
        return torch.stack([_parakeet(F, c, mel, v, case["batch"] == 1) for mel, v in zip(s["mel"], s["valid"])])
    if kind == "gigaam":
        mel, logits = _gigaam(F, c, s["pcm"])
        return {"mel": mel, "logits": logits, "ids": None}
    if not case["tokens"]:
        return _whisper_window(F, c, s["mel"])
    return _whisper_tokens(F, c, s["enc"], s["tokens"])
