"""The work that programs give this framework, as cases that can be timed and checked.

A case is a dict of plain values; ``listed()`` gives the standing ones and ``draw(rng)`` one more of the
same ranges. ``prepare(case, seed)`` makes what a program has in hand before the call (weights uploaded
once, buffers, inputs), ``run(state)`` makes one pass through the public entry points and returns its
outputs, ``exact(case, seed)`` the same outputs in 64-bit arithmetic by plain torch, ``work(case)`` the
bytes and operations the pass cannot do without, and ``tolerance(case)`` how far another correct
implementation at the same precision may be from it.

The kinds of case:

gemv         one product of a few rows by a decoder matrix (``linear_device``)
predict      one call of the prediction network for a beam's hypotheses (``TdtDecoder.predict_rows``)
decode       the greedy TDT decode of one or several utterances (``TdtDecoder.decode``, ``decode_streams``)
layer        Conformer layers over utterances stacked along the rows (``ConformerLayer.run_stack``)
block        one block of the 2048-channel encoder, strided or not (``GraniteBlock.forward``)
conditioning the CTC head, softmax and injection between two blocks (``self_conditioning``)
feedforward  the two products of a feed-forward module called one by one, in any weight precision, or
             with 8-bit weights in the exact mode (``linear_device``)
attention    the attention core on the f32 products of row-major views and the softmax
             (``matmul_rowmajor_device``, ``softmax_device``)

Sizes are those of the encoders and decoder the benchmark runs: width 1024, feed-forward 4096, 8 heads of
128, 12.5 frames per second after subsampling; decoder width 640, 8193 tokens and 5 durations. Weights
and activations have the benchmark's distributions: int8 values over the whole range with scales in
[0.001, 0.01), N(0, 1) rows."""
import math

import numpy as np
import torch

import telmo_amd
from telmo_amd import Act, Epilogue, PackedWeights, Precision
from telmo_amd.conformer import ConformerLayer, LayerWeights
from telmo_amd.granite import BlockWeights, GraniteBlock, self_conditioning
from telmo_amd.kernels import TdtDecoder

D, FF, HEADS = 1024, 4096, 8
EPS = 1e-5
LAYER_TAPS = 9
BLOCK_CHANNELS, BLOCK_TAPS, BLOCK_VOCAB = 2048, 7, 16384
H, VOCAB, DURATIONS, MAX_SYMBOLS = 640, 8193, (0, 1, 2, 3, 4), 10

PRECISIONS = {p.name_(): p for p in Precision}
VALUE_BYTES = {"f32": 4.0, "f16": 2.0, "bf16": 2.0, "int8": 1.0, "q8_0": 1.0 + 4.0 / 32}


# ------------------------------------------------------------------------------------------ cases

def listed():
    return [
        # One joint evaluation of a decoder loop that the caller runs itself: the smallest call.
        {"name": "joint, one row", "kind": "gemv", "precision": "int8", "m": 1, "k": 640, "n": 8198},
        # A beam search extends eight hypotheses by a token each.
        {"name": "predict, 8 hypotheses", "kind": "predict", "precision": "int8", "rows": 8},
        # One minute of one speaker, decoded offline.
        {"name": "decode, 60 s", "kind": "decode", "precision": "int8", "streams": 1, "frames": 750},
        # Eight half-minute utterances decoded together by a server.
        {"name": "decode, 8 x 30 s", "kind": "decode", "precision": "int8", "streams": 8, "frames": 375},
        # One encoder layer over a minute of audio, the ordinary offline call.
        {"name": "layer, 60 s", "kind": "layer", "precision": "int8", "rows": 750, "utterances": 1, "layers": 1},
        # A shorter utterance of odd length with block-scaled weights.
        {"name": "layer q8_0, 413 frames", "kind": "layer", "precision": "q8_0", "rows": 413, "utterances": 1,
         "layers": 1},
        # Batch transcription: 32 half-minute utterances through two layers of the stack.
        {"name": "2 layers, 32 x 30 s", "kind": "layer", "precision": "int8", "rows": 12000, "utterances": 32,
         "layers": 2},
        # The first, strided block of the wide encoder over a minute (50 frames per second there), odd.
        {"name": "strided block, 3001 frames", "kind": "block", "precision": "int8", "rows": 3001, "utterances": 1,
         "strided": True},
        # The same encoder's self-conditioning after its two strided blocks.
        {"name": "self-conditioning, 60 s", "kind": "conditioning", "rows": 750},
        # A feed-forward module of a pack stored in half precision.
        {"name": "f16 feed-forward, 60 s", "kind": "feedforward", "precision": "f16", "exact": False, "rows": 750},
        # The same of an int8 pack in the mode that gives the reference's bits, on a short streaming chunk.
        {"name": "exact int8 feed-forward, 93", "kind": "feedforward", "precision": "int8", "exact": True,
         "rows": 93},
        # The attention core of a layer over half a minute.
        {"name": "attention, 375 frames", "kind": "attention", "rows": 375},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "predict", "decode", "layer", "block", "conditioning", "feedforward", "attention"])
    if kind == "gemv":
        precision = rng.choice(["int8", "q8_0"])
        if rng.random() < 0.5:
            k, n = rng.choice([(640, 8198), (640, 2560), (1280, 2560), (640, 640)])
        else:  # k in whole Q8_0 blocks, the odd sizes in n
            k, n = 32 * rng.randint(4, 60), _log(rng, 48, 16384)
        return {"kind": kind, "precision": precision, "m": _log(rng, 1, 16), "k": k, "n": n}
    if kind == "predict":
        return {"kind": kind, "precision": rng.choice(["int8", "q8_0"]), "rows": rng.randint(1, 12)}
    if kind == "decode":
        streams = rng.choice([1, 1, 2, 3, 4, 6, 8])
        precision = rng.choice(["int8", "q8_0"]) if streams == 1 else "int8"
        return {"kind": kind, "precision": precision, "streams": streams,
                "frames": _log(rng, 25, 750 if streams <= 2 else 400)}
    if kind == "layer":
        utterances = rng.choice([1, 1, 1, 2, 3, 8, 16, 32])
        rows = utterances * _log(rng, max(8, 32 // utterances), min(7500, 12000 // utterances))
        layers = 1 if rows < 400 else rng.choice([1, 2])
        return {"kind": kind, "precision": rng.choice(["int8", "int8", "q8_0"]), "rows": rows,
                "utterances": utterances, "layers": layers}
    if kind == "block":
        utterances = rng.choice([1, 1, 1, 2, 4])
        return {"kind": kind, "precision": rng.choice(["int8", "int8", "q8_0"]), "strided": rng.random() < 0.5,
                "rows": utterances * _log(rng, 40, 6000 // utterances), "utterances": utterances}
    if kind == "conditioning":
        return {"kind": kind, "rows": _log(rng, 20, 1500)}
    if kind == "feedforward":
        precision = rng.choice(["f32", "f16", "bf16", "int8", "q8_0"])
        exact_mode = precision in ("int8", "q8_0")
        return {"kind": kind, "precision": precision, "exact": exact_mode, "rows": _log(rng, 1, 1000)}
    return {"kind": kind, "rows": _log(rng, 16, 900)}


# ------------------------------------------------------------------------------- inputs from a seed

class _Source:
    """Tensors drawn on the GPU from one seed, in the order asked for."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed) * 1000003 + 17)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device="cuda")

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda")

    def int8(self, *shape):
        return torch.randint(-127, 128, shape, generator=self.gen, device="cuda", dtype=torch.int8)

    def norm(self, n):
        return 1.0 + 0.1 * self.normal(n), 0.1 * self.normal(n)

    def matrix(self, precision, n, k, lo=0.001, hi=0.01):
        """A weight matrix: (its values [n, k], their scales or None) as the precision stores them."""
        if precision == "int8":
            return self.int8(n, k), lo + (hi - lo) * self.uniform(n)
        if precision == "q8_0":  # scales exact in half precision, one per 32 inputs
            return self.int8(n, k), (lo + (hi - lo) * self.uniform(n, k // 32)).half().float()
        w = self.normal(n, k) / math.sqrt(k)
        return w.to({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[precision]), None


def _panels(w):
    """[n, c] rows as panels of 16 rows, each panel's c columns one after another."""
    n, c = w.shape
    panels = -(-n // 16)
    pad = torch.zeros((panels * 16, c), dtype=w.dtype, device=w.device)
    pad[:n] = w
    return pad.view(panels, 16, c).transpose(1, 2).contiguous()


def _upload(kern, precision, matrix):
    values, scales = matrix
    n, k = values.shape
    if precision == "int8":
        scales = scales[:, None]
    return PackedWeights.from_device(kern, n, k, PRECISIONS[precision], _panels(values).view(torch.uint8).reshape(-1),
                                     None if scales is None else _panels(scales).reshape(-1))


def _wide(matrix):
    """The matrix's values in 64 bits, [n, k]."""
    values, scales = matrix
    w = values.double()
    if scales is not None:
        s = scales.double()
        w = w * (s[:, None] if s.dim() == 1 else s.repeat_interleave(32, dim=1))
    return w


_LAYER_MATS = {"ff1_in": (FF, D), "ff1_out": (D, FF), "qkv": (3 * D, D), "out": (D, D), "pw1": (2 * D, D),
               "pw2": (D, D), "ff2_in": (FF, D), "ff2_out": (D, FF)}
_LAYER_NORMS = ("norm_ff1", "norm_att", "norm_conv", "norm_ff2", "norm_out")
_BLOCK_MATS = {"ff1_up": (FF, D), "ff1_down": (D, FF), "qkv": (3 * D, D), "out": (D, D),
               "pw1": (2 * BLOCK_CHANNELS, D), "pw2": (D, BLOCK_CHANNELS), "ff2_up": (FF, D), "ff2_down": (D, FF)}
_BLOCK_NORMS = ("ff1_norm", "norm_att", "norm_conv", "ff2_norm", "norm_out")


def _data(case, seed):
    """The case's inputs as tensors, before any upload: what prepare and exact both start from."""
    src, kind = _Source(seed), case["kind"]
    p = case.get("precision", "int8")
    if kind == "gemv":
        return {"w": src.matrix(p, case["n"], case["k"]), "a": src.normal(case["m"], case["k"]).relu_(),
                "bias": src.normal(case["n"])}
    if kind in ("predict", "decode"):
        d = {"joint": src.matrix(p, VOCAB + len(DURATIONS), H), "joint_b": 0.5 * src.normal(VOCAB + len(DURATIONS)),
             "emb": 0.5 * src.normal(VOCAB, H), "lstm": [src.matrix(p, 4 * H, 2 * H, 0.0004, 0.0008) for _ in range(2)],
             "lstm_b": [0.1 * src.normal(4 * H) for _ in range(2)], "proj": src.matrix(p, H, H, 0.001, 0.003),
             "proj_b": 0.1 * src.normal(H)}
        if kind == "predict":
            d["tokens"] = torch.randint(0, VOCAB, (case["rows"],), generator=src.gen, device="cuda").tolist()
            d["states"] = 0.5 * src.normal(case["rows"], 4 * H)
            return d
        # A trained joint is sure of most frames: each row is turned towards one token (the blank for
        # a fifth of them) and one duration, about two frames on average as speech has them.
        joint = _wide(d["joint"]).float().relu_()
        shape = (case["streams"], case["frames"])
        tok = torch.randint(0, VOCAB - 1, shape, generator=src.gen, device="cuda")
        tok[src.uniform(*shape) < 0.2] = VOCAB - 1
        dur = 1 + torch.multinomial(torch.tensor([0.5, 0.3, 0.15, 0.05], device="cuda"), shape[0] * shape[1], True,
                                    generator=src.gen).view(shape)
        d["enc"] = (0.5 * src.normal(*shape, H) + joint[tok] + joint[VOCAB + dur]).contiguous()
        return d
    if kind in ("layer", "block"):
        mats, names = (_LAYER_MATS, _LAYER_NORMS) if kind == "layer" else (_BLOCK_MATS, _BLOCK_NORMS)
        channels, taps = (D, LAYER_TAPS) if kind == "layer" else (BLOCK_CHANNELS, BLOCK_TAPS)
        layers = []
        for _ in range(case.get("layers", 1)):
            m = {name: src.matrix(p, n, k) for name, (n, k) in mats.items()}
            layers.append({"mats": m, "norms": {name: src.norm(D) for name in names},
                           "biases": {name: 0.1 * src.normal(n) for name, (n, _) in mats.items() if name != "qkv"},
                           "dw_w": 0.3 * src.normal(taps, channels), "dw_b": 0.1 * src.normal(channels)})
        return {"layers": layers, "x": src.normal(case["rows"], D)}
    if kind == "conditioning":
        return {"head": src.matrix(p, BLOCK_VOCAB, D), "head_b": 0.1 * src.normal(BLOCK_VOCAB),
                "mid": src.matrix(p, D, BLOCK_VOCAB), "mid_b": 0.1 * src.normal(D), "x": src.normal(case["rows"], D)}
    if kind == "feedforward":
        return {"w_in": src.matrix(p, FF, D), "b_in": 0.1 * src.normal(FF), "w_out": src.matrix(p, D, FF),
                "b_out": 0.1 * src.normal(D), "h": src.normal(case["rows"], D), "x": src.normal(case["rows"], D)}
    t = case["rows"]
    return {"qkv": src.normal(t, 3 * D)}


# ----------------------------------------------------------------------------------- prepare and run

_stream = None


def _kernels(mode=telmo_amd.Kernels.FAST):
    """A context on the program's one stream, which is torch's current stream from the first call on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
        torch.cuda.synchronize()
    torch.cuda.set_stream(_stream)
    return telmo_amd.Kernels(0, stream=_stream.cuda_stream, mode=mode)


def prepare(case, seed):
    kern = _kernels(telmo_amd.Kernels.EXACT if case.get("exact") else telmo_amd.Kernels.FAST)
    kind, d, s = case["kind"], _data(case, seed), {"kind": case["kind"], "case": case, "kern": kern}
    p = case.get("precision", "int8")
    empty = lambda *shape: torch.empty(shape, device="cuda")  # noqa: E731
    if kind == "gemv":
        s.update(a=d["a"], w=_upload(kern, p, d["w"]), c=empty(case["m"], case["n"]), epi=Epilogue(bias=d["bias"]))
    elif kind in ("predict", "decode"):
        up = lambda m: _upload(kern, p, m)  # noqa: E731
        s["dec"] = dec = TdtDecoder(kern, H, VOCAB, DURATIONS, MAX_SYMBOLS, up(d["joint"]), d["joint_b"], d["emb"],
                                    [up(w) for w in d["lstm"]], d["lstm_b"], up(d["proj"]), d["proj_b"])
        if kind == "predict":
            s.update(tokens=d["tokens"], states0=d["states"], states=d["states"].clone(), preds=empty(case["rows"], H))
        else:  # every stream starts from the blank's prediction
            state0, pred0 = torch.zeros(1, 4 * H, device="cuda"), empty(1, H)
            dec.predict_rows([VOCAB - 1], state0, pred0)
            s.update(encs=list(d["enc"]), state0=state0, pred0=pred0,
                     states=[empty(1, 4 * H) for _ in range(case["streams"])],
                     preds=[empty(1, H) for _ in range(case["streams"])])
    elif kind == "layer":
        s["layers"] = [LayerWeights({name: _upload(kern, p, m) for name, m in w["mats"].items()}, w["norms"],
                                    w["dw_w"], w["dw_b"]) for w in d["layers"]]
        s.update(layer=ConformerLayer(kern, D, FF, LAYER_TAPS, case["rows"], EPS), x=d["x"])
    elif kind == "block":
        w = d["layers"][0]
        s["w"] = BlockWeights({name: _upload(kern, p, m) for name, m in w["mats"].items()}, w["biases"], w["norms"],
                              w["dw_w"], w["dw_b"], case["strided"])
        s.update(block=GraniteBlock(kern, D, FF, BLOCK_CHANNELS, BLOCK_TAPS, case["rows"], EPS), x0=d["x"],
                 x=d["x"].clone(), out=empty(case["rows"], D) if case["strided"] else None)
    elif kind == "conditioning":
        s.update(head=_upload(kern, p, d["head"]), head_b=d["head_b"], mid=_upload(kern, p, d["mid"]),
                 mid_b=d["mid_b"], x0=d["x"], x=d["x"].clone(), logits=empty(case["rows"], BLOCK_VOCAB))
    elif kind == "feedforward":
        s.update(w_in=_upload(kern, p, d["w_in"]), w_out=_upload(kern, p, d["w_out"]), h=d["h"], x0=d["x"],
                 x=d["x"].clone(), hid=empty(case["rows"], FF), epi_in=Epilogue(bias=d["b_in"], act=Act.SILU),
                 epi_out=Epilogue(bias=d["b_out"], scale=0.5, accumulate=True))
    else:
        t = case["rows"]
        tp = -(-t // 16) * 16  # a view's rows hold whole panels of 16 columns
        keys = torch.zeros(D, tp, device="cuda")
        keys[:, :t] = d["qkv"][:, D:2 * D].t()
        s.update(qkv=d["qkv"], keys=keys, probs=torch.zeros(HEADS, t, tp, device="cuda"), out=empty(t, D),
                 scale=Epilogue(scale=1.0 / math.sqrt(D // HEADS)))
    return s


def run(s):
    kern, case, kind = s["kern"], s["case"], s["kind"]
    if kind == "gemv":
        kern.linear_device(s["a"], case["m"], s["w"], s["c"], s["epi"])
        return s["c"]
    if kind == "predict":  # a beam search keeps the states its hypotheses came from
        s["states"].copy_(s["states0"])
        s["dec"].predict_rows(s["tokens"], s["states"], s["preds"])
        return s["states"], s["preds"]
    if kind == "decode":
        for state, pred in zip(s["states"], s["preds"]):
            state.copy_(s["state0"])
            pred.copy_(s["pred0"])
        if case["streams"] == 1:
            got = [s["dec"].decode(s["encs"][0], s["states"][0], s["preds"][0])]
        else:
            got = s["dec"].decode_streams(s["encs"], s["states"], s["preds"])
        emitted = np.full((len(got), case["frames"] * MAX_SYMBOLS, 3), -1, np.int32)  # the most there can be
        for i, (tokens, _, _) in enumerate(got):
            if tokens:
                emitted[i, :len(tokens)] = tokens
        return {"tokens": emitted, "states": s["states"], "preds": s["preds"]}
    if kind == "layer":  # in place: the next pass is the next layers of a stack
        s["layer"].run_stack(s["x"], case["rows"], s["layers"], utterances=case["utterances"])
        return s["x"]
    if kind == "block":
        s["x"].copy_(s["x0"])
        y, n = s["block"].forward(s["x"], case["rows"], s["w"], utterances=case["utterances"], out=s["out"])
        return y[:n]
    if kind == "conditioning":
        s["x"].copy_(s["x0"])
        self_conditioning(kern, s["x"], case["rows"], s["head"], s["head_b"], s["mid"], s["mid_b"], s["logits"])
        return s["x"], s["logits"]
    if kind == "feedforward":
        t = case["rows"]
        s["x"].copy_(s["x0"])
        kern.linear_device(s["h"], t, s["w_in"], s["hid"], s["epi_in"])
        kern.linear_device(s["hid"], t, s["w_out"], s["x"], s["epi_out"])
        return s["x"], s["hid"]
    t, dh = case["rows"], D // HEADS
    qkv, keys, probs, out = s["qkv"], s["keys"], s["probs"], s["out"]
    tp, span = probs.shape[2], (t - 1) * 3 * D + dh
    for i in range(HEADS):
        kern.matmul_rowmajor_device(qkv[:, i * dh:(i + 1) * dh], 3 * D, t, keys[i * dh:(i + 1) * dh], dh, t, tp,
                                    probs[i], tp, s["scale"], a_len=span)
    kern.softmax_device(probs, tp, HEADS * t, t)
    for i in range(HEADS):
        kern.matmul_rowmajor_device(probs[i], tp, t, qkv[:, 2 * D + i * dh:2 * D + (i + 1) * dh], t, dh, 3 * D,
                                    out[:, i * dh:(i + 1) * dh], D, a_len=t * tp, b_len=span,
                                    c_len=(t - 1) * D + dh)
    return out, probs


# ------------------------------------------------------------------------------------- in 64 bits

def _silu(v):
    return v * torch.sigmoid(v)


def _norm(x, gb):
    g, b = (v.double() for v in gb)
    c = x - x.mean(1, keepdim=True)
    return c / torch.sqrt((c * c).mean(1, keepdim=True) + EPS) * g + b


def _conv(u, w, utterances, stride):
    """The depthwise convolution of each utterance's rows, frames 0, stride, 2 stride, ..., then SiLU."""
    taps, channels = w["dw_w"].shape
    frames = u.shape[0] // utterances
    rows = frames // stride
    padded = torch.zeros(utterances, frames + 2 * (taps // 2), channels, dtype=torch.float64, device="cuda")
    padded[:, taps // 2:taps // 2 + frames] = u.view(utterances, frames, channels)
    y = w["dw_b"].double().expand(utterances, rows, channels).clone()
    for j in range(taps):
        y += padded[:, j:j + (rows - 1) * stride + 1:stride] * w["dw_w"][j].double()
    return _silu(y).reshape(utterances * rows, channels)


def _exact_encoder(x, w, case, strided, names):
    """One layer or block: names are the (norm, in, out) of its two feed-forward modules."""
    biases = w["biases"] if case["kind"] == "block" else {}

    def product(a, name):
        y = a @ _wide(w["mats"][name]).t()
        return y + biases[name].double() if name in biases else y

    def feed_forward(y, norm, w_in, w_out):
        return y + 0.5 * product(_silu(product(_norm(y, w["norms"][norm]), w_in)), w_out)

    x = feed_forward(x, *names[0])
    x = x + product(product(_norm(x, w["norms"]["norm_att"]), "qkv")[:, 2 * D:], "out")
    a, b = product(_norm(x, w["norms"]["norm_conv"]), "pw1").chunk(2, dim=1)
    u = _conv(a * torch.sigmoid(b), w, case["utterances"], 2 if strided else 1)
    if strided:
        frames = x.shape[0] // case["utterances"]
        pairs = x.view(case["utterances"], frames, D)[:, :frames // 2 * 2].reshape(-1, 2, D)
        x = (pairs[:, 0] + pairs[:, 1]) / 2
    x = x + product(u, "pw2")
    x = feed_forward(x, *names[1])
    return _norm(x, w["norms"]["norm_out"])


def _exact_predict(d, wide, tokens, states):
    """predict_rows in 64 bits: (states, predictions) after the tokens."""
    x, out = d["emb"].double()[tokens], []
    for i in range(2):
        h, c = states[:, 2 * i * H:(2 * i + 1) * H], states[:, (2 * i + 1) * H:(2 * i + 2) * H]
        gi, gf, gg, go = (torch.cat([x, h], 1) @ wide["lstm"][i].t() + d["lstm_b"][i].double()).chunk(4, dim=1)
        c = torch.sigmoid(gf) * c + torch.sigmoid(gi) * torch.tanh(gg)
        x = torch.sigmoid(go) * torch.tanh(c)
        out += [x, c]
    return torch.cat(out, 1), x @ wide["proj"].t() + d["proj_b"].double()


def _exact_decode(d, wide, enc):
    state = torch.zeros(1, 4 * H, dtype=torch.float64, device="cuda")
    state, pred = _exact_predict(d, wide, [VOCAB - 1], state)
    t = on_frame = 0
    while t < enc.shape[0]:
        logits = wide["joint"] @ torch.relu(enc[t].double() + pred[0]) + d["joint_b"].double()
        token, step = torch.stack([logits[:VOCAB].argmax(), logits[VOCAB:].argmax()]).tolist()
        step = DURATIONS[step]
        if token == VOCAB - 1:
            t, on_frame = t + max(step, 1), 0
            continue
        state, pred = _exact_predict(d, wide, [token], state)
        on_frame = 0 if step else on_frame + 1
        t += step
        if on_frame >= MAX_SYMBOLS:
            t, on_frame = t + 1, 0
    return state, pred


def exact(case, seed):
    kind, d = case["kind"], _data(case, seed)
    if kind == "gemv":
        return d["a"].double() @ _wide(d["w"]).t() + d["bias"].double()
    if kind in ("predict", "decode"):
        wide = {"joint": _wide(d["joint"]), "lstm": [_wide(w) for w in d["lstm"]], "proj": _wide(d["proj"])}
        if kind == "predict":
            return _exact_predict(d, wide, d["tokens"], d["states"].double())
        ends = [_exact_decode(d, wide, enc) for enc in d["enc"]]
        return {"tokens": None, "states": [e[0] for e in ends], "preds": [e[1] for e in ends]}
    if kind == "layer":
        x = d["x"].double()
        for w in d["layers"]:
            x = _exact_encoder(x, w, case, False, (("norm_ff1", "ff1_in", "ff1_out"), ("norm_ff2", "ff2_in", "ff2_out")))
        return x
    if kind == "block":
        return _exact_encoder(d["x"].double(), d["layers"][0], case, case["strided"],
                              (("ff1_norm", "ff1_up", "ff1_down"), ("ff2_norm", "ff2_up", "ff2_down")))
    if kind == "conditioning":
        x = d["x"].double()
        probs = torch.softmax(x @ _wide(d["head"]).t() + d["head_b"].double(), 1)
        return x + probs @ _wide(d["mid"]).t() + d["mid_b"].double(), probs
    if kind == "feedforward":
        hid = _silu(d["h"].double() @ _wide(d["w_in"]).t() + d["b_in"].double())
        return d["x"].double() + 0.5 * (hid @ _wide(d["w_out"]).t() + d["b_out"].double()), hid
    t, dh = case["rows"], D // HEADS
    q, k, v = (m.double().reshape(t, HEADS, dh).transpose(0, 1).contiguous() for m in d["qkv"].split(D, dim=1))
    probs = torch.softmax(torch.stack([q[i] @ k[i].t() for i in range(HEADS)]) / math.sqrt(dh), 2)
    out = torch.stack([probs[i] @ v[i] for i in range(HEADS)]).transpose(0, 1).reshape(t, D)
    padded = torch.zeros(HEADS, t, -(-t // 16) * 16, dtype=torch.float64, device="cuda")
    padded[:, :, :t] = probs
    return out, padded


# -------------------------------------------------------------------------------- work and tolerance

def work(case):
    """Each weight, input and output once; 2 operations per multiply-add of the products."""
    kind, wb = case["kind"], VALUE_BYTES[case.get("precision", "int8")]
    if kind == "gemv":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": wb * n * k + 4 * (n + m * k + m * n), "flops": 2 * m * n * k}
    net = 2 * (4 * H * 2 * H) + H * H
    if kind == "predict":
        r = case["rows"]
        return {"bytes": wb * net + 4 * r * (H + 2 * 4 * H + H), "flops": 2 * r * net}
    if kind == "decode":
        # The weights once (they fit on the chip); about 0.6 steps and 0.5 tokens per frame.
        joint, frames = (VOCAB + len(DURATIONS)) * H, case["streams"] * case["frames"]
        return {"bytes": wb * (net + joint) + 4 * frames * H, "flops": 2 * frames * (0.6 * joint + 0.5 * net)}
    if kind in ("layer", "block"):
        mats, rows = (_LAYER_MATS if kind == "layer" else _BLOCK_MATS), case["rows"]
        half = case.get("strided", False)
        out = case["utterances"] * (rows // case["utterances"] // 2) if half else rows
        late = ("pw2", "ff2_up", "ff2_down")
        flops = sum(2 * n * k * (out if name in late else rows) for name, (n, k) in mats.items())
        weights = sum(n * k for n, k in mats.values())
        layers = case.get("layers", 1)
        return {"bytes": layers * wb * weights + 4 * D * (rows + out), "flops": layers * flops}
    if kind == "conditioning":
        t = case["rows"]
        return {"bytes": 2 * BLOCK_VOCAB * D + 4 * t * (2 * D + BLOCK_VOCAB), "flops": 4 * t * BLOCK_VOCAB * D}
    if kind == "feedforward":
        t = case["rows"]
        return {"bytes": 2 * wb * FF * D + 4 * t * (3 * D + FF), "flops": 4 * t * FF * D}
    t = case["rows"]
    return {"bytes": 4 * t * (4 * D + HEADS * t), "flops": 4 * t * t * D}


def tolerance(case):
    """About four times the distance from exact() that the path shows. The fast path keeps 15 bits of
    each activation (its error is 1e-4 of a row's norm on these inputs) and a layer adds up several
    products; the exact mode and the other precisions sum in f32."""
    return {"rel": {"gemv": 2e-4, "predict": 3e-4, "decode": 5e-4, "layer": 8e-4, "block": 8e-4,
                    "conditioning": 1e-3, "feedforward": 5e-6, "attention": 5e-6}[case["kind"]]}
