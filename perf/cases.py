"""The work that is timed: what programs built on this framework have it do, each case through
the public layer API on one stream with tensors that stay on the GPU.

Every case names its entry point in "op"; sizes are those of the HTDemucs-shaped workloads of
bench.py and tests/ (7.8 s stereo chunks of 343 980 samples, 60 s of audio, widths 48..768 and
384 / 512) or generic, and lengths that are no multiple of anything. `draw` gives more cases of
the same operations over the ranges from a few rows or milliseconds of audio up to those sizes.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch
import torch.nn.functional as F

from metalaudio_amd import _lib, nn

CHUNK = 343980  # samples of a 7.8 s chunk at 44.1 kHz
TIME_CHANNELS = [2, 48, 96, 192, 384]
SEP_CHANNELS = [48, 96, 192, 384, 768]
# Squared-window sums below this are raised to it, so that the first and last samples of a signal,
# which hardly any window weight covers, fade instead of dividing rounding errors by almost nothing.
WINDOW_FLOOR = 1e-3


# ------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # One second of stereo audio through a model's first stage (Sequential of Conv1D 2->48
        # k8 s4, GroupNorm(1), GELU): the smallest call, as a streaming front end makes it.
        {"name": "conv_front_1s", "op": "conv_front", "batch": 1, "length": 44100},
        # A short sequence through a transformer's first feed-forward map with its GELU: small
        # batches of frames, where a launch and the first loads are most of the time.
        {"name": "linear_gelu_short", "op": "linear", "rows": 67, "fin": 384, "fout": 1536,
         "act": "gelu", "precision": "f32"},
        # A wide map and its LayerNorm over a full sequence (Sequential of Linear, LayerNorm).
        {"name": "linear_layernorm", "op": "linear_ln", "rows": 2048, "fin": 512, "fout": 2048},
        # The half-precision linear layer on bf16 input, the same size.
        {"name": "linear_bf16", "op": "linear", "rows": 2048, "fin": 512, "fout": 2048,
         "act": "none", "precision": "bf16"},
        # Cross-attention between two sequences of odd lengths, head dim 64.
        {"name": "cross_attention", "op": "attention", "batch": 2, "embed": 512, "heads": 8,
         "sq": 777, "sk": 1501, "cross": True},
        # The whole cross-domain bottleneck on four chunks (5 layers, head dim 48): the largest.
        {"name": "cross_transformer", "op": "cross_transformer", "batch": 4, "time": 1344,
         "freq": 2688, "layers": 5},
        # The whole time-branch encoder (4 levels with rewrite and GLU) on one 7.8 s chunk.
        {"name": "time_encoder", "op": "time_encoder", "batch": 1, "length": CHUNK},
        # One level of the time-branch decoder with its skip (8 groups), an odd length.
        {"name": "time_decoder", "op": "time_decoder", "batch": 1, "cin": 192, "cout": 96,
         "length": 5375, "groups": 8},
        # One level of the frequency branch's encoder at a chunk's spectrogram.
        {"name": "freq_encoder", "op": "freq_encoder", "batch": 1, "cin": 48, "cout": 96,
         "height": 1032, "width": 168},
        # One level of its decoder with the skip, at a width that is no multiple of 4.
        {"name": "freq_decoder", "op": "freq_decoder", "batch": 1, "cin": 192, "cout": 96,
         "height": 258, "width": 42},
        # A stereo chunk to its spectrogram and back (bin-major, as the frequency branch has it).
        {"name": "stft_roundtrip", "op": "stft", "batch": 2, "length": CHUNK, "nfft": 4096,
         "layout": "bins"},
        # 60 s of audio through the 5-level separation model in overlapping 30 s segments.
        {"name": "separate_60s", "op": "separate", "frames": 60 * 44100, "segment": 30 * 44100,
         "overlap": 2 * 44100},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["conv_front", "linear", "linear", "linear_ln", "attention", "attention",
                     "cross_transformer", "time_encoder", "time_decoder", "freq_encoder",
                     "freq_decoder", "stft", "separate"])
    if op == "conv_front":
        return {"op": op, "batch": rng.choice([1, 1, 2]), "length": _log(rng, 2000, CHUNK)}
    if op == "linear":
        prec = rng.choice(["f32", "f32", "f32", "bf16"])
        fin, fout = rng.choice([(384, 384), (384, 1152), (384, 1536), (1536, 384), (512, 2048),
                                (2048, 512), (512, 1536), (128, 96), (320, 200)])
        return {"op": op, "rows": _log(rng, 1, 10752), "fin": fin, "fout": fout,
                "act": rng.choice(["none", "none", "gelu", "relu"]), "precision": prec}
    if op == "linear_ln":
        fin, fout = rng.choice([(384, 384), (512, 2048), (1536, 384), (2048, 512), (384, 1000)])
        return {"op": op, "rows": _log(rng, 4, 8192), "fin": fin, "fout": fout}
    if op == "attention":
        cross = rng.random() < 0.5
        sq = _log(rng, 24, 2688)
        return {"op": op, "batch": rng.choice([1, 1, 2, 4]), "embed": rng.choice([384, 512]),
                "heads": 8, "sq": sq, "sk": _log(rng, 24, 2688) if cross else sq, "cross": cross}
    if op == "cross_transformer":
        return {"op": op, "batch": rng.choice([1, 2, 4]), "time": _log(rng, 40, 1344),
                "freq": _log(rng, 80, 2688), "layers": rng.choice([2, 3, 5])}
    if op == "time_encoder":
        return {"op": op, "batch": rng.choice([1, 1, 2]), "length": _log(rng, 6000, CHUNK)}
    if op == "time_decoder":
        i = rng.randrange(4)
        cout = TIME_CHANNELS[i]
        return {"op": op, "batch": rng.choice([1, 1, 2]), "cin": TIME_CHANNELS[i + 1],
                "cout": cout, "length": max(33, _log(rng, 300, CHUNK // 4) >> (2 * i)),
                "groups": min(8, cout)}
    if op in ("freq_encoder", "freq_decoder"):
        i = rng.randrange(4)
        lo, hi = TIME_CHANNELS[i], TIME_CHANNELS[i + 1]
        enc = op == "freq_encoder"
        h = max(12, _log(rng, 200, 2064) >> (i if enc else i + 1))
        w = max(6, _log(rng, 40, 336) >> (i if enc else i + 1))
        return {"op": op, "batch": 1, "cin": lo if enc else hi, "cout": hi if enc else lo,
                "height": h, "width": w}
    if op == "stft":
        nfft = rng.choice([512, 1024, 2048, 4096])
        return {"op": op, "batch": rng.choice([1, 2]), "length": _log(rng, 2 * nfft, CHUNK),
                "nfft": nfft, "layout": rng.choice(["bins", "frames"])}
    n = _log(rng, 3 * 44100, 60 * 44100)
    seg = min(n, _log(rng, 3 * 44100, 30 * 44100))
    return {"op": op, "frames": n, "segment": seg, "overlap": seg // 15}


# ------------------------------------------------------------------ parameters, from a seed alone
class _Rand:
    """Seeded float32 host tensors, drawn in a fixed order."""

    def __init__(self, case, seed):
        text = ",".join(f"{k}={v}" for k, v in sorted(case.items()) if k != "name")
        mix = sum((i + 1) * ord(c) for i, c in enumerate(text))
        self.g = torch.Generator().manual_seed(int(seed) * 1000003 + mix)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g).mul_(std)

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.g).mul_(2).sub_(1)

    def bias(self, n):
        return self.normal(n, std=0.05)

    def affine(self, n):
        return 1 + self.normal(n, std=0.1), self.normal(n, std=0.1)


def _conv_params(r, cout, cin, *k):
    return r.normal(cout, cin, *k, std=math.sqrt(2 / (cin * math.prod(k)))), r.bias(cout)


def _linear_params(r, fout, fin):
    return r.normal(fout, fin, std=1 / math.sqrt(fin)), r.bias(fout)


def _mha_params(r, E):
    wi, bi = _linear_params(r, 3 * E, E)
    wo, bo = _linear_params(r, E, E)
    return {"in_proj_weight": wi, "in_proj_bias": bi, "out_proj_weight": wo, "out_proj_bias": bo}


def _sep_levels(L):
    chans = [2] + SEP_CHANNELS
    return [(chans[i], chans[i + 1]) for i in range(5)]


def _data(case, seed):
    """The inputs and parameters of a case as float32 host tensors."""
    r, op = _Rand(case, seed), case["op"]
    d = {}
    if op == "conv_front":
        d["x"] = r.uniform(case["batch"], 2, case["length"])
        d["conv"] = _conv_params(r, 48, 2, 8)
        d["norm"] = r.affine(48)
    elif op in ("linear", "linear_ln"):
        d["x"] = r.normal(case["rows"], case["fin"])
        d["lin"] = _linear_params(r, case["fout"], case["fin"])
        if op == "linear_ln":
            d["norm"] = r.affine(case["fout"])
    elif op == "attention":
        E = case["embed"]
        d["q"] = r.normal(case["batch"], case["sq"], E)
        d["kv"] = r.normal(case["batch"], case["sk"], E) if case["cross"] else d["q"]
        d["mha"] = _mha_params(r, E)
    elif op == "cross_transformer":
        E, Hd, B = 384, 1536, case["batch"]
        d["t"], d["f"] = r.normal(B, case["time"], E), r.normal(B, case["freq"], E)
        p = d["p"] = {}
        for i in range(case["layers"]):
            for br in ("time", "freq"):
                pre = f"layers.{i}.{br}."
                for n in ("norm1", "norm2", "norm3") if i % 2 else ("norm1", "norm2"):
                    p[pre + n + ".weight"], p[pre + n + ".bias"] = r.affine(E)
                for k, v in _mha_params(r, E).items():
                    p[pre + "attn." + k] = v
                p[pre + "linear1.weight"], p[pre + "linear1.bias"] = _linear_params(r, Hd, E)
                p[pre + "linear2.weight"], p[pre + "linear2.bias"] = _linear_params(r, E, Hd)
                # LayerScale as training leaves it (it starts at 1e-4): updates that count
                p[pre + "gamma_1.scale"] = 0.2 + r.normal(E, std=0.05)
                p[pre + "gamma_2.scale"] = 0.2 + r.normal(E, std=0.05)
    elif op == "time_encoder":
        d["x"] = r.uniform(case["batch"], 2, case["length"])
        d["levels"] = []
        for ci, co in zip(TIME_CHANNELS[:-1], TIME_CHANNELS[1:]):
            d["levels"].append(_conv_params(r, co, ci, 8) + r.affine(co) +
                               _conv_params(r, 2 * co, co, 1))
    elif op == "time_decoder":
        ci, co = case["cin"], case["cout"]
        # what the level below and the encoder hand over: GELU and GLU outputs, mostly small
        d["x"] = F.gelu(r.normal(case["batch"], ci, case["length"]))
        d["skip"] = r.normal(case["batch"], ci, case["length"], std=0.5)
        d["w"] = r.normal(2 * ci, co, 8, std=math.sqrt(1 / (2 * ci)))
        d["b"] = r.bias(co)
        d["norm"] = r.affine(co)
    elif op in ("freq_encoder", "freq_decoder"):
        ci, co, B, H, W = (case[k] for k in ("cin", "cout", "batch", "height", "width"))
        d["x"] = r.normal(B, ci, H, W) if ci <= 2 else F.gelu(r.normal(B, ci, H, W))
        if op == "freq_decoder":
            d["skip"] = F.gelu(r.normal(B, ci, H, W))
            d["w"] = r.normal(2 * ci, co, 3, 3, std=math.sqrt(2 / (2 * ci * 9 / 4)))
        else:
            d["w"] = r.normal(co, ci, 3, 3, std=math.sqrt(2 / (9 * ci)))
        d["b"] = r.bias(co)
        d["norm"] = r.affine(co)
    elif op == "stft":
        d["x"] = r.uniform(case["batch"], case["length"])
    else:
        # a 60 s programme needs no 60 s of fresh noise: 4 s of it repeated with a slow gain
        n = case["frames"]
        base = r.uniform(min(n, 4 * 44100), 2)
        x = base.repeat(-(-n // base.shape[0]), 1)[:n]
        x *= (0.6 + 0.4 * torch.cos(torch.arange(n) * (2 * math.pi / 300007.0)))[:, None]
        d["x"] = x.contiguous()
        d["enc"] = [_conv_params(r, co, ci, 8) + r.affine(co) for ci, co in _sep_levels(n)]
        d["dec"] = []
        for ci, co in reversed(_sep_levels(n)):
            d["dec"].append((r.normal(2 * co, ci, 8, std=math.sqrt(1 / (2 * co))), r.bias(ci)) +
                            r.affine(ci))
        d["heads"] = [(r.normal(2, 2, 1), r.bias(2)) for _ in range(4)]
    return d


# --------------------------------------------------------------------------- the framework's side
_dev = _stream = None


def _context():
    """The one device and stream a program keeps."""
    global _dev, _stream
    if _dev is None:
        _dev = nn.AudioDevice(0)
        _stream = nn.Stream(_dev)
    return _dev, _stream


class _View:
    def __init__(self, t, owner):
        self.keep = (t, owner)  # the memory lives as long as a torch tensor over it does
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": "<f4", "strides": None,
                                         "data": (t.device_ptr, False), "version": 2}


def _torch(t, owner=None):
    """The framework's fp32 tensor as a torch tensor over the same memory."""
    return torch.as_tensor(_View(t, owner), device="cuda")


def _tensor(dev, x, dtype="f32"):
    return nn.Tensor.from_numpy(dev, x.numpy(), dtype=dtype)


def _freq_groups(case):
    return min(8, case["cin"], case["cout"]) if case["cin"] <= 2 else min(8, case["cout"])


def prepare(case, seed):
    dev, stream = _context()
    d, op = _data(case, seed), case["op"]
    s = {"op": op, "stream": stream}
    if op in ("conv_front", "linear_ln"):
        m = nn.Sequential(dev)
        if op == "conv_front":
            conv = nn.DynamicConv1D(dev, 2, 48, 8, stride=4)
            conv.load_weights(*d["conv"])
            norm = nn.GroupNorm(dev, 1, 48)
            layers = [conv, norm, nn.GELU(dev, (48, 0))]
        else:
            lin = nn.Linear(dev, case["fin"], case["fout"])
            lin.load_weights(*d["lin"])
            norm = nn.LayerNorm(dev, case["fout"])
            layers = [lin, norm]
        norm.load_parameters(*d["norm"])
        for layer in layers:
            m.add_unchecked(layer)
        m.build()
        s.update(model=m, x=_tensor(dev, d["x"]), out=None)
        return s
    if op == "linear":
        bf = case["precision"] == "bf16"
        m = nn.Linear(dev, case["fin"], case["fout"], activation=case["act"],
                      precision=case["precision"])
        m.load_weights(*d["lin"])
        s["args"] = (_tensor(dev, d["x"], "bf16" if bf else "f32"),)
        outs = [nn.Tensor(dev, (case["rows"], case["fout"]))]
        s["call"] = m.forward
    elif op == "attention":
        m = nn.MultiHeadAttention(dev, case["embed"], case["heads"])
        m.load_weights(*(d["mha"][k] for k in ("in_proj_weight", "in_proj_bias",
                                               "out_proj_weight", "out_proj_bias")))
        s["args"] = (_tensor(dev, d["q"]),)
        if case["cross"]:
            s["args"] += (_tensor(dev, d["kv"]),)
        outs = [nn.Tensor(dev, d["q"].shape)]
        s["call"] = m.forward_cross if case["cross"] else m.forward
    elif op == "cross_transformer":
        m = nn.CrossTransformerEncoder(dev, 384, 8, 1536, case["layers"])
        m.load_state(d["p"])
        s["args"] = (_tensor(dev, d["t"]), _tensor(dev, d["f"]))
        outs = [nn.Tensor(dev, d["t"].shape), nn.Tensor(dev, d["f"].shape)]
        s["call"] = m.forward_cross
    elif op == "time_encoder":
        blocks, x, outs = [], _tensor(dev, d["x"]), []
        shape = x.shape
        for (ci, co), lv in zip(zip(TIME_CHANNELS[:-1], TIME_CHANNELS[1:]), d["levels"]):
            b = nn.UNetEncoderBlock(dev, ci, co, 8, 4, 1, rewrite=True)
            b.load_weights(*lv)
            shape = b.infer_output_shape(shape)
            outs.append(nn.Tensor(dev, shape))
            blocks.append(b)
        m = list(zip(blocks, [x] + outs[:-1], outs))
        s["args"] = ()
    elif op == "time_decoder":
        m = nn.UNetDecoderBlock(dev, case["cin"], case["cin"], case["cout"], 8, 4, case["groups"])
        m.load_weights(d["w"], d["b"], *d["norm"])
        s["args"] = (_tensor(dev, d["x"]), _tensor(dev, d["skip"]))
        outs = [nn.Tensor(dev, m.infer_output_shape(d["x"].shape))]
        s["call"] = m.forward
    elif op == "freq_encoder":
        m = nn.FreqUNetEncoderBlock2D(dev, case["cin"], case["cout"], 3, 2, _freq_groups(case))
        m.load_weights(d["w"], d["b"], *d["norm"])
        s["args"] = (_tensor(dev, d["x"]),)
        outs = [nn.Tensor(dev, m.infer_output_shape(d["x"].shape))]
        s["call"] = m.forward
    elif op == "freq_decoder":
        m = nn.FreqUNetDecoderBlock2D(dev, case["cin"], case["cin"], case["cout"], 3, 2,
                                      _freq_groups(case))
        m.load_weights(d["w"], d["b"], *d["norm"])
        s["args"] = (_tensor(dev, d["x"]), _tensor(dev, d["skip"]))
        outs = [nn.Tensor(dev, m.infer_output_shape(d["x"].shape))]
        s["call"] = m.forward
    elif op == "stft":
        m = nn.STFT(dev, case["nfft"])
        nf, bins = m.frame_count(case["length"]), case["nfft"] // 2 + 1
        shape = (nf, bins) if case["layout"] == "frames" else (bins, nf)
        s["args"] = (_tensor(dev, d["x"]),)
        s["layout"] = 0 if case["layout"] == "frames" else 1
        outs = [nn.Tensor(dev, (case["batch"],) + shape), nn.Tensor(dev, (case["batch"],) + shape),
                nn.Tensor(dev, (case["batch"], m.output_length(nf)))]
    else:
        m = nn.Separator(dev)
        for i, (w, b, g, be) in enumerate(d["enc"]):
            m.load_state({f"time_encoder.{i}": {"conv.weight": w, "conv.bias": b,
                                                "norm.weight": g, "norm.bias": be}})
        for i, (w, b, g, be) in enumerate(d["dec"]):
            m.load_state({f"time_decoder.{i}": {"conv_transpose.weight": w,
                                                "conv_transpose.bias": b, "norm.weight": g,
                                                "norm.bias": be}})
        for i, (w, b) in enumerate(d["heads"]):
            m.load_state({f"output_heads.{i}": {"weight": w, "bias": b}})
        x = _tensor(dev, d["x"].reshape(-1))
        outs = [nn.Tensor(dev, (4, x.shape[0]))]
        s["args"] = (x,)
        s["cut"] = (case["segment"], case["overlap"])
    s.update(model=m, outs=outs, views=[_torch(t) for t in outs])
    return s


def run(s):
    op, stream = s["op"], s["stream"]
    if op in ("conv_front", "linear_ln"):
        y = s["model"].forward(s["x"], stream)  # the model's own output buffer
        if s["out"] is None:
            s["out"] = _torch(y, s["model"])
        return s["out"]
    if op == "time_encoder":
        for block, x, y in s["model"]:
            block.forward(x, y, stream)
    elif op == "stft":
        # the C entry points, which take the caller's output tensors
        L, plan, (re, im, y) = _lib.lib(), s["model"].handle, s["outs"]
        _lib.check(L.mnn_stft_forward(plan, s["args"][0].handle, re.handle, im.handle, 1,
                                      s["layout"], stream.handle))
        _lib.check(L.mnn_stft_inverse(plan, re.handle, im.handle, 1, s["layout"],
                                      ctypes.c_float(WINDOW_FLOOR), y.handle, stream.handle))
    elif op == "separate":
        _lib.check(_lib.lib().mnn_separator_separate_long(
            s["model"].handle, s["args"][0].handle, s["outs"][0].handle, *s["cut"],
            stream.handle))
    else:
        s["call"](*s["args"], *s["outs"], stream)
    return s["views"]


# ------------------------------------------------------------------------------- bytes and flops
def _enc_len(L):
    return (L + 6 - 8) // 4 + 1


def _unet_pad(n):
    """(left padding, padded length): zeros to the next multiple of 4^5."""
    unit = 4 ** 5
    total = -(-n // unit) * unit - n
    return total // 2, n + total


def _segments(case):
    n, seg, ov = case["frames"], case["segment"], case["overlap"]
    if seg <= 0 or seg >= n:
        return [(0, n)]
    out, start = [], 0
    while True:
        out.append((start, min(start + seg, n)))
        if start + seg >= n:
            return out
        start += seg - ov


def work(case):
    op = case["op"]
    if op == "conv_front":
        B, L = case["batch"], case["length"]
        lo = (L - 8) // 4 + 1
        return {"bytes": 4.0 * B * (2 * L + 48 * lo), "flops": 2.0 * B * 48 * lo * 16}
    if op in ("linear", "linear_ln"):
        M, K, N = case["rows"], case["fin"], case["fout"]
        e = 2.0 if case.get("precision") == "bf16" else 4.0
        return {"bytes": e * (M * K + N * K) + 4.0 * M * N, "flops": 2.0 * M * N * K}
    if op == "attention":
        B, E, Sq, Sk = case["batch"], case["embed"], case["sq"], case["sk"]
        rows = Sq + (Sk if case["cross"] else 0)
        return {"bytes": 4.0 * (B * E * (rows + Sq) + 4 * E * E),
                "flops": B * (2.0 * E * E * (2 * Sq + 2 * Sk) + 4.0 * Sq * Sk * E)}
    if op == "cross_transformer":
        B, E, Hd, n = case["batch"], 384, 1536, case["layers"]
        flops = 0.0
        for i in range(n):
            for a, b in ((case["time"], case["freq"]), (case["freq"], case["time"])):
                kv = b if i % 2 else a
                flops += B * (2.0 * E * E * (2 * a + 2 * kv) + 4.0 * a * kv * E +
                              4.0 * a * E * Hd)
        act = B * E * (case["time"] + case["freq"])
        return {"bytes": 4.0 * (2 * act + n * 2 * (4 * E * E + 2 * E * Hd)), "flops": flops}
    if op == "time_encoder":
        B, L, flops, byts = case["batch"], case["length"], 0.0, 0.0
        for ci, co in zip(TIME_CHANNELS[:-1], TIME_CHANNELS[1:]):
            lo = _enc_len(L)
            flops += B * lo * (2.0 * co * ci * 8 + 2.0 * 2 * co * co)
            byts += 4.0 * (B * (ci * L + co * lo) + co * ci * 8 + 2 * co * co)
            L = lo
        return {"bytes": byts, "flops": flops}
    if op == "time_decoder":
        B, ci, co, L = (case[k] for k in ("batch", "cin", "cout", "length"))
        return {"bytes": 4.0 * (B * (2 * ci * L + 4 * co * L) + 16 * ci * co),
                "flops": 2.0 * B * 2 * ci * co * 8 * L}
    if op == "freq_encoder":
        B, ci, co, H, W = (case[k] for k in ("batch", "cin", "cout", "height", "width"))
        ho, wo = (H - 1) // 2 + 1, (W - 1) // 2 + 1
        return {"bytes": 4.0 * (B * (ci * H * W + co * ho * wo) + 9 * ci * co),
                "flops": 2.0 * B * co * ci * 9 * ho * wo}
    if op == "freq_decoder":
        B, ci, co, H, W = (case[k] for k in ("batch", "cin", "cout", "height", "width"))
        return {"bytes": 4.0 * (B * (2 * ci * H * W + 4 * co * H * W) + 18 * ci * co),
                "flops": 2.0 * B * 2 * ci * co * 9 * H * W}
    if op == "stft":
        B, N, L = case["batch"], case["nfft"], case["length"]
        nf = (L - N) // (N // 4) + 1
        spec = 8.0 * B * nf * (N // 2 + 1)
        return {"bytes": 4.0 * B * (L + (nf - 1) * (N // 4) + N) + 2 * spec,
                "flops": 2 * B * nf * 2.5 * N * math.log2(N)}
    flops, byts = 0.0, 8.0 * case["frames"] * (1 + 4)
    for a, b in _segments(case):
        L = _unet_pad(b - a)[1]
        flops += 4 * 2.0 * 2 * 2 * L
        for ci, co in _sep_levels(L):
            L //= 4
            flops += 2.0 * ci * co * 8 * L + 2.0 * 2 * co * ci * 8 * L
            byts += 4.0 * (2 * co * L + 2 * 4 * ci * L)
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    # relative 2-norm errors of fp32 sums in another order, about four times the distance that the
    # fp32 path shows from 64-bit arithmetic
    return {"rel": {"conv_front": 1e-6, "linear": 4e-6, "linear_ln": 4e-6, "attention": 4e-6,
                    "cross_transformer": 2e-6, "time_encoder": 4e-6, "time_decoder": 4e-6,
                    "freq_encoder": 3e-6, "freq_decoder": 3e-6, "stft": 1e-6,
                    "separate": 4e-6}[case["op"]]}


# ------------------------------------------------------------------------- the same in 64 bits
def _f64(v):
    return v.to("cuda", torch.float64)


def _bf16(v):
    return v.to(torch.bfloat16).float()


def _gelu(x):
    return F.gelu(x, approximate="tanh")


def _affine_norm(x, groups, gamma, beta):
    B, C = x.shape[:2]
    y = x.reshape(B, groups, -1)
    v, m = torch.var_mean(y, dim=2, correction=0, keepdim=True)
    y = ((y - m) / torch.sqrt(v + 1e-5)).reshape(x.shape)
    shape = (1, C) + (1,) * (x.dim() - 2)
    return y * _f64(gamma).reshape(shape) + _f64(beta).reshape(shape)


def _layer_norm(x, gamma, beta):
    v, m = torch.var_mean(x, dim=-1, correction=0, keepdim=True)
    return (x - m) / torch.sqrt(v + 1e-5) * _f64(gamma) + _f64(beta)


def _linear64(x, w, b):
    return x.reshape(-1, x.shape[-1]).matmul(_f64(w).t()).reshape(*x.shape[:-1], -1) + _f64(b)


def _reflect(x, p, dim):
    n = x.shape[dim]
    i = torch.arange(-p, n + p, device=x.device).abs()
    return x.index_select(dim, torch.where(i >= n, 2 * (n - 1) - i, i))


def _conv1d64(x, w, b, stride, pad):
    if pad:
        x = _reflect(x, pad, 2)
    u = x.unfold(2, w.shape[2], stride)  # [B, C, Lo, k]
    w2 = _f64(w).reshape(w.shape[0], -1)
    y = [w2 @ ub.permute(0, 2, 1).reshape(w2.shape[1], -1) for ub in u]
    return torch.stack(y) + _f64(b)[None, :, None]


def _conv_t1d64(x, w, b):
    """k8 s4, padding 3, output padding 2: output length 4 L."""
    B, _, L = x.shape
    y = torch.zeros(B, w.shape[1], 4 * L + 8, dtype=x.dtype, device=x.device)
    for k in range(8):
        wk = _f64(w[:, :, k]).t()
        for i in range(B):
            y[i, :, k:k + 4 * L:4] += wk @ x[i]
    return y[:, :, 3:3 + 4 * L] + _f64(b)[None, :, None]


def _conv2d64(x, w, b):
    """3x3, stride 2, reflect padding 1."""
    x = _reflect(_reflect(x, 1, 2), 1, 3)
    w2 = _f64(w).reshape(w.shape[0], -1)
    ho, wo = (x.shape[2] - 3) // 2 + 1, (x.shape[3] - 3) // 2 + 1
    out = []
    for xi in x:
        u = xi.unfold(1, 3, 2).unfold(2, 3, 2)  # [C, ho, wo, 3, 3]
        out.append((w2 @ u.permute(0, 3, 4, 1, 2).reshape(w2.shape[1], -1)).reshape(-1, ho, wo))
    return torch.stack(out) + _f64(b)[None, :, None, None]


def _conv_t2d64(x, w, b):
    """3x3, stride 2, padding 1, output padding 1: output 2 H x 2 W."""
    B, C, H, W = x.shape
    y = torch.zeros(B, w.shape[1], 2 * H + 2, 2 * W + 2, dtype=x.dtype, device=x.device)
    for kh in range(3):
        for kw in range(3):
            wk = _f64(w[:, :, kh, kw]).t()
            for i in range(B):
                y[i, :, kh:kh + 2 * H:2, kw:kw + 2 * W:2] += \
                    (wk @ x[i].reshape(C, -1)).reshape(-1, H, W)
    return y[:, :, 1:1 + 2 * H, 1:1 + 2 * W] + _f64(b)[None, :, None, None]


def _mha64(q, kv, p, heads):
    E = q.shape[-1]
    wi, bi = p["in_proj_weight"], p["in_proj_bias"]
    Q, K, V = (_linear64(x, wi[i * E:(i + 1) * E], bi[i * E:(i + 1) * E])
               for i, x in enumerate((q, kv, kv)))
    hd, out = E // heads, torch.empty_like(Q)
    for b in range(q.shape[0]):
        for h in range(heads):
            c = slice(h * hd, (h + 1) * hd)
            s = Q[b, :, c].contiguous() @ K[b, :, c].t().contiguous() / math.sqrt(hd)
            out[b, :, c] = torch.softmax(s, dim=-1) @ V[b, :, c].contiguous()
    return _linear64(out, p["out_proj_weight"], p["out_proj_bias"])


def _transformer64(d, layers):
    t, f, p = _f64(d["t"]), _f64(d["f"]), d["p"]
    for i in range(layers):
        new = []
        for br, x, other in (("time", t, f), ("freq", f, t)):
            pre = f"layers.{i}.{br}."
            q = {k[len(pre):]: v for k, v in p.items() if k.startswith(pre)}
            attn = {k[5:]: v for k, v in q.items() if k.startswith("attn.")}
            a = _layer_norm(x, q["norm1.weight"], q["norm1.bias"])
            kv = _layer_norm(other, q["norm2.weight"], q["norm2.bias"]) if i % 2 else a
            x = x + _f64(q["gamma_1.scale"]) * _mha64(a, kv, attn, 8)
            last = "norm3" if i % 2 else "norm2"
            h = _layer_norm(x, q[last + ".weight"], q[last + ".bias"])
            h = _gelu(_linear64(h, q["linear1.weight"], q["linear1.bias"]))
            new.append(x + _f64(q["gamma_2.scale"]) *
                       _linear64(h, q["linear2.weight"], q["linear2.bias"]))
        t, f = new
    return [t, f]


def _stft64(d, case):
    N, hop = case["nfft"], case["nfft"] // 4
    x = d["x"].double()
    n = torch.arange(N, dtype=torch.float64)
    win = (0.5 * (1 - torch.cos(2 * math.pi * n / (N - 1)))).float().double()
    X = torch.fft.rfft(x.unfold(1, N, hop) * win, dim=-1)
    fr = torch.fft.irfft(X, n=N, dim=-1) * win
    L = (X.shape[1] - 1) * hop + N
    y, ws = torch.zeros(x.shape[0], L, dtype=torch.float64), torch.zeros(L, dtype=torch.float64)
    for i in range(X.shape[1]):
        y[:, i * hop:i * hop + N] += fr[:, i]
        ws[i * hop:i * hop + N] += win * win
    y = y / ws.clamp_min(WINDOW_FLOOR)
    re, im = X.real, X.imag
    if case["layout"] == "bins":
        re, im = re.transpose(1, 2), im.transpose(1, 2)
    return [re.contiguous(), im.contiguous(), y]


def _separate64(d, case):
    x, out, prev = _f64(d["x"]), None, 0
    out = torch.zeros(4, case["frames"], 2, dtype=torch.float64, device="cuda")
    for a, b in _segments(case):
        n = b - a
        lp, Lp = _unet_pad(n)
        y = torch.zeros(1, 2, Lp, dtype=torch.float64, device="cuda")
        y[0, :, lp:lp + n] = x[a:b].t()
        skips = []
        for i, (w, bias, g, be) in enumerate(d["enc"]):
            y = _gelu(_affine_norm(_conv1d64(y, w, bias, 4, 3), 2 if i == 0 else 8, g, be))
            skips.append(y)
        for j, (w, bias, g, be) in enumerate(d["dec"]):
            z = torch.cat([y, skips.pop()], dim=1)
            y = _gelu(_affine_norm(_conv_t1d64(z, w, bias), min(8, w.shape[1]), g, be))
        fade = max(0, prev - a)
        k = (torch.arange(fade, device="cuda", dtype=torch.float64)[:, None] + 1) / (fade + 1)
        for h, (w, bias) in enumerate(d["heads"]):
            st = (_f64(w[:, :, 0]) @ y[0] + _f64(bias)[:, None])[:, lp:lp + n].t()
            o = out[h, a:b]
            o[:fade] = o[:fade] * (1 - k) + st[:fade] * k
            o[fade:] = st[fade:]
        prev = b
    return [out.reshape(4, -1)]


def exact(case, seed):
    d, op = _data(case, seed), case["op"]
    if op == "conv_front":
        return _gelu(_affine_norm(_conv1d64(_f64(d["x"]), *d["conv"], 4, 0), 1, *d["norm"]))
    if op == "linear":
        x, (w, b) = d["x"], d["lin"]
        if case["precision"] == "bf16":  # the layer's operands are bf16 values
            x, w = _bf16(x), _bf16(w)
        y = _linear64(_f64(x), w, b)
        return [{"none": lambda v: v, "gelu": _gelu, "relu": torch.relu}[case["act"]](y)]
    if op == "linear_ln":
        return _layer_norm(_linear64(_f64(d["x"]), *d["lin"]), *d["norm"])
    if op == "attention":
        return [_mha64(_f64(d["q"]), _f64(d["kv"]), d["mha"], case["heads"])]
    if op == "cross_transformer":
        return _transformer64(d, case["layers"])
    if op == "time_encoder":
        y, out = _f64(d["x"]), []
        for w, b, g, be, rw, rb in d["levels"]:
            y = _gelu(_affine_norm(_conv1d64(y, w, b, 4, 3), 1, g, be))
            y = F.glu(_conv1d64(y, rw, rb, 1, 0), dim=1)
            out.append(y)
        return out
    if op == "time_decoder":
        z = torch.cat([_f64(d["x"]), _f64(d["skip"])], dim=1)
        return [_gelu(_affine_norm(_conv_t1d64(z, d["w"], d["b"]), case["groups"], *d["norm"]))]
    if op == "freq_encoder":
        y = _conv2d64(_f64(d["x"]), d["w"], d["b"])
        return [_gelu(_affine_norm(y, _freq_groups(case), *d["norm"]))]
    if op == "freq_decoder":
        z = torch.cat([_f64(d["x"]), _f64(d["skip"])], dim=1)
        return [_gelu(_affine_norm(_conv_t2d64(z, d["w"], d["b"]), _freq_groups(case),
                                   *d["norm"]))]
    if op == "stft":
        return _stft64(d, case)
    return _separate64(d, case)
