"""Timed cases of the framework's public entry points (nspeech_amd.abi), over the sizes the speech models use.

  decode     one token of the Moonshine decoder, captured as a HIP graph: per layer LayerNorm, q|k|v projection,
             rotary + K/V cache append, self-attention, output projection + residual + LayerNorm, cross-attention
             over the encoder's K/V, fc1 + GLU, fc2 + residual + LayerNorm; then the vocabulary projection
  utterance  the elementwise and norm ops of an encoder layer on one utterance, called one by one
  resln      residual add + LayerNorm + activation over a batch of frames
  gather     Q8_0 token embedding lookup of a batch of prompts
  adain      AdaIN1d + Snake of a Kokoro generator stage, as its own op (f32 or f16 activations)
  resblock   a Kokoro generator ResBlock: AdaIN + Snake + conv twice per dilation, row statistics handed along
  tail       the generator's end: the average of its three ResBlocks with the leaky ReLU, and the inverse STFT

F frames of Kokoro audio (40 a second) are rows of 20 F columns after the first upsampling (256 channels) and of
120 F + 1 after the second (128 channels; the reflection pad adds the odd column).
"""
import math

import torch

from nspeech_amd import abi

ROT, THETA, EPS = 32, 10000.0, 1e-5
N_FFT, HOP = 20, 5
MAX_FLOPS, MAX_BYTES = 5.6e11, 1.6e9  # a drawn case costs no more than the largest listed one


def listed():
    return [
        # one token through 6 layers of the 640-wide decoder, 300 positions in, 30 s of encoder frames
        {"name": "decode_token", "kind": "decode", "dim": 640, "heads": 10, "layers": 6, "pos": 299, "enc": 1500,
         "splits": 32, "vocab": 32768, "tiles": True},
        # one 10 s utterance in the 1024-wide conformer encoder: small calls, one after the other
        {"name": "utterance_ops", "kind": "utterance", "frames": 125, "dim": 1024, "heads": 8},
        # a batch of 32 minutes-long utterances, bf16 activations
        {"name": "resln_batch_bf16", "kind": "resln", "rows": 24000, "cols": 1024, "dtype": "bf16", "act": "gelu"},
        # prompts of a serving batch through the embedding table of the 640-wide decoder
        {"name": "gather_prompts", "kind": "gather", "vocab": 32768, "d": 640, "n": 16384, "act": "silu", "i64": False},
        # eight 24 s clips after the second upsampling, rows cut to whole vectors
        {"name": "adain_f32_batch", "kind": "adain", "B": 8, "C": 128, "T": 115200, "dtype": "f32"},
        # one 4 s sentence after the second upsampling: the odd row length that the reflection pad gives
        {"name": "adain_f32_sentence", "kind": "adain", "B": 1, "C": 128, "T": 19201, "dtype": "f32"},
        # four 12 s clips with f16 activations
        {"name": "adain_f16_batch", "kind": "adain", "B": 4, "C": 128, "T": 57601, "dtype": "f16"},
        # one 4 s sentence through the widest ResBlock of each upsampling stage
        {"name": "resblock_k11_sentence_up1", "kind": "resblock", "B": 1, "C": 256, "T": 3200, "K": 11, "iters": 3},
        {"name": "resblock_k7_sentence_up2", "kind": "resblock", "B": 1, "C": 128, "T": 19201, "K": 7, "iters": 3},
        # a batch through the narrowest ResBlock, whole-vector rows
        {"name": "resblock_k3_batch", "kind": "resblock", "B": 8, "C": 128, "T": 115200, "K": 3, "iters": 3},
        # four 12 s clips through the widest ResBlock of the second stage
        {"name": "resblock_k11_batch", "kind": "resblock", "B": 4, "C": 128, "T": 57601, "K": 11, "iters": 3},
        # the end of the generator for one 12 s clip
        {"name": "tail_clip", "kind": "tail", "B": 1, "C": 128, "T": 57601},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return c


def _draw(rng):
    kind = rng.choice(["resblock"] * 7 + ["adain"] * 5 + ["decode"] * 3 + ["resln"] * 2 + ["gather", "tail", "utterance"])
    F = _log(rng, 20, 960)  # 0.5 to 24 s of audio
    if kind == "resblock":
        up1 = rng.random() < 0.4
        return {"kind": kind, "B": rng.randint(1, 8), "C": 256 if up1 else 128, "T": 20 * F if up1 else 120 * F + 1,
                "K": rng.choice([3, 7, 11]), "iters": rng.randint(1, 3)}
    if kind == "adain":
        up1 = rng.random() < 0.3
        T = 20 * F if up1 else 120 * F + rng.choice([1, 1, 0])
        return {"kind": kind, "B": rng.randint(1, 8), "C": 256 if up1 else 128, "T": T,
                "dtype": rng.choice(["f32", "f32", "f16"])}
    if kind == "decode":
        dim, heads = rng.choice([(288, 8), (416, 8), (640, 10)])
        return {"kind": kind, "dim": dim, "heads": heads, "layers": rng.randint(1, 8), "pos": _log(rng, 1, 447) - 1,
                "enc": _log(rng, 40, 1500), "splits": rng.choice([8, 16, 32]), "vocab": 32768,
                "tiles": rng.random() < 0.75}
    if kind == "resln":
        return {"kind": kind, "rows": _log(rng, 500, 24000), "cols": rng.choice([288, 416, 512, 640, 1024]),
                "dtype": rng.choice(["bf16", "f16", "f32"]), "act": rng.choice(["none", "gelu", "silu"])}
    if kind == "gather":
        return {"kind": kind, "vocab": 32768, "d": rng.choice([288, 416, 640]), "n": _log(rng, 256, 16384),
                "act": rng.choice(["none", "silu"]), "i64": rng.random() < 0.5}
    if kind == "tail":
        return {"kind": kind, "B": rng.randint(1, 8), "C": 128, "T": 120 * F + 1}
    dim, heads = rng.choice([(288, 8), (416, 8), (640, 10), (1024, 8)])
    return {"kind": kind, "frames": _log(rng, 20, 1500), "dim": dim, "heads": heads}


_DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


class _Rng:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, mean=0.0, std=1.0, dtype=torch.float32):
        t = torch.randn(shape, generator=self.g, device="cuda").mul_(std).add_(mean)
        return t.to(dtype)

    def uniform(self, lo, hi, *shape, dtype=torch.float32):
        t = torch.rand(shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo)
        return t.to(dtype)

    def ints(self, lo, hi, *shape, dtype=torch.int64):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=dtype)

    def q8_0(self, n, k):
        """A GGUF Q8_0 weight [n, k]: (block bytes, int8 values [n, k], f16 scales [n, k / 32])."""
        qs = self.ints(-127, 128, n, k // 32, 32, dtype=torch.int8)
        d = self.uniform(0.5, 1.5, n, k // 32, 1).div_(73.0 * math.sqrt(k)).to(torch.float16)
        blocks = torch.cat([d.view(torch.uint8), qs.view(torch.uint8)], dim=2).contiguous().view(-1)
        return blocks, qs, d


# ------------------------------------------------------------------ inputs --


def _decode_inputs(c, r):
    D, H, L = c["dim"], c["heads"], max(448, c["pos"] + 1)
    Dh = D // H
    lin = lambda n, k: r.q8_0(n, k)  # noqa: E731
    f16 = torch.float16
    d = {"x": r.normal(D), "ln0": r.normal(D, mean=1.0, std=0.05, dtype=f16), "layers": []}
    for _ in range(c["layers"]):
        d["layers"].append({
            "wqkv": lin(3 * D, D), "wo": lin(D, D), "wq2": lin(D, D), "wo2": lin(D, D), "w1": lin(8 * D, D),
            "w2": lin(D, 4 * D), "b1": r.normal(8 * D, std=0.1),
            "ln1": r.normal(D, mean=1.0, std=0.05, dtype=f16), "ln2": r.normal(D, mean=1.0, std=0.05, dtype=f16),
            "ln3": r.normal(D, mean=1.0, std=0.05, dtype=f16),
            "ck": r.normal(H, L, Dh, dtype=f16), "cv": r.normal(H, L, Dh, dtype=f16),
            "ek": r.normal(c["enc"], H, Dh, dtype=f16), "ev": r.normal(c["enc"], H, Dh, dtype=f16)})
    d["wv"] = lin(c["vocab"], D)
    return d


def _resblock_inputs(c, r):
    B, C, K = c["B"], c["C"], c["K"]
    d = {"x": r.normal(B, C, c["T"], mean=0.3, std=1.5), "stages": []}
    for _ in range(2 * c["iters"]):
        d["stages"].append({"gamma": r.normal(B, C, std=0.1), "beta": r.normal(B, C, std=0.1),
                            "alpha": r.uniform(0.5, 1.5, C),
                            "w": r.normal(C, C, K, std=1.0 / math.sqrt(C * K), dtype=torch.float16),
                            "bias": r.normal(C, std=0.1, dtype=torch.float16)})
    return d


def _adain_inputs(c, r):
    p = torch.float16 if c["dtype"] == "f16" else torch.float32
    return {"x": r.normal(c["B"], c["C"], c["T"], dtype=_DT[c["dtype"]]), "gamma": r.normal(c["B"], c["C"], std=0.1, dtype=p),
            "beta": r.normal(c["B"], c["C"], std=0.1, dtype=p), "alpha": r.uniform(0.5, 1.5, c["C"], dtype=p)}


def _resln_inputs(c, r):
    dt = _DT[c["dtype"]]
    bf = lambda t: t.to(torch.bfloat16).to(torch.float32)  # noqa: E731
    return {"x": r.normal(c["rows"], c["cols"], dtype=dt), "res": r.normal(c["rows"], c["cols"], dtype=dt),
            "gamma": bf(r.normal(c["cols"], mean=1.0, std=0.02)), "beta": bf(r.normal(c["cols"], std=0.02))}


def _gather_inputs(c, r):
    blocks, qs, d = r.q8_0(c["vocab"], c["d"])
    return {"blocks": blocks, "qs": qs, "d": d, "ids": r.ints(0, c["vocab"], c["n"], dtype=torch.int64 if c["i64"] else torch.int32)}


def _tail_inputs(c, r):
    n = (c["B"], c["C"], c["T"])
    return {"r": [r.normal(*n) for _ in range(3)],
            "spec": [torch.cat([r.normal(N_FFT // 2 + 1, c["T"], mean=-2.0), r.normal(N_FFT // 2 + 1, c["T"], std=2.0)])
                     for _ in range(c["B"])]}


def _utterance_inputs(c, r):
    T, D, H = c["frames"], c["dim"], c["heads"]
    return {"x": r.normal(T, D), "res": r.normal(T, D), "g": r.normal(D, mean=1.0, std=0.02), "b": r.normal(D, std=0.02),
            "q": r.normal(1, H, T, 64), "k": r.normal(1, H, T, 64), "h": r.normal(T, 4 * D)}


_INPUTS = {"decode": _decode_inputs, "resblock": _resblock_inputs, "adain": _adain_inputs, "resln": _resln_inputs,
           "gather": _gather_inputs, "tail": _tail_inputs, "utterance": _utterance_inputs}


def _inputs(case, seed):
    return _INPUTS[case["kind"]](case, _Rng(seed))


# --------------------------------------------------------------- the cases --


class _Weight:
    """A decoder weight as a program keeps it: t4 tiles, or the repacked-Q8 layout."""

    def __init__(self, blocks, n, k, tiles, glu=False):
        self.tiles = tiles
        self.w = abi.Q8T4.from_q8_0(blocks, n, k, glu=glu) if tiles else abi.q8_0_to_gemv_q8(blocks, n, k)

    def mul(self, x, **kw):
        return abi.gemv_q8_t4(x, self.w, **kw) if self.tiles else abi.gemv_q8(x, *self.w, **kw)

    def glu(self, x, bias):
        return abi.gemv_q8_t4_bias_glu(x, self.w, bias) if self.tiles else abi.gemv_q8_bias_glu(x, *self.w, bias)

    def resadd_ln(self, x, residual, ln):
        if self.tiles:
            return abi.gemv_q8_t4_resadd_ln(x, self.w, residual, ln, eps=EPS)
        return abi.gemv_q8_resadd_ln(x, *self.w, residual, ln, eps=EPS)


def _decode_prepare(c, d):
    D, H, t = c["dim"], c["heads"], c["tiles"]
    Dh, pos, E = D // H, c["pos"], c["enc"]
    abi.init()
    table = abi.rope_table(448, ROT, THETA).cuda()
    layers = []
    for a in d["layers"]:
        layers.append({**a, "wqkv": _Weight(a["wqkv"][0], 3 * D, D, t), "wo": _Weight(a["wo"][0], D, D, t),
                       "wq2": _Weight(a["wq2"][0], D, D, t), "wo2": _Weight(a["wo2"][0], D, D, t),
                       "w1": _Weight(a["w1"][0], 8 * D, D, t, glu=True), "w2": _Weight(a["w2"][0], D, 4 * D, t),
                       "partial": torch.empty(H * c["splits"] * (Dh + 2), device="cuda")})
    wv = _Weight(d["wv"][0], c["vocab"], D, t)
    sm = Dh ** -0.5

    def step():
        h = d["x"]
        n = abi.layernorm(h.view(1, D), d["ln0"], eps=EPS, out_dtype=torch.float16).view(D)
        for a in layers:
            L = a["ck"].shape[1]
            qkv = a["wqkv"].mul(n).view(3, H, Dh)
            abi.rope_qk_cache_append(qkv[0], qkv[1], qkv[2], table, a["ck"], a["cv"], pos, ROT)
            o = abi.attention_decode(qkv[0], a["ck"], a["cv"], pos + 1, H, sm, stride_kv_head=L * Dh, stride_kv_seq=Dh)
            h, n = a["wo"].resadd_ln(o.view(D), h, a["ln1"])
            q2 = a["wq2"].mul(n).view(H, Dh)
            o = abi.attention_decode(q2, a["ek"], a["ev"], E, H, sm, stride_kv_head=Dh, stride_kv_seq=H * Dh,
                                     n_splits=c["splits"], partial=a["partial"])
            h, n = a["wo2"].resadd_ln(o.view(D), h, a["ln2"])
            h, n = a["w2"].resadd_ln(a["w1"].glu(n, a["b1"]), h, a["ln3"])
        return {"logits": wv.mul(n, out_dtype=torch.float32), "h": h}

    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    out["ck"], out["cv"] = [a["ck"] for a in layers], [a["cv"] for a in layers]
    return {"graph": graph, "out": out, "keep": (layers, wv, table, d)}


def _resblock_prepare(c, d):
    for s in d["stages"]:
        s["wp"] = abi.conv1d_pack_f16(s["w"])
    return d


def _utterance_prepare(c, d):
    d["table"] = abi.rope_table(c["frames"], ROT, THETA).cuda()
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    if case["kind"] == "decode":
        s = _decode_prepare(case, d)
    elif case["kind"] == "resblock":
        s = _resblock_prepare(case, d)
    elif case["kind"] == "utterance":
        s = _utterance_prepare(case, d)
    else:
        s = d
    s["case"] = case
    return s


def _resblock_run(c, s):
    x, stats, K = s["x"], None, c["K"]
    for it, dil in enumerate((1, 3, 5)[:c["iters"]]):
        a, b = s["stages"][2 * it], s["stages"][2 * it + 1]
        h, hs = abi.adain_snake_conv1d_chain(x, a["gamma"], a["beta"], a["alpha"], a["wp"], a["bias"], x_stats=stats,
                                             padding=(K - 1) * dil // 2, dilation=dil, eps=EPS)
        x, stats = abi.adain_snake_conv1d_chain(h, b["gamma"], b["beta"], b["alpha"], b["wp"], b["bias"], x, x_stats=hs,
                                                want_stats=it + 1 < c["iters"], padding=(K - 1) // 2, eps=EPS)
    return x


def run(state):
    c, s = state["case"], state
    kind = c["kind"]
    if kind == "decode":
        s["graph"].replay()
        return s["out"]
    if kind == "resblock":
        return _resblock_run(c, s)
    if kind == "adain":
        return abi.adain_snake(s["x"], s["gamma"], s["beta"], s["alpha"], eps=EPS)
    if kind == "resln":
        return abi.residual_add_layernorm(s["x"], s["res"], s["gamma"], s["beta"], eps=EPS, act=c["act"])
    if kind == "gather":
        return abi.q8_0_embed_gather(s["blocks"], c["vocab"], c["d"], s["ids"], act=c["act"])
    if kind == "tail":
        avg = abi.resblock_average_f32(*s["r"], leaky_slope=0.01)
        return [avg] + [abi.istft_f32(x, n_fft=N_FFT, hop=HOP) for x in s["spec"]]
    y = abi.layernorm(s["x"], s["g"], s["b"], eps=EPS)
    q, k = abi.rotary(s["q"], s["k"], ROT, THETA, table=s["table"])
    h, z = abi.residual_add_layernorm(s["x"], s["res"], s["g"], s["b"], eps=EPS)
    return [y, q, k, h, z, abi.activation(s["h"], "silu")]


# ------------------------------------------------------------ work, limits --


def work(case):
    c, kind = case, case["kind"]
    if kind == "decode":
        D, H = c["dim"], c["heads"]
        weights = c["layers"] * (3 * D * D + 3 * D * D + 8 * D * D + 4 * D * D) + c["vocab"] * D
        kv = c["layers"] * 2 * D * (c["pos"] + 1 + c["enc"])
        return {"bytes": weights * 34 / 32 + 2 * kv + 4 * c["vocab"], "flops": 2.0 * (weights + kv)}
    if kind == "resblock":
        n = c["B"] * c["C"] * c["T"]
        return {"bytes": 8.0 * n + 4.0 * c["iters"] * c["C"] * c["C"] * c["K"], "flops": 4.0 * c["iters"] * n * c["C"] * c["K"]}
    if kind == "adain":
        n = c["B"] * c["C"] * c["T"]
        return {"bytes": (8.0 if c["dtype"] == "f32" else 4.0) * n, "flops": 20.0 * n}
    if kind == "resln":
        n = c["rows"] * c["cols"]
        return {"bytes": (16.0 if c["dtype"] == "f32" else 8.0) * n, "flops": 20.0 * n}
    if kind == "gather":
        return {"bytes": c["n"] * (c["d"] * 34 / 32 + 4.0 * c["d"] + (8 if c["i64"] else 4)), "flops": 6.0 * c["n"] * c["d"]}
    if kind == "tail":
        n, f = c["B"] * c["C"] * c["T"], c["B"] * c["T"]
        return {"bytes": 16.0 * n + f * (4.0 * (N_FFT + 2) + 4 * HOP), "flops": 5.0 * n + f * 4.0 * N_FFT * (N_FFT // 2 + 1)}
    T, D, H = c["frames"], c["dim"], c["heads"]
    return {"bytes": 4.0 * (2 * T * D + 4 * T * D + 8 * T * D + 4 * H * T * 64), "flops": T * (60.0 * D + 8 * H * 64)}


def tolerance(case):
    """About four times the error measured against 64 bits; "max" allows a whole unit in the last place of a rounded output."""
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 3e-3}
    if kind == "resblock":
        return {"rel": 3e-6, "max": 1e-4}
    if kind == "adain":
        return {"rel": 9e-4, "max": 4e-3} if case["dtype"] == "f16" else {"rel": 4e-7, "max": 2e-5}
    if kind == "resln":
        return {"f32": {"rel": 4e-7, "max": 2e-5}, "f16": {"rel": 9e-4, "max": 4e-3}, "bf16": {"rel": 7e-3, "max": 4e-2}}[case["dtype"]]
    if kind == "gather":
        return {"rel": 3e-7, "max": 2e-5}
    if kind == "tail":
        return {"rel": 1e-6, "max": 1e-4}
    return {"rel": 4e-7, "max": 2e-5}


# --------------------------------------------- the same in 64 bits, plain torch --


def _ln(x, g=None, b=None):
    m = x.mean(-1, keepdim=True)
    y = (x - m) / torch.sqrt((x - m).square().mean(-1, keepdim=True) + EPS)
    y = y if g is None else y * g.double()
    return y if b is None else y + b.double()


def _act(x, act):
    if act == "gelu":
        return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))
    return x * torch.sigmoid(x) if act == "silu" else x


def _adain_snake(x, gamma, beta, alpha):
    m = x.mean(-1, keepdim=True)
    y = (x - m) / torch.sqrt((x - m).square().mean(-1, keepdim=True) + EPS)
    y = y * (1.0 + gamma.double()[:, :, None]) + beta.double()[:, :, None]
    al = alpha.double()[None, :, None]
    return y + torch.sin(al * y).square() / (al + 1e-9)


def _conv(x, w, bias, padding, dilation):
    T = x.shape[-1]
    xp = torch.nn.functional.pad(x, (padding, padding))
    wd, out = w.double(), bias.double()[None, :, None].expand(x.shape[0], -1, T).contiguous()
    for b in range(x.shape[0]):
        for k in range(w.shape[2]):
            out[b] += wd[:, :, k].contiguous() @ xp[b, :, k * dilation:k * dilation + T].contiguous()
    return out


def _rotate(x, pos):
    """x [..., T, Dh], positions pos [T]: interleaved pairs of the first ROT dims."""
    inv = 1.0 / (torch.tensor(THETA, dtype=torch.float32) ** (torch.arange(0, ROT, 2, dtype=torch.float32) / ROT))
    ang = (pos.float()[:, None] * inv.to(pos.device)[None, :]).double()  # the f32 angle that the op defines
    a, b = x[..., 0:ROT:2], x[..., 1:ROT:2]
    y = x.clone()
    y[..., 0:ROT:2] = a * ang.cos() - b * ang.sin()
    y[..., 1:ROT:2] = b * ang.cos() + a * ang.sin()
    return y


def _dequant(w):
    _, qs, d = w
    return (qs.double() * d.double()).flatten(1)


def _attend(q, k, v, sm):
    """q [H, Dh], k and v [H, n, Dh]."""
    p = torch.softmax((k * q[:, None, :]).sum(-1) * sm, dim=-1)
    return (p[:, :, None] * v).sum(1)


def _decode_exact(c, d):
    D, H = c["dim"], c["heads"]
    Dh, pos = D // H, c["pos"]
    at = torch.tensor([pos], device="cuda")
    h, cks, cvs = d["x"].double(), [], []
    n = _ln(h, d["ln0"])
    for a in d["layers"]:
        q, k, v = (_dequant(a["wqkv"]) @ n).view(3, H, Dh)
        q, k = _rotate(q[:, None, :], at)[:, 0], _rotate(k[:, None, :], at)[:, 0]
        ck, cv = a["ck"].double(), a["cv"].double()
        ck[:, pos], cv[:, pos] = k, v
        o = _attend(q, ck[:, :pos + 1], cv[:, :pos + 1], Dh ** -0.5)
        h = h + _dequant(a["wo"]) @ o.reshape(D)
        q2 = (_dequant(a["wq2"]) @ _ln(h, a["ln1"])).view(H, Dh)
        o = _attend(q2, a["ek"].double().transpose(0, 1), a["ev"].double().transpose(0, 1), Dh ** -0.5)
        h = h + _dequant(a["wo2"]) @ o.reshape(D)
        x, gate = (_dequant(a["w1"]) @ _ln(h, a["ln2"]) + a["b1"].double()).view(2, 4 * D)
        h = h + _dequant(a["w2"]) @ (_act(gate, "silu") * x)
        n = _ln(h, a["ln3"])
        cks.append(ck)
        cvs.append(cv)
    return {"logits": _dequant(d["wv"]) @ n, "h": h, "ck": cks, "cv": cvs}


def _istft(spec):
    nb, n = N_FFT // 2 + 1, spec.shape[1]
    mag, ph = torch.exp(spec[:nb].double()), torch.sin(spec[nb:].double())
    frames = torch.fft.irfft(torch.complex(mag * ph.cos(), mag * ph.sin()), n=N_FFT, dim=0)  # [N_FFT, n]
    win = torch.hann_window(N_FFT, periodic=True, dtype=torch.float64, device=spec.device)
    total = N_FFT + (n - 1) * HOP
    at = (torch.arange(n, device=spec.device) * HOP)[None, :] + torch.arange(N_FFT, device=spec.device)[:, None]
    out = torch.zeros(total, dtype=torch.float64, device=spec.device).index_add_(0, at.reshape(-1), (frames * win[:, None]).reshape(-1))
    norm = torch.zeros_like(out).index_add_(0, at.reshape(-1), win.square()[:, None].expand(-1, n).reshape(-1))
    out = torch.where(norm > 1e-8, out / norm.clamp_min(1e-8), torch.zeros_like(out))
    return out[N_FFT // 2:N_FFT // 2 + (n - 1) * HOP]


def exact(case, seed):
    c, d = case, _inputs(case, seed)
    kind = c["kind"]
    if kind == "decode":
        return _decode_exact(c, d)
    if kind == "resblock":
        x, K = d["x"].double(), c["K"]
        for it, dil in enumerate((1, 3, 5)[:c["iters"]]):
            a, b = d["stages"][2 * it], d["stages"][2 * it + 1]
            h = _conv(_adain_snake(x, a["gamma"], a["beta"], a["alpha"]), a["w"], a["bias"], (K - 1) * dil // 2, dil)
            x = x + _conv(_adain_snake(h, b["gamma"], b["beta"], b["alpha"]), b["w"], b["bias"], (K - 1) // 2, 1)
        return x
    if kind == "adain":
        return _adain_snake(d["x"].double(), d["gamma"], d["beta"], d["alpha"])
    if kind == "resln":
        h = (d["x"].double() + d["res"].double()).to(d["x"].dtype)  # rounded to the activation type by definition
        return [h.double(), _act(_ln(h.double(), d["gamma"], d["beta"]), c["act"])]
    if kind == "gather":
        ids = d["ids"].long()
        return _act((d["qs"][ids].double() * d["d"][ids].double()).flatten(1), c["act"])
    if kind == "tail":
        avg = (d["r"][0].double() + d["r"][1].double() + d["r"][2].double()) / 3.0
        return [torch.where(avg > 0, avg, 0.01 * avg)] + [_istft(x) for x in d["spec"]]
    pos = torch.arange(c["frames"], device="cuda")
    h = d["x"].double() + d["res"].double()
    return [_ln(d["x"].double(), d["g"], d["b"]), _rotate(d["q"].double(), pos), _rotate(d["k"].double(), pos), h,
            _ln(h, d["g"], d["b"]), _act(d["h"].double(), "silu")]
