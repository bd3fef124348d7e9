"""The calls that a user of this library makes, as cases that can be timed and
compared: the quantized linears of a text encoder and of a DiT block at one
token up to a long video's, the block's two attentions, the patch projection
and the weight decoder, through the entry points of include/fh3/fh3_hip.h and
the reference's own fh3_matmul.

A case is a dict of plain values.  prepare() makes its inputs on the GPU (on
the host for fh3_matmul), run() is one pass, exact() the same result in 64-bit
torch, from the packed bytes, without this library.
"""
import ctypes
import math

import numpy as np
import torch

from fasth3inc_amd import fh3 as F

DEV = "cuda"
TYPES = {"Q4_K": F.FH3_QUANT_Q4_K, "Q5_K": F.FH3_QUANT_Q5_K, "Q6_K": F.FH3_QUANT_Q6_K, "F16": F.FH3_QUANT_F16}
SUPER_BYTES = {"Q4_K": 144, "Q5_K": 176, "Q6_K": 210}  # per 256 weights
EPS = 1e-6


def listed():
    return [
        # one token through an attention projection: the decode step's smallest call
        {"name": "linear_m1", "kind": "linear", "type": "Q4_K", "M": 1, "K": 5120, "N": 5120, "form": "plain"},
        # a short batch through the text encoder's MLP
        {"name": "linear_m16", "kind": "linear", "type": "Q4_K", "M": 16, "K": 5120, "N": 17408, "form": "plain"},
        # the reference's own benchmark call: fh3_matmul on host arrays, weights registered once
        {"name": "host_m64", "kind": "host", "type": "Q4_K", "M": 64, "K": 4096, "N": 4096},
        # the text encoder's long down rows, Q6_K, an odd prompt length
        {"name": "q6k_m37", "kind": "linear", "type": "Q6_K", "M": 37, "K": 25600, "N": 5120, "form": "plain"},
        # a whole prompt prefilled through the text encoder's MLP
        {"name": "prompt_m300", "kind": "linear", "type": "Q4_K", "M": 300, "K": 5120, "N": 17408, "form": "plain"},
        # the video patch projection: short F16 rows and a bias, once per forward
        {"name": "patch_f16", "kind": "linear", "type": "F16", "M": 2880, "K": 96, "N": 5376, "form": "bias"},
        # a weight matrix decoded to fp32 rows
        {"name": "dequant_q6k", "kind": "dequant", "type": "Q6_K", "K": 8192, "N": 5120},
        # a DiT block's first linear: rmsnorm + modulate folded into the preparation, then fused QKV
        {"name": "dit_qkv", "kind": "linear", "type": "Q4_K", "M": 8192, "K": 5120, "N": 15360, "form": "norm"},
        # a DiT block's gated up projection at the shortest video's token count
        {"name": "dit_fc1", "kind": "linear", "type": "Q4_K", "M": 3016, "K": 5376, "N": 28672, "form": "swiglu"},
        # the down projection at a long sequence: the largest product
        {"name": "dit_down", "kind": "linear", "type": "Q4_K", "M": 32768, "K": 13824, "N": 5120, "form": "plain"},
        # a DiT block's dense attention from the QKV projection's output: q/k rmsnorm, rope, attention
        {"name": "attention", "kind": "attention", "n": 16384, "heads": 40, "hd": 128, "rot": 96},
        # the same with video sparse attention and its gate, the DiT's default (1024x576, 73 frames)
        {"name": "vsa", "kind": "vsa", "text": 6, "audio": 244, "gt": 22, "gh": 18, "gw": 32, "heads": 56, "hd": 128,
         "rot": 96, "sparsity": 0.8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["host", "patch", "dequant", "attention", "vsa", "vsa"])
    if kind == "linear":
        M = _log_int(rng, 1, 32768)
        K = rng.choice([1024, 2560, 4096, 5120, 5376, 7168, 8192, 13824, 14336, 25600])
        N = _log_int(rng, 1000, 28672)
        qt = rng.choice(["Q4_K"] * 5 + ["Q5_K", "Q6_K"])
        form = rng.choice(["plain", "bias", "norm", "swiglu"]) if qt == "Q4_K" else "plain"
        if form == "swiglu":
            N = (N + 127) // 128 * 128
        M = max(1, min(M, int(4.5e12 / (2.0 * K * N)), 400_000_000 // max(K, N)))
        return {"kind": "linear", "type": qt, "M": M, "K": K, "N": N, "form": form}
    if kind == "host":
        return {"kind": "host", "type": "Q4_K", "M": _log_int(rng, 1, 512), "K": rng.choice([1024, 4096, 5120]),
                "N": _log_int(rng, 1000, 8192)}
    if kind == "patch":
        return {"kind": "linear", "type": "F16", "M": _log_int(rng, 100, 16384), "K": rng.choice([32, 96, 5376]),
                "N": rng.choice([5120, 5376]), "form": "bias"}
    if kind == "dequant":
        return {"kind": "dequant", "type": rng.choice(["Q4_K", "Q5_K", "Q6_K"]),
                "K": rng.choice([4096, 5120, 8192, 25600]), "N": _log_int(rng, 500, 16384)}
    if kind == "attention":
        hd = rng.choice([64, 128, 128])
        return {"kind": "attention", "n": _log_int(rng, 300, 12000), "heads": rng.choice([16, 40, 56]), "hd": hd,
                "rot": rng.choice([0, 3 * hd // 4, 3 * hd // 4])}
    gt, gh, gw = rng.randint(6, 22), rng.randint(8, 18), rng.randint(12, 32)
    return {"kind": "vsa", "text": rng.randint(1, 90), "audio": rng.randint(40, 250), "gt": gt, "gh": gh, "gw": gw,
            "heads": rng.choice([16, 40, 56]), "hd": 128, "rot": 96, "sparsity": rng.choice([0.5, 0.8, 0.9])}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _activations(g, rows, cols):
    """LayerNorm-scale rows with 1 % of outliers at 8 sigma, as transformer activations have."""
    x = _randn(g, rows, cols)
    hit = torch.rand(rows, cols, generator=g, device=DEV) < 0.01
    return torch.where(hit, 8.0 * torch.sign(x), x)


def _groups(w, size):
    return w.reshape(w.shape[0], -1, 256 // size, size)


def _pack_scales(sc, mn):
    """The 12 bytes of eight 6-bit scales and mins of Q4_K / Q5_K."""
    out = torch.empty(*sc.shape[:-1], 12, dtype=torch.uint8, device=sc.device)
    out[..., 0:4] = sc[..., 0:4] | ((sc[..., 4:8] >> 4) << 6)
    out[..., 4:8] = mn[..., 0:4] | ((mn[..., 4:8] >> 4) << 6)
    out[..., 8:12] = (sc[..., 4:8] & 15) | ((mn[..., 4:8] & 15) << 4)
    return out


def _half_bytes(h):
    return h.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _quantize(w, qtype):
    """Rows of fp32 weights -> packed rows (uint8 [N][row bytes]), plain round-to-nearest quantisers."""
    if qtype == "F16":
        return w.to(torch.float16).view(torch.uint8)
    if qtype in ("Q4_K", "Q5_K"):
        top = 15 if qtype == "Q4_K" else 31
        g = _groups(w, 32)
        lo, hi = g.amin(-1).clamp(max=0), g.amax(-1)
        scale, mn = (hi - lo) / top, -lo
        d = (scale.amax(-1, keepdim=True) / 63).half().float()
        dmin = (mn.amax(-1, keepdim=True) / 63).half().float()
        sc = (scale / d).round().clamp(1, 63)
        m = (mn / dmin.clamp(min=1e-8)).round().clamp(0, 63)
        q = ((g + (dmin * m)[..., None]) / (d * sc)[..., None]).round().clamp(0, top).to(torch.uint8)
        parts = [_half_bytes(d[..., 0]), _half_bytes(dmin[..., 0]), _pack_scales(sc.to(torch.uint8), m.to(torch.uint8))]
        if qtype == "Q5_K":  # bit j of high byte l: bit 4 of weight l of group j
            hb = torch.zeros_like(q[..., 0, :])
            for j in range(8):
                hb |= (q[..., j, :] >> 4) << j
            parts.append(hb)
        q = q & 15
        parts.append((q[..., 0::2, :] | (q[..., 1::2, :] << 4)).flatten(-2))
        return torch.cat(parts, -1).flatten(1)
    g = _groups(w, 16)  # Q6_K
    scale = g.abs().amax(-1) / 31
    d = (scale.amax(-1, keepdim=True) / 127).half().float()
    sc = (scale / d).round().clamp(1, 127)
    q = ((g / (d * sc)[..., None]).round().clamp(-32, 31) + 32).to(torch.uint8)
    q = q.reshape(*q.shape[:2], 2, 4, 32)  # halves of 128, quarters of 32
    ql = torch.cat([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4), (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)], -1)
    qh = (q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) | ((q[..., 3, :] >> 4) << 6)
    return torch.cat([ql.flatten(-2), qh.flatten(-2), sc.to(torch.uint8), _half_bytes(d[..., 0])], -1).flatten(1)


def _weights(g, qtype, N, K):
    rows = []
    for r in range(0, N, 4096):  # bounded scratch
        rows.append(_quantize(0.02 * _randn(g, min(4096, N - r), K), qtype))
    return torch.cat(rows) if len(rows) > 1 else rows[0]


def _tables(n, rot):
    ang = torch.arange(n, device=DEV)[:, None] * 10000.0 ** (-torch.arange(rot // 2, device=DEV) / (rot // 2))
    ang = torch.cat([ang, ang], -1)
    return torch.cos(ang).float().contiguous(), torch.sin(ang).float().contiguous()


class _Registered:
    """Host weights registered with the library for as long as this lives."""

    def __init__(self, raw):
        self.raw = raw
        if F.lib().fh3_hip_register_weights(raw.ctypes.data, raw.nbytes, None) != F.FH3_OK:
            raise RuntimeError("fh3_hip_register_weights")

    def __del__(self):
        F.lib().fh3_hip_unregister_weights(self.raw.ctypes.data)


def _linear_inputs(case, seed):
    M, K, N, form = case["M"], case["K"], case["N"], case.get("form", "plain")
    g = _gen(seed)
    s = {"w": _weights(g, case["type"], N, K), "x": _activations(g, M, K)}
    if form == "bias":
        s["bias"] = 0.1 * _randn(g, N)
    if form in ("norm", "swiglu"):  # the block's prologue: rmsnorm weight, AdaLN shift and scale
        s["nw"] = 1.0 + 0.1 * _randn(g, K)
        s["shift"], s["scale"] = 0.1 * _randn(g, M, K), 0.1 * _randn(g, M, K)
    return s


def _attention_inputs(case, seed):
    g = _gen(seed)
    heads, hd, rot = case["heads"], case["hd"], case["rot"]
    n = case["n"] if case["kind"] == "attention" else sum(_counts(case))
    s = {"n": n, "qkv": _randn(g, n, 3 * heads * hd), "qn": 1.0 + 0.1 * _randn(g, hd), "kn": 1.0 + 0.1 * _randn(g, hd)}
    if rot:
        s["cos"], s["sin"] = _tables(n, rot)
    if case["kind"] == "vsa":
        s["gate"] = torch.sigmoid(_randn(g, n, heads * hd))
    return s


def _counts(case):
    return case["text"], case["audio"], case["gt"] * case["gh"] * case["gw"]


def prepare(case, seed):
    F.init(0)
    kind = case["kind"]
    if kind in ("attention", "vsa"):
        s = _attention_inputs(case, seed)
        s["o"] = torch.empty(s["n"], case["heads"] * case["hd"], device=DEV)
        if kind == "vsa":
            text, audio, _ = _counts(case)
            s["seq"] = F.seq_of(s["n"], text, audio, grid=(case["gt"], case["gh"], case["gw"]))
    elif kind == "dequant":
        s = {"w": _weights(_gen(seed), case["type"], case["N"], case["K"]),
             "y": torch.empty(case["N"], case["K"], device=DEV)}
    elif kind == "host":
        d = _linear_inputs(case, seed)
        reg = _Registered(d["w"].cpu().numpy())
        s = {"reg": reg, "x": d["x"].cpu().numpy(), "y": np.zeros((case["M"], case["N"]), np.float32),
             "w": F.Fh3W(TYPES[case["type"]], case["K"], case["N"], reg.raw.ctypes.data)}
    else:
        s = _linear_inputs(case, seed)
        out = case["N"] // 2 if case["form"] == "swiglu" else case["N"]
        s["y"] = torch.empty(case["M"], out, device=DEV)
        if case["form"] in ("norm", "swiglu"):
            s["prep"] = torch.empty(F.prepared_bytes(case["M"], case["K"]), dtype=torch.uint8, device=DEV)
    s["case"] = case
    return s


def _at(s, name):
    return s[name].data_ptr() if name in s else None


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "attention":
        F.attention_qkv_dev(_at(s, "qkv"), s["n"], c["heads"], c["hd"], _at(s, "o"), _at(s, "qn"), _at(s, "kn"), EPS,
                            _at(s, "cos"), _at(s, "sin"), c["rot"])
        return s["o"]
    if kind == "vsa":
        F.vsa_attention_qkv_dev(_at(s, "qkv"), _at(s, "gate"), _at(s, "o"), s["seq"], c["heads"], c["hd"],
                                c["sparsity"], 64, _at(s, "qn"), _at(s, "kn"), EPS, _at(s, "cos"), _at(s, "sin"),
                                c["rot"])
        return s["o"]
    if kind == "dequant":
        F.dequant_dev(_at(s, "w"), _at(s, "y"), c["N"], c["K"], qtype=TYPES[c["type"]])
        return s["y"]
    if kind == "host":
        F.lib().fh3_matmul(ctypes.byref(s["w"]), s["x"].ctypes.data, s["y"].ctypes.data, c["M"], None)
        return s["y"]
    M, K, N, qt = c["M"], c["K"], c["N"], TYPES[c["type"]]
    if c["form"] in ("norm", "swiglu"):
        F.prepare_x_norm_dev(_at(s, "x"), M, K, _at(s, "nw"), EPS, _at(s, "prep"), _at(s, "shift"), _at(s, "scale"))
        if c["form"] == "norm":
            F.matmul_prepared_dev(_at(s, "w"), K, N, _at(s, "prep"), _at(s, "y"), M, qtype=qt)
        else:
            F.matmul_prepared_epi_dev(_at(s, "w"), K, N, _at(s, "prep"), M, F.EPI_SWIGLU, _at(s, "y"), qtype=qt)
    else:
        F.matmul_dev(_at(s, "w"), K, N, _at(s, "x"), _at(s, "y"), M, _at(s, "bias"), qtype=qt)
    return s["y"]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _weight_bytes(case):
    n = case["N"] * case["K"]
    return 2 * n if case["type"] == "F16" else n // 256 * SUPER_BYTES[case["type"]]


def work(case):
    kind = case["kind"]
    if kind == "dequant":
        return {"bytes": _weight_bytes(case) + 4 * case["N"] * case["K"], "flops": 0}
    if kind in ("linear", "host"):
        M, K, N, form = case["M"], case["K"], case["N"], case.get("form", "plain")
        out = N // 2 if form == "swiglu" else N
        rows = 3 if form in ("norm", "swiglu") else 1  # x, shift, scale
        return {"bytes": _weight_bytes(case) + 4 * M * (rows * K + out), "flops": 2 * M * N * K}
    inner = case["heads"] * case["hd"]
    if kind == "attention":
        n = case["n"]
        return {"bytes": 4 * n * (4 * inner + 2 * case["rot"]), "flops": 4 * n * n * inner}
    text, audio, video = _counts(case)
    n, pre = text + audio + video, text + audio
    tiles = -(-case["gt"] // 4) * -(-case["gh"] // 4) * -(-case["gw"] // 4)
    kept = max(1, math.ceil((1 - case["sparsity"]) * tiles)) / tiles
    pairs = pre * n + video * (pre + kept * video)
    return {"bytes": 4 * n * (5 * inner + 2 * case["rot"]), "flops": 4 * pairs * inner}


def tolerance(case):
    """Decoding is exact.  Products and attentions take fp16 operands (one rounding of 2^-11 each) into fp32 sums:
    2e-4 to 4e-4 from the 64-bit result, so two correct forms may be about 4 x 4e-4 apart."""
    return "exact" if case["kind"] == "dequant" else {"rel": 1.6e-3, "max": 3e-2}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _f16_at(b, at):
    return b[..., at:at + 2].contiguous().view(torch.float16).double()


def _decode(raw, qtype):
    """Packed rows -> float64 weights [N][K]."""
    if qtype == "F16":
        return raw.view(torch.float16).double()
    b = raw.reshape(raw.shape[0], -1, SUPER_BYTES[qtype])
    if qtype == "Q6_K":
        ql, qh = b[..., 0:128].reshape(*b.shape[:2], 2, 64), b[..., 128:192].reshape(*b.shape[:2], 2, 32)
        lo = torch.stack([ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4], -2)
        hi = torch.stack([(qh >> s) & 3 for s in (0, 2, 4, 6)], -2)
        q = (lo | (hi << 4)).double().reshape(*b.shape[:2], 16, 16) - 32
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        return (_f16_at(b, 208) * sc).unsqueeze(-1).mul(q).flatten(1)
    s = b[..., 4:16]
    sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1).double()
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
    qs = b[..., 16:144] if qtype == "Q4_K" else b[..., 48:176]
    qs = qs.reshape(*b.shape[:2], 4, 32)
    q = torch.stack([qs & 15, qs >> 4], -2).reshape(*b.shape[:2], 8, 32)
    if qtype == "Q5_K":
        q = q | (torch.stack([(b[..., 16:48] >> j) & 1 for j in range(8)], -2) << 4)
    return ((_f16_at(b, 0) * sc)[..., None] * q.double() - (_f16_at(b, 2) * mn)[..., None]).flatten(1)


def _exact_linear(case, s):
    w, form = _decode(s["w"], case["type"]), case.get("form", "plain")
    out = []
    for r in range(0, case["M"], 4096):
        x = s["x"][r:r + 4096].double()
        if "nw" in s:
            x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * s["nw"].double()
            x = x * (1 + s["scale"][r:r + 4096].double()) + s["shift"][r:r + 4096].double()
        y = x @ w.t()
        if "bias" in s:
            y = y + s["bias"].double()
        if form == "swiglu":
            val, gate = y.chunk(2, -1)
            y = val * gate * torch.sigmoid(gate)
        out.append(y)
    return torch.cat(out)


def _exact_qkv(case, s, h):
    """q, k, v of head h in 64 bits, after norm and rope."""
    heads, hd, rot = case["heads"], case["hd"], case["rot"]
    inner = heads * hd
    q, k, v = (s["qkv"][:, i * inner + h * hd:i * inner + (h + 1) * hd].double() for i in range(3))
    done = []
    for x, w in ((q, s["qn"]), (k, s["kn"])):
        x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
        if rot:
            half = rot // 2
            lo, hi = x[:, :half], x[:, half:rot]
            c, t = s["cos"].double(), s["sin"].double()
            x = torch.cat([lo * c[:, :half] - hi * t[:, :half], hi * c[:, half:] + lo * t[:, half:], x[:, rot:]], -1)
        done.append(x)
    return done[0], done[1], v


def _tile_of(case):
    """The tile of each token: text and audio in runs of 64, the video in 4x4x4 cubes; and the prefix tiles."""
    text, audio, _ = _counts(case)
    runs = [torch.arange(text) // 64, torch.arange(audio) // 64 + -(-text // 64)]
    prefix = -(-text // 64) + -(-audio // 64)
    t, h, w = torch.meshgrid(torch.arange(case["gt"]) // 4, torch.arange(case["gh"]) // 4,
                             torch.arange(case["gw"]) // 4, indexing="ij")
    cube = (t * -(-case["gh"] // 4) + h) * -(-case["gw"] // 4) + w
    return torch.cat(runs + [cube.flatten() + prefix]).to(DEV), prefix


def _exact_attention(case, s):
    n, heads, hd = s["n"], case["heads"], case["hd"]
    sparse = case["kind"] == "vsa"
    out = torch.empty(n, heads, hd, dtype=torch.float64, device=DEV)
    if sparse:
        tile, prefix = _tile_of(case)
        T = int(tile.max()) + 1
        count = torch.bincount(tile, minlength=T).double()[:, None]
        keep = min(T - prefix, max(1, math.ceil(np.float32(1 - np.float32(case["sparsity"])) * np.float32(T - prefix))))
    for h in range(heads):
        q, k, v = _exact_qkv(case, s, h)
        if sparse:
            pooled = [torch.zeros(T, hd, dtype=torch.float64, device=DEV).index_add_(0, tile, x) / count for x in (q, k, v)]
            score = pooled[0] @ pooled[1].t() / math.sqrt(hd)
            sel = torch.ones(T, T, dtype=torch.bool, device=DEV)
            sel[prefix:, prefix:] = False
            top = score[prefix:, prefix:].topk(keep, -1).indices + prefix
            sel[prefix:].scatter_(1, top, True)
        for r in range(0, n, 4096):
            a = q[r:r + 4096] @ k.t() / math.sqrt(hd)
            if sparse:
                a = a.masked_fill(~sel[tile[r:r + 4096]][:, tile], -math.inf)
            out[r:r + 4096, h] = torch.softmax(a, -1) @ v
        if sparse:
            coarse = torch.softmax(score, -1) @ pooled[2]
            out[:, h] += coarse[tile] * s["gate"].reshape(n, heads, hd)[:, h].double()
    return out.reshape(n, heads * hd)


def exact(case, seed):
    if case["kind"] == "dequant":
        return _decode(_weights(_gen(seed), case["type"], case["N"], case["K"]), case["type"])
    if case["kind"] in ("attention", "vsa"):
        return _exact_attention(case, _attention_inputs(case, seed))
    y = _exact_linear(case, _linear_inputs(case, seed))
    return y.cpu().numpy() if case["kind"] == "host" else y
