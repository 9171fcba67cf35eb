"""What this framework's users have it do, as timed cases on one GPU.

Every case goes through the public host interface (vokra_amd.hip): the
quantized linears of the per-op seam, fused attention, decode attention over
the paged cache, the audio front end, and the three model-level calls (encoder
forward, batched decoder step, batched speech-LLM decode step). Sizes are those
of the repository's own configurations (Whisper-base and Whisper-large-v3
dims, a 2048-wide speech-LLM with 16/2 x 128 heads) and of the models between
them; `draw` spreads them over the ranges the listed cases stand for.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from vokra_amd import hip

DEV = "cuda"
WD = {"q4_0": hip.WDtype.Q4_0, "q5_0": hip.WDtype.Q5_0, "q8_0": hip.WDtype.Q8_0,
      "q4_k": hip.WDtype.Q4_K, "q5_k": hip.WDtype.Q5_K, "q6_k": hip.WDtype.Q6_K}
WIRE_BYTES = {"q4_0": 18 / 32, "q5_0": 22 / 32, "q8_0": 34 / 32,
              "q4_k": 144 / 256, "q5_k": 176 / 256, "q6_k": 210 / 256}  # per weight

_CTX = None


def _ctx():
    """The one device context a program holds."""
    global _CTX
    if _CTX is None:
        torch.cuda.init()
        _CTX = hip.HipContext(0)
    return _CTX


class _Dev:
    """A torch tensor as the device-pointer argument of a resident call."""

    def __init__(self, t):
        assert t.is_contiguous()
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * scale


def _empty(*shape, dtype=torch.float32):
    return _Dev(torch.zeros(*shape, device=DEV, dtype=dtype))


def _i32(x):
    return _Dev(torch.as_tensor(x, dtype=torch.int32, device=DEV).contiguous())


# ---- quantized weights: wire bytes and, for exact(), their values in 64 bits

def _le16(d):
    return d.to(torch.float16).contiguous().view(torch.uint8).reshape(*d.shape, 2)


def _block_weight(fmt, w):
    """Q4_0 / Q5_0 / Q8_0: 32-element blocks, f16 scale first."""
    n, k = w.shape
    b = w.reshape(n, k // 32, 32)
    div, lo, hi = {"q4_0": (7.0, -8, 7), "q5_0": (15.0, -16, 15), "q8_0": (127.0, -127, 127)}[fmt]
    d = (b.abs().amax(-1) / div).to(torch.float16)
    df = d.float().clamp_min(1e-12)
    q = torch.round(b / df[..., None]).clamp(lo, hi).to(torch.int32)
    parts = [_le16(d)]
    if fmt == "q8_0":
        parts.append(q.to(torch.int8).view(torch.uint8))
    else:
        u = q - lo
        if fmt == "q5_0":
            bits = ((u >> 4) & 1).reshape(n, k // 32, 4, 8)
            parts.append((bits << torch.arange(8, device=DEV)).sum(-1).to(torch.uint8))
        nib = (u & 15).reshape(n, k // 32, 16, 2)
        parts.append((nib[..., 0] | (nib[..., 1] << 4)).to(torch.uint8))
    return torch.cat(parts, -1).reshape(-1), (q.double() * d.double()[..., None]).reshape(n, k)


def _k_weight(fmt, w):
    """Q4_K / Q5_K / Q6_K: 256-element super-blocks."""
    n, k = w.shape
    if fmt == "q6_k":
        b = w.reshape(n, k // 256, 16, 16)
        sc_f = b.abs().amax(-1) / 31.0
        d = (sc_f.amax(-1) / 127.0).to(torch.float16)
        df = d.float().clamp_min(1e-12)
        sc = torch.round(sc_f / df[..., None]).clamp(1, 127).to(torch.int32)
        q = torch.round(b / (df[..., None, None] * sc[..., None].float())).clamp(-32, 31).to(torch.int32)
        w64 = d.double()[..., None, None] * sc.double()[..., None] * q.double()
        u = (q + 32).reshape(n, k // 256, 2, 4, 32)  # [half][quarter][l]
        lo, hi = u & 15, u >> 4
        ql = torch.cat([lo[..., 0, :] | (lo[..., 2, :] << 4), lo[..., 1, :] | (lo[..., 3, :] << 4)], -1)
        qh = hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)
        parts = [ql.reshape(n, k // 256, 128).to(torch.uint8), qh.reshape(n, k // 256, 64).to(torch.uint8),
                 sc.to(torch.int8).view(torch.uint8), _le16(d)]
        return torch.cat(parts, -1).reshape(-1), w64.reshape(n, k)
    top = 15 if fmt == "q4_k" else 31
    b = w.reshape(n, k // 256, 8, 32)
    mn = (-b.amin(-1)).clamp_min(0.0)
    sc_f = (b.amax(-1) + mn) / top
    d, dmin = (sc_f.amax(-1) / 63.0).to(torch.float16), (mn.amax(-1) / 63.0).to(torch.float16)
    df, mf = d.float().clamp_min(1e-12), dmin.float().clamp_min(1e-12)
    sc = torch.round(sc_f / df[..., None]).clamp(1, 63).to(torch.int32)
    m = torch.round(mn / mf[..., None]).clamp(0, 63).to(torch.int32)
    deff, meff = df[..., None] * sc.float(), dmin.float()[..., None] * m.float()
    q = torch.round((b + meff[..., None]) / deff[..., None]).clamp(0, top).to(torch.int32)
    w64 = (d.double()[..., None] * sc.double())[..., None] * q.double() - \
        (dmin.double()[..., None] * m.double())[..., None]
    packed = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                        (sc[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1)
    lo = (q & 15).reshape(n, k // 256, 4, 2, 32)  # 64-element chunk: low nibbles, then high
    parts = [_le16(d), _le16(dmin), packed.to(torch.uint8)]
    if fmt == "q5_k":
        parts.append(((q >> 4) << torch.arange(8, device=DEV)[:, None]).sum(-2).to(torch.uint8))
    parts.append((lo[..., 0, :] | (lo[..., 1, :] << 4)).reshape(n, k // 256, 128).to(torch.uint8))
    return torch.cat(parts, -1).reshape(-1), w64.reshape(n, k)


def _weight(fmt, g, n, k, scale=None):
    """(wire bytes on the host, weight in 64 bits) of a random [n, k] linear."""
    w = _randn(g, n, k, scale=0.7 / math.sqrt(k) if scale is None else scale)
    wire, w64 = (_k_weight if fmt.endswith("_k") else _block_weight)(fmt, w)
    return wire, w64


def _round_away(x):
    return torch.sign(x) * torch.floor(x.abs() + 0.5)


def _quantized(x32, group):
    """The INT8 activations the linears are defined on: per group s = amax / 127,
    q = clamp(round(x / s)); returns s * q in 64 bits."""
    v = x32.float().reshape(*x32.shape[:-1], -1, group)
    s = v.abs().amax(-1, keepdim=True) / 127.0
    q = _round_away(v / torch.where(s == 0, torch.ones_like(s), s)).clamp(-127, 127)
    return (q.double() * s.double()).reshape(x32.shape)


def _lin64(fmt, x, w64, b=None):
    y = _quantized(x, 16 if fmt.endswith("_k") else 32) @ w64.T
    return y if b is None else y + b.double()


def _q8_rows64(x):
    """Rows as the paged cache stores them (Q8_0 blocks of 32)."""
    v = x.float().reshape(*x.shape[:-1], -1, 32)
    d = v.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(d == 0, torch.zeros_like(d), 1.0 / d)
    q = _round_away((v * inv).clamp(-127, 127))
    return (q.double() * d.to(torch.float16).double()).reshape(x.shape)


def _attend64(q, k, v, mask=None):
    """[..., t_q, hd] x [..., t_kv, hd] softmax attention in 64 bits, q already scaled."""
    s = q @ k.transpose(-1, -2).contiguous()
    if mask is not None:
        s = s.masked_fill(~mask, -math.inf)
    return torch.softmax(s, -1) @ v


def _ln64(x, g, b):
    x = x.double()
    return torch.nn.functional.layer_norm(x, x.shape[-1:], g.double(), b.double(), 1e-5)


def _rms64(x, g, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * g.double()


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


# ---- family "linear": one quantized linear of the per-op seam (gemm_q_f32 on
# resident weights and device activations; the activation pass is inside)

def _linear_inputs(c, seed):
    g = _gen(seed)
    wire, w64 = _weight(c["fmt"], g, c["n"], c["k"])
    # hidden activations: unit scale with a few large channels, as after a norm
    a = _randn(g, c["m"], c["k"]) * (1.0 + 4.0 * (torch.rand(c["k"], generator=g, device=DEV) > 0.98))
    b = _randn(g, c["n"], scale=0.1) if c["bias"] else None
    return wire, w64, a, b


def _linear_prepare(c, seed):
    wire, _, a, b = _linear_inputs(c, seed)
    w = _ctx().upload_qweight(WD[c["fmt"]], c["n"], c["k"], wire.cpu().numpy())
    torch.cuda.synchronize()
    return {"w": w, "a": _Dev(a), "b": None if b is None else _Dev(b), "o": _empty(c["m"], c["n"]), "m": c["m"]}


def _linear_run(c, s):
    _ctx().gemm_q_f32_dev(s["w"], s["m"], s["a"], s["o"], d_bias=s["b"])
    return s["o"].t


def _linear_exact(c, seed):
    _, w64, a, b = _linear_inputs(c, seed)
    return _lin64(c["fmt"], a, w64, b)


def _linear_work(c):
    m, n, k = c["m"], c["n"], c["k"]
    return {"bytes": n * k * WIRE_BYTES[c["fmt"]] + 4 * (m * k + m * n + (n if c["bias"] else 0)), "flops": 2 * m * n * k}


# ---- family "attention": fused SDPA over several queries (attn_f32 on device
# arrays): encoder self-attention, a causal GQA prompt, cross-attention

def _attention_inputs(c, seed):
    g = _gen(seed)
    q = _randn(g, c["batch"], c["t_q"], c["heads"] * c["hd"])
    k = _randn(g, c["batch"], c["t_kv"], c["kv_heads"] * c["hd"])
    v = _randn(g, c["batch"], c["t_kv"], c["kv_heads"] * c["hd"])
    return q, k, v


def _attention_prepare(c, seed):
    q, k, v = _attention_inputs(c, seed)
    _ctx()
    return {"q": _Dev(q), "k": _Dev(k), "v": _Dev(v), "o": _Dev(torch.zeros_like(q))}


def _attention_run(c, s):
    _ctx().attn_f32_dev(c["batch"], c["t_q"], c["t_kv"], c["heads"], c["kv_heads"], c["hd"], s["q"], s["k"], s["v"],
                        c["hd"] ** -0.5, c["causal"], c["t_kv"] - c["t_q"] if c["causal"] else 0, s["o"])
    return s["o"].t


def _heads(x, h):
    b, t, w = x.shape
    return x.reshape(b, t, h, w // h).transpose(1, 2).contiguous()


def _attention_exact(c, seed):
    q, k, v = _attention_inputs(c, seed)
    rep = c["heads"] // c["kv_heads"]
    mask = None
    if c["causal"]:
        i = torch.arange(c["t_q"], device=DEV)[:, None] + (c["t_kv"] - c["t_q"])
        mask = torch.arange(c["t_kv"], device=DEV)[None] <= i
    out = []
    for b in range(c["batch"]):
        qh = _heads(q[b:b + 1].double() * c["hd"] ** -0.5, c["heads"])
        kh, vh = (_heads(x[b:b + 1].double(), c["kv_heads"]).repeat_interleave(rep, 1) for x in (k, v))
        out.append(_attend64(qh, kh, vh, mask).transpose(1, 2).reshape(1, c["t_q"], -1))
    return torch.cat(out)


def _attention_work(c):
    tq, tk = c["t_q"], c["t_kv"]
    pairs = tq * tk - (tq * (tq - 1) // 2 if c["causal"] else 0)
    return {"bytes": 4 * c["batch"] * c["hd"] * (2 * tq * c["heads"] + 2 * tk * c["kv_heads"]),
            "flops": 4 * c["batch"] * c["heads"] * c["hd"] * pairs}


# ---- family "paged": a decode step's cache append and attention over the paged
# Q8_0 cache, for every layer of a session in turn (its layers' caches rotate,
# as in a step; pages placed as on a long-running server)

def _spread(lo, hi, n, seed):
    """n lengths spread evenly over lo..hi, in an order of the seed's."""
    lens = np.round(np.linspace(lo, hi, n)).astype(np.int32)
    return np.random.default_rng(int(seed)).permutation(lens)


def _paged_inputs(c, seed):
    g = _gen(seed)
    lens = _spread(c["len_lo"], c["len_hi"], c["streams"], seed)  # keys after this step's append
    w = c["kv_heads"] * c["hd"]
    t = int(lens.max())
    hist = _randn(g, 2, c["layers"], t, w)  # every stream's history starts as these rows, rolled by the stream
    q = _randn(g, c["layers"], c["streams"], c["heads"] * c["hd"])
    new = _randn(g, 2, c["layers"], c["streams"], w)
    return lens, hist, q, new


def _paged_prepare(c, seed):
    lens, hist, q, new = _paged_inputs(c, seed)
    n, ppl = c["streams"], -(-c["len_hi"] // 16)
    kv = _ctx().kv_cache(c["layers"], c["kv_heads"], c["hd"], n, c["len_hi"], 16)
    kv.set_free_order(np.random.default_rng(int(seed)).permutation(c["layers"] * ppl).astype(np.int32))
    st = np.concatenate([np.full(int(lens[s]) - 1, s, np.int32) for s in range(n)])
    tt = np.concatenate([np.arange(int(lens[s]) - 1, dtype=np.int32) for s in range(n)])
    d_st, d_tt = torch.as_tensor(st, device=DEV), torch.as_tensor(tt, device=DEV)
    src = ((d_tt + 7 * d_st) % hist.shape[2]).long()
    for layer in range(c["layers"]):
        rows = [hist[j, layer][src].contiguous() for j in (0, 1)]
        torch.cuda.synchronize()
        for i in range(0, st.size, 1024):
            j = min(st.size, i + 1024)
            kv.append_dev(layer, j - i, _Dev(d_st[i:j]), _Dev(d_tt[i:j]), _Dev(rows[0][i:j]), _Dev(rows[1][i:j]))
        kv.status()
    streams, times, dl = _i32(np.arange(n)), _i32(lens - 1), _i32(lens)
    torch.cuda.synchronize()
    return {"kv": kv, "streams": streams, "times": times, "lens": dl, "max": int(lens.max()),
            "q": [_Dev(q[i]) for i in range(c["layers"])], "k": [_Dev(new[0, i]) for i in range(c["layers"])],
            "v": [_Dev(new[1, i]) for i in range(c["layers"])],
            "o": [_empty(n, c["heads"] * c["hd"]) for _ in range(c["layers"])]}


def _paged_run(c, s):
    n = c["streams"]
    for layer in range(c["layers"]):
        s["kv"].append_dev(layer, n, s["streams"], s["times"], s["k"][layer], s["v"][layer])
        s["kv"].attn_dev(layer, n, s["streams"], s["lens"], s["max"], c["heads"], s["q"][layer], c["hd"] ** -0.5,
                         s["o"][layer])
    return [o.t for o in s["o"]]


def _paged_exact(c, seed):
    lens, hist, q, new = _paged_inputs(c, seed)
    rep, hd = c["heads"] // c["kv_heads"], c["hd"]
    out = []
    for layer in range(c["layers"]):
        rows = []
        for s in range(c["streams"]):
            src = (torch.arange(int(lens[s]) - 1, device=DEV) + 7 * s) % hist.shape[2]
            k, v = (_heads(_q8_rows64(torch.cat([hist[j, layer][src], new[j, layer, s:s + 1]]))[None], c["kv_heads"])
                    .repeat_interleave(rep, 1) for j in (0, 1))
            qh = _heads(q[layer, s][None, None].double() * hd ** -0.5, c["heads"])
            rows.append(_attend64(qh, k, v).transpose(1, 2).reshape(1, -1))
        out.append(torch.cat(rows))
    return out


def _paged_keys(c):
    return int(np.round(np.linspace(c["len_lo"], c["len_hi"], c["streams"])).sum())


def _paged_work(c):
    w, keys = c["kv_heads"] * c["hd"], _paged_keys(c)
    return {"bytes": c["layers"] * (2 * keys * w * 34 / 32 + 4 * c["streams"] * (2 * w + 2 * c["heads"] * c["hd"])),
            "flops": c["layers"] * 4 * keys * c["heads"] * c["hd"]}


# ---- family "frontend": audio samples -> log-mel -> the encoder's conv stem

def _frontend_inputs(c, seed):
    g = _gen(seed)
    t = torch.arange(c["samples"], device=DEV, dtype=torch.float64) / 16000.0
    f = 100.0 + 3000.0 * torch.rand(c["batch"], 3, generator=g, device=DEV).double()
    tones = 0.1 * torch.sin(2 * math.pi * f[..., None] * t).sum(1)
    pcm = (tones.float() + _randn(g, c["batch"], c["samples"], scale=0.05)).contiguous()
    d, m = c["d"], c["mels"]
    w = {"w1": _randn(g, d, m, 3, scale=0.02), "b1": _randn(g, d, scale=0.02),
         "w2": _randn(g, d, d, 3, scale=0.02), "b2": _randn(g, d, scale=0.02), "pos": _randn(g, 1500, d, scale=0.02)}
    return pcm, w


def _frontend_prepare(c, seed):
    pcm, w = _frontend_inputs(c, seed)
    one, zero = np.ones(c["d"], np.float32), np.zeros(c["d"], np.float32)
    enc = hip.Encoder(_ctx(), hip.WDtype.Q8_0, c["d"], c["d"] // 64, 4 * c["d"], [], one, zero, c["batch"] * 1500)
    enc.set_stem(c["mels"], 3000, *[w[n].cpu().numpy() for n in ("w1", "b1", "w2", "b2", "pos")])
    return {"enc": enc, "pcm": _Dev(pcm), "mel": _empty(c["batch"], c["mels"], 3000),
            "x": _empty(c["batch"], 1500, c["d"])}


def _frontend_run(c, s):
    _ctx().log_mel_dev(s["pcm"], c["batch"], c["samples"], c["mels"], s["mel"])
    s["enc"].stem_dev(c["batch"], s["mel"], s["x"])
    return {"mel": s["mel"].t, "x": s["x"].t}


def _mel_bank(n_mels):
    """Slaney mel filter bank over the 201 bins of a 400-point transform at 16 kHz, f32 as the reference builds it."""
    step = math.log(6.4) / 27.0

    def to_mel(f):
        return 15.0 + math.log(f / 1000.0) / step if f >= 1000.0 else f * 3.0 / 200.0

    def to_hz(m):
        return 1000.0 * math.exp(step * (m - 15.0)) if m >= 15.0 else m * 200.0 / 3.0

    e = np.array([to_hz(to_mel(8000.0) * i / (n_mels + 1)) for i in range(n_mels + 2)])
    f = np.arange(201) * 40.0
    lower = (f - e[:-2, None]) / (e[1:-1] - e[:-2])[:, None]
    upper = (e[2:, None] - f) / (e[2:] - e[1:-1])[:, None]
    tri = np.maximum(0.0, np.minimum(lower, upper)).astype(np.float32)
    return (tri.astype(np.float64) * (2.0 / (e[2:] - e[:-2]))[:, None]).astype(np.float32)


def _conv64(x, w, b, stride):
    """[batch, c, t] * [o, c, 3], padding 1, in 64 bits."""
    cols = torch.nn.functional.pad(x, (1, 1)).unfold(2, 3, stride)  # [batch, c, t', 3]
    cols = cols.permute(0, 2, 1, 3).reshape(x.shape[0], cols.shape[2], -1)
    return (cols @ w.double().reshape(w.shape[0], -1).T + b.double()).transpose(1, 2)


def _frontend_exact(c, seed):
    pcm, w = _frontend_inputs(c, seed)
    x = torch.zeros(c["batch"], 480000, device=DEV, dtype=torch.float64)
    n = min(480000, c["samples"])
    x[:, :n] = pcm[:, :n].double()
    win = torch.as_tensor((0.5 - 0.5 * np.cos(2 * math.pi * np.arange(400) / 400)).astype(np.float32), device=DEV).double()
    xp = torch.nn.functional.pad(x[:, None], (200, 200), mode="reflect")[:, 0]
    fr = xp.unfold(1, 400, 160)[:, :3000] * win
    i = torch.arange(400, device=DEV)
    ang = ((i[:201, None] * i[None]) % 400).double() * (2 * math.pi / 400)
    re, im = fr @ torch.cos(ang).T, fr @ torch.sin(ang).T
    bank = torch.as_tensor(_mel_bank(c["mels"]), device=DEV).double()
    mel = torch.log10(((re.square() + im.square()) @ bank.T).clamp_min(1e-10)).transpose(1, 2)
    mel = (torch.maximum(mel, mel.amax((1, 2), keepdim=True) - 8.0) + 4.0) / 4.0
    h = _gelu64(_conv64(mel, w["w1"], w["b1"], 1))
    h = _gelu64(_conv64(h, w["w2"], w["b2"], 2))
    return {"mel": mel, "x": h.transpose(1, 2) + w["pos"].double()}


def _frontend_work(c):
    b, d, m = c["batch"], c["d"], c["mels"]
    # the transform as a 400-point real FFT (about 2.5 n log2 n), the bands' nonzeros (about two per bin), the convolutions
    mel = b * 3000 * (2.5 * 400 * math.log2(400) + 3 * 201 + 4 * 201)
    return {"bytes": 4 * (b * min(c["samples"], 480000) + b * m * 3000 + 3 * d * m + 3 * d * d + 1500 * d + b * 1500 * d),
            "flops": mel + b * (2 * 3000 * d * 3 * m + 2 * 1500 * d * 3 * d)}


# ---- family "encoder": a whole call of the encoder session (pre-norm blocks
# over a batch of utterances; a few blocks, as every block is the same work)

def _norm(g, d):
    return 1.0 + _randn(g, d, scale=0.1), _randn(g, d, scale=0.1)


def _whisper_layers(c, g, decoder):
    d, ff = c["d"], 4 * c["d"]
    out = []
    for _ in range(c["layers"]):
        L, W = {}, {}
        for name in ("ln1", "ln2") + (("ln3",) if decoder else ()):
            L[name + "_gamma"], L[name + "_beta"] = _norm(g, d)
        mats = [("wq", d, d), ("wk", d, d), ("wv", d, d), ("wo", d, d)]
        if decoder:
            mats += [("cwq", d, d), ("cwk", d, d), ("cwv", d, d), ("cwo", d, d)]
        for name, n, k in mats + [("w1", ff, d), ("w2", d, ff)]:
            L[name], W[name] = _weight(c["fmt"], g, n, k)
        for name, n in (("bq", d), ("bv", d), ("bo", d), ("b1", ff), ("b2", d)) + \
                ((("cbq", d), ("cbv", d), ("cbo", d)) if decoder else ()):
            L[name] = _randn(g, n, scale=0.05)
        out.append((L, W))
    return out


def _host(L):
    return {k: v.cpu().numpy() for k, v in L.items()}


def _encoder_inputs(c, seed):
    g = _gen(seed)
    layers = _whisper_layers(c, g, False)
    return layers, _norm(g, c["d"]), _randn(g, c["batch"], c["frames"], c["d"])


def _encoder_prepare(c, seed):
    layers, (pg, pb), x = _encoder_inputs(c, seed)
    enc = hip.Encoder(_ctx(), WD[c["fmt"]], c["d"], c["d"] // 64, 4 * c["d"], [_host(L) for L, _ in layers],
                      pg.cpu().numpy(), pb.cpu().numpy(), c["batch"] * c["frames"])
    return {"enc": enc, "x": _Dev(x), "o": _Dev(torch.zeros_like(x))}


def _encoder_run(c, s):
    s["enc"].forward_dev(c["batch"], c["frames"], s["x"], s["o"])
    return s["o"].t


def _encoder_exact(c, seed):
    layers, (pg, pb), x = _encoder_inputs(c, seed)
    f, H = c["fmt"], c["d"] // 64
    h = x.double()
    for L, W in layers:
        y = _ln64(h, L["ln1_gamma"], L["ln1_beta"])
        q, k, v = _lin64(f, y, W["wq"], L["bq"]) * 64 ** -0.5, _lin64(f, y, W["wk"]), _lin64(f, y, W["wv"], L["bv"])
        a = torch.cat([_attend64(*(_heads(t[b:b + 1], H) for t in (q, k, v))).transpose(1, 2).reshape(1, *h.shape[1:])
                       for b in range(c["batch"])])
        h = h + _lin64(f, a, W["wo"], L["bo"])
        y = _ln64(h, L["ln2_gamma"], L["ln2_beta"])
        h = h + _lin64(f, _gelu64(_lin64(f, y, W["w1"], L["b1"])), W["w2"], L["b2"])
    return _ln64(h, pg, pb)


def _encoder_work(c):
    d, t, b = c["d"], c["frames"], c["batch"]
    params = 12 * d * d
    return {"bytes": c["layers"] * params * WIRE_BYTES[c["fmt"]] + 8 * b * t * d,
            "flops": c["layers"] * b * (2 * t * params + 4 * t * t * d)}


# ---- family "decoder": a whole batched decoder step (paged self-KV, cross-
# attention over each stream's encoder output, tied logits, greedy token)

def _decoder_inputs(c, seed):
    g = _gen(seed)
    layers = _whisper_layers(c, g, True)
    lens = _spread(1, c["prefix"], c["streams"], seed)  # positions before this step
    toks = torch.randint(0, c["vocab"], (c["prefix"] + 1, c["streams"]), generator=g, device=DEV, dtype=torch.int32)
    return {"layers": layers, "post": _norm(g, c["d"]), "emb": _randn(g, c["vocab"], c["d"], scale=0.05),
            "pos": _randn(g, 448, c["d"], scale=0.05), "lens": lens, "toks": toks,
            "enc": _randn(g, 4, c["audio"], c["d"])}  # stream s listens to utterance s % 4


def _decoder_prepare(c, seed):
    x = _decoder_inputs(c, seed)
    n, d = c["streams"], c["d"]
    dec = hip.Decoder(_ctx(), WD[c["fmt"]], d, d // 64, 4 * d, c["vocab"], 448, c["audio"], n,
                      [_host(L) for L, _ in x["layers"]], x["emb"].cpu().numpy(), x["pos"].cpu().numpy(),
                      x["post"][0].cpu().numpy(), x["post"][1].cpu().numpy(), block_size=16)
    dec.set_free_order(np.random.default_rng(int(seed)).permutation(sum(dec.kv_pages())).astype(np.int32))
    torch.cuda.synchronize()
    for s in range(n):
        dec.set_encoder_dev(s, _Dev(x["enc"][s % 4]))
    toks, lens = x["toks"].cpu().numpy(), x["lens"]
    for t in range(int(lens.max())):  # the prefixes, one step at a time
        live = np.nonzero(lens > t)[0].astype(np.int32)
        dec.step(live, toks[t, live], np.full(live.size, t, np.int32))
    last = x["toks"][torch.as_tensor(lens, device=DEV).long(), torch.arange(n, device=DEV)].contiguous()
    streams, pos = _i32(np.arange(n)), _i32(lens)
    torch.cuda.synchronize()
    return {"dec": dec, "streams": streams, "toks": _Dev(last), "pos": pos, "next": _empty(n, dtype=torch.int32),
            "logits": _empty(n, c["vocab"])}


def _decoder_run(c, s):
    s["dec"].step_dev(c["streams"], s["streams"], s["toks"], s["pos"], s["next"], s["logits"])
    return {"logits": s["logits"].t}  # s["next"] is their argmax


def _decoder_exact(c, seed):
    x = _decoder_inputs(c, seed)
    f, d, n = c["fmt"], c["d"], c["streams"]
    H, T = d // 64, int(x["lens"].max()) + 1
    out = torch.empty(n, c["vocab"], device=DEV, dtype=torch.float64)
    cross = [[[_heads(_lin64(f, e[None], W[m], L.get(b)), H) for m, b in (("cwk", None), ("cwv", "cbv"))]
              for e in x["enc"]] for L, W in x["layers"]]
    emb = x["emb"].double()
    for s0 in range(0, n, 8):  # every position of a stream's prefix at once: the same rows, causally masked
        ss = range(s0, min(n, s0 + 8))
        h = (emb[x["toks"][:T, s0:s0 + 8].T.long()].float() + x["pos"][:T]).double()
        mask = torch.ones(T, T, device=DEV, dtype=torch.bool).tril()
        for li, (L, W) in enumerate(x["layers"]):
            y = _ln64(h, L["ln1_gamma"], L["ln1_beta"])
            q, k, v = _lin64(f, y, W["wq"], L["bq"]) * 64 ** -0.5, _lin64(f, y, W["wk"]), _lin64(f, y, W["wv"], L["bv"])
            a = _attend64(_heads(q, H), _heads(_q8_rows64(k), H), _heads(_q8_rows64(v), H), mask)
            h = h + _lin64(f, a.transpose(1, 2).reshape(h.shape), W["wo"], L["bo"])
            y = _ln64(h, L["ln2_gamma"], L["ln2_beta"])
            q = _heads(_lin64(f, y, W["cwq"], L["cbq"]) * 64 ** -0.5, H)
            a = torch.cat([_attend64(q[i:i + 1], *cross[li][s % 4]) for i, s in enumerate(ss)])
            h = h + _lin64(f, a.transpose(1, 2).reshape(h.shape), W["cwo"], L["cbo"])
            y = _ln64(h, L["ln3_gamma"], L["ln3_beta"])
            h = h + _lin64(f, _gelu64(_lin64(f, y, W["w1"], L["b1"])), W["w2"], L["b2"])
        at = torch.as_tensor(x["lens"][s0:s0 + 8], device=DEV).long()
        out[s0:s0 + 8] = _ln64(h[torch.arange(len(ss), device=DEV), at], *x["post"]) @ emb.T
    return {"logits": out}


def _decoder_work(c):
    d, n = c["d"], c["streams"]
    params = 14 * d * d  # the cross k / v linears run once per utterance
    keys = int(np.round(np.linspace(1, c["prefix"], n)).sum()) + n
    cross = n * c["audio"] * d * 2 * 3  # K and V of every stream, 3 bytes per value as the session keeps them
    return {"bytes": c["layers"] * (params * WIRE_BYTES[c["fmt"]] + 2 * keys * d * 34 / 32 + cross)
            + 4 * c["vocab"] * (d + n),
            "flops": c["layers"] * (2 * n * params + 4 * d * (keys + n * c["audio"])) + 2 * n * c["vocab"] * d}


# ---- family "text": a whole batched speech-LLM decode step (RMSNorm, RoPE, GQA
# over the paged cache, SwiGLU, LM head, greedy token)

def _text_inputs(c, seed):
    g = _gen(seed)
    d, hd, ff = c["d"], c["hd"], c["ff"]
    layers = []
    for _ in range(c["layers"]):
        L, W = {"attn_norm_gamma": _norm(g, d)[0], "ffn_norm_gamma": _norm(g, d)[0]}, {}
        for name, n, k in (("wq", c["heads"] * hd, d), ("wk", c["kv_heads"] * hd, d), ("wv", c["kv_heads"] * hd, d),
                           ("wo", d, c["heads"] * hd), ("w_gate", ff, d), ("w_up", ff, d), ("w_down", d, ff)):
            L[name], W[name] = _weight(c["fmt"], g, n, k)
        layers.append((L, W))
    lens = _spread(c["len_lo"], c["len_hi"], c["streams"], seed)  # positions before this step
    return {"layers": layers, "emb": _randn(g, c["vocab"], d, scale=0.5), "final": _norm(g, d)[0],
            "head": _weight(c["fmt"], g, c["vocab"], d), "lens": lens,
            "hist": _randn(g, 2, c["layers"], int(lens.max()), c["kv_heads"] * hd),
            "toks": torch.randint(0, c["vocab"], (c["streams"],), generator=g, device=DEV, dtype=torch.int32)}


def _text_prepare(c, seed):
    x = _text_inputs(c, seed)
    n = c["streams"]
    dec = hip.TextDecoder(_ctx(), WD[c["fmt"]], c["d"], c["heads"], c["kv_heads"], c["hd"], c["ff"], c["vocab"],
                          c["len_hi"] + 16, n, [_host(L) for L, _ in x["layers"]], x["emb"].cpu().numpy(),
                          x["final"].cpu().numpy(), x["head"][0].cpu().numpy(), rope_base=1e6, rms_norm_eps=1e-5,
                          block_size=16)
    dec.set_free_order(np.random.default_rng(int(seed)).permutation(sum(dec.kv_pages())).astype(np.int32))
    hist = x["hist"].cpu().numpy()
    for s in range(n):  # the streams share their prompt's rows
        dec.kv_restore(s, hist[0][:, :x["lens"][s]], hist[1][:, :x["lens"][s]])
    streams, pos = _i32(np.arange(n)), _i32(x["lens"])
    torch.cuda.synchronize()
    return {"dec": dec, "streams": streams, "toks": _Dev(x["toks"]), "pos": pos, "next": _empty(n, dtype=torch.int32),
            "logits": _empty(n, c["vocab"])}


def _text_run(c, s):
    s["dec"].step_dev(c["streams"], s["streams"], s["toks"], s["pos"], s["next"], s["logits"])
    return {"logits": s["logits"].t}  # s["next"] is their argmax


def _rope64(x, pos, base):
    """[n, heads, hd] rotated at pos [n]: the angle is the f32 product of the position and the f32 frequency."""
    half = x.shape[-1] // 2
    theta = (base ** (-2.0 * torch.arange(half, device=DEV, dtype=torch.float64) / x.shape[-1])).float()
    ang = (pos.float()[:, None] * theta).double()[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * torch.cos(ang) - b * torch.sin(ang), a * torch.sin(ang) + b * torch.cos(ang)], -1)


def _text_exact(c, seed):
    x = _text_inputs(c, seed)
    f, n, hd, rep = c["fmt"], c["streams"], c["hd"], c["heads"] // c["kv_heads"]
    pos = torch.as_tensor(x["lens"], device=DEV)
    h = x["emb"][x["toks"].long()].double()
    for li, (L, W) in enumerate(x["layers"]):
        y = _rms64(h, L["attn_norm_gamma"], 1e-5)
        q = _rope64(_lin64(f, y, W["wq"]).reshape(n, c["heads"], hd), pos, 1e6)
        k = _rope64(_lin64(f, y, W["wk"]).reshape(n, c["kv_heads"], hd), pos, 1e6).reshape(n, -1)
        v = _lin64(f, y, W["wv"])
        a = []
        for s in range(n):
            kk, vv = (_heads(_q8_rows64(torch.cat([x["hist"][j, li, :x["lens"][s]].double(), t[s:s + 1]]))[None],
                             c["kv_heads"]).repeat_interleave(rep, 1) for j, t in ((0, k), (1, v)))
            a.append(_attend64(q[s][None, :, None] * hd ** -0.5, kk, vv).reshape(1, -1))
        h = h + _lin64(f, torch.cat(a), W["wo"])
        y = _rms64(h, L["ffn_norm_gamma"], 1e-5)
        u = _lin64(f, y, W["w_gate"])
        h = h + _lin64(f, u * torch.sigmoid(u) * _lin64(f, y, W["w_up"]), W["w_down"])
    return {"logits": _lin64(f, _rms64(h, x["final"], 1e-5), x["head"][1])}


def _text_work(c):
    d, n, hd = c["d"], c["streams"], c["hd"]
    params = d * hd * (2 * c["heads"] + 2 * c["kv_heads"]) + 3 * d * c["ff"]
    keys = int(np.round(np.linspace(c["len_lo"], c["len_hi"], n)).sum()) + n
    return {"bytes": c["layers"] * (params * WIRE_BYTES[c["fmt"]] + 2 * keys * c["kv_heads"] * hd * 34 / 32)
            + c["vocab"] * d * WIRE_BYTES[c["fmt"]] + 4 * n * (c["vocab"] + d),
            "flops": c["layers"] * (2 * n * params + 4 * keys * c["heads"] * hd) + 2 * n * c["vocab"] * d}


# ---- the cases

def listed():
    return [
        # Whisper-large-v3's fc1 over one 30 s utterance: the largest linear of the encoder
        {"name": "linear_q8_0_utterance", "kind": "linear", "fmt": "q8_0", "m": 1500, "n": 5120, "k": 1280, "bias": True},
        # its fc2 over a short streaming window (187 frames): few rows, a long sum
        {"name": "linear_q8_0_window", "kind": "linear", "fmt": "q8_0", "m": 187, "n": 1280, "k": 5120, "bias": True},
        # a speech-LLM's gate projection over a prompt of audio and text positions
        {"name": "linear_q4_k_prompt", "kind": "linear", "fmt": "q4_k", "m": 413, "n": 5632, "k": 2048, "bias": False},
        # one decoder projection for one stream: the smallest call, latency
        {"name": "linear_q4_0_token", "kind": "linear", "fmt": "q4_0", "m": 1, "n": 1280, "k": 1280, "bias": True},
        # a decoder fc1 for a small batch of streams, five-bit weights
        {"name": "linear_q5_0_streams", "kind": "linear", "fmt": "q5_0", "m": 24, "n": 5120, "k": 1280, "bias": True},
        # encoder self-attention of one utterance
        {"name": "attention_utterance", "kind": "attention", "batch": 1, "t_q": 1500, "t_kv": 1500, "heads": 20,
         "kv_heads": 20, "hd": 64, "causal": False},
        # a speech-LLM prompt's causal attention, eight query heads per kv head
        {"name": "attention_prompt", "kind": "attention", "batch": 1, "t_q": 777, "t_kv": 777, "heads": 16,
         "kv_heads": 2, "hd": 128, "causal": True},
        # a serving batch's decode attention, layer after layer
        {"name": "paged_gqa_streams", "kind": "paged", "layers": 4, "streams": 32, "heads": 16, "kv_heads": 2, "hd": 128,
         "len_lo": 512, "len_hi": 4096},
        # audio in: four 30 s clips to the encoder's input at Whisper-large-v3 dims
        {"name": "frontend_large", "kind": "frontend", "batch": 4, "samples": 480000, "mels": 128, "d": 1280},
        # two encoder blocks at Whisper-large-v3 dims, one utterance
        {"name": "encoder_large_blocks", "kind": "encoder", "fmt": "q8_0", "layers": 2, "d": 1280, "batch": 1, "frames": 1500},
        # a batched decoder step: 64 streams, prefixes up to the text context, four layers and the tied head
        {"name": "decoder_step", "kind": "decoder", "fmt": "q4_0", "layers": 4, "d": 1280, "streams": 64, "prefix": 440,
         "audio": 1500, "vocab": 51866},
        # a batched speech-LLM step: 32 streams, long histories, four layers and the LM head
        {"name": "text_step", "kind": "text", "fmt": "q4_k", "layers": 4, "d": 2048, "heads": 16, "kv_heads": 2, "hd": 128,
         "ff": 5632, "streams": 32, "len_lo": 256, "len_hi": 2048, "vocab": 32000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    # the linears carry most calls of every model here, so they come most often
    kind = rng.choice(["linear"] * 5 + ["attention"] * 2 + ["paged", "frontend", "encoder", "decoder", "text"])
    c = {"kind": kind}
    if kind == "linear":
        c["fmt"] = rng.choice(["q4_0", "q5_0", "q8_0", "q4_k", "q5_k", "q6_k"])
        k, n = rng.choice([(512, 512), (512, 2048), (2048, 512), (768, 768), (768, 3072), (3072, 768), (1024, 1024),
                           (1024, 4096), (4096, 1024), (1280, 1280), (1280, 5120), (5120, 1280), (2048, 2048),
                           (2048, 256), (2048, 5632), (5632, 2048)] +
                          ([(384, 384), (384, 1536), (1536, 384)] if c["fmt"][-1] == "0" else []))
        # decode batches, windows and prompts, whole utterances
        m = rng.choice([_log(rng, 1, 64), _log(rng, 65, 600), _log(rng, 600, 1500)])
        m = min(m, max(1, 1500 * 5120 * 1280 // (n * k)))
        c.update(m=m, n=n, k=k, bias=rng.random() < 0.7)
    elif kind == "attention":
        way = rng.choice(["self", "prompt", "cross"])
        if way == "prompt":  # causal, perhaps after a history
            heads, kv, hd = rng.choice([(16, 2, 128), (32, 8, 128), (16, 16, 64)])
            t = _log(rng, 32, 1200)
            c.update(batch=1, t_q=t, t_kv=t + rng.choice([0, 0, _log(rng, 16, 300)]), heads=heads, kv_heads=kv, hd=hd, causal=True)
        else:
            heads = rng.choice([6, 8, 12, 16, 20])
            t = rng.choice([1500, _log(rng, 100, 1500)])
            batch = rng.choice([1, 1, 2]) if t * heads <= 15000 else 1
            tq = t if way == "self" else _log(rng, 2, 64)
            c.update(batch=batch, t_q=tq, t_kv=t, heads=heads, kv_heads=heads, hd=64, causal=False)
    elif kind == "paged":
        heads, kv, hd = rng.choice([(16, 2, 128), (32, 8, 128), (20, 20, 64), (8, 8, 64)])
        hi = _log(rng, 128, 448) if hd == 64 else _log(rng, 400, 4096)
        c.update(layers=4, streams=_log(rng, 1, 32), heads=heads, kv_heads=kv, hd=hd, len_lo=max(2, hi // 8), len_hi=hi)
    elif kind == "frontend":
        c.update(batch=rng.randint(1, 4), samples=rng.choice([480000, rng.randint(16000, 480000)]), mels=rng.choice([80, 128]),
                 d=rng.choice([384, 512, 768, 1024, 1280]))
    elif kind == "encoder":
        c.update(fmt=rng.choice(["q8_0", "q8_0", "q4_0", "q5_0", "q4_k", "q6_k"]), layers=2,
                 d=rng.choice([512, 768, 1024, 1280]), batch=1, frames=rng.choice([1500, _log(rng, 100, 1499)]))
    elif kind == "decoder":
        d, vocab = rng.choice([(512, 51865), (768, 51865), (1024, 51865), (1280, 51866)])
        c.update(fmt=rng.choice(["q4_0", "q8_0", "q5_0"]), layers=rng.randint(2, 4), d=d, streams=_log(rng, 1, 64),
                 prefix=_log(rng, 8, 200), audio=1500, vocab=vocab)
    else:
        hi = _log(rng, 64, 2048)
        c.update(fmt=rng.choice(["q4_k", "q4_k", "q6_k"]), layers=rng.randint(2, 4), d=2048, heads=16, kv_heads=2, hd=128,
                 ff=5632, streams=_log(rng, 1, 32), len_lo=max(1, hi // 8), len_hi=hi, vocab=32000)
    return c


_FAMILY = {k: {n: globals()["_%s_%s" % (k, n)] for n in ("prepare", "run", "exact", "work")}
           for k in ("linear", "attention", "paged", "frontend", "encoder", "decoder", "text")}


def prepare(case, seed):
    s = _FAMILY[case["kind"]]["prepare"](case, seed)
    torch.cuda.synchronize()
    return case, s


def run(state):
    case, s = state
    return _FAMILY[case["kind"]]["run"](case, s)


def exact(case, seed):
    with torch.no_grad():
        return _FAMILY[case["kind"]]["exact"](case, seed)


def work(case):
    return _FAMILY[case["kind"]]["work"](case)


def tolerance(case):
    # About four times the distance from exact() that a correct run shows. Linears: exact integer block sums, one f32
    # multiply-add chain over the blocks; attention: f32-level products. The sessions: a last-bit change that moves an
    # activation across an INT8 rounding boundary (one step of 127) spreads through the layers and the Q8_0 cache.
    return {"linear": {"rel": 1e-6}, "attention": {"rel": 2e-6}, "paged": {"rel": 2e-5}, "frontend": {"rel": 5e-6},
            "encoder": {"rel": 7e-3}, "decoder": {"rel": 3e-2}, "text": {"rel": 2.5e-2}}[case["kind"]]
