"""The calls a transcription program makes of this library, as cases to time.

One 30 s window goes through the encoder (t = 1500 rows, fewer with a reduced
audio context, 8 windows stacked to 12000 rows in batched use), then through
the decoder: the cross-attention K/V once, a prompt, and one step per token
for one beam or five.  Model files are quantized (every ggml type the library
reads) or dense f32.  The widths are Whisper's: tiny 384, base 512, small 768,
medium 1024, large-v3 and turbo 1280.

Kinds of case (the "kind" field):
  linear   one quantized product, device or host pointers (matmul_t_q)
  dense    one product with an f32 weight (matmul_t_f32)
  set      the decoder's per-token linears as one prepared group
  attn     multi-head attention on device rows
  encoder  encoder layers on a window's rows
  prefill  set_audio, a prompt and the logits of its last row
  greedy   one beam: a prompt, then one-token steps with logits
  beams    five beams' steps with stacked logits, log_softmax and top-k
"""
import numpy as np
import torch

from rusty_whisper_amd import _abi as A

DEV = "cuda:0"
QK = 32
TYPES = {"Q4_0": 2, "Q4_1": 3, "Q5_0": 6, "Q5_1": 7, "Q8_0": 8}
BLOCK_BYTES = {"Q4_0": 18, "Q4_1": 20, "Q5_0": 22, "Q5_1": 24, "Q8_0": 34}
WIDTHS = (384, 512, 768, 1024, 1280)
VOCAB = 51866
TEXT_CTX = 448
PROMPT = 4  # sot, language, task, no-timestamps


# ----------------------------------------------------------------- cases

def listed():
    return [
        # tiny.en's smallest product, one decoding row: a call's own latency
        dict(name="linear_tiny_m1", kind="linear", where="device", type="Q5_1", m=1, n=384, k=384, bias=True),
        # turbo's fc1 over 8 stacked windows: the largest product
        dict(name="linear_batch", kind="linear", where="device", type="Q5_1", m=12000, n=5120, k=1280, bias=True),
        # the drop-in route of a CPU program: small.en's q on host arrays
        dict(name="linear_host", kind="linear", where="host", type="Q8_0", m=1500, n=768, k=768, bias=True),
        # a dense model file (no quantization): large-v3's out projection
        dict(name="dense_window", kind="dense", m=1500, n=1280, k=1280, bias=True),
        # the same model's decoding rows: base's fc1 for one beam
        dict(name="dense_m1", kind="dense", m=1, n=2048, k=512, bias=True),
        # large-v3's decoder linears for five beams from HBM
        dict(name="decode_set", kind="set", type="Q5_0", m=5, d=1280, layers=32, vocab=VOCAB),
        # large-v3's encoder self-attention
        dict(name="attention_window", kind="attn", t_q=1500, t_kv=1500, heads=20, causal=False),
        # one large-v3 encoder layer on a whole window
        dict(name="encoder_large", kind="encoder", type="Q5_1", t=1500, d=1280, layers=1),
        # the whole tiny encoder at a reduced audio context (an odd length)
        dict(name="encoder_tiny", kind="encoder", type="Q8_0", t=749, d=384, layers=4),
        # turbo: a new window and a long prompt (previous text as context)
        dict(name="prefill_turbo", kind="prefill", type="Q5_0", d=1280, layers=4, audio=1500, vocab=VOCAB, tokens=227),
        # turbo, greedy: a prompt and 12 tokens
        dict(name="greedy_turbo", kind="greedy", type="Q5_0", d=1280, layers=4, audio=1500, vocab=VOCAB, steps=12),
        # small, beam search: five beams' first 6 positions
        dict(name="beams_small", kind="beams", type="Q8_0", d=768, layers=12, audio=1500, vocab=VOCAB, steps=6, beams=5,
             topk=5),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "dense", "set", "attn", "encoder", "encoder", "prefill", "greedy", "beams"))
    qt = rng.choice(sorted(TYPES))
    d = rng.choice(WIDTHS)
    bias = rng.random() < 0.8
    if kind == "linear":
        n, k = rng.choice(((d, d), (4 * d, d), (d, 4 * d)))
        m = rng.choice((rng.randint(1, 8), _log_int(rng, 9, 1500), _log_int(rng, 9, 12000)))
        where = "host" if rng.random() < 0.2 else "device"
        if where == "host":
            m = min(m, 1500)
        return dict(kind=kind, where=where, type=qt, m=m, n=n, k=k, bias=bias)
    if kind == "dense":
        n, k = rng.choice(((d, d), (4 * d, d), (d, 4 * d)))
        m = rng.choice((rng.randint(1, 8), _log_int(rng, 9, 1500)))
        return dict(kind=kind, m=m, n=n, k=k, bias=bias)
    if kind == "set":
        return dict(kind=kind, type=qt, m=rng.randint(1, 8), d=d, layers=rng.choice((4, 6, 12)), vocab=rng.choice((51864, 51865, VOCAB)))
    if kind == "attn":
        heads = d // 64
        causal = rng.random() < 0.4
        if causal:
            t_kv = _log_int(rng, 4, TEXT_CTX)
            t_q = rng.choice((1, t_kv, rng.randint(1, t_kv)))
        else:
            t_kv = _log_int(rng, 100, 1500)
            t_q = rng.choice((t_kv, t_kv, rng.randint(1, TEXT_CTX)))
        return dict(kind=kind, t_q=t_q, t_kv=t_kv, heads=heads, causal=causal)
    if kind == "encoder":
        return dict(kind=kind, type=qt, t=_log_int(rng, 100, 1500), d=d, layers=rng.choice((1, 2, 4)))
    layers = rng.choice((2, 4, 6))
    audio = rng.choice((1500, 1500, rng.randint(100, 1499)))
    if kind == "prefill":
        return dict(kind=kind, type=qt, d=d, layers=layers, audio=audio, vocab=VOCAB, tokens=_log_int(rng, 2, 230))
    if kind == "greedy":
        return dict(kind=kind, type=qt, d=d, layers=layers, audio=audio, vocab=VOCAB, steps=rng.randint(2, 16))
    return dict(kind=kind, type=qt, d=d, layers=layers, audio=audio, vocab=VOCAB, steps=rng.randint(2, 6),
                beams=rng.randint(2, 8), topk=rng.randint(1, 8))


# ------------------------------------------------------ quantized weights

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _randn(g, *shape, scale=1.0, shift=0.0):
    return torch.randn(*shape, device=DEV, generator=g) * scale + shift


def _codes(qt, w):
    """ggml's quantization of f32 rows w [n, k]: per 32-block the scale d and
    (Q*_1) the minimum m as f16, and the stored codes [n, nb, 32]."""
    b = w.reshape(w.shape[0], -1, QK)
    one = torch.ones((), device=w.device)
    if qt in ("Q4_1", "Q5_1"):
        top = 15.0 if qt == "Q4_1" else 31.0
        lo, hi = b.amin(-1, keepdim=True), b.amax(-1, keepdim=True)
        d = (hi - lo) / top
        q = torch.clamp(torch.round((b - lo) / torch.where(d > 0, d, one)), 0, top)
        return d.squeeze(-1).half(), lo.squeeze(-1).half(), q.to(torch.uint8)
    if qt == "Q8_0":
        d = b.abs().amax(-1, keepdim=True) / 127.0
        q = torch.clamp(torch.round(b / torch.where(d > 0, d, one)), -127, 127)
        return d.squeeze(-1).half(), None, q.to(torch.int8)
    half = 8.0 if qt == "Q4_0" else 16.0
    at = b.abs().argmax(-1, keepdim=True)
    d = b.gather(-1, at) / -half
    q = torch.clamp(torch.round(b / torch.where(d != 0, d, one)) + half, 0, 2 * half - 1)
    return d.squeeze(-1).half(), None, q.to(torch.uint8)


def _raw(qt, codes):
    """The codes as ggml blocks (a host byte array)."""
    d, m, q = codes
    put = lambda x: x.contiguous().view(torch.uint8).reshape(d.shape[0], d.shape[1], -1)  # noqa: E731
    parts = [put(d)] + ([put(m)] if m is not None else [])
    if qt == "Q8_0":
        parts.append(put(q))
    else:
        if qt in ("Q5_0", "Q5_1"):
            bits = ((q >> 4).reshape(*q.shape[:2], 4, 8).to(torch.int32) << torch.arange(8, device=q.device, dtype=torch.int32)).sum(-1)
            parts.append(bits.to(torch.uint8))
        parts.append((q[..., :16] & 15) | ((q[..., 16:] & 15) << 4))
    return torch.cat(parts, -1).reshape(-1).cpu().numpy()


def _dequant(qt, codes):
    """The values the blocks stand for, in 64 bits, [n, k]."""
    d, m, q = codes
    off = {"Q4_0": 8, "Q5_0": 16}.get(qt, 0)
    v = (q.double() - off) * d.double().unsqueeze(-1)
    if m is not None:
        v = v + m.double().unsqueeze(-1)
    return v.reshape(d.shape[0], -1)


class _Given:
    """What a case's weights are made from: quantized matrices and vectors in
    a fixed order, from the seed alone, for the library (`exact` False:
    resident handles) or in 64 bits."""

    def __init__(self, seed, exact):
        self.g, self.exact = _gen(seed), exact

    def weight(self, qt, n, k, scale=None):
        w = _randn(self.g, n, k, scale=scale if scale is not None else 0.7 / k ** 0.5)
        c = _codes(qt, w)
        if self.exact:
            return _dequant(qt, c)
        return A.DeviceWeight(TYPES[qt], n, k, _raw(qt, c))

    def vec(self, *shape, scale=0.1, shift=0.0):
        v = _randn(self.g, *shape, scale=scale, shift=shift)
        return v.double() if self.exact else v

    def encoder_layer(self, qt, d):
        p = {}
        for nm in ("q", "k", "v", "out"):
            p[nm] = self.weight(qt, d, d)
        p["fc1"], p["fc2"] = self.weight(qt, 4 * d, d), self.weight(qt, d, 4 * d)
        for nm in ("q_b", "v_b", "out_b", "fc2_b"):
            p[nm] = self.vec(d)
        p["fc1_b"] = self.vec(4 * d)
        for ln in ("attn_ln", "mlp_ln"):
            p[ln + "_w"], p[ln + "_b"] = self.vec(d, shift=1.0), self.vec(d)
        return p

    def decoder(self, c):
        qt, d = c["type"], c["d"]
        layers = []
        for _ in range(c["layers"]):
            p = self.encoder_layer(qt, d)
            for nm in ("cq", "ck", "cv", "cout"):
                p[nm] = self.weight(qt, d, d)
            for nm in ("cq_b", "cv_b", "cout_b"):
                p[nm] = self.vec(d)
            p["cross_ln_w"], p["cross_ln_b"] = self.vec(d, shift=1.0), self.vec(d)
            layers.append(p)
        emb = self.weight(qt, c["vocab"], d, scale=0.04)
        return layers, emb, self.vec(TEXT_CTX, d, scale=0.03), self.vec(d, shift=1.0), self.vec(d)

    def tokens(self, c, *shape):
        return torch.randint(0, c["vocab"], shape, device=DEV, generator=self.g).cpu().numpy()


def _stream():
    return torch.cuda.current_stream().cuda_stream


# ---------------------------------------------------------------- prepare

def _set_shapes(c):
    d = c["d"]
    return [(d, d)] * 8 + [(4 * d, d), (d, 4 * d)]


def prepare(case, seed):
    c, G = case, _Given(seed, False)
    s = {"case": c}
    kind = c["kind"]
    if kind == "linear":
        s["w"] = G.weight(c["type"], c["n"], c["k"])
        s["a"] = G.vec(c["m"], c["k"], scale=1.0)
        s["bias"] = G.vec(c["n"]) if c["bias"] else None
        if c["where"] == "host":
            s["a"] = s["a"].cpu().numpy()
            s["bias"] = None if s["bias"] is None else s["bias"].cpu().numpy()
        else:
            s["out"] = torch.empty(c["m"], c["n"], device=DEV)
            s["ws_len"] = max(1, A.workspace_size(c["m"], c["k"]))
            s["ws"] = torch.empty(s["ws_len"], dtype=torch.uint8, device=DEV)
    elif kind == "dense":
        s["b"] = G.vec(c["n"], c["k"], scale=0.7 / c["k"] ** 0.5)
        s["a"] = G.vec(c["m"], c["k"], scale=1.0)
        s["bias"] = G.vec(c["n"]) if c["bias"] else None
        s["out"] = torch.empty(c["m"], c["n"], device=DEV)
    elif kind == "set":
        m, shapes = c["m"], _set_shapes(c)
        total = c["layers"] * sum(n for n, _ in shapes) + c["vocab"]
        s["out"], s["keep"], items, at = torch.empty(m * total, device=DEV), [], [], 0
        for n, k in shapes * c["layers"] + [(c["vocab"], c["d"])]:
            w, a, b = G.weight(c["type"], n, k), G.vec(m, k, scale=1.0), G.vec(n)
            s["keep"].append((w, a, b))
            items.append((w, a, b, s["out"][at:at + m * n], m))
            at += m * n
        s["group"] = A.Group(A.make_linears(items))
    elif kind == "attn":
        n = 64 * c["heads"]
        # projections of layernormed rows: peaked in some rows, flat in others
        s["q"], s["k"], s["v"] = G.vec(c["t_q"], n, scale=1.5), G.vec(c["t_kv"], n, scale=1.5), G.vec(c["t_kv"], n, scale=1.0)
        s["out"] = torch.empty(c["t_q"], n, device=DEV)
        s["ws_len"] = max(1, A.attention_workspace_size(c["t_q"], c["t_kv"], n))
        s["ws"] = torch.empty(s["ws_len"], dtype=torch.uint8, device=DEV)
    elif kind == "encoder":
        s["layers"] = [A.EncoderLayer(c["d"] // 64, **G.encoder_layer(c["type"], c["d"])) for _ in range(c["layers"])]
        s["stem"], s["pos"] = G.vec(c["t"], c["d"], scale=0.8), G.vec(c["t"], c["d"], scale=0.3)
        s["x"] = torch.empty(c["t"], c["d"], device=DEV)
        s["ws_len"] = s["layers"][0].workspace_size(c["t"])
        s["ws"] = torch.empty(s["ws_len"], dtype=torch.uint8, device=DEV)
    else:
        d = c["d"]
        layers, emb, pos, lw, lb = G.decoder(c)
        s["emb"] = emb
        s["dec"] = A.Decoder(d // 64, TEXT_CTX, c["audio"], layers, emb, pos, lw, lb)
        s["enc"] = G.vec(c["audio"], d, scale=1.0)
        if kind == "prefill":
            s["tokens"] = G.tokens(c, c["tokens"])
            s["hidden"], s["logits"] = torch.empty(c["tokens"], d, device=DEV), torch.empty(1, c["vocab"], device=DEV)
        elif kind == "greedy":
            s["tokens"] = G.tokens(c, PROMPT + c["steps"])
            s["hidden"] = torch.empty(PROMPT + c["steps"], d, device=DEV)
            s["logits"] = torch.empty(1 + c["steps"], c["vocab"], device=DEV)
            s["dec"].set_audio(s["enc"], _stream())
        else:
            nb, k = c["beams"], c["topk"]
            s["tokens"] = G.tokens(c, c["steps"], nb)
            s["dec"].set_audio(s["enc"], _stream())
            s["beams"] = [s["dec"]] + [s["dec"].fork(_stream()) for _ in range(nb - 1)]
            s["hidden"] = torch.empty(c["steps"], nb, d, device=DEV)
            s["logits"] = torch.empty(c["steps"], nb, c["vocab"], device=DEV)
            s["ids"] = torch.empty(c["steps"], nb, k, dtype=torch.int32, device=DEV)
            s["lps"] = torch.empty(c["steps"], nb, k, device=DEV)
    return s


# -------------------------------------------------------------------- run

def run(state):
    s, c, st = state, state["case"], _stream()
    kind = c["kind"]
    if kind == "linear":
        if c["where"] == "host":
            return s["w"].matmul(s["a"], s["bias"])
        s["w"].matmul_dev(s["a"], c["m"], s["out"], s["bias"], s["ws"], s["ws_len"], st)
        return s["out"]
    if kind == "dense":
        A.matmul_t_f32_dev(s["a"], c["m"], c["k"], s["b"], c["n"], s["out"], s["bias"], st)
        return s["out"]
    if kind == "set":
        s["group"].run(st)
        return s["out"]
    if kind == "attn":
        A.attention_dev(s["q"], s["k"], s["v"], c["t_q"], c["t_kv"], 64 * c["heads"], c["heads"], c["causal"], s["out"],
                        workspace=s["ws"], workspace_len=s["ws_len"], stream=st)
        return s["out"]
    if kind == "encoder":
        torch.add(s["stem"], s["pos"], out=s["x"])  # the conv stem's rows and the positions
        for layer in s["layers"]:
            layer.run(s["x"], c["t"], s["ws"], s["ws_len"], st)
        return s["x"]
    dec, emb, hid, logits = s["dec"], s["emb"], s["hidden"], s["logits"]
    if kind == "prefill":
        dec.set_audio(s["enc"], st)
        dec.forward_hidden(s["tokens"], hid, st)
        emb.matmul_dev(hid[-1:], 1, logits, stream=st)
        return {"hidden": hid, "logits": logits}
    if kind == "greedy":
        dec.reset()
        dec.forward_hidden(s["tokens"][:PROMPT], hid[:PROMPT], st)
        emb.matmul_dev(hid[PROMPT - 1], 1, logits[0], stream=st)
        for i in range(c["steps"]):
            at = PROMPT + i
            dec.forward_hidden(s["tokens"][at:at + 1], hid[at], st)
            emb.matmul_dev(hid[at], 1, logits[1 + i], stream=st)
        return {"hidden": hid, "logits": logits}
    for b in s["beams"]:
        b.reset()
    for i in range(c["steps"]):
        A.decoder_forward_beams(s["beams"], s["tokens"][i], hid[i], st)
        emb.matmul_dev(hid[i], c["beams"], logits[i], stream=st)
        A.logits_topk_dev(logits[i], c["beams"], c["vocab"], c["topk"], s["ids"][i], s["lps"][i], st)
    return {"hidden": hid, "ids": s["ids"], "logits": logits, "logprobs": s["lps"]}


# ------------------------------------------------------------------- work

def _attn_work(t_q, t_kv, d, causal=False):
    pairs = t_q * (t_kv - t_q) + t_q * (t_q + 1) // 2 if causal else t_q * t_kv
    return 4 * pairs * d


def work(case):
    c = case
    kind = c["kind"]
    wb = lambda n, k: n * (k // QK) * BLOCK_BYTES[c["type"]]  # noqa: E731
    if kind == "linear":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": wb(n, k) + 4 * m * (n + k) + (4 * n if c["bias"] else 0), "flops": 2 * m * n * k}
    if kind == "dense":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 4 * (n * k + m * n + m * k) + (4 * n if c["bias"] else 0), "flops": 2 * m * n * k}
    if kind == "set":
        sh, m = _set_shapes(c) * c["layers"] + [(c["vocab"], c["d"])], c["m"]
        return {"bytes": sum(wb(n, k) + 4 * m * (n + k) + 4 * n for n, k in sh), "flops": sum(2 * m * n * k for n, k in sh)}
    if kind == "attn":
        d = 64 * c["heads"]
        return {"bytes": 4 * d * 2 * (c["t_q"] + c["t_kv"]), "flops": _attn_work(c["t_q"], c["t_kv"], d, c["causal"])}
    d, L = c["d"], c["layers"]
    if kind == "encoder":
        t = c["t"]
        return {"bytes": L * 12 * wb(d, d) + 12 * t * d, "flops": L * (24 * t * d * d + _attn_work(t, t, d))}
    au, V = c["audio"], c["vocab"]
    per = lambda m: L * 28 * m * d * d  # noqa: E731  q k v out, cross q and out, fc1, fc2: 14 d^2 weights per row
    cross = 2 * au * d * 4  # the window's K and V rows
    layer_w = 14 * wb(d, d)
    if kind == "prefill":
        t = c["tokens"]
        return {"bytes": L * (layer_w + 2 * wb(d, d)) + 4 * au * d + wb(V, d) + 4 * (V + t * d),
                "flops": L * 4 * au * d * d + per(t) + 2 * V * d
                + L * (_attn_work(t, t, d, True) + _attn_work(t, au, d))}
    if kind == "greedy":
        n = c["steps"]
        return {"bytes": (n + 1) * (L * (layer_w + cross) + wb(V, d) + 4 * V) + 4 * d * (PROMPT + n),
                "flops": per(PROMPT + n) + 2 * (n + 1) * V * d
                + L * (_attn_work(PROMPT + n, PROMPT + n, d, True) + _attn_work(PROMPT + n, au, d))}
    n, nb = c["steps"], c["beams"]
    return {"bytes": n * (L * (layer_w + cross) + wb(V, d) + 8 * nb * V + 4 * nb * d),
            "flops": nb * (per(n) + 2 * n * V * d + L * (_attn_work(n, n, d, True) + _attn_work(n, au, d)))}


# -------------------------------------------------------------- tolerance

def tolerance(case):
    c = case
    kind = c["kind"]
    if kind == "dense":
        return "exact"  # the entry promises the reference's bits
    if kind == "linear":
        # few rows: exact block sums combined in f32; more: f16 operands
        return {"rel": 4e-6} if c["m"] <= 8 else {"rel": 1e-3}
    if kind == "set":
        return {"rel": 4e-6}
    if kind == "attn":
        return {"rel": 3e-6}
    # activations pass through int8 blocks at every product, so a last-bit
    # difference moves a few codes by one and travels through later layers:
    # against 64 bits 0.0017 over one layer, 0.0054 over four, 0.014 over the
    # decoders' twelve; neighbours among the best ids then change places
    if kind == "encoder":
        return {"rel": 0.007 + 0.005 * (c["layers"] - 1)}
    return {"rel": 0.05, "differ": 0.6} if kind == "beams" else {"rel": 0.04}


# ------------------------------------------------------------------ exact

def _quantized(x):
    """Rows as the products see them: int8 codes per 32-block (amax / 127 in
    f32, half away from zero), back as 64-bit values."""
    b = x.float().reshape(x.shape[0], -1, QK)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    v = b * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    q = torch.clamp(torch.sign(v) * torch.floor(v.abs().double() + 0.5), -127, 127)
    return (q * d.double()).reshape(x.shape)


def _product(x, w, bias=None):
    y = _quantized(x) @ w.t().contiguous()
    return y if bias is None else y + bias


def _norm(x, w, b):
    mean = x.mean(-1, keepdim=True)
    var = ((x - mean) ** 2).mean(-1, keepdim=True)
    return (x - mean) / torch.sqrt(var + 1e-5) * w + b


def _gelu(t):
    return 0.5 * t * (1.0 + torch.tanh(0.7978846 * (t + 0.044715 * t * t * t)))


def _attention(q, k, v, heads, causal):
    out = torch.empty_like(q)
    t_q, t_kv = q.shape[0], k.shape[0]
    hide = None
    if causal:
        hide = torch.arange(t_kv, device=DEV)[None, :] > (torch.arange(t_q, device=DEV) + t_kv - t_q)[:, None]
    for h in range(heads):
        i = slice(64 * h, 64 * h + 64)
        sc = (q[:, i].contiguous() @ k[:, i].t().contiguous()) * 0.125
        if causal:
            sc = sc.masked_fill(hide, float("-inf"))
        out[:, i] = torch.softmax(sc, -1) @ v[:, i].contiguous()
    return out


def _encoder(p, x, heads):
    h = _norm(x, p["attn_ln_w"], p["attn_ln_b"])
    q, k, v = _product(h, p["q"], p["q_b"]), _product(h, p["k"]), _product(h, p["v"], p["v_b"])
    x = x + _product(_attention(q, k, v, heads, False), p["out"], p["out_b"])
    h = _gelu(_product(_norm(x, p["mlp_ln_w"], p["mlp_ln_b"]), p["fc1"], p["fc1_b"]))
    return x + _product(h, p["fc2"], p["fc2_b"])


def _decode(W, enc, tokens):
    """Hidden rows of one token sequence in one pass (the caches make the
    steps' rows the same)."""
    layers, emb, pos, lw, lb = W
    heads = emb.shape[1] // 64
    x = emb[torch.from_numpy(np.asarray(tokens, dtype=np.int64)).to(DEV)] + pos[:len(tokens)]
    for p in layers:
        h = _norm(x, p["attn_ln_w"], p["attn_ln_b"])
        q, k, v = _product(h, p["q"], p["q_b"]), _product(h, p["k"]), _product(h, p["v"], p["v_b"])
        x = x + _product(_attention(q, k, v, heads, True), p["out"], p["out_b"])
        q = _product(_norm(x, p["cross_ln_w"], p["cross_ln_b"]), p["cq"], p["cq_b"])
        a = _attention(q, _product(enc, p["ck"]), _product(enc, p["cv"], p["cv_b"]), heads, False)
        x = x + _product(a, p["cout"], p["cout_b"])
        h = _gelu(_product(_norm(x, p["mlp_ln_w"], p["mlp_ln_b"]), p["fc1"], p["fc1_b"]))
        x = x + _product(h, p["fc2"], p["fc2_b"])
    return _norm(x, lw, lb)


def exact(case, seed):
    c, G = case, _Given(seed, True)
    kind = c["kind"]
    if kind == "linear":
        w, a = G.weight(c["type"], c["n"], c["k"]), G.vec(c["m"], c["k"], scale=1.0)
        y = _product(a, w, G.vec(c["n"]) if c["bias"] else None)
        return y.cpu().numpy() if c["where"] == "host" else y
    if kind == "dense":
        b, a = G.vec(c["n"], c["k"], scale=0.7 / c["k"] ** 0.5), G.vec(c["m"], c["k"], scale=1.0)
        y = a @ b.t().contiguous()
        return y + G.vec(c["n"]) if c["bias"] else y
    if kind == "set":
        out = []
        for n, k in _set_shapes(c) * c["layers"] + [(c["vocab"], c["d"])]:
            w, a, b = G.weight(c["type"], n, k), G.vec(c["m"], k, scale=1.0), G.vec(n)
            out.append(_product(a, w, b).reshape(-1))
        return torch.cat(out)
    if kind == "attn":
        n = 64 * c["heads"]
        q, k, v = G.vec(c["t_q"], n, scale=1.5), G.vec(c["t_kv"], n, scale=1.5), G.vec(c["t_kv"], n, scale=1.0)
        return _attention(q, k, v, c["heads"], c["causal"])
    if kind == "encoder":
        layers = [G.encoder_layer(c["type"], c["d"]) for _ in range(c["layers"])]
        x = G.vec(c["t"], c["d"], scale=0.8) + G.vec(c["t"], c["d"], scale=0.3)
        for p in layers:
            x = _encoder(p, x, c["d"] // 64)
        return x
    W = G.decoder(c)
    enc = G.vec(c["audio"], c["d"], scale=1.0)
    if kind == "prefill":
        hid = _decode(W, enc, G.tokens(c, c["tokens"]))
        return {"hidden": hid, "logits": _product(hid[-1:], W[1])}
    if kind == "greedy":
        hid = _decode(W, enc, G.tokens(c, PROMPT + c["steps"]))
        return {"hidden": hid, "logits": _product(hid[PROMPT - 1:], W[1])}
    tok = G.tokens(c, c["steps"], c["beams"])
    hid = torch.stack([_decode(W, enc, tok[:, b]) for b in range(c["beams"])], 1)
    logits = _product(hid.reshape(-1, c["d"]), W[1]).reshape(c["steps"], c["beams"], -1)
    return {"hidden": hid, "ids": None, "logits": logits, "logprobs": torch.log_softmax(logits, -1).topk(c["topk"]).values}
