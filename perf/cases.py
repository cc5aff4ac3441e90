"""The work that users of this framework have it do, as timed cases.

A case is a call (or the few calls) that a program makes through the package's
public entry points, at the decoder widths of the 0.3B configuration (hidden
1024, 16 query and 2 KV heads of 128, SwiGLU 3072): token decode, prompt
prefill, batched and continuous-batching decode, the vision projector, and the
op-level calls of a host that keeps its own loop.  Whole-model cases run its 18
layers with the 103,424-row head; the others run stacks of 3 layers with small
vocabularies, whose rounding travels less far.
"""
import math

import numpy as np
import torch

from rapidocrvl_amd import lib
from rapidocrvl_amd.config import DecoderConfig

HIDDEN, INTER, HEADS, KV_HEADS, HEAD_DIM = 1024, 3072, 16, 2, 128
Q_ROWS, KV_ROWS = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
EPS, THETA, SECTIONS = 1e-5, 500000.0, (16, 24, 24)
VOCAB = 103424
VISION = 1152
QT = {"q8": lib.Q8, "q6": lib.Q6, "q4": lib.Q4}
BITS = {"q8": 8, "q6": 6, "q4": 4}
LIM = {"q8": 127, "q6": 31, "q4": 7}
SHAPES = {"q": (Q_ROWS, HIDDEN), "k": (KV_ROWS, HIDDEN), "v": (KV_ROWS, HIDDEN), "o": (HIDDEN, Q_ROWS),
          "gate": (INTER, HIDDEN), "up": (INTER, HIDDEN), "down": (HIDDEN, INTER)}
ROLES = {"q": lib.W_Q, "k": lib.W_K, "v": lib.W_V, "o": lib.W_O, "gate": lib.W_GATE, "up": lib.W_UP,
         "down": lib.W_DOWN}


def listed():
    return [
        # one user's page: decode after a 5 + 1332 + 8 row image prompt, batch 1, the 4-bit model
        {"name": "decode_q4_image", "kind": "decode", "q": "q4", "layers": 18, "vocab": VOCAB, "rows": 1345, "n": 32},
        # short text continuation in the 8-bit model: launches and latency, hardly any cache
        {"name": "decode_q8_text", "kind": "decode", "q": "q8", "layers": 3, "vocab": 5008, "rows": 64, "n": 16},
        # the end of a long document: the cache of 8,192 rows dominates, 6-bit
        {"name": "decode_q6_long", "kind": "decode", "q": "q6", "layers": 3, "vocab": 5000, "rows": 8192, "n": 24},
        # four concurrent requests decoded together at about 2.4k rows of context each
        {"name": "batch4_q6", "kind": "batch", "q": "q6", "layers": 3, "vocab": 5008, "rows": 2403, "seqs": 4,
         "n": 24},
        # a server's full house: 16 image requests in the continuous batch, whole model
        {"name": "serve16_q4", "kind": "serve", "q": "q4", "layers": 18, "vocab": VOCAB, "rows": 1345, "seqs": 16,
         "n": 16},
        # the image prompt of one page through the whole model, with its logits
        {"name": "prefill_q4_image", "kind": "prefill", "q": "q4", "layers": 18, "vocab": VOCAB, "n": 1345, "grid": 36},
        # a 64-id text prompt in the 8-bit model
        {"name": "prefill_q8_text", "kind": "prefill", "q": "q8", "layers": 3, "vocab": 5008, "n": 64, "grid": 0},
        # a long ragged prompt, 6-bit
        {"name": "prefill_q6_long", "kind": "prefill", "q": "q6", "layers": 3, "vocab": 5000, "n": 2403, "grid": 0},
        # the image prompt in the mode that repeats a CPU host's u8-activation results to the bit
        {"name": "prefill_q4_vnni", "kind": "prefill", "q": "q4", "layers": 3, "vocab": 5008, "n": 1345, "grid": 36,
         "vnni": True},
        # the vision projector on one page's 72 x 74 patch grid, host rows in and out
        {"name": "project_page", "kind": "project", "t": 1, "h": 72, "w": 74},
        # the MLP half of a layer as an op-level host calls it, host vectors in and out: the smallest call
        {"name": "mlp_op_q4", "kind": "mlp", "q": "q4"},
        # the candidates of one sampled token from the 6-bit head, op level
        {"name": "head_top40_q6", "kind": "topk", "q": "q6", "vocab": VOCAB, "k": 40},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "batch", "serve", "prefill", "prefill", "prefill", "project", "mlp", "topk"])
    q = rng.choice(["q4", "q6", "q8"])
    if kind == "decode":
        whole = rng.random() < 0.4
        return {"kind": kind, "q": q, "layers": 18 if whole else 3, "vocab": VOCAB if whole else rng.choice([5000, 5008]),
                "rows": _log_int(rng, 5, 2048 if whole else 8192), "n": rng.randint(6, 32)}
    if kind == "batch":
        return {"kind": kind, "q": q, "layers": 3, "vocab": rng.choice([5000, 5008]), "rows": _log_int(rng, 48, 2500),
                "seqs": rng.randint(2, 4), "n": rng.randint(8, 24)}
    if kind == "serve":
        return {"kind": kind, "q": q, "layers": 3, "vocab": rng.choice([5000, 5008]), "rows": _log_int(rng, 48, 2500),
                "seqs": rng.randint(3, 16), "n": rng.randint(8, 24)}
    if kind == "prefill":
        vnni = q != "q8" and rng.random() < 0.2
        n = _log_int(rng, 7, 1400 if vnni else 2500)
        side = int(math.sqrt(n * 0.9)) if n > 200 and rng.random() < 0.5 else 0
        return {"kind": kind, "q": q, "layers": 3, "vocab": rng.choice([5000, 5008]), "n": n, "grid": side, "vnni": vnni}
    if kind == "project":
        return {"kind": kind, "t": rng.choice([1, 1, 2]), "h": _log_int(rng, 8, 64), "w": _log_int(rng, 8, 64)}
    if kind == "mlp":
        return {"kind": kind, "q": q, "residual": round(rng.uniform(0.2, 4.0), 3)}
    return {"kind": kind, "q": q, "vocab": rng.choice([VOCAB, _log_int(rng, 5000, VOCAB)]), "k": rng.randint(2, 64)}


# ---------------------------------------------------------------------------
# inputs: everything from the seed, drawn on the GPU
# ---------------------------------------------------------------------------


def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1009 + part)
    return g


def _normal(g, shape, std=0.02):
    """Checkpoint-like values: normal, rounded to bf16, held in f32."""
    return (torch.randn(shape, generator=g, device="cuda") * std).bfloat16().float()


def _quantized(g, shape, q, w=None):
    """Row-quantized codes: scale = max|w| / limit, rounded half away from zero."""
    w = _normal(g, shape) if w is None else w
    scale = w.abs().amax(1) / torch.full((1,), float(LIM[q]), device="cuda")  # by a tensor: correctly rounded
    v = w * (1.0 / scale)[:, None]
    codes = torch.where(v >= 0, (v + 0.5).floor(), (v - 0.5).ceil()).clamp(-LIM[q], LIM[q]).to(torch.int8)
    return scale, codes


def _packed(q, codes):
    if q == "q8":
        return codes.view(torch.uint8)
    if q == "q4":
        u = (codes + 8).to(torch.uint8)
        return u[:, 0::2] | (u[:, 1::2] << 4)
    u = (codes.to(torch.int32) + 32).view(codes.shape[0], -1, 4)
    bits = u[..., 0] | (u[..., 1] << 6) | (u[..., 2] << 12) | (u[..., 3] << 18)
    return torch.stack([bits & 255, (bits >> 8) & 255, (bits >> 16) & 255], -1).to(torch.uint8).view(codes.shape[0], -1)


def _matrix(q, scale, codes):
    rows, cols = codes.shape
    return lib.QMatrix(QT[q], rows, cols, scale.cpu().numpy(), _packed(q, codes).cpu().numpy())


def _weights(case, seed):
    """The decoder's tensors one after another: (layer, name, value)."""
    g, q = _gen(seed, 1), case["q"]
    for li in range(case["layers"]):
        for name, shape in SHAPES.items():
            yield li, name, _quantized(g, shape, q)
        yield li, "ln1", 1.0 + _normal(g, HIDDEN)
        yield li, "ln2", 1.0 + _normal(g, HIDDEN)
    yield -1, "final", 1.0 + _normal(g, HIDDEN)
    yield -1, "head", _quantized(g, (case["vocab"], HIDDEN), q)
    yield -1, "embed", _normal(g, (case["vocab"], HIDDEN))


def _model(case, seed):
    """A model on the device with its weights, and the host's embedding table."""
    ctx = lib.Context(0)
    m = lib.Model(ctx, DecoderConfig(hidden=HIDDEN, inter=INTER, layers=case["layers"], heads=HEADS, kv_heads=KV_HEADS,
                                     head_dim=HEAD_DIM, vocab=case["vocab"], eps=EPS, rope_theta=THETA,
                                     mrope_section=SECTIONS))
    embed = None
    for li, name, value in _weights(case, seed):
        if name in ROLES:
            m.set_weight(li, ROLES[name], _matrix(case["q"], *value))
        elif name == "head":
            m.set_weight(-1, lib.W_LM_HEAD, _matrix(case["q"], *value))
        elif name == "embed":
            embed = value.cpu().numpy()
            m.set_embed(embed)
        else:
            m.set_norm(li, {"ln1": lib.N_LN1, "ln2": lib.N_LN2, "final": lib.N_FINAL}[name], value.cpu().numpy())
    if case.get("vnni"):
        m.set_vnni(True)
    return m, embed


def _cache(case, seed, member):
    """The K and V rows a prompt left behind, layer by layer: what unit-RMS
    rows through the projections give (0.02 * sqrt(1024) = 0.64)."""
    g = _gen(seed, 100 + member)
    for li in range(case["layers"]):
        kv = torch.randn((2, case["rows"], KV_ROWS), generator=g, device="cuda") * 0.64
        yield li, kv[0], kv[1]


def _member_rows(case, i):
    """Requests of one batch differ in length, as their prompts do."""
    return max(1, case["rows"] - 3 * i)


def _firsts(case, seed):
    """First token and position of each member (an image's rows span few positions)."""
    rng = np.random.default_rng([seed, 3])
    n = case.get("seqs", 1)
    first = [int(t) for t in rng.integers(0, case["vocab"], n)]
    return first, [_member_rows(case, i) // 20 + 3 for i in range(n)]


def _sequences(case, seed, m):
    seqs = []
    for i in range(case.get("seqs", 1)):
        s = m.seq(case["rows"] + case["n"] + 8)
        for li, k, v in _cache(case, seed, i):
            s.write_kv(li, k.cpu().numpy(), v.cpu().numpy(), case["rows"])
        s.truncate(_member_rows(case, i))
        seqs.append(s)
    return seqs


def _positions(n, side):
    """(T, H, W) positions of a prompt: 5 text rows, a side x side image block,
    text again (the block's three axes count from its start), or text only."""
    pos = []
    if side:
        pos = [(i, i, i) for i in range(5)]
        for r in range(side):
            pos += [(5, 5 + r, 5 + c) for c in range(side)]
    at = 5 + side if side else 0
    while len(pos) < n:
        pos.append((at, at, at))
        at += 1
    return np.array(pos[:n], np.int32)


def _prompt(case, seed):
    """Prompt rows: image rows of unit scale between text embeddings."""
    g = _gen(seed, 2)
    x = torch.randn((case["n"], HIDDEN), generator=g, device="cuda")
    image = 5 + case["grid"] ** 2
    if case["grid"]:
        x[:5] *= 0.02
        x[image:] *= 0.02
    else:
        x *= 0.02
    return x


def _vision(case, seed):
    g = _gen(seed, 4)
    k = 4 * VISION
    return {"norm_w": 1.0 + _normal(g, VISION), "norm_b": _normal(g, VISION), "w1": _normal(g, (k, k)),
            "b1": _normal(g, k), "w2": _normal(g, (HIDDEN, k)), "b2": _normal(g, HIDDEN),
            "rows": torch.randn((case["t"] * case["h"] * case["w"], VISION), generator=g, device="cuda")}


def _mlp(case, seed):
    g = _gen(seed, 5)
    w = {name: _quantized(g, SHAPES[name], case["q"]) for name in ("gate", "up", "down")}
    return w, {"x": torch.randn(HIDDEN, generator=g, device="cuda"),
               "residual": torch.randn(HIDDEN, generator=g, device="cuda") * case.get("residual", 1.0),
               "norm": 1.0 + _normal(g, HIDDEN)}


def _head(case, seed):
    g = _gen(seed, 6)
    return _quantized(g, (case["vocab"], HIDDEN), case["q"]), torch.randn(HIDDEN, generator=g, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind in ("decode", "batch", "serve"):
        m, embed = _model(case, seed)
        first, pos = _firsts(case, seed)
        seqs = _sequences(case, seed, m)
        if kind == "serve":
            st["batch"] = lib.Batch(m)
        st.update(seqs=seqs, first=first, pos=pos, embed=embed, model=m)
    elif kind == "prefill":
        m, _ = _model(case, seed)
        st.update(seq=m.seq(case["n"] + 256), rows=_prompt(case, seed).cpu().numpy(),
                  pos=_positions(case["n"], case["grid"]), model=m)
    elif kind == "project":
        v = {k: t.cpu().numpy() for k, t in _vision(case, seed).items()}
        rows = v.pop("rows")
        st.update(proj=lib.Projector(lib.Context(0), v["norm_w"], v["norm_b"], v["w1"], v["b1"], v["w2"], v["b2"], EPS),
                  rows=rows)
    elif kind == "mlp":
        w, v = _mlp(case, seed)
        ctx = lib.Context(0)
        st.update({name: ctx.upload(_matrix(case["q"], *w[name])) for name in w})
        st.update({name: t.cpu().numpy() for name, t in v.items()}, ctx=ctx)
    else:
        w, x = _head(case, seed)
        ctx = lib.Context(0)
        st.update(head=ctx.upload(_matrix(case["q"], *w)), x=x.cpu().numpy(), ctx=ctx)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def _next_logits(st, i, token, pos):
    """What follows a generated token, as a program asks that ranks continuations itself."""
    return st["seqs"][i].step(st["embed"][token], (pos, pos, pos))[1]


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "decode":
        s, n = st["seqs"][0], case["n"]
        s.truncate(case["rows"])
        tokens = s.decode_greedy(st["first"][0], st["pos"][0], n, eos=())
        return {"tokens": tokens, "logits": _next_logits(st, 0, tokens[-1], st["pos"][0] + n - 1)}
    if kind in ("batch", "serve"):
        n = case["n"]
        for i, s in enumerate(st["seqs"]):
            s.truncate(_member_rows(case, i))
        if kind == "batch":
            tokens = lib.decode_batch(st["seqs"], st["first"], st["pos"], n, eos=())
        else:
            b = st["batch"]
            for s, t, p in zip(st["seqs"], st["first"], st["pos"]):
                b.join(s, t, p, n, eos=())
            while b.step(16):
                pass
            tokens = [b.leave(s) for s in st["seqs"]]
        last = len(tokens) - 1
        return {"tokens": tokens, "logits": _next_logits(st, last, tokens[last][-1], st["pos"][last] + n - 1)}
    if kind == "prefill":
        st["seq"].reset()
        token, logits = st["seq"].prefill(st["rows"], st["pos"], want_logits=True)
        return {"token": token, "logits": logits}
    if kind == "project":
        return st["proj"].project(st["rows"], (case["t"], case["h"], case["w"]))
    if kind == "mlp":
        return st["ctx"].swiglu_down_add_rmsnorm(st["gate"], st["up"], st["down"], st["x"], st["residual"], st["norm"],
                                                 EPS, True)
    return st["ctx"].matvec_topk(st["head"], st["x"], case["k"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def _matrix_bytes(q, rows, cols):
    return rows * (cols * BITS[q] // 8 + 4)


def work(case):
    kind = case["kind"]
    if kind == "project":
        rows = case["t"] * (case["h"] // 2) * (case["w"] // 2)
        k = 4 * VISION
        return {"bytes": 4 * case["t"] * case["h"] * case["w"] * VISION + k * k + HIDDEN * k + 4 * rows * HIDDEN,
                "flops": 2 * rows * (k * k + HIDDEN * k)}
    if kind == "mlp":
        return {"bytes": sum(_matrix_bytes(case["q"], *SHAPES[n]) for n in ("gate", "up", "down")) + 5 * 4 * HIDDEN,
                "flops": 6 * HIDDEN * INTER}
    if kind == "topk":
        return {"bytes": _matrix_bytes(case["q"], case["vocab"], HIDDEN) + 4 * HIDDEN + 8 * case["k"],
                "flops": 2 * case["vocab"] * HIDDEN}
    layer = sum(_matrix_bytes(case["q"], *s) for s in SHAPES.values())
    layer_macs = sum(r * c for r, c in SHAPES.values())
    head, head_macs = _matrix_bytes(case["q"], case["vocab"], HIDDEN), case["vocab"] * HIDDEN
    row = 2 * 4 * KV_ROWS
    if kind == "prefill":
        n = case["n"]
        pairs = n * (n + 1) // 2
        return {"bytes": case["layers"] * (layer + n * row) + head + 4 * n * HIDDEN + 4 * case["vocab"],
                "flops": 2 * case["layers"] * (n * layer_macs + 2 * pairs * Q_ROWS) + 2 * head_macs}
    # the tokens of a decode come one after another: each reads the weights once for all members, and each member's cache
    seqs, n = case.get("seqs", 1), case["n"]
    steps = n - 1
    cached = sum(_member_rows(case, i) * steps + steps * (steps + 1) // 2 for i in range(seqs))
    last = _member_rows(case, seqs - 1) + n
    return {"bytes": (steps + 1) * (case["layers"] * layer + head) + case["layers"] * row * (cached + last) + 4 * case["vocab"],
            "flops": 2 * (seqs * steps + 1) * (case["layers"] * layer_macs + head_macs)
            + 4 * case["layers"] * Q_ROWS * (cached + last)}


def tolerance(case):
    if case.get("vnni"):
        return "exact"  # the mode is defined by its bits
    # four times the distance from float64 sums that was measured, stacks of 3
    # layers and all 18: f32 sums, and in a prompt's attention products of
    # 16 + 16 bit halves
    whole = case.get("layers", 0) > 3
    if case["kind"] in ("decode", "batch", "serve"):
        return {"rel": 2.5e-5 if whole else 1.2e-5}
    if case["kind"] == "prefill":
        return {"rel": 7e-5 if whole else 4e-5}
    return {"rel": 4e-6 if case["kind"] == "project" else 1.2e-6}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------


def _dequant(value):
    scale, codes = value
    return codes.double() * scale.double()[:, None]


def _rsqrt64(x):
    """The decoder's 1/sqrt: the bit-shift estimate and two Newton steps, which
    are part of its definition (up to 5e-6 from the true root)."""
    y = (0x5F3759DF - (x.float().view(torch.int32) >> 1)).to(torch.int32).view(torch.float32).double()
    for _ in range(2):
        y = y * (1.5 - 0.5 * x * y * y)
    return y


def _exp2_64(t):
    """2^t as the decoder defines it: a fifth-degree polynomial of the fraction
    (up to 3e-6 from the true power)."""
    n = t.round()
    f = t - n
    c = (1.0, 0.6931471824645996, 0.24022650718688965, 0.05550410971045494, 0.009618128649890423,
         0.0013352063251659274)
    p = torch.zeros_like(f)
    for a in reversed(c):
        p = p * f + a
    return torch.ldexp(p, n.to(torch.int32))


def _rms64(x, w):
    return x * _rsqrt64((x * x).mean(-1, keepdim=True) + EPS) * w


def _silu64(x):
    return x / (1.0 + _exp2_64(-x * math.log2(math.e)))


class _Decoder64:
    """The decoder in float64, prompt rows or single tokens of one sequence at a time."""

    def __init__(self, case, seed):
        self.layers = [{} for _ in range(case["layers"])]
        self.top = {}
        self.out_only = case["q"] != "q8"
        for li, name, value in _weights(case, seed):
            into = self.top if li < 0 else self.layers[li]
            into[name] = _dequant(value) if isinstance(value, tuple) else value.double()
        half = HEAD_DIM // 2
        self.freq = THETA ** (-torch.arange(half, device="cuda", dtype=torch.float64) * 2 / HEAD_DIM)
        ends = np.cumsum(SECTIONS)
        self.axis = torch.tensor([min(int(np.searchsorted(ends, i, side="right")), 2) for i in range(half)], device="cuda")

    def rope(self, x, pos):
        a = pos[:, self.axis] * self.freq
        c, s = a.cos()[:, None], a.sin()[:, None]
        x1, x2 = x.chunk(2, -1)
        return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], -1)

    def rows(self, x, pos, cache):
        """Rows x [n][hidden] after the cached ones; returns the logits of the last."""
        n, h = x.shape[0], x
        pos = torch.as_tensor(np.asarray(pos), device="cuda").double()
        for li, L in enumerate(self.layers):
            y = _rms64(h, L["ln1"])
            q = self.rope((y @ L["q"].T).view(n, HEADS, HEAD_DIM), pos)
            k = self.rope((y @ L["k"].T).view(n, KV_HEADS, HEAD_DIM), pos)
            v = (y @ L["v"].T).view(n, KV_HEADS, HEAD_DIM)
            if li in cache:
                k, v = torch.cat([cache[li][0], k]), torch.cat([cache[li][1], v])
            cache[li] = (k, v)
            total = k.shape[0]
            clen = torch.arange(total - n, total, device="cuda")
            hidden = torch.arange(total, device="cuda")[None] > clen[:, None]
            att = torch.empty((n, HEADS, HEAD_DIM), dtype=torch.float64, device="cuda")
            for hd in range(HEADS):
                kv = hd // (HEADS // KV_HEADS)
                sc = (q[:, hd] @ k[:, kv].T.contiguous()) / math.sqrt(HEAD_DIM)
                att[:, hd] = torch.softmax(sc.masked_fill(hidden, -math.inf), -1) @ v[:, kv]
            both = h + att.view(n, Q_ROWS) @ L["o"].T
            y = _rms64(both, L["ln2"])
            if self.out_only:  # 4- and 6-bit rows keep the residual before attention at these cache lengths
                both = torch.where(((clen == 0) | (clen >= 6))[:, None], h, both)
            h = both + (_silu64(y @ L["gate"].T) * (y @ L["up"].T)) @ L["down"].T
        return self.top["head"] @ _rms64(h[-1], self.top["final"])

    def token(self, t, pos, cache):
        return self.rows(self.top["embed"][t][None], [(pos, pos, pos)], cache)


def _exact_decode(case, seed):
    dec = _Decoder64(case, seed)
    first, at = _firsts(case, seed)
    streams = []
    for i, (t, p) in enumerate(zip(first, at)):
        rows = _member_rows(case, i)
        cache = {li: (k[:rows].double().view(rows, KV_HEADS, HEAD_DIM), v[:rows].double().view(rows, KV_HEADS, HEAD_DIM))
                 for li, k, v in _cache(case, seed, i)}
        out = [t]
        for j in range(case["n"] - 1):
            out.append(int(dec.token(out[-1], p + j, cache).argmax()))
        streams.append(out)
        if i + 1 == len(first):
            logits = dec.token(out[-1], p + case["n"] - 1, cache).cpu().numpy()
    return streams, logits


def exact(case, seed):
    kind = case["kind"]
    if case.get("vnni"):
        return None  # quantized activations: no 64-bit counterpart
    if kind in ("decode", "batch", "serve"):
        streams, logits = _exact_decode(case, seed)
        streams = [np.array(s, np.int32) for s in streams]
        return {"tokens": streams[0] if kind == "decode" else streams, "logits": logits}
    if kind == "prefill":
        logits = _Decoder64(case, seed).rows(_prompt(case, seed).double(), _positions(case["n"], case["grid"]), {})
        return {"token": int(logits.argmax()), "logits": logits.cpu().numpy()}
    if kind == "project":
        v = _vision(case, seed)
        w1, w2 = _dequant(_quantized(None, None, "q8", v["w1"])), _dequant(_quantized(None, None, "q8", v["w2"]))
        v = {k: t.double() for k, t in v.items()}
        d = v["rows"] - v["rows"].mean(1, keepdim=True)
        y = d * _rsqrt64((d * d).mean(1, keepdim=True) + EPS) * v["norm_w"] + v["norm_b"]
        t, h, w = case["t"], case["h"] // 2, case["w"] // 2
        y = y.view(t, case["h"], case["w"], VISION)[:, :2 * h, :2 * w].reshape(t, h, 2, w, 2, VISION)
        y = y.permute(0, 1, 3, 2, 4, 5).reshape(t * h * w, 4 * VISION)
        y = y @ w1.T + v["b1"]
        e = _exp2_64(2 * math.log2(math.e) * math.sqrt(2 / math.pi) * (y + 0.044715 * y ** 3))
        return ((0.5 * y * (1 + (e - 1) / (e + 1))) @ w2.T + v["b2"]).cpu().numpy()
    if kind == "mlp":
        w, v = _mlp(case, seed)
        w, v = {k: _dequant(t) for k, t in w.items()}, {k: t.double() for k, t in v.items()}
        r = v["residual"] + w["down"] @ (_silu64(w["gate"] @ v["x"]) * (w["up"] @ v["x"]))
        return _rms64(r, v["norm"]).cpu().numpy(), r.cpu().numpy()
    w, x = _head(case, seed)
    s = _dequant(w) @ x.double()
    top = torch.sort(s, descending=True, stable=True)
    return top.indices[:case["k"]].to(torch.int32).cpu().numpy(), top.values[:case["k"]].cpu().numpy()
