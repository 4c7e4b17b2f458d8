"""The calls that a user of this library makes, as measured cases.

The shapes are those of the Qwen3.5-9B decoder that the library serves
(hidden size 4096, MLP size 12288, projections of 1024 to 12288 outputs, a
vocabulary of 248,320), the weight types are those of its mixed GGUF files
(most matrices Q4_K; Q5_K, Q6_K, Q8_0 and IQ4_XS among them), activations are
fp32 or fp16.  Rows run from one token of one sequence, over decode batches of
up to 8 sequences with 1 to 5 rows each (speculative verification), short
prompts and prompt tails, the engine's 128-row prefill chunks and ragged
batches, to a 2048-row prefill.

A case is a dict: ``kind`` (the entry points called), ``m`` rows split over
``queries`` sequences, ``k`` and ``n`` of the projection, ``type`` (and
``down_type``, ``head_type``) of the weights, ``dtype`` of the activations,
``post`` (0 store, 1 residual added, 2 gated by the auxiliary) and ``norm``
(the projection's RMS norm given with it).
"""
import math

import torch

import mtlqwen_amd as q4k
from mtlqwen_amd.linear import linear_norm

HIDDEN, FFN, VOCAB = 4096, 12288, 248320
Q4_K, Q6_K, Q5_K, Q8_0, IQ4_XS = "q4_k", "q6_k", "q5_k", "q8_0", "iq4_xs"
TYPES = {Q4_K: (12, 144), Q6_K: (14, 210), Q5_K: (13, 176), Q8_0: (8, 272), IQ4_XS: (23, 136)}  # ggml type, bytes per 256 weights
EPS = 1e-6

# (k, n) of the projections: key/value, output, query and its GDN relatives,
# the joined query/key/value, one of the MLP, the MLP's way back.
PROJECTIONS = [(4096, 1024), (4096, 4096), (4096, 6144), (4096, 8192), (4096, 12288), (12288, 4096)]


def _case(kind, m, queries, dtype, type=Q4_K, **more):
    return {"kind": kind, "m": m, "queries": queries, "dtype": dtype, "type": type, **more}


def listed():
    return [
        # One token of one conversation: the attention output projection with its residual.
        {"name": "o_m1_f32", **_case("linear", 1, 1, "f32", k=4096, n=4096, post=1, norm=False)},
        # Eight conversations, one token each: the whole MLP block with its norm.
        {"name": "mlp_m8_f32", **_case("mlp", 8, 8, "f32", down_type=Q4_K)},
        # One conversation verifying four drafted tokens: the value projection, kept at a higher precision in mixed files.
        {"name": "v_q6k_m5_f16", **_case("linear", 5, 1, "f16", Q6_K, k=4096, n=1024, post=0, norm=True)},
        # Eight conversations, one token each: final norm and vocabulary projection.
        {"name": "head_q6k_m8_f32", **_case("head", 8, 8, "f32", Q6_K)},
        # Eight conversations verifying four drafted tokens each: embedding, one layer's projections, norm and logits of every row.
        {"name": "pass_m40_f16", **_case("pass", 40, 8, "f16", down_type=Q5_K, head_type=Q6_K)},
        # A short prompt (or the tail of a long one): the MLP of a layer in 4- and 5-bit types.
        {"name": "mlp_iq4xs_q5k_m19_f16", **_case("mlp", 19, 1, "f16", IQ4_XS, down_type=Q5_K)},
        # An odd number of prompt tokens from two conversations: the MLP's way back in 6 bits.
        {"name": "down_q6k_m77_f32", **_case("linear", 77, 2, "f32", Q6_K, k=12288, n=4096, post=1, norm=False)},
        # The reference engine's prefill chunk: 128 rows, fp16, the whole MLP block.
        {"name": "mlp_m128_f16", **_case("mlp", 128, 1, "f16", down_type=Q4_K)},
        # A ragged prompt batch: the query projection with its norm.
        {"name": "q_m333_f16", **_case("linear", 333, 3, "f16", k=4096, n=8192, post=0, norm=True)},
        # Ragged prompts of eight conversations: the whole MLP block.
        {"name": "mlp_m821_f32", **_case("mlp", 821, 8, "f32", down_type=Q4_K)},
        # A long prompt: a projection whose weights are kept in 8 bits.
        {"name": "up_q8_0_m1531_f16", **_case("linear", 1531, 1, "f16", Q8_0, k=4096, n=12288, post=2, norm=False)},
        # The longest prefill: the whole MLP block.
        {"name": "mlp_m2048_f32", **_case("mlp", 2048, 8, "f32", down_type=Q4_K)},
    ]


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["mlp"] * 3 + ["gate_up", "head"])
    if kind == "head":
        m = int(round(math.exp(rng.uniform(0, math.log(64)))))
    else:
        m = int(round(math.exp(rng.uniform(0, math.log(2048)))))
    # A decode batch has at most 5 rows a sequence; others are prompts of any length.
    queries = rng.randint(max(1, -(-m // 5)), min(8, m)) if m <= 40 and rng.random() < 0.7 else rng.randint(1, min(8, m))
    dtype = rng.choice(["f32", "f16"])
    weight = rng.choice([Q4_K] * 4 + [Q5_K, Q6_K, Q8_0, IQ4_XS])
    if kind == "linear":
        k, n = rng.choice(PROJECTIONS * 3 + [(32768, 4096)])
        if k == 32768:
            weight = Q4_K
        post = rng.choice([0, 0, 1, 2])
        return _case(kind, m, queries, dtype, weight, k=k, n=n, post=post, norm=k == HIDDEN and post == 0 and rng.random() < 0.5)
    if kind == "mlp":
        down = rng.choice([Q4_K, Q4_K, Q5_K, Q6_K, Q8_0, IQ4_XS])
        return _case(kind, m, queries, dtype, weight, down_type=down)
    return _case(kind, m, queries, dtype, weight)


# ---- inputs -----------------------------------------------------------------

def _dtype(case):
    return torch.float32 if case["dtype"] == "f32" else torch.float16


def _counts(case):
    """Rows of each sequence: alike for a decode batch, ragged for prompts."""
    m, q = case["m"], case["queries"]
    if m <= 5 * q:
        return [m // q + (1 if i < m % q else 0) for i in range(q)]
    total = q * (q + 1) // 2
    counts = [max(1, m * (i + 1) // total) for i in range(q)]
    counts[-1] += m - sum(counts)
    return counts


def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * int(seed) + part)
    return g


def _quantized(seed, part, n, k, kind):
    """GGUF bytes [n, blocks, bytes] of an n x k matrix: uniform quants and
    sub-block scales, block scales that give centred weights of about
    1/sqrt(k), as trained projections have."""
    g, nb = _gen(seed, part), k // 256
    size = TYPES[kind][1]
    w = torch.randint(0, 256, (n, nb, size), generator=g, device="cuda", dtype=torch.uint8)
    std = {Q4_K: 340.0, Q5_K: 700.0, Q6_K: 1365.0, Q8_0: 73.9, IQ4_XS: 1290.0}[kind]  # of the weights at a block scale of 1

    def scales(cols):
        d = (0.5 + torch.rand((n, nb, cols), generator=g, device="cuda")) / (std * math.sqrt(k))
        return d.to(torch.float16)

    if kind in (Q4_K, Q5_K):
        d = scales(1)
        both = torch.cat([d, (d.float() * (7.5 if kind == Q4_K else 15.5)).to(torch.float16)], dim=2)
        w[:, :, 0:4] = both.view(torch.uint8)
    elif kind == Q6_K:
        w[:, :, 208:210] = scales(1).view(torch.uint8)
    elif kind == Q8_0:
        r = w.view(n, nb, 8, 34)
        r[:, :, :, 0:2] = scales(8).view(torch.uint8).view(n, nb, 8, 2)
    else:
        w[:, :, 0:2] = scales(1).view(torch.uint8)
    return w


def _weight(seed, part, n, k, kind):
    return q4k.Weight(_quantized(seed, part, n, k, kind).view(-1), n, k, ggml_type=TYPES[kind][0])


def _acts(seed, part, m, k, dtype):
    """Activations: normal, with one channel in 256 ten times larger, as a
    decoder's hidden state has."""
    g = _gen(seed, part)
    x = torch.randn((m, k), generator=g, device="cuda")
    return (x * (1.0 + 9.0 * (torch.rand((k,), generator=g, device="cuda") < 1 / 256))).to(dtype)


def _norm(seed, part, k):
    return 0.5 + torch.rand((k,), generator=_gen(seed, part), device="cuda")


def _inputs(case, seed):
    """The tensors of a case, and its weights as (n, k, type, part) of _quantized."""
    m, kind, dt = case["m"], case["kind"], _dtype(case)
    t, w = {}, {}
    if kind == "linear":
        t["x"] = _acts(seed, 1, m, case["k"], dt)
        if case["post"]:
            t["aux"] = _acts(seed, 2, m, case["n"], dt)
        if case["norm"]:
            t["norm"] = _norm(seed, 3, case["k"])
        w["w"] = (case["n"], case["k"], case["type"], 11)
    elif kind in ("gate_up", "mlp"):
        t["x"] = _acts(seed, 1, m, HIDDEN, dt)
        w["gate"] = (FFN, HIDDEN, case["type"], 11)
        w["up"] = (FFN, HIDDEN, case["type"], 12)
        if kind == "mlp":
            t["norm"] = _norm(seed, 3, HIDDEN)
            w["down"] = (HIDDEN, FFN, case["down_type"], 13)
    elif kind == "head":
        t["x"] = _acts(seed, 1, m, HIDDEN, dt)
        t["norm"] = _norm(seed, 3, HIDDEN)
        w["head"] = (VOCAB, HIDDEN, case["type"], 14)
    else:
        tokens = torch.randint(0, VOCAB, (case["queries"], 64), generator=_gen(seed, 4), device="cuda", dtype=torch.int32)
        t["tokens"] = tokens
        t["attn"] = _acts(seed, 5, m, HIDDEN, dt)
        for i, name in enumerate(("attn_norm", "ffn_norm", "out_norm")):
            t[name] = _norm(seed, 6 + i, HIDDEN)
        w["table"] = (VOCAB, HIDDEN, Q4_K, 15)
        w["qkv"] = (6144, HIDDEN, case["type"], 16)
        w["o"] = (HIDDEN, HIDDEN, case["type"], 17)
        w["gate"] = (FFN, HIDDEN, case["type"], 11)
        w["up"] = (FFN, HIDDEN, case["type"], 12)
        w["down"] = (HIDDEN, FFN, case["down_type"], 13)
        w["head"] = (VOCAB, HIDDEN, case["head_type"], 14)
    return t, w


def prepare(case, seed):
    t, w = _inputs(case, seed)
    m, dt = case["m"], _dtype(case)
    s = dict(t, case=case, counts=_counts(case))
    for name, (n, k, kind, part) in w.items():
        s[name] = _weight(seed, part, n, k, kind)

    def empty(rows, cols):
        return torch.empty((rows, cols), device="cuda", dtype=dt)

    kind = case["kind"]
    if kind == "linear":
        s["y"] = empty(m, case["n"])
    if kind in ("gate_up", "mlp", "pass"):
        s["buffer"] = empty(m, FFN)
    if kind in ("mlp", "head", "pass"):
        s["hidden"] = empty(m, HIDDEN)
    if kind in ("head", "pass"):
        s["rows"] = empty(m, HIDDEN)
        s["logits"] = empty(m, VOCAB)
    if kind == "pass":
        s["qkv_out"] = empty(m, 6144)
    return s


# ---- one pass -----------------------------------------------------------------

def run(s):
    c = s["case"]
    m, counts, kind = c["m"], s["counts"], c["kind"]
    if kind == "linear":
        gated, aux = c["post"] == 2, s.get("aux")
        if c["norm"]:
            return linear_norm(s["x"], s["w"], s["norm"], m, s["y"], auxiliary=aux, gated=gated, query_counts=counts, eps=EPS)
        return q4k.linear(s["x"], s["w"], m, s["y"], auxiliary=aux, gated=gated, query_counts=counts)
    if kind == "gate_up":
        return q4k.mlp_gate_up(s["x"], s["gate"], s["up"], m, s["buffer"], query_counts=counts)
    if kind == "mlp":
        # The residual stream enters the block as its own copy; the block adds to it in place.
        s["hidden"].copy_(s["x"])
        q4k.mlp(s["hidden"], s["gate"], s["up"], s["down"], s["hidden"], s["buffer"], m, query_counts=counts, norm_weight=s["norm"], eps=EPS)
        return s["hidden"], s["buffer"]
    if kind == "head":
        q4k.rms_norm_gather(s["x"], s["norm"], s["rows"], counts, counts, eps=EPS)
        return q4k.linear(s["rows"], s["head"], m, s["logits"], query_counts=counts)
    h = s["hidden"]
    nq = len(counts)
    q4k.embedding_batch(s["table"], s["tokens"], s["tokens"].shape[1], counts, [7] * nq, list(range(nq)), h)
    linear_norm(h, s["qkv"], s["attn_norm"], m, s["qkv_out"], query_counts=counts, eps=EPS)
    q4k.linear(s["attn"], s["o"], m, h, auxiliary=h, query_counts=counts)
    q4k.mlp(h, s["gate"], s["up"], s["down"], h, s["buffer"], m, query_counts=counts, norm_weight=s["ffn_norm"], eps=EPS)
    q4k.rms_norm_gather(h, s["out_norm"], s["rows"], counts, counts, eps=EPS)
    q4k.linear(s["rows"], s["head"], m, s["logits"], query_counts=counts)
    return s["qkv_out"], h, s["logits"]


def work(case):
    """Weights read once, activations read once, outputs written once; two
    operations per weight and row."""
    m, e, kind = case["m"], 4 if case["dtype"] == "f32" else 2, case["kind"]

    def proj(n, k, t):
        return n * (k // 256) * TYPES[t][1], 2 * m * n * k

    if kind == "linear":
        parts, acts = [(case["n"], case["k"], case["type"])], case["k"] + case["n"] * (2 if case["post"] else 1)
    elif kind == "gate_up":
        parts, acts = [(FFN, HIDDEN, case["type"])] * 2, HIDDEN + FFN
    elif kind == "mlp":
        parts, acts = [(FFN, HIDDEN, case["type"])] * 2 + [(HIDDEN, FFN, case["down_type"])], HIDDEN + FFN + HIDDEN
    elif kind == "head":
        parts, acts = [(VOCAB, HIDDEN, case["type"])], HIDDEN + VOCAB
    else:
        parts = [(6144, HIDDEN, case["type"]), (HIDDEN, HIDDEN, case["type"])] + [(FFN, HIDDEN, case["type"])] * 2
        parts += [(HIDDEN, FFN, case["down_type"]), (VOCAB, HIDDEN, case["head_type"])]
        acts = HIDDEN + 6144 + HIDDEN + FFN + VOCAB
    both = [proj(*p) for p in parts]
    return {"bytes": sum(b for b, _ in both) + m * e * acts, "flops": sum(f for _, f in both)}


def tolerance(case):
    """About four times the largest error against 64 bits that was measured.
    fp16 outputs round at each step (gated ones three times): 6e-4, and 7e-4
    through a whole pass.  fp32 outputs of more than 24 rows carry the one
    rounding of activations (and prefill weights) to fp16: 4e-4.  Up to 24
    rows the activations keep 22 bits: 3e-7 where quant times scale is exact
    (4- and 5-bit K types), 2.5e-4 where that product rounds to fp16."""
    if case["kind"] == "pass":
        return {"rel": 3e-3}
    if case["dtype"] == "f16":
        return {"rel": 2.2e-3}
    if case["m"] > 24:
        return {"rel": 1.6e-3}
    exact_products = {case["type"], case.get("down_type", Q4_K)} <= {Q4_K, Q5_K}
    return {"rel": 1e-5 if exact_products else 1e-3}


# ---- the same in 64 bits ---------------------------------------------------------

IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _scale_min(s):
    """The eight 6-bit scales and mins of 12 packed bytes: [..., 12] -> two [..., 8]."""
    lo, hi, top = s[..., 0:4], s[..., 4:8], s[..., 8:12]
    sc = torch.cat([lo & 63, (top & 15) | ((lo >> 6) << 4)], dim=-1)
    mn = torch.cat([hi & 63, (top >> 4) | ((hi >> 6) << 4)], dim=-1)
    return sc.double(), mn.double()


def _dequantized(w, kind):
    """[rows, blocks, bytes] -> the weights [rows, k] in 64 bits."""
    n, nb = w.shape[:2]
    if kind in (Q4_K, Q5_K):
        d, dmin = _half(w[..., 0:2]), _half(w[..., 2:4])
        sc, mn = _scale_min(w[..., 4:16])
        qs = w[..., (16 if kind == Q4_K else 48):].reshape(n, nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], dim=3).reshape(n, nb, 8, 32)
        if kind == Q5_K:
            bit = torch.arange(8, device=w.device, dtype=torch.uint8).view(1, 1, 8, 1)
            q = q + 16 * ((w[..., 16:48].unsqueeze(2) >> bit) & 1)
        v = q.double() * (d * sc).unsqueeze(-1) - (dmin * mn).unsqueeze(-1)
    elif kind == Q6_K:
        ql, qh = w[..., 0:128].reshape(n, nb, 2, 2, 32), w[..., 128:192].reshape(n, nb, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], dim=3)  # quarters 0..3 of each half
        shift = torch.tensor([0, 2, 4, 6], device=w.device, dtype=torch.uint8).view(1, 1, 1, 4, 1)
        q = (lo | (((qh >> shift) & 3) << 4)).double() - 32.0
        sc = w[..., 192:208].contiguous().view(torch.int8).double().unsqueeze(-1)
        v = q.reshape(n, nb, 16, 16) * sc * _half(w[..., 208:210]).unsqueeze(-1)
    elif kind == Q8_0:
        r = w.reshape(n, nb, 8, 34)
        v = r[..., 2:].contiguous().view(torch.int8).double() * _half(r[..., 0:2])
    else:
        high = w[..., 2].int() | (w[..., 3].int() << 8)
        low = w[..., 4:8].int()
        j = torch.arange(8, device=w.device)
        ls = ((low[..., j // 2] >> (4 * (j % 2))) & 15) | (((high.unsqueeze(-1) >> (2 * j)) & 3) << 4)
        qs = w[..., 8:].reshape(n, nb, 8, 16)
        q = torch.cat([qs & 15, qs >> 4], dim=3).long()
        table = torch.tensor(IQ4, device=w.device, dtype=torch.float64)
        v = table[q] * ((ls.double() - 32.0) * _half(w[..., 0:2])).unsqueeze(-1)
    return v.reshape(n, nb * 256)


def exact(case, seed):
    t, w = _inputs(case, seed)
    kind = case["kind"]
    f = {name: v.double() for name, v in t.items() if v.is_floating_point()}

    def product(x, name):
        n, k, qt, part = w[name]
        q = _quantized(seed, part, n, k, qt)
        y = torch.empty((x.shape[0], n), device="cuda", dtype=torch.float64)
        for i in range(0, n, 4096):
            y[:, i:i + 4096] = x @ _dequantized(q[i:i + 4096], qt).t().contiguous()
        return y

    def norm(x, name):
        return x * torch.rsqrt((x * x).mean(dim=1, keepdim=True) + EPS) * f[name]

    def silu(v):
        return v / (1.0 + torch.exp(-v))

    if kind == "linear":
        y = product(norm(f["x"], "norm") if case["norm"] else f["x"], "w")
        return y + f["aux"] if case["post"] == 1 else silu(f["aux"]) * y if case["post"] == 2 else y
    if kind == "gate_up":
        return silu(product(f["x"], "gate")) * product(f["x"], "up")
    if kind == "mlp":
        xn = norm(f["x"], "norm")
        gate = silu(product(xn, "gate")) * product(xn, "up")
        return f["x"] + product(gate, "down"), gate
    if kind == "head":
        return product(norm(f["x"], "norm"), "head")
    counts = _counts(case)
    ids = torch.cat([t["tokens"][q, 7:7 + c] for q, c in enumerate(counts)]).long()
    n, k, qt, part = w["table"]
    h = _dequantized(_quantized(seed, part, n, k, qt)[ids], qt)
    qkv = product(norm(h, "attn_norm"), "qkv")
    h = h + product(f["attn"], "o")
    xn = norm(h, "ffn_norm")
    h = h + product(silu(product(xn, "gate")) * product(xn, "up"), "down")
    return qkv, h, product(norm(h, "out_norm"), "head")
