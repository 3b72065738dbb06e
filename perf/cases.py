"""Performance cases of the MiniLM-L6 embedding engine.

Each case is one call (or one short chain of calls) that a user of this
framework makes through `bbh.engine`, at sizes taken from the repository's own
configurations, tests and benchmark.  `listed()` names the fixed cases,
`draw(rng)` gives more of the same ranges, `prepare` makes what a user's
program holds before the call, `run` makes the call, `exact` restates it in
64-bit torch without this repository's kernels.

Kinds:
  embed        bert_embed: one padded batch -> embeddings (online queries,
               fixed-length batches, long documents)
  encode       bert_encode: one padded batch -> the final hidden rows
  corpus       a corpus of short sentences, one bert_embed per batch of 64
               over a pool of 4 slots (embed_each)
  packed       the same corpus without its padding rows (embed_packed)
  attn_block   attention_block of one layer (QKV, attention, O-proj + LN)
  ffn_block    ffn_block of one layer (FFN1 + GELU, FFN2 + LN)
  linear       launch_matmul: one Linear with bias, with or without GELU
  unfused      scores -> masked softmax -> context, for callers that want the
               attention probabilities
  rowops       embedding -> LayerNorm -> mean pool -> L2 normalise
"""

import functools
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bert-by-hand_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from bbh import engine, synth  # noqa: E402

H, F, HEADS, D, LAYERS, VOCAB = 384, 1536, 12, 32, 6, 30522
EPS = 1e-12
MAX_ROWS = 256 * 512
# The encoder's four Linears (N, K), and a 20-way classifier head on the
# embeddings (any N and K are accepted).
SHAPES = {"qkv": (1152, 384), "o_proj": (384, 384), "ffn1": (1536, 384), "ffn2": (384, 1536),
          "head": (20, 384)}


def listed():
    return [
        # one short query at a time: an online service's latency
        {"name": "embed_1x16", "kind": "embed", "batch": 1, "seq": 16, "lo": 9, "hi": 9},
        # the reference's fixed batch of short sentences (9 tokens at 16)
        {"name": "embed_64x16", "kind": "embed", "batch": 64, "seq": 16, "lo": 9, "hi": 9},
        # a batch of paragraphs padded to the reference's full length
        {"name": "embed_64x128", "kind": "embed", "batch": 64, "seq": 128, "lo": 9, "hi": 128},
        # the benchmark corpus: 2000 sentences in padded batches of 64
        {"name": "corpus_2000", "kind": "corpus", "n": 2000, "batch": 64, "median": 12},
        # the same corpus without padding, for indexing jobs
        {"name": "packed_2000", "kind": "packed", "n": 2000, "batch": 64, "median": 12},
        # long documents, the largest batch: indexing at the position limit
        {"name": "embed_256x512", "kind": "embed", "batch": 256, "seq": 512, "lo": 256, "hi": 512},
        # token-level features of a few mid-length documents
        {"name": "encode_21x304", "kind": "encode", "batch": 21, "seq": 304, "lo": 100, "hi": 304},
        # one layer's blocks, for callers that run the encoder layer by layer
        {"name": "attn_block_40x384", "kind": "attn_block", "batch": 40, "seq": 384, "lo": 200, "hi": 384},
        {"name": "ffn_block_256x80", "kind": "ffn_block", "batch": 256, "seq": 80},
        # a Linear on an odd number of rows
        {"name": "linear_qkv_2003", "kind": "linear", "rows": 2003, "shape": "qkv", "gelu": False},
        # attention with its probabilities kept
        {"name": "unfused_32x128", "kind": "unfused", "batch": 32, "seq": 128, "lo": 40, "hi": 128},
        # the memory-bound operators one by one
        {"name": "rowops_128x112", "kind": "rowops", "batch": 128, "seq": 112, "lo": 20, "hi": 112},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["embed", "embed", "encode", "corpus", "packed", "attn_block", "ffn_block",
                       "linear", "unfused", "rowops"])
    if kind in ("corpus", "packed"):
        return {"kind": kind, "n": _log(rng, 200, 2000), "batch": 64, "median": rng.randint(8, 16)}
    if kind == "linear":
        shape = rng.choice(sorted(SHAPES))
        return {"kind": kind, "rows": _log(rng, 1, 40000 if shape != "head" else 4000),
                "shape": shape, "gelu": shape == "ffn1" and rng.random() < 0.7}
    seq = 16 * rng.randint(1, 32)
    rows = {"embed": 65536, "encode": 32768, "attn_block": 65536, "ffn_block": MAX_ROWS,
            "unfused": 16384, "rowops": 65536}[kind]
    batch = _log(rng, 1, max(1, min(512, rows // seq)))
    case = {"kind": kind, "batch": batch, "seq": seq}
    if kind != "ffn_block":
        case["lo"] = max(3, int(seq * rng.uniform(0.2, 1.0)))
        case["hi"] = rng.randint(max(case["lo"], seq - 15), seq)
    return case


# ---- what a user's program holds ---------------------------------------------

@functools.lru_cache(maxsize=None)
def _weights():
    """fp16 weights of the MiniLM-L6 shape: the seeded N(0, 0.02) tensors,
    with LayerNorm gammas and betas that are not 1 and 0 and with query / key
    weights large enough for attention to be peaked, as in a trained model."""
    w = synth.make_weights(0)
    rng = np.random.default_rng(11)
    for k, v in w.items():
        if k.endswith("LayerNorm.weight"):
            v = rng.uniform(0.6, 1.4, v.shape)
        elif k.endswith("LayerNorm.bias"):
            v = rng.normal(0.0, 0.1, v.shape)
        elif ".query.weight" in k or ".key.weight" in k:
            v = v * 4.0
        w[k] = np.asarray(v, np.float32).astype(np.float16)
    return w


@functools.lru_cache(maxsize=None)
def _model():
    return engine.load_model_weights(_weights())


@functools.lru_cache(maxsize=None)
def _pool(slots, batch, seq):
    return engine.Pool(slots, batch, seq)  # one pool for a program's life


@functools.lru_cache(maxsize=None)
def _table(name):
    return torch.from_numpy(_weights()[name]).cuda()


def _lengths(case, rng):
    n = rng.integers(case["lo"], case["hi"] + 1, size=case["batch"])
    n[rng.integers(0, case["batch"])] = case["hi"]
    return n


def _sentence(rng, n):
    return np.concatenate([[synth.CLS_ID], rng.integers(synth.ID_LO, synth.ID_HI + 1, max(0, n - 2)),
                           [synth.SEP_ID]])[:n].astype(np.int32)


def _tokens(case, seed):
    rng = np.random.default_rng(seed)
    rows = [_sentence(rng, int(n)) for n in _lengths(case, rng)]
    ids, types, mask = synth.pack(rows, case["seq"])
    types[:, case["seq"] // 2:] = mask[:, case["seq"] // 2:]  # sentence pairs
    return ids, types, mask


def _corpus(case, seed):
    """Batches of (ids, types, mask): lognormal lengths, sigma 0.5, in [5, 64]."""
    rng = np.random.default_rng(seed)
    n = np.clip(np.round(rng.lognormal(np.log(case["median"]), 0.5, case["n"])), 5, 64)
    return [b[:3] for b in synth.batches_of([_sentence(rng, int(x)) for x in n], case["batch"])]


def _hidden(rows, seed):
    """Hidden rows as a LayerNorm leaves them."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((rows, H), device="cuda", generator=g)
    x *= 0.6 + 0.8 * torch.rand((H,), device="cuda", generator=g)
    return x.half()


def _mask(case, seed):
    n = torch.from_numpy(_lengths(case, np.random.default_rng(seed)))
    return (torch.arange(case["seq"])[None] < n[:, None]).int().cuda()


def _linear_input(case, seed):
    n, k = SHAPES[case["shape"]]
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn((case["rows"], k), device="cuda", generator=g).half()
    w = (torch.randn((n, k), device="cuda", generator=g) * 0.05).half()
    b = (torch.randn((n,), device="cuda", generator=g) * 0.05).half()
    return a, w, b


def _qkv(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    qkv = torch.randn((case["batch"] * case["seq"], 3 * H), device="cuda", generator=g)
    qkv[:, :2 * H] *= 1.5
    return qkv.half()


def prepare(case, seed):
    kind = case["kind"]
    half = lambda *s: torch.empty(s, dtype=torch.float16, device="cuda")  # noqa: E731
    st = {"case": case, "kind": kind}
    if kind in ("embed", "encode"):
        st["tok"] = [torch.from_numpy(a).cuda() for a in _tokens(case, seed)]
        st["ws"] = engine.make_workspace(case["batch"], case["seq"])
        st["out"] = half(case["batch"] * (case["seq"] if kind == "encode" else 1), H)
    elif kind in ("corpus", "packed"):
        st["pb"] = engine.PackedBatches(_corpus(case, seed), group_by_seq=kind == "packed")
        st["pool"] = _pool(4, 64, 64) if kind == "corpus" else _pool(1, 1024, 64)
        st["out"] = half(st["pb"].rows, H)
    elif kind in ("attn_block", "ffn_block"):
        rows = case["batch"] * case["seq"]
        st["ws"] = engine.make_workspace(case["batch"], case["seq"])
        st["x"], st["out"] = _hidden(rows, seed), half(rows, H)
        if kind == "attn_block":
            st["mask"] = _mask(case, seed)
    elif kind == "linear":
        st["a"], st["w"], st["b"] = _linear_input(case, seed)
        st["out"] = half(case["rows"], SHAPES[case["shape"]][0])
    elif kind == "unfused":
        b, s = case["batch"], case["seq"]
        st["qkv"], st["mask"] = _qkv(case, seed), _mask(case, seed)
        st["scores"], st["out"] = half(b * HEADS, s, s), half(b * s, H)
    else:  # rowops
        b, s = case["batch"], case["seq"]
        st["tok"] = [torch.from_numpy(a).cuda() for a in _tokens(case, seed)]
        st["tab"] = [_table("embeddings." + n) for n in (
            "word_embeddings.weight", "position_embeddings.weight", "token_type_embeddings.weight",
            "LayerNorm.weight", "LayerNorm.bias")]
        st["emb"], st["ln"], st["out"] = half(b * s, H), half(b * s, H), half(b, H)
    if kind not in ("linear", "unfused", "rowops"):
        st["model"] = _model()
    return st


def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "embed":
        return engine.bert_embed(st["ws"], st["model"], *st["tok"], emb=st["out"])
    if kind == "encode":
        return engine.bert_encode(st["ws"], st["model"], *st["tok"], out=st["out"])
    if kind == "corpus":
        return engine.embed_each(st["pool"], st["model"], st["pb"], emb=st["out"])
    if kind == "packed":
        return engine.embed_packed(st["pool"], st["model"], st["pb"], emb=st["out"])
    if kind == "attn_block":
        return engine.attention_block(st["ws"], st["model"], 2, st["x"], st["mask"], st["out"],
                                      case["batch"], case["seq"])
    if kind == "ffn_block":
        return engine.ffn_block(st["ws"], st["model"], 2, st["x"], st["out"], case["batch"],
                                case["seq"])
    if kind == "linear":
        n, k = SHAPES[case["shape"]]
        return engine.launch_matmul(st["a"], st["w"], st["out"], case["rows"], n, k, bias=st["b"],
                                    gelu=case["gelu"])
    if kind == "unfused":
        b, s = case["batch"], case["seq"]
        engine.launch_attention_scores(st["qkv"], st["scores"], b, HEADS, s, D, 3 * H, 0, H,
                                       D ** -0.5)
        engine.launch_softmax(st["scores"], b * HEADS * s, s, mask=st["mask"],
                              mask_stride=HEADS * s)
        engine.launch_attention_context(st["scores"], st["qkv"], st["out"], b, HEADS, s, D, 3 * H,
                                        2 * H)
        return {"probs": st["scores"], "context": st["out"]}
    b, s = case["batch"], case["seq"]
    word, pos, typ, gamma, beta = st["tab"]
    engine.launch_embedding(st["tok"][0], st["tok"][1], word, pos, typ, st["emb"], s, H, b)
    engine.launch_layernorm(st["emb"], gamma, beta, st["ln"], b * s, H)
    engine.launch_mean_pool(st["ln"], st["tok"][2], st["out"], s, H, b)
    engine.launch_l2_normalize(st["out"], H, b)
    return {"embedding": st["emb"], "layernorm": st["ln"], "pooled": st["out"]}


# ---- least work -----------------------------------------------------------------

def _mean_len(case):
    return (case["lo"] + case["hi"]) / 2


def work(case):
    kind = case["kind"]
    layer = 3 * H * H + H * H + 2 * H * F  # weights of a layer, without biases
    if kind in ("corpus", "packed"):
        # the expected token count; padding is not part of what is needed
        tokens = case["n"] * case["median"] * 1.133
        per = case["median"] * 1.133
        return {"bytes": 2 * LAYERS * layer + tokens * (2 * H + 12) + case["n"] * 2 * H,
                "flops": LAYERS * (2 * layer * tokens + 4 * H * per * tokens)}
    if kind == "linear":
        (n, k), m = SHAPES[case["shape"]], case["rows"]
        return {"bytes": 2 * (m * k + n * k + n + m * n), "flops": 2 * m * n * k}
    b, s = case["batch"], case["seq"]
    rows = b * s
    if kind in ("embed", "encode"):
        keys = _mean_len(case)
        # bert_embed also leaves the hidden rows in the workspace
        out = rows if kind == "encode" else rows + b
        return {"bytes": 2 * LAYERS * layer + b * keys * 2 * H + 12 * rows + out * 2 * H,
                "flops": LAYERS * (2 * layer * rows + 4 * H * keys * rows)}
    if kind == "attn_block":
        return {"bytes": 2 * (4 * H * H + 2 * rows * H) + 4 * rows,
                "flops": 2 * rows * 4 * H * H + 4 * H * _mean_len(case) * rows}
    if kind == "ffn_block":
        return {"bytes": 2 * (2 * H * F + 2 * rows * H), "flops": 4 * rows * H * F}
    if kind == "unfused":
        keys = _mean_len(case)
        return {"bytes": 2 * (4 * rows * H + HEADS * rows * s) + 4 * rows,
                "flops": 4 * H * keys * rows + 5 * HEADS * rows * keys}
    tokens = b * _mean_len(case)
    return {"bytes": 2 * H * (tokens + 2 * rows + b) + 12 * rows, "flops": 16 * rows * H}


def tolerance(case):
    # about four times the error against exact() seen over listed and drawn cases
    return {"embed": {"rel": 2e-3}, "encode": {"rel": 3e-3}, "corpus": {"rel": 2e-3},
            "packed": {"rel": 2e-3}, "attn_block": {"rel": 1.2e-3}, "ffn_block": {"rel": 1.2e-3},
            "linear": {"rel": 9e-4}, "unfused": {"rel": 4e-3}, "rowops": {"rel": 1.2e-3}}[case["kind"]]


# ---- the same in 64 bits ----------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _w64(name):
    return torch.from_numpy(_weights()[name]).cuda().double()


def _ln64(x, name):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + EPS) * _w64(name + ".weight") + _w64(name + ".bias")


def _lin64(x, name):
    return torch.addmm(_w64(name + ".bias"), x, _w64(name + ".weight").t().contiguous())


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.erf(x * 0.5 ** 0.5))


def _probs64(q, k, mask):
    """q, k (b, heads, s, D), mask (b, s) -> (b, heads, s, s)."""
    s = torch.matmul(q.contiguous(), k.transpose(-1, -2).contiguous()) * D ** -0.5
    return torch.softmax(s.masked_fill(mask[:, None, None, :] == 0, float("-inf")), -1)


def _heads64(x, b, s):
    return x.reshape(b, s, HEADS, D).permute(0, 2, 1, 3)


def _merge64(x, b, s):
    return x.permute(0, 2, 1, 3).reshape(b * s, H)


def _attn_block64(x, i, mask):
    b, s = mask.shape
    p = "encoder.layer.%d.attention." % i
    q, k, v = (_heads64(_lin64(x, p + "self." + n), b, s) for n in ("query", "key", "value"))
    c = torch.empty((b, HEADS, s, D), dtype=torch.float64, device="cuda")
    for j in range(0, b, 16):
        pr = _probs64(q[j:j + 16], k[j:j + 16], mask[j:j + 16])
        c[j:j + 16] = torch.matmul(pr, v[j:j + 16].contiguous())
    return _ln64(_lin64(_merge64(c, b, s), p + "output.dense") + x, p + "output.LayerNorm")


def _ffn_block64(x, i):
    p = "encoder.layer.%d." % i
    out = torch.empty_like(x)
    for j in range(0, x.shape[0], 32768):
        y = x[j:j + 32768]
        out[j:j + 32768] = _ln64(_lin64(_gelu64(_lin64(y, p + "intermediate.dense")),
                                        p + "output.dense") + y, p + "output.LayerNorm")
    return out


def _encode64(ids, types, mask):
    b, s = ids.shape
    t = lambda a: torch.as_tensor(a, device="cuda").long()  # noqa: E731
    ids, types, mask = t(ids), t(types), t(mask)
    e = "embeddings."
    x = _w64(e + "word_embeddings.weight")[ids] + _w64(e + "token_type_embeddings.weight")[types]
    x = _ln64((x + _w64(e + "position_embeddings.weight")[:s]).reshape(b * s, H), e + "LayerNorm")
    for i in range(LAYERS):
        x = _ffn_block64(_attn_block64(x, i, mask), i)
    return x


def _pool64(x, mask, b, s):
    m = torch.as_tensor(mask, device="cuda").double().reshape(b, s, 1)
    y = (x.reshape(b, s, H) * m).sum(1) / m.sum(1).clamp(min=1)
    return y / y.norm(dim=-1, keepdim=True).clamp(min=1e-12)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("embed", "encode"):
        ids, types, mask = _tokens(case, seed)
        b, s = ids.shape
        step = max(1, 32768 // s)
        x = torch.cat([_encode64(ids[j:j + step], types[j:j + step], mask[j:j + step])
                       for j in range(0, b, step)])
        return x if kind == "encode" else _pool64(x, mask, b, s)
    if kind in ("corpus", "packed"):
        batches = _corpus(case, seed)
        if kind == "packed":  # outputs come in the packed (length-grouped) order
            batches = sorted(batches, key=lambda b: b[0].shape[1])
        return torch.cat([_pool64(_encode64(*b), b[2], *b[0].shape) for b in batches])
    if kind == "attn_block":
        x = _hidden(case["batch"] * case["seq"], seed).double()
        return _attn_block64(x, 2, _mask(case, seed))
    if kind == "ffn_block":
        return _ffn_block64(_hidden(case["batch"] * case["seq"], seed).double(), 2)
    if kind == "linear":
        a, w, b = (t.double() for t in _linear_input(case, seed))
        y = torch.addmm(b, a, w.t().contiguous())
        return _gelu64(y) if case["gelu"] else y
    b, s = case["batch"], case["seq"]
    if kind == "unfused":
        q, k, v = (_heads64(t, b, s) for t in _qkv(case, seed).double().split(H, dim=1))
        p = _probs64(q, k, _mask(case, seed))
        return {"probs": p.reshape(b * HEADS, s, s),
                "context": _merge64(torch.matmul(p, v.contiguous()), b, s)}
    ids, types, mask = (torch.as_tensor(a, device="cuda").long() for a in _tokens(case, seed))
    e = "embeddings."
    x = _w64(e + "word_embeddings.weight")[ids] + _w64(e + "token_type_embeddings.weight")[types]
    x = (x + _w64(e + "position_embeddings.weight")[:s]).reshape(b * s, H)
    y = _ln64(x, e + "LayerNorm")
    return {"embedding": x, "layernorm": y, "pooled": _pool64(y, mask, b, s)}
