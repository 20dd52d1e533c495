"""The calls whose speed this framework is judged by: whole encoder passes as
a program makes them (EncodeSeqs, EncodeTokens, the decision heads), from one
short query to eight 8,192-token documents, and the int8 linear layer with
outlier channels. Models are random-init int8 weights of the three shapes the
repository measures (ModernBERT-base, its own 384-wide backbone, the small
test shape); ids are uniform over the vocabulary, as in bench.py.

A model is loaded once a process and kept, as a program keeps it; `prepare`
makes the batch. Results are pinned to the reference's CPU path bit for bit,
so every tolerance is "exact".
"""
import math

import numpy as np
import torch

from indecis_amd import _lib, heads, linalg
from indecis_amd.modernbert import EMB_BF16, EMB_F32, EMB_I8, Config, Model, Weights

SHAPES = {
    # ModernBERT-base, and the reference's own backbone width (bench.py's w384)
    "base": dict(hidden=768, layers=22, heads=12, intermediate=1152, vocab=50368),
    "w384": dict(hidden=384, layers=22, heads=6, intermediate=1152, vocab=32768),
    "small": dict(hidden=256, layers=6, heads=4, intermediate=512, vocab=32768),
}
FORMATS = {"f32": EMB_F32, "bf16": EMB_BF16, "i8": EMB_I8}
# decision heads (rows, per token): Choice-8, Noul and a 5-option Score on
# the pooled row; a Spans head over 4 types on every token
HEADS = {"decide": ((8, False), (1, False), (4, False)), "spans": ((heads.span_tag_count(4), True),)}
RATIO = 6.0  # the outlier ratio of the linear layers


def listed():
    enc = dict(emb="f32", lanes=8, pooling="mean")
    return [
        # one short query embedded on the reference's own backbone, its table
        # compacted to int8: the smallest call, latency only
        dict(enc, name="query_w384", call="seqs", shape="w384", seqs=1, lo=15, hi=15, emb="i8"),
        # one sentence on the base shape, as an interactive caller sends it
        dict(enc, name="sentence_base", call="seqs", shape="base", seqs=1, lo=24, hi=24),
        # the small shape's batch of 64 sentences of 15 tokens
        dict(enc, name="sentences_small", call="seqs", shape="small", seqs=64, lo=15, hi=15),
        # one document at the length limit that Open sets (256 tokens), every
        # token's state returned to the host
        dict(enc, name="document_base", call="tokens", shape="base", seqs=1, lo=256, hi=256),
        # what a serving batcher groups: a dozen requests of a sentence or a
        # paragraph; bf16 table, CLS pooling
        dict(enc, name="serving_base", call="seqs", shape="base", seqs=12, lo=16, hi=128, emb="bf16", pooling="cls"),
        # the decision path over many short inputs, heads on the device
        dict(enc, name="decide_base", call="decide", shape="base", seqs=256, lo=8, hi=256),
        # indexing with the small shape, ids and result in device memory
        dict(enc, name="index_small", call="device", shape="small", seqs=256, lo=16, hi=256),
        # indexing with the 384-wide backbone; results of an AVX-512 host
        dict(enc, name="index_w384", call="device", shape="w384", seqs=256, lo=64, hi=512, lanes=16),
        # the headline batch: 256 sequences of 64 to 512 tokens, base shape
        dict(enc, name="index_base", call="device", shape="base", seqs=256, lo=64, hi=512),
        # one long document with a Spans head on every token
        dict(enc, name="spans_base", call="spans", shape="base", seqs=1, lo=4096, hi=4096),
        # eight documents of the longest length
        dict(enc, name="long_base", call="device", shape="base", seqs=8, lo=8192, hi=8192),
        # a vision tower's MLP product (four images of 196 patches) with
        # massive input channels split off, host rows in and out
        dict(name="linear_outliers", call="linear", rows=784, k=3072, n=768, outliers=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.12:
        return dict(call="linear", rows=_log(rng, 1, 4096), k=rng.choice([768, 1152, 3072]),
                    n=rng.choice([96, 768, 1152, 3072]), outliers=rng.random() < 0.7)
    shape = rng.choice(["base", "base", "w384", "small"])
    hi = _log(rng, 8, 8192)
    lo = max(1, min(hi, _log(rng, max(1, hi // 16), hi)))
    tokens = _log(rng, hi, 49152)
    return dict(call=rng.choice(["seqs", "tokens", "device", "device", "decide", "spans"]), shape=shape,
                seqs=max(1, min(512, 2 * tokens // (lo + hi))), lo=lo, hi=hi, emb=rng.choice(["f32", "bf16", "i8"]),
                lanes=rng.choice([8, 8, 16, 4]), pooling=rng.choice(["mean", "mean", "cls"]))


_weights, _models = {}, {}


def _shape_weights(shape, emb):
    """The shape's weights with the table in one format (the same matrices
    and the same float32 table whatever the format)."""
    if (shape, emb) not in _weights:
        _weights[shape, emb] = Weights.random(Config(**SHAPES[shape]), seed=4, emb_format=FORMATS[emb])
    return _weights[shape, emb]


def _head_weights(shape, which):
    rng = np.random.default_rng(11)
    out = []
    for rows, per_token in HEADS[which]:
        w, _ = heads.random_head(rows, SHAPES[shape]["hidden"], rng)
        out.append((w, rng.standard_normal(rows).astype(np.float32), per_token))
    return out


def _model(case):
    """The loaded model of a case, kept for the process."""
    call = case["call"] if case["call"] in HEADS else ""
    key = (case["shape"], case["emb"], case["lanes"], case["pooling"], call)
    if key not in _models:
        w = _shape_weights(case["shape"], case["emb"])
        cfg = Config(**SHAPES[case["shape"]], pooling=case["pooling"])
        m = Model(None, device=0, lanes=case["lanes"], cfg=cfg)
        m.upload(w)
        if call:
            m.set_heads(_head_weights(case["shape"], call))
        _models[key] = m
    return _models[key]


def _lengths(case):
    """Sequence lengths of a batch; they follow the case, not the seed, so
    that batches of two seeds hold the same number of tokens."""
    rng = np.random.default_rng([case["seqs"], case["lo"], case["hi"]])
    return rng.integers(case["lo"], case["hi"] + 1, size=case["seqs"])


def _ids(case, seed):
    rng = np.random.default_rng([seed, 1])
    vocab = SHAPES[case["shape"]]["vocab"]
    return [rng.integers(0, vocab, size=int(n), dtype=np.int32) for n in _lengths(case)]


def _linear_weights(case):
    """The layer's weights: one matrix a shape, as a loaded tower has it."""
    key = (case["k"], case["n"])
    if key not in _weights:
        rng = np.random.default_rng(5)
        q, s = linalg.pack_b8(rng.standard_normal((case["n"], case["k"]), dtype=np.float32) * np.float32(0.03))
        bias = (rng.standard_normal(case["n"]) * 0.1).astype(np.float32)
        _weights[key] = (q, s, bias)
        _models[key] = linalg.PackedB8(q, s)
    return _weights[key], _models[key]


def _linear_rows(case, seed):
    """Activation rows with massive channels: a few columns 20-60 times the others."""
    rng = np.random.default_rng([seed, 2])
    x = rng.standard_normal((case["rows"], case["k"]), dtype=np.float32)
    massive = rng.choice(case["k"], size=max(1, case["k"] // 256), replace=False)
    x[:, massive] *= rng.uniform(20, 60, size=len(massive)).astype(np.float32)
    return x


def prepare(case, seed):
    if case["call"] == "linear":
        (_, _, bias), packed = _linear_weights(case)
        return dict(case=case, packed=packed, x=_linear_rows(case, seed), bias=bias)
    model = _model(case)
    seqs = _ids(case, seed)
    state = dict(case=case, model=model, seqs=seqs)
    if case["call"] == "device":
        state["offs"] = np.concatenate([[0], np.cumsum([len(s) for s in seqs])]).astype(np.int32)
        state["ids"] = torch.from_numpy(np.concatenate(seqs)).to("cuda")
        state["out"] = torch.empty((len(seqs), model.cfg.hidden), dtype=torch.float32, device="cuda")
    return state


def run(state):
    call = state["case"]["call"]
    if call == "linear":
        return linalg.linear8(state["x"], state["packed"], state["bias"], state["case"]["outliers"], RATIO)
    model = state["model"]
    if call == "seqs":
        return model.encode_seqs(state["seqs"])
    if call == "tokens":
        return model.encode_tokens(state["seqs"])
    if call == "decide":
        return model.encode_heads(state["seqs"], tokens=False)[0]
    if call == "spans":
        return model.encode_heads(state["seqs"], mean=True, pooled=False)[1]
    model.encode_device(state["ids"].data_ptr(), state["offs"], state["out"].data_ptr(), _lib.OUT_POOLED,
                        torch.cuda.current_stream().cuda_stream)
    return state["out"]


def work(case):
    if case["call"] == "linear":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": 4.0 * m * k + k * n + 8.0 * n + 4.0 * m * n, "flops": 2.0 * m * k * n}
    s = SHAPES[case["shape"]]
    H, L, I, nh = s["hidden"], s["layers"], s["intermediate"], s["heads"]
    lens = _lengths(case).astype(np.float64)
    N, B = lens.sum(), len(lens)
    per_layer = 4 * H * H + 3 * H * I
    d = np.minimum(64, lens - 1)  # local layers: 64 keys either side
    pairs_local = (lens + 2 * (d * lens - d * (d + 1) / 2)).sum()
    pairs_global = (lens * lens).sum()
    n_global = len([l for l in range(L) if l % 3 == 0])
    pairs = n_global * pairs_global + (L - n_global) * pairs_local
    row = {"f32": 4 * H, "bf16": 2 * H, "i8": H + 4}[case["emb"]]
    rows = sum(r for r, _ in HEADS.get(case["call"], ()))
    out = {"tokens": 4 * N * H, "decide": 8 * B * rows, "spans": 8 * N * rows}.get(case["call"], 4 * B * H)
    return {"bytes": float(L * per_layer + N * (4 + row) + out),
            "flops": float(2 * N * L * per_layer + 4 * 64 * nh * pairs)}


def tolerance(case):
    return "exact"


# ---- the same results in 64 bits ---------------------------------------------
# The int8 path's own definition (where it rounds to integers) with every
# other step in float64; plain torch, on the GPU where there is one.

_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_DEV).double()


def _quant(x, dim=-1):
    """Symmetric int8 along dim: rounded values and scales."""
    s = x.abs().amax(dim, keepdim=True) / 127
    return torch.round(x / torch.where(s > 0, s, torch.ones_like(s))), s


def _mm(x, q, s):
    """Rows of x quantised, times int8 weight rows q with scales s."""
    a, sa = _quant(x)
    return (a @ q.T.contiguous()) * s * sa


def _norm(x, gamma, eps):
    c = x - x.mean(-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + eps) * gamma


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _attend(q, k, v, window):
    """One sequence: q, k, v [heads, n, 64]."""
    n = q.shape[1]
    qi, sq = _quant(q)
    ki, sk = _quant(k - k.mean(1, keepdim=True))
    vi, sv = _quant(v, 1)
    out = torch.empty_like(v)
    near = None
    if window >= 0 and n > window + 1:
        i = torch.arange(n, device=q.device)
        near = (i[:, None] - i[None, :]).abs() <= window
    for h in range(q.shape[0]):
        z = (qi[h] @ ki[h].T.contiguous()) * sk[h].T * (sq[h] * 0.125)
        if near is not None:
            z = z.masked_fill(~near, -math.inf)
        p = torch.round(255 * torch.exp(z - z.amax(1, keepdim=True)))
        out[h] = (p @ vi[h]) * sv[h] / p.sum(1, keepdim=True)
    return out


def _states(case, seed):
    w = _shape_weights(case["shape"], case["emb"])
    c = w.cfg
    H, nh = c.hidden, c.heads
    seqs = _ids(case, seed)
    ids = np.concatenate(seqs)
    if case["emb"] == "f32":
        x = _f64(w.emb_f32[ids])
    elif case["emb"] == "bf16":
        rows = (w.emb_bf16[ids].astype(np.uint32) << 16).view(np.float32)
        for t, e in zip(w.emb_exact_ids, w.emb_exact_rows):
            rows[ids == t] = e
        x = _f64(rows)
    else:
        x = _f64(w.emb_i8[ids]) * _f64(w.emb_i8_scale[ids])[:, None]
    x = _norm(x, _f64(w.emb_norm), c.norm_eps)
    pos = torch.arange(max(len(s) for s in seqs), device=_DEV).double()
    for l in range(c.layers):
        glob = l % c.global_every == 0
        theta = c.global_theta if glob else c.local_theta
        inv = (1.0 / theta ** (np.arange(32) * 2.0 / 64)).astype(np.float32)
        ang = pos[:, None] * _f64(inv)[None, :]
        cos, sin = torch.cos(ang), torch.sin(ang)
        y = x if l == 0 else _norm(x, _f64(w.attn_norm[l]), c.norm_eps)
        qkv = _mm(y, _f64(w.wqkv_q[l]), _f64(w.wqkv_s[l]))
        ctx, t = torch.empty_like(x), 0
        for s in seqs:
            n = len(s)
            q, k, v = (u.reshape(n, nh, 64).transpose(0, 1).contiguous() for u in qkv[t:t + n].split(H, dim=1))
            q, k = _rotate(q, cos[:n], sin[:n]), _rotate(k, cos[:n], sin[:n])
            o = _attend(q, k, v, -1 if glob else c.window())
            ctx[t:t + n] = o.transpose(0, 1).reshape(n, H)
            t += n
        x = x + _mm(ctx, _f64(w.wo_q[l]), _f64(w.wo_s[l]))
        z = _mm(_norm(x, _f64(w.mlp_norm[l]), c.norm_eps), _f64(w.wi_q[l]), _f64(w.wi_s[l]))
        a, g = z.chunk(2, dim=1)
        a = 0.5 * a * (1 + torch.erf(a / math.sqrt(2.0)))
        x = x + _mm(a * g, _f64(w.womlp_q[l]), _f64(w.womlp_s[l]))
    return _norm(x, _f64(w.final_norm), c.norm_eps), [len(s) for s in seqs]


def _exact_linear(case, seed):
    (q, s, bias), _ = _linear_weights(case)
    x, q, s = _f64(_linear_rows(case, seed)), _f64(q), _f64(s)
    extra = 0.0
    if case["outliers"]:
        top = x.abs().amax(0)
        cols = torch.nonzero(top > RATIO * top.mean())[:, 0]
        cols = cols[torch.argsort(top[cols], descending=True)[:32]]
        extra = x[:, cols] @ (q[:, cols] * s[:, None]).T.contiguous()
        x = x.clone()
        x[:, cols] = 0
    return (_mm(x, q, s) + extra + _f64(bias)).cpu().numpy()


def exact(case, seed):
    if case["call"] == "linear":
        return _exact_linear(case, seed)
    x, lens = _states(case, seed)
    if case["call"] == "tokens":
        return x.cpu().numpy()
    if case["call"] == "spans":
        (w, b, _), = _head_weights(case["shape"], "spans")
        return (x @ _f64(w).T.contiguous() + _f64(b)).cpu().numpy()
    cls = case["pooling"] == "cls"
    pooled = torch.stack([r[0] if cls else r.mean(0) for r in x.split(lens)])
    if case["call"] == "decide":
        hs = _head_weights(case["shape"], "decide")
        w = _f64(np.concatenate([h[0] for h in hs]))
        b = _f64(np.concatenate([h[1] for h in hs]))
        pooled = pooled @ w.T.contiguous() + b
    return pooled.cpu().numpy()
