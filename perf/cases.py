"""The workloads this framework is timed on: what a program that trains or runs a GPT with it has the GPU do.

Every case goes through public entry points: the engine's operators and the GPT session (nnengine.py over
include/nnhip_engine.h) and, for the optimizer's update, the kernel library (include/nnhip_kernels.h). A case is a
plain dict; `kind` names the path and the other entries are its sizes and options.

  train      gradient accumulation: per micro-batch load_batch, forward_loss, backward_scaled; then the gradients
  decode     incremental inference: one token after another through the KV caches, logits of each
  linear     one Linear layer: forward with bias, and its three gradients
  attention  softmax attention forward and backward, one shared mask per packed row of heads
  head       the output head: logits, sparse cross-entropy and the head's gradients
  adamw      one AdamW update of a model's parameter list
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "neuralnet.cpp_amd"))

import nnengine  # noqa: E402

NORM_EPS = 1e-5
ADAM = dict(lr=1e-3, beta1=0.9, beta2=0.999, eps=1e-8, wd=0.01, t=100)
_ENGINE = None


def engine():
    """The program's one engine."""
    global _ENGINE
    if _ENGINE is None:
        _ENGINE = nnengine.Engine()
    return _ENGINE


# -- the cases ---------------------------------------------------------------
def listed():
    return [
        # A first training step on a small model (the repository's tiny GPT: 2 layers, d 128, T 128, batch 8): hundreds
        # of short launches, so call overheads and launch latency.
        dict(name="train_tiny", kind="train", layers=2, d=128, heads=4, ff=512, vocab=1024, seq=128, batch=8, micro=1,
             pos="learned", norm="rmsnorm", act="swiglu", docs=False),
        # The GPT-2 style options (learned positions, LayerNorm, QuickGeLU) at a middle size, an odd vocabulary and
        # a sequence length that is no multiple of a tile.
        dict(name="train_layernorm_gelu", kind="train", layers=3, d=512, heads=8, ff=2048, vocab=5003, seq=500, batch=6,
             micro=2, pos="learned", norm="layernorm", act="gelu", docs=False),
        # The benchmark model's layer shape (d 768, 12 heads, SwiGLU 3072, RMSNorm, ALiBi, context 1024), four layers
        # deep, with four accumulated micro-batches.
        dict(name="train_alibi_swiglu", kind="train", layers=4, d=768, heads=12, ff=3072, vocab=8192, seq=1024, batch=4,
             micro=4, pos="alibi", norm="rmsnorm", act="swiglu", docs=False),
        # Serving one stream: tokens in the middle of a 1024 context, the benchmark's layer shape.
        dict(name="decode_768", kind="decode", layers=6, d=768, heads=12, ff=3072, vocab=8192, seq=1024, cur=512, steps=8,
             pos="alibi", norm="rmsnorm", act="swiglu"),
        # The smallest products that are launched: a projection of a tiny model over 128 tokens.
        dict(name="linear_small", kind="linear", d_in=128, d_out=512, tokens=128),
        # Odd sizes in every dimension, as a vocabulary or a packed batch leaves them.
        dict(name="linear_odd", kind="linear", d_in=333, d_out=1001, tokens=2777),
        # The feed-forward's first product at the benchmark's 8192 tokens a step: the largest of a layer.
        dict(name="linear_ffn", kind="linear", d_in=768, d_out=6144, tokens=8192),
        # Causal attention, batch 16 x 8 heads at T 512 (the repository's attention benchmark), with its backward.
        dict(name="attention_causal", kind="attention", rows=1, heads=128, seq=512, dk=64, docs=False),
        # Packed documents in a 2048 context, each row with its own mask (the document-masked benchmark).
        dict(name="attention_docs", kind="attention", rows=8, heads=12, seq=2048, dk=64, docs=True),
        # Wide heads and an odd length: d 128 heads of a 1024-wide model at T 777.
        dict(name="attention_wide_odd", kind="attention", rows=1, heads=16, seq=777, dk=128, docs=False),
        # The output head over the benchmark's 32000 classes for two sequences of 1024.
        dict(name="head_32000", kind="head", d=768, vocab=32000, tokens=2048),
        # The optimizer over the benchmark's layer shapes: one layer, the embedding and the head.
        dict(name="adamw", kind="adamw", layers=1, d=768, ff=3072, vocab=8192),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "decode", "linear", "linear", "linear", "attention", "attention", "head",
                       "adamw"])
    if kind in ("train", "decode"):
        pos = rng.choice(["learned", "sinusoidal", "alibi", "rope"])
        heads = rng.choice([2, 4, 6, 8, 12])
        dk = rng.choice([16, 32, 40, 64, 64])
        c = dict(kind=kind, layers=rng.randint(1, 4), d=heads * dk, heads=heads, ff=_log(rng, 64, 3072),
                 vocab=_log(rng, 50, 8192), pos=pos, norm=rng.choice(["rmsnorm", "layernorm"]),
                 act=rng.choice(["swiglu", "gelu"]))
        if kind == "decode":
            seq = _log(rng, 64, 1024)
            steps = rng.randint(1, 8)
            return dict(c, seq=seq, cur=rng.randint(0, seq - steps), steps=steps)
        return dict(c, seq=_log(rng, 17, 1024), batch=rng.randint(1, 4), micro=rng.randint(1, 3),
                    docs=rng.random() < 0.3)
    if kind == "linear":
        return dict(kind=kind, d_in=_log(rng, 32, 3072), d_out=_log(rng, 32, 6144), tokens=_log(rng, 16, 8192))
    if kind == "attention":
        dk = rng.choice([16, 32, 40, 64, 64, 96, 128])
        docs = rng.random() < 0.4
        return dict(kind=kind, rows=rng.randint(2, 6) if docs else 1, heads=rng.choice([2, 4, 8, 12, 16, 32]),
                    seq=_log(rng, 33, 2048 if dk <= 64 else 1024), dk=dk, docs=docs)
    if kind == "head":
        return dict(kind=kind, d=_log(rng, 64, 1024), vocab=_log(rng, 256, 32000), tokens=_log(rng, 32, 2048))
    return dict(kind=kind, layers=1, d=_log(rng, 32, 768), ff=_log(rng, 64, 3072),
                vocab=_log(rng, 64, 8192))


# -- inputs ------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _randint(g, hi, *shape):
    return torch.randint(0, hi, shape, generator=g, device="cuda")


def _up(x):
    return engine().tensor(x.cpu().numpy())


class _DeviceArray:
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr="<f4", strides=None, version=2)


def _view(t):
    """An engine tensor as a torch tensor on the same memory, everything it depends on queued."""
    return torch.as_tensor(_DeviceArray(t.device_ptr(), t.shape), device="cuda")


def _gpt_shapes(c):
    """(shape, role) of each parameter in the session's order."""
    d, v, ff = c["d"], c["vocab"], c["ff"]
    norm = [((d, 1), "gain")] + ([((d, 1), "shift")] if c["norm"] == "layernorm" else [])
    up = 2 * ff if c["act"] == "swiglu" else ff
    out = [((v, d), "weight")]
    if c["pos"] == "learned":
        out.append(((c["seq"], d), "weight"))
    for _ in range(c["layers"]):
        out += [((d, d), "weight"), ((d, 1), "bias")] * 4 + norm
        out += [((up, d), "weight"), ((up, 1), "bias"), ((d, ff), "weight"), ((d, 1), "bias")] + norm
    return out + norm + [((v, d), "weight"), ((v, 1), "bias")]


def _gpt_params(c, g):
    """Weights as after some training: matrices N(0, 0.02) to N(0, 0.04), gains about 1, biases about 0."""
    out = []
    for shape, role in _gpt_shapes(c):
        if role == "gain":
            out.append(1.0 + _randn(g, *shape, std=0.1))
        else:
            out.append(_randn(g, *shape, std=0.03 if role == "weight" else 0.01))
    return out


def _session(c, params):
    s = engine().gpt(vocab_size=c["vocab"], d_model=c["d"], seq_len=c["seq"], num_heads=c["heads"], d_ff=c["ff"],
                     num_layers=c["layers"], pos_enc=c["pos"], activation=c["act"], norm=c["norm"])
    s.set_params([p.cpu().numpy() for p in params])
    return s


def _doc_ids(c, g, row_len, rows):
    """Document numbers of packed rows: lengths uniform in [row_len / 32, row_len / 2]."""
    out = np.empty((rows, row_len), np.uint64)
    r = np.random.default_rng(int(_randint(g, 1 << 30, 1).item()))
    for b in range(rows):
        at, n = 0, 0
        while at < row_len:
            step = int(r.integers(max(1, row_len // 32), max(2, row_len // 2 + 1)))
            n += 1
            out[b, at:at + step] = n
            at += step
    return out


def _train_inputs(c, seed):
    g = _gen(seed)
    params = _gpt_params(c, g)
    toks = [_randint(g, c["vocab"], c["seq"] + 1, c["batch"]).cpu().numpy() for _ in range(c["micro"])]
    docs = _doc_ids(c, g, c["seq"], c["batch"]) if c["docs"] else None
    return params, toks, docs


def _decode_inputs(c, seed):
    g = _gen(seed)
    params = _gpt_params(c, g)
    return params, _randint(g, c["vocab"], c["cur"] + c["steps"]).cpu().tolist()


def _linear_inputs(c, seed):
    g = _gen(seed)
    return (_randn(g, c["d_out"], c["d_in"], std=0.03), _randn(g, c["d_out"], 1, std=0.01),
            _randn(g, c["d_in"], c["tokens"]), _randn(g, c["d_out"], c["tokens"], std=1e-3))


def _attention_inputs(c, seed):
    g = _gen(seed)
    t, n = c["seq"], c["heads"] * c["dk"]
    rows = [tuple(_randn(g, n, t) for _ in range(4)) for _ in range(c["rows"])]
    docs = _doc_ids(c, g, t, c["rows"]) if c["docs"] else None
    return rows, docs


def _head_inputs(c, seed):
    g = _gen(seed)
    return (_randn(g, c["vocab"], c["d"], std=0.05), _randn(g, c["vocab"], 1, std=0.01),
            _randn(g, c["d"], c["tokens"]), _randint(g, c["vocab"], c["tokens"]))


def _adam_shapes(c):
    return [s for s, _ in _gpt_shapes(dict(c, norm="rmsnorm", act="swiglu", pos="alibi"))]


def _adam_inputs(c, seed):
    g = _gen(seed)
    shapes = _adam_shapes(c)
    p = [_randn(g, *s, std=0.03) for s in shapes]
    m = [_randn(g, *s, std=1e-4) for s in shapes]
    v = [_randn(g, *s, std=1e-4) ** 2 for s in shapes]
    gr = [_randn(g, *s, std=1e-3) for s in shapes]
    return p, m, v, gr


def _adam_scalars():
    a = ADAM
    f = np.float32
    b1, b2 = f(a["beta1"]), f(a["beta2"])
    return dict(decay=f(1 - a["lr"] * a["wd"]), beta1=b1, one_minus_beta1=f(1) - b1, beta2=b2, one_minus_beta2=f(1) - b2,
                inv_bc1=f(1 / (1 - float(b1) ** a["t"])), inv_bc2=f(1 / (1 - float(b2) ** a["t"])), eps=f(a["eps"]),
                neg_lr=f(-a["lr"]))


def prepare(case, seed):
    c, e = case, engine()
    if c["kind"] == "train":
        params, toks, docs = _train_inputs(c, seed)
        s = _session(c, params)
        if docs is not None:
            s.set_doc_ids(docs)
        batches = [(t[:-1].astype(np.float32), np.ascontiguousarray(t[1:].T).reshape(-1)) for t in toks]
        s.load_batch(*batches[0])
        s.forward_loss()
        return dict(case=c, s=s, batches=batches, shapes=_gpt_shapes(c))
    if c["kind"] == "decode":
        params, toks = _decode_inputs(c, seed)
        s = _session(c, params)
        s.reset_cache()
        for i in range(c["cur"]):
            s.forward_step(toks[i], i, i)
        return dict(case=c, s=s, toks=toks[c["cur"]:])
    if c["kind"] == "linear":
        w, b, x, gr = _linear_inputs(c, seed)
        return dict(case=c, w=_up(w), b=_up(b), x=_up(x), g=_up(gr), gw=e.create_tensor(*w.shape),
                    gb=e.create_tensor(*b.shape))
    if c["kind"] == "attention":
        rows, docs = _attention_inputs(c, seed)
        up = []
        for r, qkvg in enumerate(rows):
            ids = docs[r] if docs is not None else ()
            up.append([_up(x) for x in qkvg] + [e.tensor(e.build_attention_mask(1, c["seq"], 1, False, doc_ids=ids))])
        return dict(case=c, rows=up)
    if c["kind"] == "head":
        w, b, x, lab = _head_inputs(c, seed)
        return dict(case=c, w=_up(w), b=_up(b), x=_up(x), lab=_up(lab.float().reshape(1, -1)),
                    gw=e.create_tensor(*w.shape), gb=e.create_tensor(*b.shape))
    p, m, v, gr = _adam_inputs(c, seed)
    lib = nnengine.hip_library()
    fn = lib.nnhip_adam_update_list
    f = ctypes.c_float
    fn.argtypes = [ctypes.c_void_p] * 5 + [ctypes.c_size_t, ctypes.c_int] + [f] * 9 + [ctypes.c_void_p]
    n = len(p)
    lists = [(ctypes.c_void_p * n)(*[t.data_ptr() for t in ts]) for ts in (p, m, v, gr)]
    lists.append((ctypes.c_size_t * n)(*[t.numel() for t in p]))
    return dict(case=c, fn=fn, lists=lists, n=n, scalars=[float(x) for x in _adam_scalars().values()], p=p, m=m, v=v,
                g=gr)


# -- one pass ----------------------------------------------------------------
def _gather_grads(shapes, grads):
    """Weight gradients one by one; the vectors (biases, gains) as one, as an optimizer's flat group holds them."""
    mats = [a for (_, role), a in zip(shapes, grads) if role == "weight"]
    return mats + [np.concatenate([a.reshape(-1) for (_, role), a in zip(shapes, grads) if role != "weight"])]


def _run_train(st):
    s, n = st["s"], len(st["batches"])
    s.zero_grad()
    losses = []
    for tokens, labels in st["batches"]:
        s.load_batch(tokens, labels)
        losses.append(s.forward_loss())
        s.backward_scaled(1.0 / n)
    return [np.array(losses, np.float32)] + _gather_grads(st["shapes"], s.grads())


def _run_decode(st):
    s, cur = st["s"], st["case"]["cur"]
    return [s.forward_step(t, cur + i, cur + i) for i, t in enumerate(st["toks"])]


def _linear_backward(e, st, g):
    dx = e.matmul(st["w"], g, True, False)
    e.add_inplace(st["gw"], e.matmul(g, st["x"], False, True))
    e.add_inplace(st["gb"], e.row_reduce_sum(g))
    return dx


def _run_linear(st):
    e = engine()
    e.zero(st["gw"])
    e.zero(st["gb"])
    y = e.matmul(st["w"], st["x"])
    e.broadcast_row_inplace(y, st["b"], "Add")
    dx = _linear_backward(e, st, st["g"])
    st["out"] = [y, dx, st["gw"], st["gb"]]
    return [_view(t) for t in st["out"]]


def _attention_row(e, c, q, k, v, g, mask):
    """The attention layer's calls for one row of heads; its temporaries end with it."""
    h, t, d = c["heads"], c["seq"], c["dk"]
    alpha = 1.0 / math.sqrt(d)
    m = e.batched_matmul_reduce(q, k, h, "Max", True, False, alpha, True, mask)
    l = e.batched_matmul_softmax_denom(q, k, m, h, True, False, alpha, mask)
    vt = e.rearrange_3d(e.transpose(v), t, h, d)
    o = e.batched_matmul_softmax_apply(q, k, vt, m, l, h, True, False, alpha, mask)
    p = e.batched_matmul(g, v, h, True, False)
    gt = e.rearrange_3d(e.transpose(g), t, h, d)
    dq, r = e.batched_matmul_softmax_backward_q(q, k, p, m, l, h, True, False, alpha, mask)
    dk, dv = e.batched_matmul_softmax_backward_kv(q, k, p, gt, r, m, l, h, True, False, alpha, mask)
    return [o, dq, dk, dv]


def _run_attention(st):
    st["out"] = [x for row in st["rows"] for x in _attention_row(engine(), st["case"], *row)]
    return [_view(x) for x in st["out"]]


def _run_head(st):
    c, e = st["case"], engine()
    e.zero(st["gw"])
    e.zero(st["gb"])
    y = e.matmul(st["w"], st["x"])
    e.broadcast_row_inplace(y, st["b"], "Add")
    g, lv = e.col_softmax_sparse_forward(y, st["lab"], None, c["vocab"], 1.0 / c["tokens"])
    dx = _linear_backward(e, st, g)
    st["out"] = [y, lv, dx, st["gw"], st["gb"]]
    return [_view(t) for t in st["out"]]


def _run_adamw(st):
    rc = st["fn"](*st["lists"], st["n"], 1, *st["scalars"], torch.cuda.current_stream().cuda_stream)
    if rc != 0:
        raise RuntimeError(f"nnhip_adam_update_list: {rc}")
    return st["p"] + st["m"] + st["v"]


def run(state):
    return {"train": _run_train, "decode": _run_decode, "linear": _run_linear, "attention": _run_attention,
            "head": _run_head, "adamw": _run_adamw}[state["case"]["kind"]](state)


# -- what a pass cannot do without -------------------------------------------
def _pairs(c, docs=None):
    """Allowed (query, key) pairs of one row of T tokens: causal, or causal within the mean document length."""
    t = c["seq"]
    if not c.get("docs"):
        return t * (t + 1) / 2
    mean = max(1.0, (max(1, t // 32) + max(2, t // 2 + 1) - 1) / 2)
    return t * (mean + 1) / 2


def work(case):
    c = case
    if c["kind"] in ("train", "decode"):
        shapes = [s for s, _ in _gpt_shapes(c)]
        params = sum(a * b for a, b in shapes)
        products = sum(a * b for (a, b), (_, role) in zip(shapes, _gpt_shapes(c)) if role == "weight") - c["vocab"] * c["d"]
        if c["pos"] == "learned":
            products -= c["seq"] * c["d"]
        if c["kind"] == "decode":
            kv = sum(2 * c["layers"] * (c["cur"] + i + 1) * c["d"] for i in range(c["steps"]))
            rest = params - c["vocab"] * c["d"]
            return dict(bytes=4.0 * (c["steps"] * rest + kv + c["steps"] * c["vocab"]),
                        flops=2.0 * c["steps"] * products + 2.0 * kv)
        n = c["batch"] * c["seq"]
        attn = 12.0 * c["layers"] * c["d"] * c["batch"] * _pairs(c)
        return dict(bytes=4.0 * 2 * params, flops=c["micro"] * (6.0 * products * n + attn))
    if c["kind"] == "linear":
        i, o, n = c["d_in"], c["d_out"], c["tokens"]
        return dict(bytes=4.0 * (2 * o * i + 2 * o + 2 * i * n + 2 * o * n), flops=6.0 * i * o * n)
    if c["kind"] == "attention":
        n = c["rows"] * c["heads"] * c["dk"] * c["seq"]
        return dict(bytes=4.0 * (8 * n + c["rows"] * c["seq"] ** 2),
                    flops=12.0 * c["rows"] * c["heads"] * c["dk"] * _pairs(c))
    if c["kind"] == "head":
        d, v, n = c["d"], c["vocab"], c["tokens"]
        return dict(bytes=4.0 * (2 * v * d + 2 * d * n + v * n + 2 * n), flops=6.0 * d * v * n)
    count = sum(a * b for a, b in _adam_shapes(c))
    return dict(bytes=4.0 * 7 * count, flops=14.0 * count)


def tolerance(case):
    # Four times the largest error against 64 bits that float32 sums in another order showed over the ranges.
    return {"train": dict(rel=2e-5, max=2e-3), "decode": dict(rel=1e-5, max=1e-4), "linear": dict(rel=1e-5, max=1e-4),
            "attention": dict(rel=1e-5, max=1e-3), "head": dict(rel=1e-5, max=1e-3), "adamw": dict(rel=1e-6, max=1e-4)}[
                case["kind"]]


# -- the same results in 64 bits ---------------------------------------------
def _exact_norm(c, x, it):
    if c["norm"] == "rmsnorm":
        return x / torch.sqrt((x * x).mean(0, keepdim=True) + NORM_EPS) * next(it)
    z = x - x.mean(0, keepdim=True)
    return z / torch.sqrt((z * z).mean(0, keepdim=True) + NORM_EPS) * next(it) + next(it)


def _exact_rope(x, t):
    """(B, H, dk, T): rows j and j + dk/2 turned by position * 10000^(-2j/dk)."""
    half = x.shape[2] // 2
    j = torch.arange(half, dtype=torch.float64, device="cuda")[:, None]
    ang = torch.arange(t, dtype=torch.float64, device="cuda")[None, :] * 10000.0 ** (-2.0 * j / (2 * half))
    lo, hi, co, si = x[:, :, :half], x[:, :, half:], torch.cos(ang), torch.sin(ang)
    return torch.cat([lo * co - hi * si, hi * co + lo * si], dim=2)


def _exact_gpt(c, params, tokens, docs=None):
    """Logits (vocab, batch * T) of tokens (T, batch), column b*T + t."""
    t, b = tokens.shape
    d, h = c["d"], c["heads"]
    dk = d // h
    f64 = dict(dtype=torch.float64, device="cuda")
    it = iter(params)
    x = next(it)[tokens.T.reshape(-1)]
    if c["pos"] == "learned":
        x = x + next(it)[:t].repeat(b, 1)
    elif c["pos"] == "sinusoidal":
        i = torch.arange(d, **f64)
        ang = torch.arange(t, **f64)[:, None] / 10000.0 ** (2 * torch.floor(i / 2) / d)[None, :]
        x = x + torch.where(i % 2 == 0, torch.sin(ang), torch.cos(ang)).repeat(b, 1)
    x = x.T
    i = torch.arange(t, device="cuda")
    allowed = (i[None, :] <= i[:, None])[None, None]
    if docs is not None:
        ids = torch.as_tensor(docs.astype(np.int64), device="cuda")
        allowed = allowed & (ids[:, None, :, None] == ids[:, None, None, :])
    bias = torch.zeros(1, 1, 1, 1, **f64)
    if c["pos"] == "alibi":
        slope = 2.0 ** (-8.0 * torch.arange(h, **f64) / h)
        bias = -slope[None, :, None, None] * (i[:, None] - i[None, :]).double()[None, None]
    heads = lambda z: z.reshape(h, dk, b, t).permute(2, 0, 1, 3)   # (B, H, dk, T)  # noqa: E731
    for _ in range(c["layers"]):
        wq, bq, wk, bk, wv, bv, wo, bo = (next(it) for _ in range(8))
        n = _exact_norm(c, x, it)
        q, k, v = heads(wq @ n + bq), heads(wk @ n + bk), heads(wv @ n + bv)
        if c["pos"] == "rope":
            q, k = _exact_rope(q, t), _exact_rope(k, t)
        s = (q.transpose(2, 3).contiguous() @ k / math.sqrt(dk) + bias).masked_fill(~allowed, -math.inf)
        o = v @ torch.softmax(s, dim=3).transpose(2, 3).contiguous()
        x = x + wo @ o.permute(1, 2, 0, 3).reshape(d, b * t) + bo
        w1, b1, w2, b2 = (next(it) for _ in range(4))
        u = w1 @ _exact_norm(c, x, it) + b1
        if c["act"] == "swiglu":
            gate, up = u[:c["ff"]], u[c["ff"]:]
            u = gate * torch.sigmoid(gate) * up
        else:
            u = u * torch.sigmoid(1.702 * u)
        x = x + w2 @ u + b2
    x = _exact_norm(c, x, it)
    return next(it) @ x + next(it)


def _exact_train(c, seed):
    params, toks, docs = _train_inputs(c, seed)
    shapes = _gpt_shapes(c)
    params = [p.double().requires_grad_(True) for p in params]
    losses = []
    for t in toks:
        t = torch.as_tensor(t, device="cuda")
        labels = t[1:].T.reshape(-1)
        loss = torch.nn.functional.cross_entropy(_exact_gpt(c, params, t[:-1], docs).T, labels)
        (loss / len(toks)).backward()
        losses.append(float(loss.detach()))
    # A gain's gradient is kept times the gain, as the layers accumulate it.
    grads = [(p.grad * p.detach() if role == "gain" else p.grad).cpu().numpy() for (_, role), p in zip(shapes, params)]
    return [np.array(losses)] + _gather_grads(shapes, grads)


def _exact_decode(c, seed):
    params, toks = _decode_inputs(c, seed)
    with torch.no_grad():
        logits = _exact_gpt(c, [p.double() for p in params], torch.tensor(toks, device="cuda")[:, None])
    return [logits[:, c["cur"] + i].cpu().numpy() for i in range(c["steps"])]


def _exact_linear(c, seed):
    w, b, x, g = (t.double() for t in _linear_inputs(c, seed))
    return [w @ x + b, w.T @ g, g @ x.T, g.sum(1, keepdim=True)]


def _exact_attention(c, seed):
    rows, docs = _attention_inputs(c, seed)
    h, t, d = c["heads"], c["seq"], c["dk"]
    i = torch.arange(t, device="cuda")
    out = []
    for r, row in enumerate(rows):
        q, k, v, g = (x.double().reshape(h, d, t) for x in row)
        allowed = i[None, :] <= i[:, None]
        if docs is not None:
            ids = torch.as_tensor(docs[r].astype(np.int64), device="cuda")
            allowed = allowed & (ids[:, None] == ids[None, :])
        s = (q.transpose(1, 2).contiguous() @ k / math.sqrt(d)).masked_fill(~allowed[None], -math.inf)
        p = torch.softmax(s, dim=2)
        dp = g.transpose(1, 2).contiguous() @ v
        o = p @ v.transpose(1, 2).contiguous()          # (H, T, d)
        ds = p * (dp - (p * dp).sum(2, keepdim=True)) / math.sqrt(d)
        dq = k @ ds.transpose(1, 2).contiguous()
        dk = q @ ds
        dv = g @ p
        out += [o.reshape(h * t, d), dq.reshape(h * d, t), dk.reshape(h * d, t), dv.reshape(h * d, t)]
    return out


def _exact_head(c, seed):
    w, b, x, lab = _head_inputs(c, seed)
    w, b, x = w.double(), b.double(), x.double()
    n = c["tokens"]
    y = w @ x + b
    logp = torch.log_softmax(y, dim=0)
    at = torch.arange(n, device="cuda")
    g = torch.exp(logp)
    g[lab, at] -= 1.0
    g /= n
    return [y, logp[lab, at].reshape(1, n), w.T @ g, g @ x.T, g.sum(1, keepdim=True)]


def _exact_adamw(c, seed):
    p, m, v, g = _adam_inputs(c, seed)
    a = {k: float(x) for k, x in _adam_scalars().items()}
    new = ([], [], [])
    for pi, mi, vi, gi in zip(p, m, v, g):
        pi, mi, vi, gi = (t.double() for t in (pi, mi, vi, gi))
        mi = mi * a["beta1"] + a["one_minus_beta1"] * gi
        vi = vi * a["beta2"] + gi * gi * a["one_minus_beta2"]
        pi = pi * a["decay"] + a["neg_lr"] * (mi * a["inv_bc1"]) / (torch.sqrt(vi * a["inv_bc2"]) + a["eps"])
        for out, t in zip(new, (pi, mi, vi)):
            out.append(t)
    return new[0] + new[1] + new[2]


def exact(case, seed):
    return {"train": _exact_train, "decode": _exact_decode, "linear": _exact_linear, "attention": _exact_attention,
            "head": _exact_head, "adamw": _exact_adamw}[case["kind"]](case, seed)
