"""Workloads of the gpt-oss layers and of the decode loop, for timing and comparison.

Five kinds, each through the entry point a serving program calls:

  moe      MLPBlock(x): RMSNorm, router, top-4, both MXFP4 expert matmuls, combine and
           residual, at the 20B (32 experts) and 120B (128 experts) shapes, from one decode
           token to a 4096-token prefill, with uniform or Zipf-skewed routing
  decode   AttentionBlock(x, cache), one new token for each of a ragged batch of sequences
           over the paged KV cache
  prefill  AttentionBlock(x, cache), the prompts of one or a few sequences, over nothing or
           over a cached prefix (the next turn of a chat)
  head     final norm, unembedding and top-p sampling of up to 8 sequences
  loop     Engine.decode_sample: one whole 24-layer decode step replayed from its graph,
           after the previous token was rolled back and sampled again

Inputs come from the seed alone, by functions that `exact` shares.  The distributions are the
benchmark's: MXFP4 bytes uniform, E8M0 scales 118..122, dense weights N(0, 0.02), biases
N(0, 0.01), activations N(0, 1).
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpt-oss-tvm_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

import attn_native  # noqa: E402
from engine import Engine  # noqa: E402
from model.attention import AttentionBlock  # noqa: E402
from model.config import GPTOssConfig, gpt_oss_20b  # noqa: E402
from model.kv_cache import PagedKVCache  # noqa: E402
from model.mlp import MLPBlock  # noqa: E402

DEV = "cuda"
BF = torch.bfloat16
HIDDEN, TOP_K, VOCAB, LAYERS = 2880, 4, 201088, 24
QH, KVH, DIM, PAGE = 64, 8, 64, 16
QKV = (QH + 2 * KVH) * DIM
EPS, LIMIT, ALPHA = 1e-5, 7.0, 1.702
WINDOW = 128
ROUND = 256            # tokens by which the sequences of a batch grow in turn
EXPERT_BYTES = 3 * HIDDEN * (HIDDEN // 32) * 17 + 3 * HIDDEN * 2


# -- the cases ---------------------------------------------------------------------------

def listed():
    return [
        # one chat at a time: every layer of every token of a single user's answer
        {"name": "moe20b_decode1", "kind": "moe", "experts": 32, "tokens": 1, "zipf": 0.0},
        # a lightly loaded server
        {"name": "moe20b_decode7", "kind": "moe", "experts": 32, "tokens": 7, "zipf": 0.0},
        # the benchmark's headline: a full decode batch
        {"name": "moe20b_decode64", "kind": "moe", "experts": 32, "tokens": 64, "zipf": 0.0},
        # an ordinary chat prompt, or decode tokens mixed with a short chunk
        {"name": "moe20b_prompt333", "kind": "moe", "experts": 32, "tokens": 333, "zipf": 0.0},
        # a long prompt, skewed over the experts as real text is
        {"name": "moe20b_prefill4096", "kind": "moe", "experts": 32, "tokens": 4096, "zipf": 0.5},
        # the large model: a decode batch, and a prefill chunk
        {"name": "moe120b_decode256", "kind": "moe", "experts": 128, "tokens": 256, "zipf": 0.0},
        {"name": "moe120b_prefill2048", "kind": "moe", "experts": 128, "tokens": 2048,
         "zipf": 0.0},
        # a full layer of a decode batch with chats of all lengths
        {"name": "attn_decode64", "kind": "decode", "sequences": 64, "context": 4096,
         "window": False},
        # a full layer of a long prompt
        {"name": "attn_prefill4096", "kind": "prefill", "sequences": 1, "tokens": 4096,
         "prefix": 0, "window": False},
        # a full layer of a chat's next turn: a short text over what is cached
        {"name": "attn_extend300", "kind": "prefill", "sequences": 1, "tokens": 300,
         "prefix": 6000, "window": False},
        # the end of a small decode step: next-token logits and the sampled tokens
        {"name": "head5", "kind": "head", "sequences": 5},
        # the whole decode step of a single user, 20B model
        {"name": "loop20b_context1000", "kind": "loop", "context": 1000},
    ]


def _spread(rng, lo, hi):
    """An integer of lo..hi, uniform in its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    u = rng.random()
    if u < 0.45:
        experts = rng.choice([32, 32, 128])
        n = _spread(rng, 1, 4096 if experts == 32 else 2048)
        return {"kind": "moe", "experts": experts, "tokens": n, "zipf": rng.choice([0.0, 0.5])}
    if u < 0.65:
        return {"kind": "decode", "sequences": _spread(rng, 1, 64),
                "context": _spread(rng, 16, 4096), "window": rng.random() < 0.3}
    if u < 0.85:
        tokens = _spread(rng, 9, 4096)
        sequences = rng.choice([1, 1, 2, 3])
        # no more query-key pairs than the longest listed prompt has
        most = max(0, min(8192, 4096 * 2048 // tokens - tokens // 2))
        return {"kind": "prefill", "sequences": sequences, "tokens": tokens,
                "prefix": rng.choice([0, rng.randint(0, most)]), "window": rng.random() < 0.3}
    if u < 0.93:
        return {"kind": "head", "sequences": rng.randint(1, 8)}
    return {"kind": "loop", "context": _spread(rng, 32, 2000)}


# -- inputs, from the seed alone ------------------------------------------------------------

def _gen(seed, *parts):
    g = torch.Generator(device=DEV)
    value = 1469598103934665603
    for p in (seed, *parts):
        value = ((value ^ (int(p) + 7)) * 1099511628211) % (1 << 63)
    g.manual_seed(value)
    return g


def _normal(g, shape, std=1.0, mean=0.0):
    return (torch.randn(shape, generator=g, device=DEV) * std + mean).to(BF)


def _bytes(g, shape, lo, hi):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=torch.uint8)


def _moe_params(g, experts, zipf, low=(118, 118)):
    """The nine tensors of a block by its parameter names; `low`: the smallest scale byte of
    mlp1 and of mlp2."""
    h, groups = HIDDEN, HIDDEN // 32
    bias = torch.randn(experts, generator=g, device=DEV) * 0.01
    if zipf:
        p = torch.arange(1, experts + 1, device=DEV, dtype=torch.float64) ** -1.1
        bias = bias + (zipf * torch.log(p / p.sum())).float()
    return {
        "norm.weight": _normal(g, (h,), 0.1, 1.0),
        "gate.weight": _normal(g, (experts, h), 0.02),
        "gate.bias": bias.to(BF),
        "mlp1_weight_blocks": _bytes(g, (experts, 2 * h, groups, 16), 0, 256),
        "mlp1_weight_scales": _bytes(g, (experts, 2 * h, groups), low[0], low[0] + 5),
        "mlp1_bias": _normal(g, (experts, 2 * h), 0.01),
        "mlp2_weight_blocks": _bytes(g, (experts, h, groups, 16), 0, 256),
        "mlp2_weight_scales": _bytes(g, (experts, h, groups), low[1], low[1] + 5),
        "mlp2_bias": _normal(g, (experts, h), 0.01),
    }


def _attn_params(g):
    return {
        "sinks": _normal(g, (QH,)),
        "norm.weight": _normal(g, (HIDDEN,), 0.1, 1.0),
        "qkv.weight": _normal(g, (QKV, HIDDEN), 0.02),
        "qkv.bias": _normal(g, (QKV,), 0.01),
        "out.weight": _normal(g, (HIDDEN, QH * DIM), 0.02),
        "out.bias": _normal(g, (HIDDEN,), 0.01),
    }


def _fill(module, params):
    with torch.no_grad():
        for name, value in params.items():
            module.get_parameter(name).copy_(value)
    return module


def _lengths(case):
    """(cached, new) tokens of each sequence, the same for every seed."""
    b = case["sequences"]
    rng = random.Random("%d %d" % (b, case.get("context", case.get("tokens"))))
    if case["kind"] == "decode":  # the new token included, a context is at most "context" long
        return [(max(0, round(case["context"] * rng.uniform(0.25, 1.0)) - 1), 1)
                for _ in range(b)]
    cuts = sorted(rng.sample(range(1, case["tokens"]), b - 1))
    return [(case["prefix"], hi - lo) for lo, hi in zip([0] + cuts, cuts + [case["tokens"]])]


def _pages(lengths):
    """The pages of each sequence of a pool that hands them out in order, when the cached
    tokens came in turns of ROUND and the new ones in one forward."""
    pages, used, done = [[] for _ in lengths], 0, 0
    turns = []
    while any(done < c for c, _ in lengths):
        done += ROUND
        turns.append([min(c, done) for c, _ in lengths])
    turns.append([c + n for c, n in lengths])
    for turn in turns:
        for p, length in zip(pages, turn):
            while len(p) * PAGE < length:
                p.append(used)
                used += 1
    return pages, used


def _head_inputs(seed, b):
    """Hidden states whose logits have a clear favourite, as a trained model's do."""
    g = _gen(seed, 5)
    w = _normal(g, (VOCAB, HIDDEN), 0.02)
    norm = _normal(g, (HIDDEN,), 0.1, 1.0)
    tokens = torch.randint(0, VOCAB, (b,), generator=g, device=DEV)
    toward = w[tokens].float()
    toward = toward / toward.norm(dim=1, keepdim=True)
    x = torch.randn((b, HIDDEN), generator=g, device=DEV)
    x = x + toward * (0.3 * math.sqrt(HIDDEN))
    return w, norm, x.to(BF)


def _loop_token(seed):
    """The last step's logits [1, 1, vocab] (bf16 values in fp32) and the token they yield:
    it has most of the probability."""
    g = _gen(seed, 6)
    logits = torch.randn(VOCAB, generator=g, device=DEV)
    token = int(torch.randint(0, VOCAB, (1,), generator=g, device=DEV).item())
    logits[token] = 14.0
    return logits.to(BF).float().view(1, 1, VOCAB), token


def _loop_layer(seed, i):
    """A layer's parameters.  mlp2's scales are eight binades below the benchmark's: a layer
    changes the residual stream a little, as in a trained model (at the benchmark's the MoE
    output is twelve times its input)."""
    g = _gen(seed, 7, i)
    return _attn_params(g), _moe_params(g, 32, 0.0, (118, 110))


def _loop_ends(seed):
    g = _gen(seed, 8)
    return (_normal(g, (VOCAB, HIDDEN)), _normal(g, (HIDDEN,), 0.1, 1.0),
            _normal(g, (VOCAB, HIDDEN), 0.02))


# -- what a program holds before the call -----------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "moe":
            g = _gen(seed, 1)
            block = MLPBlock(GPTOssConfig(num_experts=case["experts"]), device=DEV)
            _fill(block, _moe_params(g, case["experts"], case["zipf"]))
            x = _normal(g, (1, case["tokens"], HIDDEN))
            block.reserve(case["tokens"])
            return {"kind": kind, "block": block, "x": x}
        if kind in ("decode", "prefill"):
            return _prepare_attention(case, seed)
        if kind == "head":
            w, norm, x = _head_inputs(seed, case["sequences"])
            return {"kind": kind, "w": w, "norm": norm, "x": x,
                    "workspace": attn_native.sample_workspace(case["sequences"], DEV)}
        return _prepare_loop(case, seed)


def _prepare_attention(case, seed):
    g = _gen(seed, 2)
    lengths = _lengths(case)
    layer = 0 if case["window"] else 1     # even layers slide
    block = _fill(AttentionBlock(GPTOssConfig(), layer_idx=layer, device=DEV), _attn_params(g))
    new = sum(n for _, n in lengths)
    x = _normal(g, (1, new, HIDDEN))
    _, used = _pages(lengths)
    ids = list(range(len(lengths)))
    cache = PagedKVCache(2, used, len(ids), max(new, ROUND * len(ids)), device=DEV)
    cache.data[layer].copy_(_normal(g, tuple(cache.data[layer].shape)))
    for i in ids:
        cache.add_sequence(i)
        cache.enable_sliding_window(i, WINDOW)
    done = 0
    while any(done < c for c, _ in lengths):
        grow = [(i, min(c - done, ROUND)) for i, (c, _) in enumerate(lengths) if c > done]
        cache.begin_forward([i for i, _ in grow], [n for _, n in grow])
        cache.end_forward()
        done += ROUND
    # a forward's tables serve all of its layers: they are there before this one
    cache.begin_forward(ids, [n for _, n in lengths])
    return {"kind": case["kind"], "block": block, "x": x, "cache": cache, "layer": layer}


def _prepare_loop(case, seed):
    cfg = gpt_oss_20b()
    cfg.context_window_size = cfg.prefill_chunk_size = 4096
    eng = Engine(config=cfg, max_total_seq_len=case["context"] + 64)
    for i, layer in enumerate(eng.model.model.block):
        attn, moe = _loop_layer(seed, i)
        _fill(layer.attn, attn)
        _fill(layer.mlp, moe)
    emb, norm, unembed = _loop_ends(seed)
    eng.model.model.embedding.weight.copy_(emb)
    eng.model.model.norm.weight.copy_(norm)
    eng.model.unembedding.weight.copy_(unembed)
    seq = eng.begin_sequence()
    cache = eng.paged_kv_cache
    cache.begin_forward([seq], [case["context"]])
    cache.end_forward()
    for i in range(LAYERS):
        data = cache.layer(i)
        data.copy_(_normal(_gen(seed, 9, i), tuple(data.shape)))
    logits, _ = _loop_token(seed)
    eng.sample_device(logits)
    eng.capture_decode(seq)
    return {"kind": "loop", "engine": eng, "seq": seq, "logits": logits}


# -- one pass ------------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    with torch.no_grad():
        if kind == "moe":
            return state["block"](state["x"])
        if kind in ("decode", "prefill"):
            out = state["block"](state["x"], state["cache"])
            return out, state["cache"].layer(state["layer"])
        if kind == "head":
            logits = attn_native.gemv(state["x"], state["w"], norm_w=state["norm"], eps=EPS)
            return logits, attn_native.sample_top_p(logits, 0.7, 0.9, 0.5, state["workspace"])
        eng, seq = state["engine"], state["seq"]
        eng.sample_device(state["logits"])
        eng.decode_sample(seq)
        logits = eng.graph_logits
        eng.popn(seq, 1)
        return logits


# -- what a pass cannot do without -------------------------------------------------------------

def _attended(cached, new, window):
    """(query-key pairs, keys read) of one head and one sequence."""
    w = window or (cached + new)
    pairs = sum(min(p + 1, w) for p in range(cached, cached + new))
    return pairs, min(cached + new, w + new - 1)


def work(case):
    kind = case["kind"]
    if kind == "moe":
        e, n = case["experts"], case["tokens"]
        touched = e * (1.0 - (1.0 - TOP_K / e) ** n)
        return {"bytes": touched * EXPERT_BYTES + e * (HIDDEN + 1) * 2 + HIDDEN * 2
                + n * HIDDEN * 4,
                "flops": n * (2.0 * TOP_K * 3 * HIDDEN * HIDDEN + 2.0 * HIDDEN * e)}
    if kind in ("decode", "prefill"):
        lengths = _lengths(case)
        each = [_attended(c, n, WINDOW if case["window"] else 0) for c, n in lengths]
        n = sum(m for _, m in lengths)
        dense = QKV * HIDDEN + HIDDEN * QH * DIM
        return {"bytes": 2.0 * dense + n * HIDDEN * 4 + 2 * (n + sum(k for _, k in each))
                * KVH * DIM * 2,
                "flops": 2.0 * n * dense + sum(p for p, _ in each) * QH * 4.0 * DIM}
    if kind == "head":
        b = case["sequences"]
        return {"bytes": 2.0 * VOCAB * HIDDEN + b * (2 * HIDDEN + 2 * VOCAB),
                "flops": 2.0 * b * VOCAB * HIDDEN}
    dense = QKV * HIDDEN + HIDDEN * QH * DIM
    keys = LAYERS // 2 * (case["context"] + 1 + min(case["context"] + 1, WINDOW))
    return {"bytes": LAYERS * (2.0 * dense + TOP_K * EXPERT_BYTES + 64 * HIDDEN)
            + 2.0 * VOCAB * HIDDEN + keys * KVH * DIM * 4 + 4 * VOCAB,
            "flops": LAYERS * (2.0 * dense + 2.0 * TOP_K * 3 * HIDDEN * HIDDEN)
            + 2.0 * VOCAB * HIDDEN + keys * QH * DIM * 4.0}


# -- how close another correct implementation comes --------------------------------------------

def tolerance(case):
    """About four times what the outputs differ from `exact` (which rounds to bf16 where the
    model does): a last bit here and there.  Measured: moe 0.0004, attention 0.001, head 0.0017
    (exact logits are not rounded).  Over the loop's 24 layers such bits move later roundings
    and now and then an expert near a tie: 0.014 to 0.016, and two implementations that are both
    this far off differ by 1.4 times that."""
    return {"moe": {"rel": 0.002, "max": 0.03, "differ": 0.0},
            "decode": {"rel": 0.004, "max": 0.03, "differ": 0.0},
            "prefill": {"rel": 0.004, "max": 0.03, "differ": 0.0},
            "head": {"rel": 0.004, "max": 0.03, "differ": 0.0},
            "loop": {"rel": 0.03, "max": 0.4, "differ": 0.0}}[case["kind"]]


# -- the same in 64 bits, in plain torch ---------------------------------------------------------
# The tensors that the model's definition keeps in bf16 (a norm's output, q, k and v, the
# attention output, each block's output, router logits) are rounded where it rounds them;
# everything between them is float64.

_FP4 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _r(x):
    return x.to(torch.float32).to(BF).to(torch.float64)


def _norm64(x, weight):
    x = x.double()
    return _r(x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * weight.double())


def _expert64(blocks, scales):
    table = torch.tensor(_FP4 + [-v for v in _FP4], dtype=torch.float64, device=DEV)
    b = blocks.long()
    v = torch.stack([table[b & 15], table[b >> 4]], dim=-1)          # [N, K/32, 16, 2]
    v = v.flatten(-2) * torch.exp2(scales.double() - 127.0)[..., None]
    return v.flatten(-2)


def _moe64(x, p):
    """x [n, H] float64 -> x + MoE(norm(x))."""
    t = _norm64(x, p["norm.weight"])
    logits = _r(_r(t @ p["gate.weight"].double().t()) + p["gate.bias"].double())
    top, idx = torch.sort(logits, dim=-1, descending=True, stable=True)
    weight = _r(torch.softmax(top[:, :TOP_K], dim=-1))
    idx = idx[:, :TOP_K]
    out = torch.zeros_like(x)
    for e in idx.unique().tolist():
        rows, slot = torch.nonzero(idx == e, as_tuple=True)
        w1 = _expert64(p["mlp1_weight_blocks"][e], p["mlp1_weight_scales"][e])
        h = t[rows] @ w1.t() + p["mlp1_bias"][e].double()
        glu = h[:, 0::2].clamp(max=LIMIT)
        lin = h[:, 1::2].clamp(-LIMIT, LIMIT)
        act = glu * torch.sigmoid(ALPHA * glu) * (lin + 1.0)
        w2 = _expert64(p["mlp2_weight_blocks"][e], p["mlp2_weight_scales"][e])
        y = act @ w2.t() + p["mlp2_bias"][e].double()
        out.index_add_(0, rows, y * weight[rows, slot][:, None])
    return _r(x + _r(out))


def _rope64(x, positions):
    """YaRN RoPE (theta 150000, factor 32, betas 32 and 1, 4096 positions) of x [n, heads, 64]:
    tables in float32 as the checkpoint's model has them, cos and sin rounded to bf16."""
    theta, factor, half = 150000.0, 32.0, DIM // 2
    d = torch.arange(half, dtype=torch.float32, device=DEV)
    freq = theta ** (2.0 * d.double() / DIM)
    low, high = (DIM * math.log(4096 / (rot * 2 * math.pi)) / (2 * math.log(theta))
                 for rot in (32.0, 1.0))
    ramp = ((d - max(low, 0.0)) / (min(high, DIM - 1.0) - max(low, 0.0))).clamp(0, 1)
    inv = (ramp.double() / (factor * freq) + (1.0 - ramp.double()) / freq).float()
    angle = (positions.float()[:, None] * inv).double()
    scale = 0.1 * math.log(factor) + 1.0
    cos, sin = ((_r(f) * scale)[:, None, :] for f in (torch.cos(angle), torch.sin(angle)))
    a, b = x[..., :half], x[..., half:]
    return _r(torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1))


def _attend64(q, k, v, first, window, sinks):
    """q [n, 64, 64] at positions first.. over k, v [m, 8, 64]: softmax, then the sink's factor."""
    n, m = q.shape[0], k.shape[0]
    at = torch.arange(first, first + n, device=DEV)[:, None]
    key = torch.arange(m, device=DEV)[None, :]
    hidden = (key > at) | (key <= at - window) if window else key > at
    outs = []
    for h in range(QH):
        s = (q[:, h] @ k[:, h // (QH // KVH)].t()) / math.sqrt(DIM)
        s = s.masked_fill(hidden, -math.inf)
        lse = torch.logsumexp(s, dim=-1, keepdim=True)
        o = torch.exp(s - lse) @ v[:, h // (QH // KVH)]
        outs.append(_r(_r(o) * _r(torch.sigmoid(lse - sinks[h].double()))))
    return torch.stack(outs, dim=1)


def _attention64(x, p, data, pages, lengths, window):
    """x [n, H] float64 through an attention block over `data` [pages, 2, 8, 16, 64] float64,
    to which the new keys and values are added."""
    t = _norm64(x, p["norm.weight"])
    qkv = _r(_r(t @ p["qkv.weight"].double().t()) + p["qkv.bias"].double())
    outs, row = [], 0
    for mine, (cached, new) in zip(pages, lengths):
        part = qkv[row:row + new].view(new, QH + 2 * KVH, DIM)
        pos = torch.arange(cached, cached + new, device=DEV)
        q = _rope64(part[:, :QH], pos)
        k, v = _rope64(part[:, QH:QH + KVH], pos), part[:, QH + KVH:]
        table = torch.tensor(mine, device=DEV)
        data[table[pos // PAGE], 0, :, pos % PAGE] = k
        data[table[pos // PAGE], 1, :, pos % PAGE] = v
        kv = data[table].permute(1, 0, 3, 2, 4).reshape(2, -1, KVH, DIM)[:, :cached + new]
        outs.append(_attend64(q, kv[0], kv[1], cached, window, p["sinks"]))
        row += new
    o = torch.cat(outs).reshape(-1, QH * DIM)
    y = _r(_r(o @ p["out.weight"].double().t()) + p["out.bias"].double())
    return _r(x + y)


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "moe":
            g = _gen(seed, 1)
            p = _moe_params(g, case["experts"], case["zipf"])
            x = _normal(g, (1, case["tokens"], HIDDEN))
            return _moe64(x[0].double(), p)[None]
        if kind in ("decode", "prefill"):
            g = _gen(seed, 2)
            lengths = _lengths(case)
            p = _attn_params(g)
            x = _normal(g, (1, sum(n for _, n in lengths), HIDDEN))
            pages, used = _pages(lengths)
            data = _normal(g, (used, 2, KVH, PAGE, DIM)).double()
            out = _attention64(x[0].double(), p, data, pages, lengths,
                               WINDOW if case["window"] else 0)
            return out[None], data
        if kind == "head":
            w, norm, x = _head_inputs(seed, case["sequences"])
            t = _norm64(x, norm)
            logits = torch.cat([t @ part.double().t() for part in w.split(25000)], dim=1)
            return logits, None
        return _loop64(case, seed)


def _loop64(case, seed):
    _, token = _loop_token(seed)
    emb, norm, unembed = _loop_ends(seed)
    x = emb[token:token + 1].double()
    pool = -(-(case["context"] + 64) // PAGE) + 1
    lengths = [(case["context"], 1)]
    pages = [list(range(-(-(case["context"] + 1) // PAGE)))]
    for i in range(LAYERS):
        attn, moe = _loop_layer(seed, i)
        data = _normal(_gen(seed, 9, i), (pool, 2, KVH, PAGE, DIM)).double()
        x = _attention64(x, attn, data, pages, lengths, WINDOW if i % 2 == 0 else 0)
        x = _moe64(x, moe)
    t = _norm64(x, norm)
    return torch.cat([t @ part.double().t() for part in unembed.split(25000)],
                     dim=1).view(1, 1, VOCAB)
