"""The work a serving program gives this library, as cases that can be timed
and whose results can be compared.

Five kinds, each through the entry point a program calls:

  decode   one layer's decode tick: ``PagedKVBatch.decode_layer`` (q/k norm,
           rope, append and attention of one token per sequence)
  tick     one layer's tick with prompt chunks, and decode tokens beside
           them: ``norm_rope_write_layer`` then ``attend_layer``
  block    a whole transformer block on such a tick: ``TransformerBlock``
  model    a decode tick of a whole model from its captured graph, planning
           and token upload included: ``TickGraphRunner.run`` (what
           ``Engine(compile=True)`` runs per tick), logits returned
  sample   the next token of every request: ``sampler.sample_batch``
  pages    a prefix copied into the pool and back out: ``import_cache`` and
           ``snapshot``

The geometry is the default model's (32 query heads over 8 kv heads of 128,
hidden size 2560, MLP 9728, vocabulary 151,936); the attention kinds are also
drawn with other head groups and page sizes. Lengths belong to the case
(``lens`` seeds them), the values to the seed. Projections reach the
attention calls as a program has them: strided views of one fused q/k/v
buffer.
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hayate-exp_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

D = 128  # head size
HIDDEN, MID = 2560, 9728
VOCAB = 151_936
EPS = 1e-6
THETA = 1_000_000
POSITIONS = 40_960
DEV = "cuda"


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one user, a short chat: the smallest call, latency and launches
        _decode("decode 1x512", batch=1, lo=512, hi=512),
        # a served batch whose contexts are spread out
        _decode("decode 32 ragged", batch=32, lo=256, hi=4096),
        # long documents: the largest reads
        _decode("decode 8x32768", batch=8, lo=32_768, hi=32_768),
        # a follow-up question of odd length on a cached conversation
        _tick("question 77 on 1500", chunks=1, chunk_lo=77, chunk_hi=77, cached_lo=1500,
              cached_hi=1500),
        # four requests in the middle of their prompts, full chunks
        _tick("prefill 4x512", chunks=4, chunk_lo=512, chunk_hi=512, cached_lo=0, cached_hi=3584),
        # a busy tick: prompt chunks beside decoding requests
        _tick("mixed 8x512 + 56", chunks=8, chunk_lo=512, chunk_hi=512, cached_lo=1024,
              cached_hi=4096, decodes=56, ctx_lo=512, ctx_hi=8192),
        # a block of a decode tick at the default batch limit
        _tick("block decode 20", kind="block", decodes=20, ctx_lo=500, ctx_hi=1100),
        # a block of one default prompt chunk
        _tick("block prompt 512", kind="block", chunks=1, chunk_lo=512, chunk_hi=512),
        # a block of a busy tick: the largest products
        _tick("block 4x512 + 16", kind="block", chunks=4, chunk_lo=512, chunk_hi=512,
              cached_lo=0, cached_hi=2048, decodes=16, ctx_lo=300, ctx_hi=3000),
        # a few users decoding through a whole (shallow) model and its head
        _tick("model decode 4", kind="model", layers=8, decodes=4, ctx_lo=200, ctx_hi=900),
        # the sampling of the default batch: greedy, top-k and top-p rows
        {"name": "sample 20", "kind": "sample", "rows": 20, "vocab": VOCAB, "greedy": 0.25,
         "lens": 5},
        # a cached prompt copied in and out, all layers
        {"name": "pages 36x1999", "kind": "pages", "layers": 36, "tokens": 1999, "page": 128},
    ]


def _decode(name, batch, lo, hi, **kw):
    return _tick(name, kind="decode", decodes=batch, ctx_lo=lo, ctx_hi=hi, **kw)


def _tick(name, kind="tick", layers=1, chunks=0, chunk_lo=0, chunk_hi=0, cached_lo=0, cached_hi=0,
          decodes=0, ctx_lo=0, ctx_hi=0, page=128, q_heads=32, kv_heads=8, lens=11):
    """`chunks` prompt chunks of chunk_lo..chunk_hi tokens on cached_lo..
    cached_hi cached ones, and `decodes` decode tokens whose contexts (the
    token included) are ctx_lo..ctx_hi long."""
    case = {"kind": kind, "chunks": chunks, "chunk_lo": chunk_lo, "chunk_hi": chunk_hi,
            "cached_lo": cached_lo, "cached_hi": cached_hi, "decodes": decodes, "ctx_lo": ctx_lo,
            "ctx_hi": ctx_hi, "page": page, "q_heads": q_heads, "kv_heads": kv_heads,
            "lens": lens}
    if kind == "model":
        case["layers"] = layers
    return dict(case, name=name) if name else case


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "tick", "tick", "block", "block", "model", "sample",
                       "pages"])
    lens = rng.randrange(1 << 20)
    if kind == "sample":
        return {"kind": "sample", "rows": _log(rng, 1, 20),
                "vocab": rng.choice([VOCAB, VOCAB, VOCAB, _log(rng, 1000, VOCAB)]),
                "greedy": rng.choice([0.0, 0.0, 0.25, 0.5, 1.0]), "lens": lens}
    if kind == "pages":
        return {"kind": "pages", "layers": rng.choice([36, 36, _log(rng, 1, 36)]),
                "tokens": _log(rng, 1, 1999), "page": rng.choice([128, 128, 256])}
    geometry = {"lens": lens}
    if kind in ("decode", "tick"):
        geometry["q_heads"] = rng.choice([32, 32, 32, 16, 64])
        geometry["page"] = rng.choice([128, 128, 256])
    if kind in ("decode", "model") or (kind == "block" and rng.random() < 0.5):
        n = _log(rng, 1, {"decode": 64, "block": 48, "model": 20}[kind])
        most = min(32_768, {"decode": 200_000, "block": 60_000, "model": 20_000}[kind] // n)
        hi = _log(rng, 16, most)
        return _tick(None, kind=kind, layers=_log(rng, 1, 6), decodes=n,
                     ctx_lo=max(1, int(hi * rng.choice([1.0, 0.5, 0.06]))), ctx_hi=hi, **geometry)
    tokens = _log(rng, 2, 2048)
    chunks = rng.randint(1, min(8, -(-tokens // 2)))
    hi = min(512, max(2, tokens // chunks))
    cached = rng.choice([0, _log(rng, 1, 4096)])
    return _tick(None, kind=kind, chunks=chunks, chunk_lo=max(2, int(hi * rng.choice([1.0, 0.3]))),
                 chunk_hi=hi, cached_lo=int(cached * rng.choice([1.0, 0.25])), cached_hi=cached,
                 decodes=rng.choice([0, 0, _log(rng, 1, 56)]), ctx_lo=100, ctx_hi=4000, **geometry)


def _lengths(case):
    """(cached tokens, query tokens) of every sequence: evenly spaced chunk
    depths and drawn lengths, the same for every seed."""
    r = random.Random(case["lens"])
    cached, q = [], []
    n = case["chunks"]
    for i in range(n):
        lo, hi = case["cached_lo"], case["cached_hi"]
        cached.append(lo + (hi - lo) * i // max(1, n - 1) if n > 1 else hi)
        q.append(r.randint(case["chunk_lo"], case["chunk_hi"]))
    for _ in range(case["decodes"]):
        cached.append(r.randint(case["ctx_lo"], case["ctx_hi"]) - 1)
        q.append(1)
    return cached, q


# --------------------------------------------------------------- the inputs
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)
        self.host = random.Random(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        x = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
        flat, step = x.view(-1), 1 << 27
        for i in range(0, flat.numel(), step):
            n = min(step, flat.numel() - i)
            flat[i : i + n] = torch.randn(n, generator=self.g, device=DEV) * std + mean
        return x


def _pool(case, gen, layers):
    """Pools of N(0, 1) and the pages of every sequence, in drawn order."""
    cached, q = _lengths(case)
    page = case["page"]
    need = [-(-(c + n) // page) for c, n in zip(cached, q)]
    pages = sum(need) + 4
    order = list(range(pages))
    gen.host.shuffle(order)
    lists, at = [], 0
    for n in need:
        lists.append(order[at : at + n])
        at += n
    shape = (layers, 1, case["kv_heads"], pages * page, D)
    return cached, q, lists, gen.normal(*shape), gen.normal(*shape)


def _rope_tables():
    freq = 1.0 / THETA ** (torch.arange(0, D, 2, dtype=torch.float32, device=DEV) / D)
    angle = torch.arange(POSITIONS, dtype=torch.float32, device=DEV)[:, None] * freq[None]
    angle = torch.cat([angle, angle], dim=1)
    return torch.cos(angle), torch.sin(angle)


def _block_weights(case, gen):
    hq, hkv = case["q_heads"] * D, case["kv_heads"] * D
    shapes = {"self_attn.q_proj": (hq, HIDDEN), "self_attn.k_proj": (hkv, HIDDEN),
              "self_attn.v_proj": (hkv, HIDDEN), "self_attn.o_proj": (HIDDEN, hq),
              "mlp.gate_proj": (MID, HIDDEN), "mlp.up_proj": (MID, HIDDEN),
              "mlp.down_proj": (HIDDEN, MID)}
    w = {n: gen.normal(*s, std=s[1] ** -0.5) for n, s in shapes.items()}
    for n, size in (("self_attn.q_norm", D), ("self_attn.k_norm", D), ("input_layernorm", HIDDEN),
                    ("post_attention_layernorm", HIDDEN)):
        w[n] = gen.normal(size, std=0.1, mean=1.0)
    return w


def _inputs(case, seed):
    """Everything a pass reads, as plain tensors and lists."""
    gen = _Gen(seed)
    kind = case["kind"]
    if kind == "sample":
        r = random.Random(case["lens"])
        rows = case["rows"]
        temps = [0.0 if r.random() < case["greedy"] else r.choice([0.6, 0.7, 1.0, 1.3])
                 for _ in range(rows)]
        return {"logits": gen.normal(rows, case["vocab"], std=2.5), "temps": temps,
                "ks": [r.choice([None, 20, 50]) for _ in range(rows)],
                "ps": [r.choice([None, 0.8, 0.95]) for _ in range(rows)]}
    if kind == "pages":
        shape = (case["layers"], 8, case["tokens"], D)
        n = -(-case["tokens"] // case["page"]) + 4
        order = list(range(n))
        gen.host.shuffle(order)
        return {"k": gen.normal(*shape), "v": gen.normal(*shape), "pages": order[: n - 4],
                "capacity": n * case["page"]}
    layers = case.get("layers", 1)
    cached, q, lists, kp, vp = _pool(case, gen, layers)
    cos, sin = _rope_tables()
    got = {"cached": cached, "q": q, "lists": lists, "k_pool": kp, "v_pool": vp, "cos": cos,
           "sin": sin}
    n = sum(q)
    if kind in ("decode", "tick"):
        heads = case["q_heads"] + 2 * case["kv_heads"]
        got["qkv"] = gen.normal(n, heads, D)
        got["q_norm"] = gen.normal(D, std=0.1, mean=1.0)
        got["k_norm"] = gen.normal(D, std=0.1, mean=1.0)
    elif kind == "block":
        got["weights"] = _block_weights(case, gen)
        got["x"] = gen.normal(1, n, HIDDEN)
    else:
        got["layers"] = [_block_weights(case, gen) for _ in range(layers)]
        got["embed"] = gen.normal(VOCAB, HIDDEN)
        got["head"] = gen.normal(VOCAB, HIDDEN, std=HIDDEN**-0.5)
        got["norm"] = gen.normal(HIDDEN, std=0.1, mean=1.0)
        got["tokens"] = [gen.host.randrange(VOCAB) for _ in range(n)]
    return got


# ---------------------------------------------------------------- the passes
def _manager(case, inp, layers):
    """The pool with its requests in place. The manager's tensors become the
    inputs' own (a program's pool holds what earlier ticks wrote)."""
    from hayate_amd import PagedKVCacheManager

    m = PagedKVCacheManager(layers, case["kv_heads"], D, inp["k_pool"].shape[3], case["page"],
                            len(inp["q"]), torch.bfloat16, DEV, num_q_heads=case["q_heads"])
    m.k_cache.copy_(inp.pop("k_pool"))
    m.v_cache.copy_(inp.pop("v_pool"))
    handles = []
    for c, pages in zip(inp["cached"], inp["lists"]):
        h = m.allocate()
        m.claim_pages(h, pages)
        h.length = c
        handles.append(h)
    return m, handles


def _fill(module, weights):
    with torch.no_grad():
        for name, w in weights.items():
            module.get_submodule(name).weight.copy_(w)


def prepare(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind == "sample":
        return {"case": case, **inp, "generator": torch.Generator(device=DEV).manual_seed(seed)}
    if kind == "pages":
        from hayate_amd import Cache, PagedKVCacheManager

        m = PagedKVCacheManager(case["layers"], 8, D, inp["capacity"], case["page"], 1,
                                torch.bfloat16, DEV, num_q_heads=32)
        h = m.allocate()
        m.claim_pages(h, inp["pages"])
        return {"case": case, "m": m, "h": h, "cache": Cache.from_tensors(inp["k"], inp["v"])}
    m, handles = _manager(case, inp, case.get("layers", 1))
    state = {"case": case, "m": m, "handles": handles, "cos": inp["cos"], "sin": inp["sin"]}
    if kind in ("decode", "tick"):
        hq, hkv = case["q_heads"], case["kv_heads"]
        qkv = inp["qkv"]
        state.update(q=qkv[:, :hq], k=qkv[:, hq : hq + hkv], v=qkv[:, hq + hkv :],
                     q_norm=inp["q_norm"], k_norm=inp["k_norm"])
    elif kind == "block":
        from hayate_amd.model import Qwen3Config, TransformerBlock

        with torch.device(DEV):
            block = TransformerBlock(Qwen3Config(num_heads=case["q_heads"],
                                                 num_kv_groups=case["kv_heads"]))
        _fill(block, inp["weights"])
        state.update(block=block.eval(), x=inp["x"])
    else:
        from hayate_amd.model import Qwen3Config, Qwen3Model
        from hayate_amd.tick_graph import TickGraphRunner

        with torch.device(DEV):
            model = Qwen3Model(Qwen3Config(num_layers=case["layers"]))
        for i, w in enumerate(inp["layers"]):
            _fill(model.layers[i], w)
        _fill(model, {"embed_tokens": inp["embed"], "out_head": inp["head"], "norm": inp["norm"]})
        model.eval().initialize_rope(DEV)
        state.update(runner=TickGraphRunner(model, m, POSITIONS), tokens=inp["tokens"],
                     q_lens=inp["q"])
        return state
    state["batch"] = m.begin_tick(handles, inp["q"])
    return state


def run(state):
    s = state
    kind = s["case"]["kind"]
    with torch.inference_mode():
        if kind == "decode":
            q, out = s["batch"].decode_layer(0, s["q"], s["k"], s["v"], s["q_norm"], s["k_norm"],
                                             EPS, s["cos"], s["sin"])
            return {"q": q, "out": out, "k_pool": s["m"].k_cache, "v_pool": s["m"].v_cache}
        if kind == "tick":
            q = s["batch"].norm_rope_write_layer(0, s["q"], s["k"], s["v"], s["q_norm"],
                                                 s["k_norm"], EPS, s["cos"], s["sin"])
            out = s["batch"].attend_layer(q, 0)
            return {"q": q, "out": out, "k_pool": s["m"].k_cache, "v_pool": s["m"].v_cache}
        if kind == "block":
            y, _, _ = s["block"](s["x"], s["cos"], s["sin"], None, None, None, None, s["batch"], 0)
            return {"out": y, "k_pool": s["m"].k_cache, "v_pool": s["m"].v_cache}
        if kind == "model":
            logits = s["runner"].run(s["handles"], s["q_lens"], s["tokens"])
            return {"logits": logits, "k_pool": s["m"].k_cache, "v_pool": s["m"].v_cache}
        if kind == "sample":
            from hayate_amd.sampler import sample_batch

            return sample_batch(s["logits"], s["temps"], s["ks"], s["ps"], s["generator"])
        s["m"].import_cache(s["h"], s["cache"])
        got = s["m"].snapshot(s["h"])
        return {"k": got.k, "v": got.v}


# ------------------------------------------------------------ bytes and flops
def _attention_work(case):
    """(bytes, flops) of one layer's norm, rope, append and attention; every
    cached row is read once and every row in or out moves once."""
    cached, q = _lengths(case)
    hq, hkv = case["q_heads"], case["kv_heads"]
    n = sum(q)
    kv = sum(c + t for c, t in zip(cached, q))
    pairs = sum(t * c + t * (t + 1) // 2 for c, t in zip(cached, q))
    row = 2 * D
    return kv * 2 * hkv * row + n * (3 * hq + 4 * hkv) * row, 4 * hq * D * pairs


def _weights_work(case, tokens):
    hq, hkv = case["q_heads"] * D, case["kv_heads"] * D
    params = HIDDEN * (2 * hq + 2 * hkv + 3 * MID)
    return 2 * params, 2 * params * tokens


def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": 2 * case["rows"] * case["vocab"], "flops": 0}
    if kind == "pages":
        return {"bytes": 8 * case["layers"] * 8 * case["tokens"] * D * 2, "flops": 0}
    b, f = _attention_work(case)
    if kind in ("decode", "tick"):
        return {"bytes": b, "flops": f}
    n = sum(_lengths(case)[1])
    # inside a block the projections and the context need not leave the chip
    b -= n * (3 * case["q_heads"] + 2 * case["kv_heads"]) * 2 * D
    wb, wf = _weights_work(case, n)
    if kind == "block":
        return {"bytes": b + wb + 4 * n * HIDDEN, "flops": f + wf}
    layers = case["layers"]
    head = VOCAB * HIDDEN
    return {"bytes": layers * (b + wb) + 2 * head + n * (2 * HIDDEN + 2 * VOCAB),
            "flops": layers * (f + wf) + 2 * n * head}


def tolerance(case):
    """bf16 results of sums in 32 bits. The attention kinds round the
    probabilities and the output once (about 2.5e-3 from 64 bits); a block
    rounds its five products' results, a model those of all its layers."""
    kind = case["kind"]
    if kind == "pages":
        return "exact"
    if kind == "sample":
        return {"rel": 0.0, "differ": 0.01}
    return {"decode": {"rel": 0.01, "max": 0.2}, "tick": {"rel": 0.01, "max": 0.2},
            "block": {"rel": 0.01, "max": 0.2}, "model": {"rel": 0.025, "max": 0.5}}[kind]


# ------------------------------------------------------------ 64-bit results
def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rotate(x, cos, sin):
    half = torch.cat([-x[..., D // 2 :], x[..., : D // 2]], dim=-1)
    return x * cos[:, None] + half * sin[:, None]


def _attend(case, inp, layer, q, k, v, q_norm, k_norm, kp, vp):
    """Norm, rope, append into the 64-bit pools kp, vp and causal attention;
    q, k, v are (tokens, heads, D) in 64 bits. Returns rotated q, context."""
    page, group = case["page"], case["q_heads"] // case["kv_heads"]
    outs, rots, at = [], [], 0
    for c, n, pages in zip(inp["cached"], inp["q"], inp["lists"]):
        cos, sin = inp["cos"][c : c + n].double(), inp["sin"][c : c + n].double()
        rows = slice(at, at + n)
        at += n
        qr = _rotate(_rms(q[rows], q_norm), cos, sin)
        kr = _rotate(_rms(k[rows], k_norm), cos, sin)
        t = torch.arange(c + n, device=DEV)
        where = torch.tensor(pages, device=DEV)[t // page] * page + t % page
        kp[layer, 0][:, where[c:]] = kr.transpose(0, 1)
        vp[layer, 0][:, where[c:]] = v[rows].transpose(0, 1)
        keys, values = kp[layer, 0][:, where], vp[layer, 0][:, where]
        mask = t[None, :] > (c + torch.arange(n, device=DEV))[:, None]
        out = torch.empty_like(qr)
        for h in range(case["kv_heads"]):
            qh = qr[:, h * group : (h + 1) * group].transpose(0, 1)
            score = (qh @ keys[h].T) / math.sqrt(D)
            score.masked_fill_(mask, -math.inf)
            out[:, h * group : (h + 1) * group] = (torch.softmax(score, -1) @ values[h]).transpose(
                0, 1)
        outs.append(out)
        rots.append(qr)
    return torch.cat(rots), torch.cat(outs)


def _block64(case, inp, layer, w, x, kp, vp):
    hq, hkv = case["q_heads"], case["kv_heads"]
    n = x.shape[0]
    lin = lambda a, name: a @ w[name].double().T  # noqa: E731
    h = _rms(x, w["input_layernorm"])
    q = lin(h, "self_attn.q_proj").view(n, hq, D)
    k = lin(h, "self_attn.k_proj").view(n, hkv, D)
    v = lin(h, "self_attn.v_proj").view(n, hkv, D)
    _, ctx = _attend(case, inp, layer, q, k, v, w["self_attn.q_norm"], w["self_attn.k_norm"], kp,
                     vp)
    x = x + lin(ctx.reshape(n, hq * D), "self_attn.o_proj")
    h = _rms(x, w["post_attention_layernorm"])
    gate = lin(h, "mlp.gate_proj")
    return x + lin(gate * torch.sigmoid(gate) * lin(h, "mlp.up_proj"), "mlp.down_proj")


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None  # token ids
    inp = _inputs(case, seed)
    if kind == "pages":
        return {"k": inp["k"].double(), "v": inp["v"].double()}
    kp, vp = inp["k_pool"].double(), inp["v_pool"].double()
    pools = {"k_pool": kp, "v_pool": vp}
    with torch.inference_mode():
        if kind in ("decode", "tick"):
            hq, hkv = case["q_heads"], case["kv_heads"]
            qkv = inp["qkv"].double()
            q, out = _attend(case, inp, 0, qkv[:, :hq], qkv[:, hq : hq + hkv], qkv[:, hq + hkv :],
                             inp["q_norm"], inp["k_norm"], kp, vp)
            return {"q": q, "out": out, **pools}
        if kind == "block":
            return {"out": _block64(case, inp, 0, inp["weights"], inp["x"][0].double(), kp,
                                    vp)[None], **pools}
        x = inp["embed"][torch.tensor(inp["tokens"], device=DEV)].double()
        for i, w in enumerate(inp["layers"]):
            x = _block64(case, inp, i, w, x, kp, vp)
        logits = _rms(x, inp["norm"]) @ inp["head"].double().T
        return {"logits": logits[:, None], **pools}
