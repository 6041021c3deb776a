"""The work that a program using this package has the GPU do, as measurable cases.

A speculative decoding session prefills the target and the drafter, then runs
rounds: draft (a chain or a tree), the target's verify forward, verification,
and the drafter's update pass over the accepted tokens.  Each kind below is one
of those pieces through the entry point that a program calls:

  verify_greedy  sampling.verify_chain_greedy_dev: target argmax + acceptance
  draft_chain    spec.ChainRound.enqueue_draft, replayed as the decoder does, as one graph per chain length
  draft_tree     tree_draft.TreeDrafter.draft: a greedy draft tree
  drafter_pass   Drafter.fuse + Drafter.__call__ over L tokens: a round's update (few rows) or a prompt (many)
  target_layer   target.TargetLayer: one decoder layer over a verify or prefill block of up to 64 rows
  target_model   target.TargetModel: the whole verify forward, with its logits and feature taps
  verify_sampled sampling.probs_from_logits + verify_tree_stochastic_dev: the T > 0 verification of a tree
  ops_layer      ops.*: a decoder layer out of the backend operations, as the C++ runtime composes it

Model shapes are the package's own: the Qwen3-1.7B and Qwen3-4B widths, random-init weights.
"""
from __future__ import annotations

import math

import torch

from woodcock_amd import _lib, ops
from woodcock_amd.cache import KVCache
from woodcock_amd.config import QWEN3_EOS, qwen3_1p7b_drafter, qwen3_4b_drafter
from woodcock_amd.drafter import Drafter
from woodcock_amd.runtime import ptr
from woodcock_amd.sampling import (SamplingParams, probs_from_logits, verify_chain_greedy_dev,
                                   verify_tree_stochastic_dev)
from woodcock_amd.spec import ChainRound
from woodcock_amd.synthetic import draft_vocab, random_drafter
from woodcock_amd.target import TargetConfig, TargetLayer, TargetModel, random_layer, random_target
from woodcock_amd.tree_draft import TreeDrafter

DEV = "cuda"
VOCAB = 151936
KINDS = ("verify_greedy", "draft_chain", "draft_tree", "drafter_pass", "target_layer", "target_model",
         "verify_sampled", "ops_layer")


def listed():
    return [
        # the end of a greedy chain round: 4 drafts against 5 rows of target logits
        {"name": "verify_greedy_5rows", "kind": "verify_greedy", "rows": 5, "vocab": VOCAB},
        # the drafting of a greedy chain round at the benchmarked drafter and context
        {"name": "draft_chain_1p7b_k4", "kind": "draft_chain", "model": "1.7b", "k": 4, "ctx": 512, "head": 16384},
        # tree drafting at the benchmarked tree shape (depth 6, width 4, 60 nodes verified)
        {"name": "draft_tree_1p7b_6x4", "kind": "draft_tree", "model": "1.7b", "depth": 6, "width": 4, "budget": 59,
         "ctx": 1000, "head": 16384},
        # the update that ends a round: 5 accepted tokens go through the drafter
        {"name": "update_1p7b_5rows", "kind": "drafter_pass", "model": "1.7b", "rows": 5, "ctx": 512,
         "kv": "bf16", "taps": "f32"},
        # a short chat prompt of an odd length through the drafter
        {"name": "prefill_1p7b_333rows", "kind": "drafter_pass", "model": "1.7b", "rows": 333, "ctx": 0,
         "kv": "bf16", "taps": "bf16"},
        # a document prompt through the larger drafter
        {"name": "prefill_4b_2048rows", "kind": "drafter_pass", "model": "4b", "rows": 2048, "ctx": 0,
         "kv": "bf16", "taps": "bf16"},
        # one layer of the target over a full prefill block in the middle of a prompt, its causal mask given
        {"name": "layer_1p7b_64rows_causal", "kind": "target_layer", "model": "1.7b", "rows": 64, "ctx": 1984,
         "tree": False},
        # one layer of the larger target over a 60-node draft tree late in a long session
        {"name": "layer_4b_60rows_tree", "kind": "target_layer", "model": "4b", "rows": 60, "ctx": 8000,
         "tree": True},
        # the whole verify forward of a short chain
        {"name": "model_1p7b_5rows", "kind": "target_model", "rows": 5, "ctx": 512},
        # the sampled verification of a tree: temperature, top-k and top-p at every node, then the tree rule
        {"name": "verify_sampled_60rows", "kind": "verify_sampled", "rows": 60, "vocab": VOCAB, "head": 16384,
         "temperature": 0.8, "top_k": 50, "top_p": 0.95},
        # a decoder layer of the C++ runtime decoding one token
        {"name": "ops_layer_1row", "kind": "ops_layer", "model": "1.7b", "rows": 1, "ctx": 600, "weights": "bf16"},
        # ... and prefilling a prompt
        {"name": "ops_layer_384rows", "kind": "ops_layer", "model": "1.7b", "rows": 384, "ctx": 0,
         "weights": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    model = rng.choice(("1.7b", "4b"))
    if kind == "verify_greedy":
        return {"kind": kind, "rows": rng.randint(2, 16), "vocab": _log(rng, 4096, VOCAB)}
    if kind == "draft_chain":
        return {"kind": kind, "model": model, "k": rng.randint(2, 8), "ctx": _log(rng, 16, 4096),
                "head": rng.choice((16384, 32768, 49152))}
    if kind == "draft_tree":
        return {"kind": kind, "model": model, "depth": rng.randint(2, 6), "width": rng.randint(2, 6),
                "budget": rng.randint(8, 62), "ctx": _log(rng, 16, 4096), "head": rng.choice((16384, 32768))}
    if kind == "drafter_pass":
        if rng.random() < 0.4:  # an update in a round
            return {"kind": kind, "model": model, "rows": rng.randint(1, 9), "ctx": _log(rng, 16, 4096),
                    "kv": "bf16", "taps": "f32"}
        return {"kind": kind, "model": model, "rows": _log(rng, 16, 1536), "ctx": rng.choice((0, _log(rng, 16, 512))),
                "kv": rng.choice(("bf16", "bf16", "f32")), "taps": rng.choice(("bf16", "f32"))}
    if kind == "target_layer":
        tree = rng.random() < 0.5
        return {"kind": kind, "model": model, "rows": _log(rng, 1, 64), "ctx": _log(rng, 16, 8192), "tree": tree}
    if kind == "target_model":
        rows = rng.randint(1, 8)  # a chain of up to 7 drafts, or plain decoding (then at any context)
        return {"kind": kind, "rows": rows, "ctx": _log(rng, 16, 4096 if rows <= 2 else 1000)}
    if kind == "verify_sampled":
        return {"kind": kind, "rows": rng.randint(2, 62), "vocab": rng.choice((VOCAB, _log(rng, 20000, VOCAB))),
                "head": 16384, "temperature": round(rng.uniform(0.5, 1.2), 2),
                "top_k": rng.choice((0, rng.randint(10, 200))), "top_p": rng.choice((1.0, round(rng.uniform(0.8, 0.99), 2)))}
    return {"kind": kind, "model": "1.7b", "rows": _log(rng, 1, 384), "ctx": rng.choice((0, _log(rng, 16, 1024))),
            "weights": rng.choice(("bf16", "f32"))}


# ------------------------------------------------------------------ shapes and inputs

def _drafter_cfg(case):
    return qwen3_4b_drafter() if case["model"] == "4b" else qwen3_1p7b_drafter()


def _target_cfg(case):
    if case.get("model") == "4b":
        return TargetConfig(hidden_size=2560, num_heads=32, num_kv_heads=8, head_dim=128, intermediate_size=9728,
                            num_layers=36)
    return TargetConfig()


def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + salt * 7919 + 12345) % (1 << 62))
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _fill(cache, n, g):
    for c in cache:
        c.keys[0, :, :n] = _randn(g, c.kv_heads, n, c.head_dim).to(c.keys.dtype)
        c.values[0, :, :n] = _randn(g, c.kv_heads, n, c.head_dim).to(c.values.dtype)
        c.offset = n


def _parents(n, seed, depth=6, width=4):
    """A draft tree's parents in node order: levels of at most `width` expanded nodes."""
    r = torch.Generator().manual_seed(seed)
    parents, level, front = [-1], [0], [0]
    while len(parents) < n:
        nxt = []
        for p in front:
            for _ in range(width):
                if len(parents) == n:
                    break
                parents.append(p)
                level.append(level[p] + 1)
                nxt.append(len(parents) - 1)
        pick = torch.randperm(len(nxt), generator=r)[:width].tolist() if nxt else [0]
        front = sorted(nxt[i] for i in pick) if nxt and level[nxt[0]] < depth else [0]
    return parents, level


def _tree_mask(parents, ctx):
    n = len(parents)
    m = torch.zeros(n, ctx + n, dtype=torch.uint8)
    m[:, :ctx] = 1
    for v in range(n):
        u = v
        while u >= 0:
            m[v, ctx + u] = 1
            u = parents[u]
    return m


def _drafter(case, seed, kv=torch.bfloat16, restricted=True):
    cfg = _drafter_cfg(case)
    if not restricted:  # passes that never reach the head
        return Drafter(cfg, random_drafter(cfg, seed=seed, device=DEV, head_rows=1024), DEV, kv)
    d = Drafter(cfg, random_drafter(cfg, seed=seed, device=DEV), DEV, kv)
    d.restrict_vocab(draft_vocab(cfg.vocab_size, case["head"], seed=seed % 1000, always=QWEN3_EOS))
    return d


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    s = {"kind": kind, "case": dict(case)}
    if kind == "verify_greedy":
        s["logits"] = 3 * _randn(g, case["rows"], case["vocab"])
        best = s["logits"].argmax(dim=1)[:-1]
        keep = torch.rand(best.shape, generator=g, device=DEV) < 0.8
        other = torch.randint(0, case["vocab"], best.shape, generator=g, device=DEV)
        s["drafts"] = torch.where(keep, best, other).to(torch.int32)
    elif kind == "draft_chain":
        d = _drafter(case, seed)
        k, ctx = case["k"], case["ctx"]
        rnd = ChainRound(d, k, (ctx + 64 + 255) // 256 * 256)
        _fill(rnd.cache, ctx, g)
        rnd.set_root(ctx, _randn(g, 1, d.cfg.hidden_size), 11)
        rnd.enqueue_draft(k)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            rnd.enqueue_draft(k)
        torch.cuda.current_stream().wait_stream(side)
        s.update(drafter=d, round=rnd, graph=graph)
    elif kind == "draft_tree":
        d = _drafter(case, seed)
        ctx = case["ctx"]
        cache = d.make_cache((ctx + 128 + 255) // 256 * 256)
        _fill(cache, ctx, g)
        s.update(drafter=d, cache=cache, tree=TreeDrafter(d, cache, case["depth"], case["width"], case["budget"]),
                 root=_randn(g, 1, d.cfg.hidden_size), token=torch.tensor([11], dtype=torch.int32, device=DEV),
                 offset=torch.tensor([ctx], dtype=torch.int32, device=DEV))
    elif kind == "drafter_pass":
        d = _drafter(case, seed, torch.float32 if case["kv"] == "f32" else torch.bfloat16, restricted=False)
        cfg, L, ctx = d.cfg, case["rows"], case["ctx"]
        cache = d.make_cache((ctx + L + 255) // 256 * 256)
        _fill(cache, ctx, g)
        dt = torch.bfloat16 if case["taps"] == "bf16" else torch.float32
        s.update(drafter=d, cache=cache, taps=[_randn(g, L, cfg.target_hidden_size).to(dt) for _ in range(3)],
                 tokens=torch.randint(0, cfg.vocab_size, (L,), generator=g, device=DEV, dtype=torch.int32))
    elif kind == "target_layer":
        cfg, rows, ctx = _target_cfg(case), case["rows"], case["ctx"]
        layer = TargetLayer(cfg, random_layer(cfg, seed=seed, device=DEV), DEV)
        cache = KVCache(cfg.num_kv_heads, cfg.head_dim, (ctx + 64 + 255) // 256 * 256, torch.bfloat16, DEV)
        _fill([cache], ctx, g)
        layer.rope(cache.capacity + 64)
        s.update(layer=layer, cache=cache, x0=_randn(g, rows, cfg.hidden_size),
                 x=torch.empty(rows, cfg.hidden_size, device=DEV),
                 offset=torch.tensor([ctx], dtype=torch.int32, device=DEV), positions=None, mask=None)
        wide = torch.zeros(rows, cache.capacity, dtype=torch.uint8, device=DEV)  # 16-byte rows, as the decoder's
        wide[:, :ctx + rows] = _causal(rows, ctx)
        s["mask"] = wide
        if case["tree"]:
            parents, level = _parents(rows, seed)
            wide[:, :ctx + rows] = _tree_mask(parents, ctx).to(DEV)
            s["positions"] = (torch.tensor(level, dtype=torch.int32) + ctx).to(DEV)
    elif kind == "target_model":
        cfg, rows, ctx = _target_cfg(case), case["rows"], case["ctx"]
        model = TargetModel(cfg, random_target(cfg, seed=seed, device=DEV), DEV, max_rows=16)
        cache = model.make_cache((ctx + 64 + 255) // 256 * 256)
        _fill(cache, ctx, g)
        model.rope(cache[0].capacity + 64)
        s.update(model=model, cache=cache, offset=torch.tensor([ctx], dtype=torch.int32, device=DEV),
                 logits=torch.empty(rows, cfg.vocab_size, device=DEV),
                 taps=[torch.empty(rows, cfg.hidden_size, device=DEV) for _ in model.feature_layers],
                 tokens=torch.randint(0, cfg.vocab_size, (rows,), generator=g, device=DEV, dtype=torch.int32))
    elif kind == "verify_sampled":
        n, V, H = case["rows"], case["vocab"], case["head"]
        rank = torch.rand(n, V, generator=g, device=DEV).argsort(dim=1).float()
        s["logits"] = -1.1 * torch.log(rank + 1.0)  # a Zipf law over a permutation of the vocabulary
        d2t = torch.rand(V, generator=g, device=DEV).argsort()[:H].sort().values
        s["d2t"] = d2t.to(torch.int32)
        z = s["logits"][:, d2t] + 0.5 * _randn(g, n, H)
        s["q"] = torch.softmax(z / case["temperature"], dim=1)
        parents, _ = _parents(n, seed)
        tokens = [11] * n
        for p in sorted(set(parents[1:])):
            kids = [v for v in range(n) if parents[v] == p]
            rows = torch.multinomial(s["q"][p], len(kids), generator=g)
            for v, t in zip(kids, d2t[rows].tolist()):
                tokens[v] = int(t)
        s["tokens"] = torch.tensor(tokens, dtype=torch.int32, device=DEV)
        s["parents"] = torch.tensor(parents, dtype=torch.int32, device=DEV)
        s["p"] = torch.empty_like(s["logits"])
        s["round"] = torch.tensor([3], dtype=torch.int32, device=DEV)
        s["rng"] = _lib.Uniforms(seed % (1 << 31), ptr(s["round"]), 0)
        s["sp"] = SamplingParams(case["temperature"], case["top_k"], case["top_p"])
    else:
        cfg, L, ctx = _target_cfg(case), case["rows"], case["ctx"]
        w = random_layer(cfg, seed=seed, device=DEV)
        if case["weights"] == "f32":
            w = {k: v.float() for k, v in w.items()}
        T = ctx + L
        s.update(cfg=cfg, w=w, x0=_randn(g, L, cfg.hidden_size),
                 K=_randn(g, T, cfg.num_kv_heads, cfg.head_dim), V=_randn(g, T, cfg.num_kv_heads, cfg.head_dim),
                 positions=torch.arange(ctx, T, dtype=torch.int32, device=DEV), mask=None)
        if L > 1:
            i = torch.arange(L, device=DEV)[:, None] + ctx
            s["mask"] = (torch.arange(T, device=DEV)[None] <= i).to(torch.uint8)
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "verify_greedy":
        return verify_chain_greedy_dev(s["logits"], s["drafts"])
    if kind == "draft_chain":
        s["graph"].replay()
        rnd = s["round"]
        n = case["ctx"]
        return {"drafts": rnd.drafts[:case["k"]], "root_out": rnd.upd_out[:1], "hidden": rnd.step_hid,
                "keys": rnd.cache[0].keys[0, :, n:n + case["k"] - 1],
                "values": rnd.cache[0].values[0, :, n:n + case["k"] - 1]}
    if kind == "draft_tree":
        t = s["tree"].draft(s["token"], None, None, s["offset"], root_hidden=s["root"])
        return {"tokens": t.tokens, "parents": t.parents, "depth": t.depth, "count": t.count}
    if kind == "drafter_pass":
        d, cache, n = s["drafter"], s["cache"], case["ctx"]
        for c in cache:
            c.offset = n
        g = d.fuse(s["taps"])
        hidden, out = d(s["tokens"], g, cache)
        L = case["rows"]
        return {"fused": g, "hidden": hidden, "out": out, "keys": cache[0].keys[0, :, n:n + L],
                "values": cache[0].values[0, :, n:n + L]}
    if kind == "target_layer":
        s["x"].copy_(s["x0"])
        x = s["layer"](s["x"], s["cache"], s["offset"], s["positions"], s["mask"])
        n, L = case["ctx"], case["rows"]
        return {"x": x, "keys": s["cache"].keys[0, :, n:n + L], "values": s["cache"].values[0, :, n:n + L]}
    if kind == "target_model":
        logits, taps = s["model"](s["tokens"], s["cache"], s["offset"], logits=s["logits"], taps=s["taps"])
        return {"logits": logits, "taps": taps}
    if kind == "verify_sampled":
        p = probs_from_logits(s["logits"], s["sp"], out=s["p"])
        v = verify_tree_stochastic_dev(p, s["q"], s["tokens"], s["parents"], s["rng"], s["d2t"])
        return {"p": p, "verdict": v}
    cfg, w, L, n = s["cfg"], s["w"], case["rows"], case["ctx"]
    H, Hk, D, eps = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.rms_norm_eps
    x = s["x0"].clone()
    h = ops.rmsnorm(x, w["input_layernorm.weight"], eps)
    q = ops.linear(h, w["self_attn.q_proj.weight"]).view(L, H, D)
    k = ops.linear(h, w["self_attn.k_proj.weight"]).view(L, Hk, D)
    v = ops.linear(h, w["self_attn.v_proj.weight"]).view(L, Hk, D)
    ops.rmsnorm(q, w["self_attn.q_norm.weight"], eps, out=q)
    ops.rmsnorm(k, w["self_attn.k_norm.weight"], eps, out=k)
    ops.rope(q, s["positions"], cfg.rope_theta)
    ops.rope(k, s["positions"], cfg.rope_theta)
    s["K"][n:].copy_(k)
    s["V"][n:].copy_(v)
    att = ops.attention(q, s["K"], s["V"], s["mask"], 1.0 / math.sqrt(D))
    ops.linear(att.view(L, H * D), w["self_attn.o_proj.weight"], y=x, accumulate=True)
    h = ops.rmsnorm(x, w["post_attention_layernorm.weight"], eps)
    gate = ops.linear(h, w["mlp.gate_proj.weight"])
    up = ops.linear(h, w["mlp.up_proj.weight"])
    ops.silu_mul(gate, up)
    ops.linear(gate, w["mlp.down_proj.weight"], y=x, accumulate=True)
    return {"x": x, "keys": s["K"][n:], "values": s["V"][n:]}


# ------------------------------------------------------------------ what a pass cannot do without

def _layer_work(cfg, rows, ctx, wbytes, kvbytes, streams=1):
    """(bytes, flops) of a decoder layer over `rows` tokens at context `ctx`."""
    d, H, Hk, D, F = cfg.hidden_size, cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.intermediate_size
    params = streams * (H + 2 * Hk) * D * d + H * D * d + 3 * F * d
    b = params * wbytes + 2 * Hk * D * (ctx + rows) * kvbytes + 8 * rows * d
    f = 2.0 * params * rows + 4.0 * H * D * rows * (ctx + (rows + 1) / 2)
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "verify_greedy":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4 * n, "flops": n}
    if kind == "verify_sampled":
        n = case["rows"] * case["vocab"]
        return {"bytes": 8 * n + 4 * case["rows"] * case["head"], "flops": 4 * n}
    if kind == "draft_chain":
        cfg = _drafter_cfg(case)
        b, f = _layer_work(cfg, 1, case["ctx"], 2, 2, streams=2)
        hb = case["head"] * cfg.hidden_size
        return {"bytes": (case["k"] - 1) * b + case["k"] * 2 * hb, "flops": (case["k"] - 1) * f + case["k"] * 2 * hb}
    if kind == "draft_tree":
        cfg = _drafter_cfg(case)
        w, depth = case["width"], case["depth"]
        b, f = _layer_work(cfg, w, case["ctx"], 2, 2, streams=2)
        hb = case["head"] * cfg.hidden_size
        return {"bytes": (depth - 1) * b + depth * 2 * hb,
                "flops": (depth - 1) * f + 2 * hb * (1 + (depth - 1) * w)}
    if kind == "drafter_pass":
        cfg, L = _drafter_cfg(case), case["rows"]
        b, f = _layer_work(cfg, L, case["ctx"], 2, 4 if case["kv"] == "f32" else 2, streams=2)
        fc = cfg.hidden_size * 3 * cfg.target_hidden_size
        tb = 4 if case["taps"] == "f32" else 2
        return {"bytes": b + 2 * fc + 3 * L * cfg.target_hidden_size * tb + 10 * L * cfg.hidden_size,
                "flops": f + 2.0 * fc * L}
    if kind == "target_layer":
        cfg = _target_cfg(case)
        b, f = _layer_work(cfg, case["rows"], case["ctx"], 2, 2)
        return {"bytes": b + case["rows"] * (case["ctx"] + case["rows"]), "flops": f}
    if kind == "target_model":
        cfg = _target_cfg(case)
        b, f = _layer_work(cfg, case["rows"], case["ctx"], 2, 2)
        head = cfg.vocab_size * cfg.hidden_size
        return {"bytes": cfg.num_layers * b + 2 * head + 4 * case["rows"] * cfg.vocab_size,
                "flops": cfg.num_layers * f + 2.0 * head * case["rows"]}
    cfg = _target_cfg(case)
    b, f = _layer_work(cfg, case["rows"], case["ctx"], 4 if case["weights"] == "f32" else 2, 4)
    return {"bytes": b + case["rows"] * (case["ctx"] + case["rows"]), "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind in ("verify_greedy", "draft_tree"):
        return "exact"
    if kind == "verify_sampled":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "ops_layer" or case.get("kv") == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "target_model":  # 28 layers; the activations go through the products as bf16 hi + lo
        return {"rel": 5e-5, "max": 1e-3}
    # bf16 cache rows: a value that lies at a rounding boundary lands one bf16 step off
    return {"rel": 1e-3, "max": 2e-2}


# ------------------------------------------------------------------ the same in 64 bits, in plain torch

F64 = torch.float64


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(dim=-1, keepdim=True) + eps) * w.to(F64)


def _mm(x, w):
    return x @ w.to(F64).T


def _rope(x, pos, base):
    """Rotate-half RoPE of [rows, heads, D]; the angle is the float32 product that defines the position's rotation."""
    half = x.shape[-1] // 2
    inv = torch.pow(torch.tensor(base, dtype=F64), -2.0 * torch.arange(half, dtype=F64) / x.shape[-1]).float().to(DEV)
    a = (pos.float()[:, None] * inv[None]).to(F64)[:, None]
    c, n = torch.cos(a), torch.sin(a)
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat([x1 * c - x2 * n, x2 * c + x1 * n], dim=-1)


def _attend(q, K, V, visible):
    """q [rows, H, D], K / V [Hk, T, D], visible [rows, T] -> [rows, H * D]."""
    L, H, D = q.shape
    Hk = K.shape[0]
    out = torch.empty(L, H, D, dtype=F64, device=DEV)
    for h in range(H):
        kh = h // (H // Hk)
        z = (q[:, h] @ K[kh].T) / math.sqrt(D)
        z = torch.softmax(z.masked_fill(~visible, -math.inf), dim=1)
        out[:, h] = z @ V[kh]
    return out.reshape(L, H * D)


def _layer(cfg, w, p, h, emb, K, V, ctx, pos, visible):
    """One decoder layer in 64 bits; K / V [Hk, ctx, D] as cached.  Returns (h', new keys, new values) with the new
    rows rounded to the cache's type, as the attention reads them."""
    L, H, Hk, D, eps = h.shape[0], cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.rms_norm_eps
    n = _rms(h, w[p + "input_layernorm.weight"], eps)
    parts = []
    for name in ("q", "k", "v"):
        y = _mm(n, w[p + "self_attn.%s_proj.weight" % name])
        if emb is not None:
            y = y + _mm(_rms(emb, w[p + "aux_norm.weight"], eps), w[p + "self_attn.aux_%s.weight" % name])
        parts.append(y)
    q = _rope(_rms(parts[0].view(L, H, D), w[p + "self_attn.q_norm.weight"], eps), pos, cfg.rope_theta)
    k = _rope(_rms(parts[1].view(L, Hk, D), w[p + "self_attn.k_norm.weight"], eps), pos, cfg.rope_theta)
    v = parts[2].view(L, Hk, D)
    k, v = (t.transpose(0, 1).to(K.dtype) for t in (k, v))
    att = _attend(q, torch.cat([K.to(F64), k.to(F64)], dim=1), torch.cat([V.to(F64), v.to(F64)], dim=1), visible)
    h = h + _mm(att, w[p + "self_attn.o_proj.weight"])
    n = _rms(h, w[p + "post_attention_layernorm.weight"], eps)
    act = torch.nn.functional.silu(_mm(n, w[p + "mlp.gate_proj.weight"])) * _mm(n, w[p + "mlp.up_proj.weight"])
    return h + _mm(act, w[p + "mlp.down_proj.weight"]), k.to(F64), v.to(F64)


def _causal(rows, ctx):
    i = torch.arange(rows, device=DEV)[:, None] + ctx
    return torch.arange(ctx + rows, device=DEV)[None] <= i


def exact(case, seed):
    kind = case["kind"]
    if kind in ("verify_greedy", "draft_tree"):
        return None  # whole numbers
    s = prepare(case, seed)
    if kind == "draft_chain":
        d, rnd, ctx = s["drafter"], s["round"], case["ctx"]
        cfg, w, ids = d.cfg, d.w, d.vocab_ids
        embed = w["embed_tokens.weight"]
        head = d._head
        hid = rnd.upd_hid[:1].to(F64)
        out = root = _rms(hid, w["norm.weight"], cfg.rms_norm_eps)
        K, V = (t[0, :, :ctx] for t in (rnd.cache[0].keys, rnd.cache[0].values))
        drafts, hids, ks, vs = [], [], [], []
        for i in range(case["k"]):
            drafts.append(int(ids[int(_mm(out, head).argmax())]))
            if i == case["k"] - 1:
                break
            pos = torch.tensor([ctx + i], device=DEV)
            h, k, v = _layer(cfg, w, "layers.0.", out, embed[drafts[-1]][None].to(F64), K, V, ctx + i, pos,
                             torch.ones(1, ctx + i + 1, dtype=torch.bool, device=DEV))
            K, V = torch.cat([K, k.to(K.dtype)], dim=1), torch.cat([V, v.to(V.dtype)], dim=1)
            hids.append(h)
            ks.append(k)
            vs.append(v)
            out = _rms(h, w["norm.weight"], cfg.rms_norm_eps)
        return {"drafts": None, "root_out": root, "hidden": torch.cat(hids), "keys": torch.cat(ks, dim=1),
                "values": torch.cat(vs, dim=1)}
    if kind == "drafter_pass":
        d, ctx, L = s["drafter"], case["ctx"], case["rows"]
        cfg, w = d.cfg, d.w
        taps = torch.cat([_rms(t.to(F64), w["feature_norms.%d.weight" % i], cfg.rms_norm_eps)
                          for i, t in enumerate(s["taps"])], dim=1)
        g = _mm(taps, w["fc.weight"])
        emb = w["embed_tokens.weight"][s["tokens"].long()].to(F64)
        K, V = (t[0, :, :ctx] for t in (s["cache"][0].keys, s["cache"][0].values))
        h, k, v = _layer(cfg, w, "layers.0.", g, emb, K, V, ctx, torch.arange(ctx, ctx + L, device=DEV),
                         _causal(L, ctx))
        return {"fused": g, "hidden": h, "out": _rms(h, w["norm.weight"], cfg.rms_norm_eps), "keys": k, "values": v}
    if kind == "target_layer":
        cfg, ctx, L = s["layer"].cfg, case["ctx"], case["rows"]
        K, V = (t[0, :, :ctx] for t in (s["cache"].keys, s["cache"].values))
        pos = torch.arange(ctx, ctx + L, device=DEV) if s["positions"] is None else s["positions"]
        vis = s["mask"][:, :ctx + L].bool()
        h, k, v = _layer(cfg, s["layer"].w, "", s["x0"].to(F64), None, K, V, ctx, pos, vis)
        return {"x": h, "keys": k, "values": v}
    if kind == "target_model":
        cfg, ctx, L = s["model"].cfg, case["ctx"], case["rows"]
        cache, feats = s["cache"], s["model"].feature_layers
        tokens = s["tokens"].long()
        del s
        w = random_target(cfg, seed=seed, device=DEV)
        h = w["embed_tokens.weight"][tokens].to(F64)
        pos, vis, taps = torch.arange(ctx, ctx + L, device=DEV), _causal(L, ctx), {}
        for i in range(cfg.num_layers):
            K, V = (t[0, :, :ctx] for t in (cache[i].keys, cache[i].values))
            h, _, _ = _layer(cfg, w, "layers.%d." % i, h, None, K, V, ctx, pos, vis)
            taps[i] = h
        return {"logits": _mm(_rms(h, w["norm.weight"], cfg.rms_norm_eps), w["embed_tokens.weight"]),
                "taps": [taps[i] for i in feats]}
    if kind == "verify_sampled":
        x = s["logits"].to(F64) / case["temperature"]
        if case["top_k"]:
            kth = x.topk(case["top_k"], dim=1).values[:, -1:]
            x = x.masked_fill(x < kth, -math.inf)
        p = torch.softmax(x, dim=1)
        if case["top_p"] < 1.0:
            sp, order = p.sort(dim=1, descending=True, stable=True)
            drop = sp.cumsum(dim=1) - sp >= case["top_p"]
            p = p.masked_fill(torch.zeros_like(drop).scatter(1, order, drop), 0.0)
            p = p / p.sum(dim=1, keepdim=True)
        return {"p": p, "verdict": None}
    cfg, L, ctx = s["cfg"], case["rows"], case["ctx"]
    K, V = (t[:ctx].transpose(0, 1) for t in (s["K"], s["V"]))
    vis = _causal(L, ctx)
    h, k, v = _layer(cfg, s["w"], "", s["x0"].to(F64), None, K.to(F64), V.to(F64), ctx, s["positions"], vis)
    return {"x": h, "keys": k.transpose(0, 1), "values": v.transpose(0, 1)}
