"""The measured cases of the tree-verification framework.

Each case is one call (or one recorded step) that a decode loop, a server or a
script makes through the public entry points, at widths of the configured
models (tiny fp32 Llama, Llama-2-7B with NF4 linears, Qwen2.5-14B in fp16 and
with NF4 linears) with the layer count cut to a few, so that weights are made
quickly and 16-bit roundings do not travel through tens of layers. Kinds:

  step     VerifyStep: a drafted tree over a cached prefix (masks, pass,
           acceptance, compaction), replayed from its HIP graph
  batch    BatchVerifyStep: several sequences' trees, each over its own prefix
  prefill  TargetModel.forward_cached without a mask: a prompt, a continuation
           of a cached prefix, or one token
  draft    DeviceDrafter.draft_logits: the drafter over its whole context
  attend   ops.tree_attention alone, over a long prefix
  propose  propose_tree_device on draft logits, then accept_tree of that tree

``absmax`` is the type of the NF4 block scales: "float16" (this package's
quantiser) or "float32" (what a bitsandbytes checkpoint holds).
"""

import math
from dataclasses import replace

import torch

from parallel_eagle_amd import _lib, ops
from parallel_eagle_amd.batch import BatchKVCache, BatchVerifyStep
from parallel_eagle_amd.config import LLAMA2_7B_NF4, QWEN25_14B_FP16, QWEN25_14B_NF4, TINY_LLAMA
from parallel_eagle_amd.drafter import DeviceDrafter
from parallel_eagle_amd.model import DeviceModel
from parallel_eagle_amd.target import TargetModel
from parallel_eagle_amd.tree import propose_tree_device

DEV = "cuda"
SHAPES = {"tiny": TINY_LLAMA, "7b-nf4": LLAMA2_7B_NF4, "14b-fp16": QWEN25_14B_FP16, "14b-nf4": QWEN25_14B_NF4}
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
SIZE = {"float32": 4, "bfloat16": 2, "float16": 2}
FEATURES = {1: (1, 1, 1), 2: (1, 2, 2), 3: (1, 2, 3), 4: (1, 2, 4)}
NF4 = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
       -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
       0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0]


def listed():
    return [
        # the smallest call: a small fp32 model's whole step, bound by launches
        {"name": "step-tiny-fp32", "kind": "step", "model": "tiny", "layers": 2, "nodes": 8, "depth": 4,
         "prefix": 64, "absmax": "float16"},
        # the headline workload's step: a 26-node tree at 7B width over 2048 cached tokens
        {"name": "step-7b-T26-P2048", "kind": "step", "model": "7b-nf4", "layers": 4, "nodes": 26, "depth": 5,
         "prefix": 2048, "absmax": "float16"},
        # a wide tree over a long chat
        {"name": "step-7b-T64-P8192", "kind": "step", "model": "7b-nf4", "layers": 2, "nodes": 64, "depth": 6,
         "prefix": 8192, "absmax": "float16"},
        # an unquantised 16-bit target with grouped KV heads and a large vocabulary
        {"name": "step-14b-fp16-T26-P4096", "kind": "step", "model": "14b-fp16", "layers": 2, "nodes": 26,
         "depth": 5, "prefix": 4096, "absmax": "float16"},
        # a server's step: eight sequences with prefixes of different lengths
        {"name": "batch-14b-B8-T26", "kind": "batch", "model": "14b-nf4", "layers": 2, "batch": 8, "nodes": 26,
         "depth": 5, "prefix_min": 512, "prefix": 4096, "absmax": "float16"},
        # a prompt of 2000 tokens into an empty cache (the largest case)
        {"name": "prefill-7b-2000", "kind": "prefill", "model": "7b-nf4", "layers": 2, "rows": 2000, "prefix": 0,
         "absmax": "float16"},
        # an unquantised prompt of an odd length
        {"name": "prefill-14b-fp16-777", "kind": "prefill", "model": "14b-fp16", "layers": 1, "rows": 777,
         "prefix": 0, "absmax": "float16"},
        # the next user turn of a chat on an imported bitsandbytes checkpoint
        {"name": "turn-7b-150-P900", "kind": "prefill", "model": "7b-nf4", "layers": 4, "rows": 150, "prefix": 900,
         "absmax": "float32"},
        # greedy decoding: one token after 3000 cached ones
        {"name": "token-14b-P3000", "kind": "prefill", "model": "14b-nf4", "layers": 4, "rows": 1, "prefix": 3000,
         "absmax": "float32"},
        # the drafter over a context of 1500 tokens
        {"name": "draft-7b-1500", "kind": "draft", "model": "7b-nf4", "layers": 2, "rows": 1500, "depth": 5,
         "absmax": "float16"},
        # the attention of one layer over a cache near its limit
        {"name": "attend-14b-T48-P15000", "kind": "attend", "model": "14b-nf4", "nodes": 48, "depth": 6,
         "prefix": 15000, "absmax": "float16"},
        # proposing a tree from draft logits and walking it, at the large vocabulary
        {"name": "propose-14b-k5-w5", "kind": "propose", "model": "14b-nf4", "depth": 5, "width": 5,
         "absmax": "float16"},
    ]


def draw(rng):
    def log(lo, hi):
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))

    kind = rng.choice(["step", "step", "step", "batch", "prefill", "prefill", "prefill", "draft", "attend", "propose"])
    absmax = rng.choice(["float16", "float32"])
    c = {"kind": kind}
    if kind == "step":
        model = rng.choice(["tiny", "7b-nf4", "7b-nf4", "14b-fp16", "14b-nf4"])
        nodes = log(2, 64) if rng.random() < 0.8 else rng.randint(65, 160)
        c.update(model=model, layers=2, nodes=nodes, depth=min(nodes, rng.randint(2, 7)),
                 prefix=log(16, 1024 if model == "tiny" else 8192), absmax=absmax)
    elif kind == "batch":
        lo = log(32, 2048)
        c.update(model=rng.choice(["7b-nf4", "14b-nf4"]), layers=2, batch=rng.randint(2, 8), nodes=rng.randint(6, 30),
                 depth=rng.randint(3, 6), prefix_min=lo, prefix=lo + log(16, 2048), absmax=absmax)
    elif kind == "prefill":
        model = rng.choice(["7b-nf4", "14b-nf4", "14b-fp16"])
        rows = rng.choice([1, log(2, 64), log(65, 256), log(257, 1800 if model == "7b-nf4" else 900)])
        prefix = log(16, 8192) if rows < 16 else rng.choice([0, log(16, 8192)]) if rows <= 700 else 0
        c.update(model=model, layers=1 if rows > 256 else 2, rows=rows, prefix=prefix, absmax=absmax)
    elif kind == "draft":
        c.update(model=rng.choice(["7b-nf4", "14b-fp16"]), layers=1, rows=log(8, 1500), depth=rng.randint(2, 7),
                 absmax=absmax)
    elif kind == "attend":
        nodes = log(1, 200)
        c.update(model=rng.choice(["7b-nf4", "14b-fp16", "14b-nf4"]), nodes=nodes, depth=min(nodes, rng.randint(1, 8)),
                 prefix=log(32, 16000), absmax=absmax)
    else:
        c.update(model=rng.choice(["7b-nf4", "14b-fp16", "14b-nf4"]), depth=rng.randint(2, 8), width=rng.randint(1, 8),
                 absmax=absmax)
    return c


# ------------------------------------------------------------------ inputs
def _shape(c):
    s = SHAPES[c["model"]]
    n = c.get("layers", 1)
    return replace(s, num_layers=n, feature_layers=FEATURES[n])


def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed(seed * 100003 + stream)


def _randn(gen, size, dtype, std=1.0, mean=0.0):
    return (torch.randn(size, generator=gen, device=DEV, dtype=torch.float32) * std + mean).to(dtype)


def _quantise(w, absmax_dtype):
    """fp32 [N][K] -> ("nf4", packed [N][K/2], absmax [N][K/64]): nearest code of each block's normalised values."""
    n, k = w.shape
    b = w.view(n, k // 64, 64)
    amax = b.abs().amax(-1)
    book = torch.tensor(NF4, device=DEV)
    codes = torch.bucketize(b / amax[..., None], (book[1:] + book[:-1]) / 2).to(torch.uint8).view(n, k)
    return "nf4", (codes[:, 0::2] << 4 | codes[:, 1::2]).contiguous(), amax.to(absmax_dtype)


def _layer(s, gen, nf4, bias, absmax, dtype):
    w = {"attn_norm": _randn(gen, (s.hidden,), dtype, 0.1, 1.0), "mlp_norm": _randn(gen, (s.hidden,), dtype, 0.1, 1.0)}
    for name, n, k in s.linear_shapes():
        w[name] = (_quantise(_randn(gen, (n, k), torch.float32, s.init_std), DTYPES[absmax]) if nf4
                   else _randn(gen, (n, k), dtype, s.init_std))
    if bias:
        for name, n in (("q_bias", s.q_dim), ("k_bias", s.kv_dim), ("v_bias", s.kv_dim)):
            w[name] = _randn(gen, (n,), dtype, s.init_std)
    return w


def _weights(c, seed, layers=True):
    s, gen = _shape(c), _gen(seed, 1)
    dt = DTYPES[s.dtype]
    w = {"embed": _randn(gen, (s.vocab, s.hidden), dt, s.init_std),
         "lm_head": _randn(gen, (s.vocab, s.hidden), dt, s.init_std),
         "final_norm": _randn(gen, (s.hidden,), dt, 0.1, 1.0), "layers": []}
    for li in range(s.num_layers if layers else 1):
        w["layers"].append(_layer(s, _gen(seed, 10 + li), s.weight_format == "nf4", s.qkv_bias, c["absmax"], dt))
    return w


def _draft_weights(c, seed):
    s, gen = _shape(c), _gen(seed, 40)
    dt, h = DTYPES[s.dtype], s.hidden
    return {"feat_norm": _randn(gen, (h,), dt, 0.1, 1.0), "feat_proj": _randn(gen, (h, 3 * h), dt, s.init_std),
            "in_proj": _randn(gen, (h, 2 * h), dt, s.init_std), "mask_emb": _randn(gen, (h,), dt),
            "h_shared": _randn(gen, (h,), dt),
            "layers": [_layer(s, _gen(seed, 50 + li), False, False, c["absmax"], dt) for li in range(c["layers"])]}


def _draft_inputs(c, seed):
    s, gen = _shape(c), _gen(seed, 41)
    ids = torch.randint(0, s.vocab, (c["rows"],), generator=gen, device=DEV)
    return ids, _randn(gen, (c["rows"], 3 * s.hidden), DTYPES[s.dtype], 2.0)


def _prefix(c, s, seed, rows):
    """A cached prefix's K and V, [L][nkv][rows][hd] each."""
    gen, size = _gen(seed, 2), (s.num_layers, s.num_kv_heads, rows, s.head_dim)
    return _randn(gen, size, DTYPES[s.dtype]), _randn(gen, size, DTYPES[s.dtype])


def _tree(nodes, depth, vocab, seed):
    """(tokens, parents): `depth` levels, the early ones narrow; tokens distinct. Made on the host, as a drafter's beam
    ends on the host."""
    gen = torch.Generator().manual_seed(seed * 100003 + 3)
    per = [max(1, nodes // depth)] * depth
    for i in range(nodes - sum(per)):
        per[depth - 1 - i % depth] += 1
    parents, level = [], [-1]
    for n in per:
        pick = torch.randint(0, len(level), (n,), generator=gen).sort().values.tolist()
        level, parents = [len(parents) + i for i in range(n)], parents + [level[j] for j in pick]
    return torch.randperm(vocab, generator=gen)[:nodes].tolist(), parents


def _root(s, token, seed, batch=None):
    """A root logit row whose largest entry is `token`."""
    r = _randn(_gen(seed, 4), (s.vocab,) if batch is None else (batch, s.vocab), DTYPES[s.dtype])
    if batch is None:
        r[token] = 30.0
    else:
        r[torch.arange(batch, device=DEV), torch.tensor(token, device=DEV)] = 30.0
    return r


def _batch_prefixes(c, seed):
    gen = torch.Generator().manual_seed(seed * 100003 + 5)
    return torch.randint(c["prefix_min"], c["prefix"] + 1, (c["batch"],), generator=gen).tolist()


def _accepted(parents):
    """The root child that the root logit names: the second one where there are two."""
    kids = [t for t, p in enumerate(parents) if p < 0]
    return kids[min(1, len(kids) - 1)]


def _attend_inputs(c, seed):
    s, gen = _shape(c), _gen(seed, 6)
    dt = DTYPES[s.dtype]
    cap = c["prefix"] + c["nodes"] + 64
    q = _randn(gen, (c["nodes"], s.num_heads, s.head_dim), dt, 1.3)
    return q, _randn(gen, (s.num_kv_heads, cap, s.head_dim), dt), _randn(gen, (s.num_kv_heads, cap, s.head_dim), dt)


def prepare(case, seed):
    c, s = case, _shape(case)
    kind, dt = c["kind"], DTYPES[s.dtype]
    if kind == "attend":
        q, k, v = _attend_inputs(c, seed)
        _, parents = _tree(c["nodes"], c["depth"], s.vocab, seed)
        words = (c["nodes"] + 63) // 64
        status = torch.zeros(4, dtype=torch.int32, device=DEV)
        bits, _, _ = ops.tree_masks(torch.tensor(parents, dtype=torch.int32, device=DEV), c["prefix"], words, status)
        return {"kind": kind, "q": q, "k": k, "v": v, "bits": bits, "prefix": c["prefix"],
                "scale": s.head_dim ** -0.5}
    if kind == "propose":
        gen = _gen(seed, 7)
        n = c["depth"] * c["width"]
        return {"kind": kind, "draft": _randn(gen, (c["depth"], s.vocab), dt, 2.0), "widths": [c["width"]] * c["depth"],
                "root": _randn(gen, (s.vocab,), dt, 2.0), "nodes": _randn(gen, (n, s.vocab), dt, 2.0)}
    if kind == "draft":
        w = _weights(c, seed, layers=False)
        tm = TargetModel(DeviceModel.from_weights(replace(s, num_layers=1, feature_layers=(1, 1, 1)), w, DEV))
        del w
        drafter = DeviceDrafter(tm, _draft_weights(c, seed), max_depth=c["depth"], capacity=c["rows"] + 64)
        ids, feats = _draft_inputs(c, seed)
        return {"kind": kind, "drafter": drafter, "ids": ids, "feats": feats, "k": c["depth"]}
    tm = TargetModel(DeviceModel.from_weights(s, _weights(c, seed), DEV))
    if kind == "batch":
        prefixes = _batch_prefixes(c, seed)
        cache = BatchKVCache(tm, c["batch"], max(prefixes) + c["nodes"] + 32)
        trees = [_tree(c["nodes"], c["depth"], s.vocab, seed * 64 + b) for b in range(c["batch"])]
        for b, p in enumerate(prefixes):
            k, v = _prefix(c, s, seed * 64 + b, p)
            cache.k[b, :, :, :p], cache.v[b, :, :, :p] = k, v
            cache.seq(b).seq_len = p
        step = BatchVerifyStep(tm, cache, [t for t, _ in trees], [p for _, p in trees])
        step.root.copy_(_root(s, [t[_accepted(p)] for t, p in trees], seed, c["batch"]))
        step.capture()
        return {"kind": kind, "step": step, "cache": cache, "prefixes": prefixes, "nodes": c["nodes"]}
    rows = c["nodes"] if kind == "step" else c["rows"]
    cache = tm.make_cache(c["prefix"] + rows + 32)
    cache.k[:, :, : c["prefix"]], cache.v[:, :, : c["prefix"]] = _prefix(c, s, seed, c["prefix"])
    cache.seq_len = c["prefix"]
    if kind == "step":
        tokens, parents = _tree(rows, c["depth"], s.vocab, seed)
        step = tm.verify_step(cache, rows)
        step.load_tree(tokens, parents, _root(s, tokens[_accepted(parents)], seed))
        step.capture()
        return {"kind": kind, "step": step, "cache": cache, "prefix": c["prefix"], "rows": rows}
    ids = torch.randint(0, s.vocab, (1, rows), generator=_gen(seed, 8), device=DEV)
    pos = torch.arange(c["prefix"], c["prefix"] + rows, device=DEV)[None]
    return {"kind": kind, "tm": tm, "cache": cache, "ids": ids, "pos": pos, "prefix": c["prefix"], "rows": rows}


def run(state):
    st, kind = state, state["kind"]
    if kind == "attend":
        return ops.tree_attention(st["q"], st["k"], st["v"], st["prefix"], _lib.PE_MASK_TREE, st["bits"], st["scale"])
    if kind == "propose":
        tokens, parents, _ = propose_tree_device(st["draft"], st["widths"], max(st["widths"]))
        return {"tokens": tokens, "parents": parents,
                "accepted": ops.accept_tree(st["root"], st["nodes"][: tokens.numel()], tokens, parents)[:2]}
    if kind == "draft":
        return {"logits": st["drafter"].draft_logits(st["ids"], st["feats"], st["k"])}
    cache = st["cache"]
    if kind == "batch":
        step = st["step"]
        step.run()
        rows = {"k%d" % b: cache.k[b, :, :, p: p + st["nodes"]] for b, p in enumerate(st["prefixes"])}
        rows.update({"v%d" % b: cache.v[b, :, :, p: p + st["nodes"]] for b, p in enumerate(st["prefixes"])})
        return {"logits": step.logits, "fused": step.fused, "accepted": step.accept_out[:, :1], **rows}
    p = st["prefix"]
    if kind == "step":
        step = st["step"]
        step.run()
        logits, fused, more = step.logits, step.fused, {"accepted": step.accept_out[:1]}
    else:
        cache.crop(p)  # the same prefix again
        logits, fused, _ = st["tm"].forward_cached(st["ids"], cache, st["pos"])
        more = {}
    return {"logits": logits, "fused": fused, "k": cache.k[:, :, p: p + st["rows"]],
            "v": cache.v[:, :, p: p + st["rows"]], **more}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    c, s = case, _shape(case)
    es, kind = SIZE[s.dtype], c["kind"]
    kv_row = 2 * s.kv_dim * es  # one token's K and V of one layer
    if kind == "attend":
        t, keys = c["nodes"], c["prefix"] + c["nodes"]
        return {"bytes": keys * kv_row + 2 * t * s.q_dim * es, "flops": 4 * t * keys * s.q_dim}
    if kind == "propose":
        n = c["depth"] * c["width"]
        return {"bytes": (c["depth"] + 1 + n) * s.vocab * es, "flops": 4 * (c["depth"] + 1 + n) * s.vocab}
    params = sum(n * k for _, n, k in s.linear_shapes())
    per = es if s.weight_format == "dense" else 0.5 + SIZE[c["absmax"]] / 64
    if kind == "draft":
        m, h = c["rows"] + c["depth"] - 1, s.hidden
        keys = m * (m + 1) // 2
        return {"bytes": int((c["layers"] * params + 5 * h * h + s.vocab * h) * es + c["rows"] * 4 * h * es
                             + c["depth"] * s.vocab * es + c["layers"] * m * kv_row),
                "flops": 2 * (c["layers"] * params * m + 5 * h * h * c["rows"] + s.vocab * h * c["depth"])
                + 4 * c["layers"] * keys * s.q_dim}
    if kind == "batch":
        m, prefixes = c["batch"] * c["nodes"], [(c["prefix_min"] + c["prefix"]) // 2] * c["batch"]
        pairs = sum((p + c["nodes"]) * c["nodes"] for p in prefixes)
    elif kind == "step":
        m, prefixes = c["nodes"], [c["prefix"]]
        pairs = m * (c["prefix"] + m)
    else:
        m, prefixes = c["rows"], [c["prefix"]]
        pairs = m * c["prefix"] + m * (m + 1) // 2
    nbytes = s.num_layers * (params * per + (sum(prefixes) + m) * kv_row) + s.vocab * s.hidden * es
    nbytes += m * (s.vocab + 4 * s.hidden) * es
    flops = 2 * m * (s.num_layers * params + s.vocab * s.hidden) + 4 * s.num_layers * pairs * s.q_dim
    return {"bytes": int(nbytes), "flops": int(flops)}


def tolerance(case):
    if case["kind"] == "propose":
        return "exact"
    # about four times the largest error measured against exact(): fp32 2.6e-7; one fp16 or bf16 attention 2.1e-3; fp16
    # layers 1.9e-3; the drafter (bf16, two layers) 8e-3; bf16 layers over NF4 weights 0.021 in the logits of four layers
    if case["model"] == "tiny":
        return {"rel": 1e-6}
    if case["kind"] == "attend" or case["model"] == "14b-fp16":
        return {"rel": 0.008}
    return {"rel": 0.03 if case["kind"] == "draft" else 0.08}


# ------------------------------------------------------------------ the same in 64 bits
def _double(w):
    """A weight as float64: NF4 linears are bf16 weights (code value times the block's absmax, rounded), as
    bitsandbytes hands them to its matrix product."""
    if isinstance(w, tuple):
        _, packed, absmax = w
        codes = torch.stack([packed >> 4, packed & 15], -1).view(packed.shape[0], -1)
        v = torch.tensor(NF4, device=DEV)[codes.long()].view(absmax.shape[0], -1, 64) * absmax.float()[..., None]
        return v.to(torch.bfloat16).view(packed.shape[0], -1).double()
    return w.double()


def _matmul(x, w):
    """x @ w.T in float64, a block of w's rows at a time."""
    return torch.cat([x @ _double(w[i: i + 16384]).T for i in range(0, w.shape[0], 16384)], 1) if torch.is_tensor(w) \
        else x @ _double(w).T


def _norm(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, pos, s):
    """x [M][heads][hd], rotated with the tables a 16-bit model holds: cos and sin rounded to its type."""
    inv = 1.0 / (s.rope_theta ** (torch.arange(0, s.head_dim, 2, dtype=torch.float32) / s.head_dim))
    ang = pos.cpu().float()[:, None] * inv[None]
    ang = torch.cat([ang, ang], -1)
    cos, sin = (f.to(DTYPES[s.dtype]).to(DEV).double()[:, None] for f in (ang.cos(), ang.sin()))
    a, b = x.chunk(2, -1)
    return x * cos + torch.cat([-b, a], -1) * sin


def _attention(q, k, v, allow, s):
    """q [M][nh][hd] against k, v [nkv][S][hd]; allow bool [M][S]."""
    out = torch.empty_like(q)
    for h in range(s.num_heads):
        kv = h // (s.num_heads // s.num_kv_heads)
        a = (q[:, h].contiguous() @ k[kv].T.contiguous()) * s.head_dim ** -0.5
        out[:, h] = torch.softmax(a.masked_fill(~allow, -math.inf), -1) @ v[kv]
    return out.reshape(q.shape[0], -1)


def _decoder(h, pos, allow, past, layers, s):
    """The layers over rows h; past(li) -> the cached (K, V) of layer li. Returns each layer's output and new K, V."""
    m, states, new = h.shape[0], [], []
    for li, w in enumerate(layers):
        x = _norm(h, w["attn_norm"], s.rms_eps)
        q, k, v = (_matmul(x, w[n]) + (w[n + "_bias"].double() if n + "_bias" in w else 0.0) for n in "qkv")
        q, k = _rope(q.view(m, -1, s.head_dim), pos, s), _rope(k.view(m, -1, s.head_dim), pos, s)
        k, v = k.transpose(0, 1), v.view(m, -1, s.head_dim).transpose(0, 1)
        pk, pv = past(li)
        a = _attention(q, torch.cat([pk.double(), k], 1), torch.cat([pv.double(), v], 1), allow, s)
        h = h + _matmul(a, w["o"])
        x = _norm(h, w["mlp_norm"], s.rms_eps)
        h = h + _matmul(torch.nn.functional.silu(_matmul(x, w["gate"])) * _matmul(x, w["up"]), w["down"])
        states.append(h)
        new.append((k, v))
    return states, new


def _tree_allow(parents, prefix):
    """(allow bool [T][prefix + T], depth [T])"""
    t = len(parents)
    allow = torch.zeros((t, prefix + t), dtype=torch.bool)
    allow[:, :prefix] = True
    depth = [0] * t
    for i, p in enumerate(parents):
        if p >= 0:
            allow[i] = allow[p]
            depth[i] = depth[p] + 1
        allow[i, prefix + i] = True
    return allow.to(DEV), torch.tensor(depth, device=DEV)


def _forward(c, s, w, ids, pos, allow, k, v):
    states, new = _decoder(w["embed"][ids].double(), pos, allow, lambda li: (k[li], v[li]), w["layers"], s)
    final = _norm(states[-1], w["final_norm"], s.rms_eps)
    states[-1] = final
    fused = torch.cat([states[f - 1] for f in s.feature_layers], 1)
    return _matmul(final, w["lm_head"]), fused, torch.stack([a for a, _ in new]), torch.stack([b for _, b in new])


def _verify(c, s, w, tokens, parents, seed):
    """The pass over one tree, then the accepted node's K/V moved to the prefix's end."""
    k, v = _prefix(c, s, seed, c["prefix"])
    allow, depth = _tree_allow(parents, c["prefix"])
    logits, fused, nk, nv = _forward(c, s, w, torch.tensor(tokens, device=DEV), depth + c["prefix"], allow, k, v)
    path, want = [_accepted(parents)], None
    while want != -1:
        best = int(logits[path[-1]].argmax())
        want = next((t for t, p in enumerate(parents) if p == path[-1] and tokens[t] == best), -1)
        path += [want] if want >= 0 else []
    for x in (nk, nv):
        x[:, :, : len(path)] = x[:, :, path].clone()
    return logits, fused, nk, nv


def exact(case, seed):
    c, s = case, _shape(case)
    kind = c["kind"]
    if kind == "propose":
        return None
    if kind == "attend":
        q, k, v = _attend_inputs(c, seed)
        _, parents = _tree(c["nodes"], c["depth"], s.vocab, seed)
        allow, _ = _tree_allow(parents, c["prefix"])
        n = c["prefix"] + c["nodes"]
        return _attention(q.double(), k[:, :n].double(), v[:, :n].double(), allow, s)
    if kind == "draft":
        base, w = _weights(c, seed, layers=False), _draft_weights(c, seed)
        ids, feats = _draft_inputs(c, seed)
        p, m = c["rows"], c["rows"] + c["depth"] - 1
        f = _norm(feats.double().view(p, 3, -1), w["feat_norm"], s.rms_eps).reshape(p, -1)
        x = _matmul(torch.cat([base["embed"][ids].double(), _matmul(f, w["feat_proj"])], 1), w["in_proj"])
        slot = _matmul(torch.cat([w["mask_emb"], w["h_shared"]]).double()[None], w["in_proj"])
        x = torch.cat([x, slot.expand(m - p, -1)])
        allow = torch.ones((m, m), dtype=torch.bool, device=DEV).tril()
        none = torch.zeros((s.num_kv_heads, 0, s.head_dim), device=DEV)
        states, _ = _decoder(x, torch.arange(m, device=DEV), allow, lambda li: (none, none), w["layers"], s)
        return {"logits": _matmul(_norm(states[-1][p - 1:], base["final_norm"], s.rms_eps), base["lm_head"])}
    w = _weights(c, seed)
    if kind == "batch":
        out = {"accepted": None}
        parts = []
        for b, p in enumerate(_batch_prefixes(c, seed)):
            tokens, parents = _tree(c["nodes"], c["depth"], s.vocab, seed * 64 + b)
            parts.append(_verify(dict(c, prefix=p), s, w, tokens, parents, seed * 64 + b))
            out["k%d" % b], out["v%d" % b] = parts[-1][2:]
        return {"logits": torch.cat([x[0] for x in parts]), "fused": torch.cat([x[1] for x in parts]), **out}
    if kind == "step":
        tokens, parents = _tree(c["nodes"], c["depth"], s.vocab, seed)
        logits, fused, nk, nv = _verify(c, s, w, tokens, parents, seed)
        return {"logits": logits, "fused": fused, "k": nk, "v": nv, "accepted": None}
    m, p = c["rows"], c["prefix"]
    ids = torch.randint(0, s.vocab, (1, m), generator=_gen(seed, 8), device=DEV)[0]
    k, v = _prefix(c, s, seed, p)
    allow = torch.ones((m, p + m), dtype=torch.bool, device=DEV).tril(p)
    logits, fused, nk, nv = _forward(c, s, w, ids, torch.arange(p, p + m, device=DEV), allow, k, v)
    return {"logits": logits, "fused": fused, "k": nk, "v": nv}
