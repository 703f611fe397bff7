"""Passes of more than 64 rows in every weight format: a causal pass of M rows
at once (each linear one many-row launch) against the same rows in passes of at
most 64 (the fused kernels), and a batched pass against its sequences alone."""
from dataclasses import replace

import pytest
import torch

from parallel_eagle_amd import _lib, batch, ops
from parallel_eagle_amd.batch import BatchKVCache, forward_tree_batch
from parallel_eagle_amd.config import ModelShape
from parallel_eagle_amd.model import DeviceModel
from parallel_eagle_amd.target import TargetModel

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPE = ModelShape(name="small", num_layers=2, hidden=512, num_heads=4, num_kv_heads=2, head_dim=128,
                   intermediate=768, vocab=512, qkv_bias=True, weight_format="nf4", dtype="bfloat16",
                   feature_layers=(0, 1, 2), max_positions=1024)


def _target(fmt, shape=SHAPE):
    shape = shape if fmt.startswith("nf4") else replace(shape, weight_format="dense", dtype=fmt)
    gen = torch.Generator(device=DEV).manual_seed(5)
    rnd = lambda *size, std=0.04: torch.randn(size, generator=gen, device=DEV) * std
    w = {"embed": rnd(shape.vocab, shape.hidden, std=1.0), "lm_head": rnd(shape.vocab, shape.hidden),
         "final_norm": 1 + rnd(shape.hidden), "layers": []}
    for _ in range(shape.num_layers):
        lw = {"attn_norm": 1 + rnd(shape.hidden), "mlp_norm": 1 + rnd(shape.hidden)}
        for name, n, k in shape.linear_shapes():
            lw[name] = rnd(n, k)
            if fmt.startswith("nf4"):
                packed, absmax = ops.nf4_quantize(lw[name].contiguous())
                # fp32 scales that fp16 does not hold
                lw[name] = ("nf4", packed, absmax.float() * 1.0003 if fmt == "nf4-f32abs" else absmax)
        for name, n in (("q_bias", shape.q_dim), ("k_bias", shape.kv_dim), ("v_bias", shape.kv_dim)):
            lw[name] = rnd(n)
        w["layers"].append(lw)
    return TargetModel(DeviceModel.from_weights(shape, w, DEV), cache_capacity=640)


@pytest.fixture(scope="module", params=["nf4-f16abs", "nf4-f32abs", "bfloat16", "float16"])
def target(request):
    return _target(request.param)


def _close(a, b, dtype):
    # both round at the same points; sums in another order move single roundings (2^-8 of a bf16, 2^-11 of an
    # fp16 value), which the two layers carry on
    assert bool(torch.isfinite(a).all())
    rel = ((a.double() - b.double()).norm() / b.double().norm()).item()
    assert rel <= (2.0 ** -6 if dtype == torch.bfloat16 else 2.0 ** -9), rel


@pytest.mark.parametrize("rows,prefix", [(65, 0), (97, 33), (160, 0), (193, 200), (256, 7), (257, 0), (300, 40),
                                         (545, 0)])
def test_causal_pass_at_once_equals_short_passes(target, rows, prefix):
    gen = torch.Generator(device=DEV).manual_seed(rows)
    ids = torch.randint(0, SHAPE.vocab, (prefix + rows,), generator=gen, device=DEV)
    pos = torch.arange(prefix + rows, device=DEV)
    want, caches = [], [target.make_cache(), target.make_cache()]
    for c0 in range(0, prefix + rows, 64):
        want.append(target.forward_cached(ids[c0: c0 + 64], caches[0], pos[c0: c0 + 64])[:2])
    for c0 in range(0, prefix, 64):
        c1 = min(prefix, c0 + 64)
        target.forward_cached(ids[c0:c1], caches[1], pos[c0:c1])
    logits, fused, _ = target.forward_cached(ids[prefix:], caches[1], pos[prefix:])
    n = prefix + rows
    _close(logits[0], torch.cat([x[0][0] for x in want])[prefix:], target.dtype)
    _close(fused[0], torch.cat([x[1][0] for x in want])[prefix:], target.dtype)
    _close(caches[1].k[:, :, :n], caches[0].k[:, :, :n], target.dtype)
    _close(caches[1].v[:, :, :n], caches[0].v[:, :, :n], target.dtype)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_odd_row_blocks_of_the_fp32_partials(dtype):
    """A wide q/k/v projection takes row blocks of up to eight 32-row tiles, the
    last of 1, 3, 5 or 7."""
    tm = _target(dtype, replace(SHAPE, num_layers=1, num_heads=96, num_kv_heads=48, feature_layers=(0, 1, 1)))
    for rows in (145, 209, 321, 449):
        ids = torch.randint(0, SHAPE.vocab, (rows,), generator=torch.Generator(device=DEV).manual_seed(rows), device=DEV)
        pos = torch.arange(rows, device=DEV)
        caches = [tm.make_cache(), tm.make_cache()]
        want = [tm.forward_cached(ids[c: c + 64], caches[0], pos[c: c + 64])[0][0] for c in range(0, rows, 64)]
        got = tm.forward_cached(ids, caches[1], pos)[0][0]
        _close(got, torch.cat(want), tm.dtype)
        for a, b in ((caches[1].k, caches[0].k), (caches[1].v, caches[0].v)):
            _close(a[:, :, :rows], b[:, :, :rows], tm.dtype)


@pytest.mark.parametrize("trees", [(40, 26), (64, 64, 30, 7), (60,) * 5])
def test_batched_pass_equals_its_sequences_alone(target, trees):
    gen = torch.Generator(device=DEV).manual_seed(sum(trees))
    cache = BatchKVCache(target, len(trees), 256)
    toks, pars = [], []
    for b, t in enumerate(trees):
        p = 30 + 17 * b
        ids = torch.randint(0, SHAPE.vocab, (p,), generator=gen, device=DEV)
        target.forward_cached(ids, cache.seq(b), torch.arange(p, device=DEV))
        toks.append(torch.randint(0, SHAPE.vocab, (t,), generator=gen, device=DEV).tolist())
        pars.append([-1] + [(i - 1) // 2 for i in range(1, t)])
    logits, fused, info = forward_tree_batch(target, toks, pars, cache)
    for b, t in enumerate(trees):
        p = cache.seq(b).seq_len
        depth = [0] * t
        for i in range(1, t):
            depth[i] = depth[pars[b][i]] + 1
        pos = torch.tensor([p + d for d in depth], device=DEV)
        lg, fu, _ = target.forward_cached(torch.tensor(toks[b], device=DEV), cache.seq(b), pos, parents=pars[b])
        r0, r1 = info.row0[b], info.row0[b + 1]
        _close(logits[r0:r1], lg[0], target.dtype)
        _close(fused[r0:r1], fu[0], target.dtype)


@pytest.mark.parametrize("rows", [65, 150, 256, 257])
def test_causal_pass_in_the_workspace_of_a_chunk(target, rows, monkeypatch):
    pos = torch.arange(rows, device=DEV)
    ids = pos * 7 % SHAPE.vocab
    want = target.forward_cached(ids, target.make_cache(), pos)[:2]
    small = max(target.model.workspace_bytes(64, rows), target.model.workspace_bytes(rows % 64 or 64, rows))
    monkeypatch.setattr(target, "_ws", torch.zeros(small, dtype=torch.uint8, device=DEV))
    monkeypatch.setattr(type(target.model), "workspace_bytes", lambda self, m, kv_len: small)
    if rows > 256:
        with pytest.raises(_lib.PEError):
            target.forward_cached(ids, target.make_cache(), pos)
        return
    got = target.forward_cached(ids, target.make_cache(), pos)[:2]
    _close(got[0], want[0], target.dtype)
    _close(got[1], want[1], target.dtype)


@pytest.mark.parametrize("fmt", ["nf4-f16abs", "nf4-f32abs", "bfloat16"])
def test_causal_pass_in_the_workspace_of_a_longer_one(fmt, monkeypatch):
    """512 rows take more K splits than 513 at this width."""
    tm = _target(fmt, replace(SHAPE, num_heads=8, num_kv_heads=8, intermediate=1408))
    pos = torch.arange(512, device=DEV)
    ids = pos * 7 % SHAPE.vocab
    want = tm.forward_cached(ids, tm.make_cache(), pos)[:2]
    longer = min(tm.model.workspace_bytes(m, 640) for m in range(513, 640))
    monkeypatch.setattr(tm, "_ws", torch.zeros(longer, dtype=torch.uint8, device=DEV))
    monkeypatch.setattr(type(tm.model), "workspace_bytes", lambda self, m, kv_len: longer)
    got = tm.forward_cached(ids, tm.make_cache(), pos)[:2]
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("trees", [(40, 26), (60,) * 5])
def test_batched_pass_in_a_smaller_workspace(target, trees, monkeypatch):
    cache = BatchKVCache(target, len(trees), 256)
    toks = [[(11 * i + b) % SHAPE.vocab for i in range(t)] for b, t in enumerate(trees)]
    pars = [[-1] + [(i - 1) // 2 for i in range(1, t)] for t in trees]
    for b in range(len(trees)):
        p = torch.arange(20 + b, device=DEV)
        target.forward_cached(p, cache.seq(b), p)
    want = forward_tree_batch(target, toks, pars, cache)
    need = batch.batch_workspace_bytes
    monkeypatch.setattr(batch, "batch_workspace_bytes", lambda tm, t: need(tm, t) - 256)
    if target.model.desc().weight_format == _lib.PE_WFMT_NF4 and sum(trees) <= 256:
        with pytest.raises(_lib.PEError):
            forward_tree_batch(target, toks, pars, cache)
        return
    got = forward_tree_batch(target, toks, pars, cache)
    _close(got[0], want[0], target.dtype)
    _close(got[1], want[1], target.dtype)
