"""The drafter's attention over a context at once (row blocks through an LDS
ring) against the same context drafted in extensions of fewer than 256 rows
(the one-tile kernel), at the edges of the row blocks, and both against the
oracle."""
from dataclasses import replace

import pytest
import torch

from oracle.drafter import OracleDrafter, draft_allow_mask, draft_positions, drafter_rms_norm
from oracle.model import DTYPES
from parallel_eagle_amd.drafter import DeviceDrafter
from parallel_eagle_amd.model import DeviceModel
from parallel_eagle_amd.target import TargetModel
from tests.test_gpu_many_row_pass import DEV, SHAPE, _target
from tests.test_oracle_pins import _drafter_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["bfloat16", "float16"])
def drafters(request):
    tm = _target(request.param)
    gen = torch.Generator(device=DEV).manual_seed(11)
    rnd = lambda *size, std=0.04: torch.randn(size, generator=gen, device=DEV) * std
    h = SHAPE.hidden
    w = {"feat_norm": 1 + rnd(h), "feat_proj": rnd(h, 3 * h), "in_proj": rnd(h, 2 * h), "mask_emb": rnd(h, std=1.0),
         "h_shared": rnd(h, std=1.0), "layers": []}
    for _ in range(2):
        w["layers"].append({"attn_norm": 1 + rnd(h), "mlp_norm": 1 + rnd(h),
                            **{n: rnd(a, b) for n, a, b in replace(SHAPE, qkv_bias=False).linear_shapes()}})
    return [DeviceDrafter(tm, w, max_depth=6, capacity=1000) for _ in range(2)]


@pytest.mark.parametrize("p", [257, 258, 320, 385, 513, 700, 950])
def test_context_at_once_equals_extensions(drafters, p):
    gen = torch.Generator(device=DEV).manual_seed(p)
    ids = torch.randint(0, SHAPE.vocab, (p,), generator=gen, device=DEV)
    feats = torch.randn(p, 3 * SHAPE.hidden, generator=gen, device=DEV).to(drafters[0].dtype) * 3
    at_once = drafters[0].draft_logits(ids, feats, 5)
    drafters[1].reset()
    for n in [*range(200, p, 200), p]:
        by_parts = drafters[1].draft_logits_extend(ids[:n], feats[:n], 5)
    assert bool(torch.isfinite(at_once).all())
    # the same roundings, sums in another order: single roundings move (2^-8 of a bf16, 2^-11 of an fp16 value, the
    # scores' among them) and two layers carry them on
    rel = ((at_once.double() - by_parts.double()).norm() / by_parts.double().norm()).item()
    assert rel <= (2.0 ** -5 if drafters[0].dtype == torch.bfloat16 else 2.0 ** -8), rel
    for a, b in ((drafters[0].cache.k, drafters[1].cache.k), (drafters[0].cache.v, drafters[1].cache.v)):
        a, b = a[:, :, :p].double(), b[:, :, :p].double()
        assert ((a - b).norm() / b.norm()).item() <= (2.0 ** -5 if drafters[0].dtype == torch.bfloat16 else 2.0 ** -8)


def _layer_two_values(w, shared, dt, ids, feats, k):
    """The oracle's V rows of the second layer (m rows): what the first layer's
    attention left for every row."""
    one = OracleDrafter(SHAPE, {**w, "layers": w["layers"][:1]}, shared, dt)
    p = ids.numel()
    x = torch.cat([one.real_input(ids, feats), one.mask_input(k - 1)])
    x = one.layers_forward(x, draft_positions(p, k), draft_allow_mask(p, k))
    second = w["layers"][1]
    return torch.nn.functional.linear(drafter_rms_norm(x, second["attn_norm"], SHAPE.rms_eps), second["v"])


@pytest.mark.parametrize("low_scores", [False, True])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("p", [100, 257, 300, 513])
def test_context_matches_the_oracle(dtype, p, low_scores):
    """Grouped query heads, with fewer than 256 context rows and with more.
    low_scores: every tenth token's keys have q.k past the type's lowest value
    in every head, so their scores round to -infinity and their weight is 0."""
    dt, h, hd, k = DTYPES[dtype], SHAPE.hidden, SHAPE.head_dim, 5
    w, shared = _drafter_weights(SHAPE, 2, 3, dt, seed=p)
    gen = torch.Generator().manual_seed(p)
    ids = torch.randint(0, SHAPE.vocab - 1, (p,), generator=gen)
    feats = (torch.randn(p, 3 * h, generator=gen) * 3).to(dt)
    if low_scores:
        # channel 0 of a row is 1, channel 1 is -1 for the marked token and 0 for all others; queries carry channel 0
        # and keys channel 1 in the dim that RoPE turns least (0.06 rad over 513 positions)
        ids[5::10] = SHAPE.vocab - 1
        shared["embed"][:, 0], shared["embed"][:, 1] = 1.0, 0.0
        shared["embed"][-1, 1] = -1.0
        w["in_proj"][:2] = 0.0
        w["in_proj"][0, 0] = w["in_proj"][1, 1] = 1.0
        w["mask_emb"][:2] = torch.tensor([1.0, 0.0])
        first = w["layers"][0]
        first["attn_norm"][:2] = 1.0
        big = 1000.0 if dt == torch.float16 else 1e20
        for name, channel in (("q", 0), ("k", 1)):
            heads = first[name].view(-1, hd, h)
            heads[:, [hd // 2 - 1, hd - 1]] = 0.0
            heads[:, hd // 2 - 1, channel] = big
        rows = drafter_rms_norm(OracleDrafter(SHAPE, w, shared, dt).real_input(ids, feats), first["attn_norm"],
                                SHAPE.rms_eps).double()
        assert (rows[:, 0].min() * big) * (rows[5::10, 1].max() * big) < -1.1 * torch.finfo(dt).max
    tm = TargetModel(DeviceModel.from_weights(
        replace(SHAPE, weight_format="dense", dtype=dtype, num_layers=1, feature_layers=(1, 1, 1)),
        {**shared, "layers": [dict(w["layers"][1], q_bias=torch.zeros(SHAPE.q_dim), k_bias=torch.zeros(SHAPE.kv_dim),
                                   v_bias=torch.zeros(SHAPE.kv_dim))]}, DEV))
    dr = DeviceDrafter(tm, w, max_depth=k, capacity=p + k)
    got = dr.draft_logits(ids.to(DEV), feats.to(DEV), k).cpu()
    got_v = dr.cache.v[1, :, : p + k - 1].transpose(0, 1).reshape(p + k - 1, -1).cpu()
    wide = lambda d: {n: [wide(x) for x in v] if isinstance(v, list) else v.float() for n, v in d.items()}
    logits = lambda *a: OracleDrafter(SHAPE, *a[:3]).draft_logits(*a[3:])
    for mine, oracle in ((got_v, _layer_two_values), (got, logits)):
        own = oracle(w, shared, dt, ids, feats, k)
        ref = oracle(wide(w), wide(shared), torch.float32, ids, feats.float(), k)
        err = lambda a: ((a.float() - ref).norm() / ref.norm()).item()
        print(f"relative error: device {err(mine):.4g}, the oracle's own roundings {err(own):.4g}")
        assert bool(torch.isfinite(own).all()) and bool(torch.isfinite(mine).all())
        # the same roundings, so the same distance from the fp32 evaluation; sums in another order move single ones
        assert err(mine) <= 1.1 * err(own) + 1e-6
