"""The drafter's attention over a context at once (row blocks through an LDS
ring) against the same context drafted in extensions of fewer than 256 rows
(the one-tile kernel), at the edges of the row blocks."""
from dataclasses import replace

import pytest
import torch

from parallel_eagle_amd.drafter import DeviceDrafter
from tests.test_gpu_many_row_pass import DEV, SHAPE, _target

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
