"""The fp32 kernels (linear, attention, the plain pass) at the edges of their
vector paths, against float64."""
from dataclasses import replace

import pytest
import torch

from parallel_eagle_amd import _lib, ops
from parallel_eagle_amd.config import TINY_LLAMA
from parallel_eagle_amd.target import TargetModel

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rnd(gen, *size):
    return torch.randn(size, generator=gen, device=DEV, dtype=torch.float32)


@pytest.mark.parametrize("m,n,k,pad", [(1, 5, 4, 0), (8, 64, 256, 0), (9, 67, 704, 4), (26, 33, 68, 0),
                                       (7, 10, 70, 0), (3, 8, 256, 1)])  # the last two: one-word loads
@pytest.mark.parametrize("epi", ["store", "residual", "swiglu"])
def test_fp32_linear(m, n, k, pad, epi):
    gen = torch.Generator(device=DEV).manual_seed(m * n + k)
    x = _rnd(gen, m, k + pad)[:, :k]
    if epi == "swiglu":
        n = (n + 31) // 32 * 64
    w = _rnd(gen, n, k)
    ref = x.double() @ w.double().T
    mag = x.double().abs() @ w.double().abs().T
    bound = (k + 8) * 2.0 ** -24 * mag
    if epi == "store":
        got = ops.linear(x, n, dense=w)
    elif epi == "residual":
        r = _rnd(gen, m, n)
        got = ops.linear(x, n, dense=w, epilogue=_lib.PE_EPI_RESIDUAL, resid=r)
        ref, bound = ref + r.double(), bound + 2.0 ** -23 * (mag + r.double().abs())
    else:
        got = ops.linear(x, n, dense=w, epilogue=_lib.PE_EPI_SWIGLU)
        t = ref.view(m, n // 64, 2, 32)
        e = bound.view(m, n // 64, 2, 32)
        g, u = t[:, :, 0].reshape(m, -1), t[:, :, 1].reshape(m, -1)
        eg, eu = e[:, :, 0].reshape(m, -1), e[:, :, 1].reshape(m, -1)
        s = torch.nn.functional.silu(g)
        ref = s * u
        # |silu'| <= 1.1; the exponential, quotient and products round a few times each
        bound = 1.1 * eg * (u.abs() + eu) + (s.abs() + eg) * eu + 16 * 2.0 ** -24 * ref.abs() + 1e-12
    assert bool(((got.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("hd,nh,nkv", [(64, 4, 2), (4, 2, 1), (68, 3, 3), (128, 4, 1), (200, 2, 1), (30, 2, 1)])
@pytest.mark.parametrize("t,prefix,causal", [(1, 0, True), (8, 64, False), (70, 5, False), (33, 1000, True),
                                             (2, 4200, False)])  # past the scores that stay in LDS
def test_fp32_attention(hd, nh, nkv, t, prefix, causal):
    gen = torch.Generator(device=DEV).manual_seed(hd + t + prefix)
    q, k, v = _rnd(gen, t, nh, hd), _rnd(gen, nkv, prefix + t + 3, hd), _rnd(gen, nkv, prefix + t + 3, hd)
    parents = [-1] + [(i - 1) // 2 for i in range(1, t)]
    allow = torch.ones(t, prefix + t, dtype=torch.bool).tril(prefix)
    bits = None
    if not causal:
        status = torch.zeros(4, dtype=torch.int32, device=DEV)
        bits, _, _ = ops.tree_masks(torch.tensor(parents, dtype=torch.int32, device=DEV), prefix, (t + 63) // 64, status)
        allow[:, prefix:] = False
        for i, p in enumerate(parents):
            if p >= 0:
                allow[i] |= allow[p]
            allow[i, prefix + i] = True
    mode = _lib.PE_MASK_CAUSAL if causal else _lib.PE_MASK_TREE
    got = ops.tree_attention(q, k, v, prefix, mode, bits, hd ** -0.5).view(t, nh, hd)
    s = prefix + t
    for h in range(nh):
        kk, vv = k[h // (nh // nkv), :s].double(), v[h // (nh // nkv), :s].double()
        sc = (q[:, h].double() @ kk.T) * hd ** -0.5
        ref = torch.softmax(sc.masked_fill(~allow.to(DEV), float("-inf")), -1) @ vv
        # scores of a few units with an error of hd + 8 roundings move a probability by as much, and the sum over the
        # keys rounds once per key of one lane's share
        err = ((hd + 8) * 12 + s / 4 + 16) * 2.0 ** -24
        assert float((got[:, h].double() - ref).abs().max()) <= err * (1 + float(vv.abs().max()))


def test_plain_pass_captures_every_hidden_state():
    """Features of inner layers and of the final norm, in any slot order, are the same rows."""
    ids = torch.arange(5, 14, device=DEV)
    pos = torch.arange(9, device=DEV)
    out = {}
    for layers in ((1, 2, 4), (4, 3, 1), (2, 4, 3)):
        shape = replace(TINY_LLAMA, num_layers=4, feature_layers=layers)
        tm = TargetModel.synthetic(shape, 3, DEV, norm_noise=0.1)
        assert tuple(tm.feature_layers) == layers
        logits, fused, _ = tm.forward_cached(ids, tm.make_cache(32), pos)
        parts = fused[0].view(9, 3, shape.hidden)
        for i, ly in enumerate(layers):
            assert torch.equal(parts[:, i], out.setdefault(ly, parts[:, i].clone()))
        assert torch.equal(logits[0], out.setdefault("logits", logits[0].clone()))
    assert not torch.equal(out[1], out[2])


def test_pass_of_a_model_without_layers():
    """Embeddings, the final norm and the lm_head alone."""
    tm = TargetModel.synthetic(TINY_LLAMA, seed=2, device=DEV, keep_logical=True, norm_noise=0.1)
    tm.model.desc().num_layers = 0
    ids = torch.arange(3, 14, device=DEV)
    logits = tm.forward_cached(ids, tm.make_cache(), torch.arange(11, device=DEV))[0][0]
    h = tm.model.embed[ids].double()
    x = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + TINY_LLAMA.rms_eps) * tm.model.final_norm.double()
    w = tm.model.lm_head_logical.double()
    k = TINY_LLAMA.hidden
    # the product's K roundings, and the norm's row sum (K / 256 + 12 of them) and two products
    bound = (k + k / 256 + 20) * 2.0 ** -24 * (x.abs() @ w.abs().T)
    assert bool(((logits.double() - x @ w.T).abs() <= bound).all())
