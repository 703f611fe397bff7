"""The row searches (argmax, a row's top tokens) where their fast paths change:
whole vectors and tails, aligned and unaligned rows, one and several rounds of
vectors, ties, signed zeros and NaNs of either sign."""
import numpy as np
import pytest
import torch

from parallel_eagle_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _first_max(x: torch.Tensor) -> int:
    """The first NaN, or the first of the largest values."""
    v = x.float().numpy()
    nan = np.flatnonzero(np.isnan(v))
    return int(nan[0]) if nan.size else int(np.flatnonzero(v == v.max())[0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("v", [1, 7, 8, 8191, 20000, 152067])
def test_argmax_rows(dtype, v):
    gen = torch.Generator().manual_seed(v)
    rows = []
    for kind in range(7):
        x = torch.randint(-40, 41, (v,), generator=gen).to(dtype)  # many ties
        at = torch.randint(0, v, (2,), generator=gen)
        if kind == 1:  # the maximum is a zero of both signs
            x = -x.abs()
            x[at] = torch.tensor([0.0, -0.0]).to(dtype)
        elif kind == 2:
            x[:] = float("-inf")
        elif kind == 3:
            x[at] = float("inf")
        elif kind == 4:
            x[at] = float("nan")
        elif kind == 5:
            x[at[0]] = -float("nan")
        elif kind == 6:
            x = -x.abs() - 1
        rows.append(x)
    want = [_first_max(x) for x in rows]
    for pad in (0, 1):  # with one more column every second row starts unaligned
        wide = torch.zeros(len(rows), v + pad, dtype=dtype)
        wide[:, :v] = torch.stack(rows)
        assert ops.argmax_rows(wide.to(DEV)[:, :v]).cpu().tolist() == want, pad


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("v,c,pad", [(64, 64, 0), (1030, 20, 1), (9001, 64, 0), (152064, 64, 0), (152064, 5, 1)])
def test_top_tokens_of_rows_with_many_ties(dtype, v, c, pad):
    k = 3
    gen = torch.Generator().manual_seed(v + c)
    wide = torch.zeros(k, v + pad, dtype=dtype)
    wide[:, :v] = (torch.randint(-30, 31, (k, v), generator=gen).float() / 8).to(dtype)
    wide[1, :v] = wide[1, :v].sort(descending=True).values  # the top tokens are one thread's neighbours
    scratch = torch.zeros(k * _lib.PE_PROPOSE_SCRATCH_PER_DEPTH, dtype=torch.uint8, device=DEV)
    _, _, status = ops.propose_tree(wide.to(DEV)[:, :v], [c] * k, c, scratch=scratch)
    assert int(status.item()) == 0
    W = _lib.PE_PROPOSE_MAX_WIDTH
    lp = scratch[: k * W * 4].view(torch.float32).view(k, W)[:, :c].cpu()
    ids = scratch[k * W * 4: k * W * 8].view(torch.int32).view(k, W)[:, :c].cpu()
    for d in range(k):
        x = wide[d, :v].float()
        want = np.lexsort((np.arange(v), -x.numpy()))[:c]
        assert ids[d].tolist() == want.tolist()
        ref = torch.log_softmax(x.double(), -1)[torch.from_numpy(want)]
        # a sum of v fp32 terms in 1024 partial sums: v / 1024 + 26 roundings of 2^-24, and a few of the logarithm
        assert bool(((lp[d].double() - ref).abs() <= (v / 1024 + 32) * 2.0 ** -24 * (1 + ref.abs())).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("v", [1, 63, 1024, 1025, 16384])
def test_log_probabilities_do_not_depend_on_the_row_length_rule(dtype, v):
    """A short row's sum is taken by the search's own launch: the same bits as for the same row followed by -inf up
    to a length whose sums have a launch of their own (their exponentials are zeros)."""
    gen = torch.Generator().manual_seed(v)
    x = (torch.randn(2, v, generator=gen) * 3).to(dtype)
    wide = torch.full((2, 20000), float("-inf"), dtype=dtype)
    wide[:, :v] = x
    c = min(v, 8)
    out = []
    for rows in (x, wide):
        scratch = torch.zeros(2 * _lib.PE_PROPOSE_SCRATCH_PER_DEPTH, dtype=torch.uint8, device=DEV)
        tokens, parents, status = ops.propose_tree(rows.to(DEV), [c] * 2, c, scratch=scratch)
        assert int(status.item()) == 0
        W = _lib.PE_PROPOSE_MAX_WIDTH
        out.append((tokens.cpu(), parents.cpu(), scratch[: 2 * W * 4].view(torch.int32).view(2, W)[:, :c].cpu()))
    assert all(torch.equal(a, b) for a, b in zip(*out))
