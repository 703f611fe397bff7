"""The 16-bit linear over more than 256 rows (256-column tiles fed by an LDS
ring) against the float64 product, at the edges of its row blocks, rings and
stores."""
import pytest
import torch

from parallel_eagle_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k,pad", [
    (257, 256, 128, 0),     # one K unit: fewer stages than the ring holds; a last block of one row
    (320, 512, 384, 8),     # a last block of two tiles; rows wider than N, still 16-byte aligned
    (384, 256, 640, 1),     # four tiles; rows that are not 16-byte aligned
    (417, 768, 256, 0),     # five tiles and a ragged sixth
    (777, 256, 1152, 0),    # few column tiles: small row blocks
    (2047, 8192, 256, 0),   # full row blocks, one round of workgroups
    (480, 65536, 128, 0),   # many column tiles, so large row blocks: a last one of seven tiles,
    (410, 65536, 128, 1),   # of five, the last one ragged
    (281, 65536, 128, 0),   # and of three
    (300, 384, 256, 0),     # N not a multiple of 256: the 128-column kernel
])
def test_many_row_linear_matches_the_float64_product(dtype, m, n, k, pad):
    gen = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=gen, device=DEV).to(dtype)
    w = (torch.randn(n, k, generator=gen, device=DEV) * 0.02).to(dtype)
    out = torch.full((m, n + pad), 7.0, dtype=dtype, device=DEV)
    ops.linear(x, n, dense=ops.dense_repack(w), out=out[:, :n])
    ref = x.double() @ w.double().T
    # one rounding of the result after fp32 sums of k products: half a unit in the last place is at most 2^-8 of
    # the value with bf16's 8 significant bits, 2^-11 with fp16's 11 (2^-25 below its normal range)
    half_ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = half_ulp * ref.abs() * 1.01 + k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -25
    assert bool(((out[:, :n].double() - ref).abs() <= bound).all())
    assert pad == 0 or bool((out[:, n:] == 7.0).all())


def test_rows_past_two_gib():
    """Byte offsets within X from 2 GiB on (up to 4 GiB the same kernel): the last rows of 2.2 GiB."""
    m, n, k = 72001, 256, 16384
    gen = torch.Generator(device=DEV).manual_seed(1)
    x = torch.empty(m, k, dtype=torch.bfloat16, device=DEV).normal_(generator=gen)
    w = (torch.randn(n, k, generator=gen, device=DEV) * 0.02).to(torch.bfloat16)
    out = ops.linear(x, n, dense=ops.dense_repack(w))
    rows = torch.cat([torch.arange(300, device=DEV), torch.arange(65400, 65700, device=DEV),
                      torch.arange(m - 300, m, device=DEV)])
    xr = x[rows].double()
    ref = xr @ w.double().T
    bound = 2.0 ** -8 * ref.abs() * 1.01 + k * 2.0 ** -24 * (xr.abs() @ w.double().abs().T)
    assert bool(((out[rows].double() - ref).abs() <= bound).all())
