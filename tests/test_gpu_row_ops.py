"""RMSNorm rows and the A-tiled packing at the edges of their vector paths."""
import pytest
import torch

from oracle.drafter import drafter_rms_norm
from oracle.model import rms_norm
from parallel_eagle_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,pad", [(8, 0), (1024, 8), (2048, 0), (2056, 0), (4100, 0), (5120, 1), (8192, 0),
                                   (8200, 0)])  # past the registers' share: one element at a time
def test_rmsnorm_rows(dtype, h, pad):
    gen = torch.Generator().manual_seed(h)
    wide = (torch.randn(5, h + pad, generator=gen) * 3).to(dtype)
    x, w = wide[:, :h], (1 + 0.3 * torch.randn(h, generator=gen)).to(dtype)
    for mode, want in ((_lib.PE_NORM_HF, rms_norm(x, w, 1e-5)),
                       (_lib.PE_NORM_FP32_WEIGHT, drafter_rms_norm(x, w, 1e-5))):
        got = ops.rmsnorm(wide.to(DEV)[:, :h], w.to(DEV), 1e-5, mode=mode).cpu()
        # fp32 statistics summed in another order: h / 256 + 12 roundings, which may move each rounding to 16 bits by
        # one ulp (2^-7 of a bf16, 2^-10 of an fp16 value, 2^-24 below fp16's normal range): HF's form rounds the
        # normalised value and the product, the other form once
        ulp = {torch.float32: 2.0 ** -23, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
        eps = (h / 256 + 12) * 2.0 ** -24 + (2 if mode == _lib.PE_NORM_HF else 1) * ulp
        floor = 2.0 ** -23 if dtype == torch.float16 else 1e-30
        assert bool(((got.double() - want.double()).abs() <= eps * want.double().abs() + floor).all())


@pytest.mark.parametrize("m,k,ld,off", [(257, 128, 128, 0), (288, 384, 392, 0), (290, 256, 257, 0), (385, 512, 512, 1),
                                        (513, 1152, 1160, 4), (300, 256, 256, 8)])
def test_packing_of_many_rows(m, k, ld, off):
    """pe_dense_gemm over more than 256 rows packs X (the last two columns: the
    rows' stride and first element): an identity weight returns X bit for bit."""
    gen = torch.Generator(device=DEV).manual_seed(m)
    flat = torch.randn(m * ld + 8, generator=gen, device=DEV).to(torch.bfloat16)
    x = flat[off: off + m * ld].view(m, ld)[:, :k]
    w = torch.eye(k, device=DEV).to(torch.bfloat16)
    assert torch.equal(ops.linear(x, k, dense=ops.dense_repack(w)), x)
