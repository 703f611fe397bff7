"""The eager softmax's scaling and exponential (csrc/pe_eager.h), compiled for
the host: every 16-bit score against the fp32 division, and the exponential
against the float64 one, with infinities and NaN."""
import ctypes as C
import subprocess

import numpy as np
import pytest
import torch

from parallel_eagle_amd import build

SOURCE = """
#include "pe_eager.h"
extern "C" void quotients(int f16, const float* x, float* q, int n) {
  for (int i = 0; i < n; ++i) q[i] = f16 ? eager_quotient<PE_DTYPE_F16>(x[i]) : eager_quotient<PE_DTYPE_BF16>(x[i]);
}
extern "C" void exponentials(const float* x, float* y, int n) {
  for (int i = 0; i < n; ++i) y[i] = exp_neg(x[i]);
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("eager")
    (d / "eager.hip").write_text(SOURCE)
    subprocess.run([build.hipcc(), *build.COMMON, f"-I{build.CSRC}", "--offload-host-only", "-shared",
                    str(d / "eager.hip"), "-o", str(d / "eager.so")], check=True, capture_output=True)
    return C.CDLL(str(d / "eager.so"))


def _ptr(t):
    return C.cast(t.data_ptr(), C.POINTER(C.c_float))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_score_rounds_as_its_division_does(host, dtype):
    x = torch.from_numpy(np.arange(65536, dtype=np.uint16).view(np.int16)).view(dtype)
    q = torch.empty(65536)
    xf = x.float()
    host.quotients(int(dtype == torch.float16), _ptr(xf), _ptr(q), 65536)
    got, want = q.to(dtype), (xf / float(np.sqrt(np.float32(128)))).to(dtype)
    nan = xf.isnan()
    assert bool(got[nan].isnan().all())
    assert torch.equal(got[~nan].view(torch.int16), want[~nan].view(torch.int16))  # bits: infinities, signs of zero


def test_exponential_of_negative_differences(host):
    x = torch.cat([-torch.rand(400000, generator=torch.Generator().manual_seed(0)) * 87, torch.zeros(2)])
    x[-1] = -87.0
    y = torch.empty_like(x)
    host.exponentials(_ptr(x), _ptr(y), x.numel())
    want = x.double().exp()
    # exp2 within an ulp, the first-order correction's own rounding, and its second-order term (below 2^-40)
    assert bool(((y.double() - want).abs() <= 1.5 * 2.0 ** -23 * want).all())


def test_exponential_of_scores_that_are_not_finite(host):
    inf = float("inf")
    x = torch.tensor([-inf, -3.4e38, -2.4e38, -2.3e38, -65504.0, -200.0, -128.0, float("nan"), inf - inf])
    y = torch.empty_like(x)
    host.exponentials(_ptr(x), _ptr(y), x.numel())
    assert bool((y[:7] < 2.0 ** -149).all()) and bool((y[:7] >= 0).all()) and bool(y[7:].isnan().all())
