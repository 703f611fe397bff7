"""pe_forward_workspace_bytes grows with the rows of a causal pass (65 rows and
more), so a workspace of a long prompt serves every shorter one. A call's own
workspace: one dispatched operation while it is small, its counters zero."""
import ctypes as C

import pytest
from torch.utils._python_dispatch import TorchDispatchMode

from parallel_eagle_amd import _lib, ops
from test_abi import _desc_7b_nf4


@pytest.mark.parametrize("fmt", [_lib.PE_WFMT_NF4, _lib.PE_WFMT_NF4_F32ABS, _lib.PE_WFMT_DENSE])
def test_workspace_of_a_longer_prompt_serves_shorter_ones(fmt):
    d = _desc_7b_nf4()
    d.weight_format = fmt
    lib = _lib.load()
    # beyond the 256 nodes that a tree pass, which has its own layout, can have
    rows = [257, 300, 400, 511, 512, 513, 600, 768, 769, 1024, 1025, 2000, 2048, 2049]
    need = [lib.pe_forward_workspace_bytes(C.byref(d), m, 4096) for m in rows]
    assert all(b >= a > 0 for a, b in zip(need, need[1:]))
    # up to 256 rows a smaller workspace runs the chunked pass, so nothing that fits 257 rows is refused
    chunk = lib.pe_forward_workspace_bytes(C.byref(d), 64, 4096)
    assert chunk <= need[0]


@pytest.mark.parametrize("fmt", [_lib.PE_WFMT_NF4, _lib.PE_WFMT_NF4_F32ABS, _lib.PE_WFMT_DENSE])
@pytest.mark.parametrize("hidden,heads,kv_heads,intermediate", [
    (512, 4, 2, 768), (512, 8, 8, 1408), (1024, 16, 8, 3072), (1024, 8, 2, 2816), (2048, 16, 16, 5632),
    (4096, 32, 32, 11008)])
def test_workspace_grows_with_every_row_at_every_width(fmt, hidden, heads, kv_heads, intermediate):
    d = _desc_7b_nf4()
    d.weight_format, d.hidden, d.num_heads, d.num_kv_heads = fmt, hidden, heads, kv_heads
    d.intermediate = d.intermediate_padded = intermediate
    need = [_lib.load().pe_forward_workspace_bytes(C.byref(d), m, 4096) for m in range(257, 2600)]
    assert need[0] > 0 and all(b >= a for a, b in zip(need, need[1:]))


@pytest.mark.parametrize("nbytes", [0, 4096, ops.ZEROED_BYTES, ops.ZEROED_BYTES + 1])
def test_workspace_of_one_call(nbytes):
    calls = []

    class Count(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            calls.append(func)
            return func(*args, **(kwargs or {}))

    with Count():
        ws = ops._workspace(nbytes, "cpu")
    assert ws.numel() == max(nbytes, 256) and int(ws[: ops.COUNTER_BYTES].count_nonzero()) == 0
    if nbytes <= ops.ZEROED_BYTES:
        assert len(calls) == 1
