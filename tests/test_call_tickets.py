"""Arrival-flag values: workgroups that merge their partials in one launch
tell each other by a value in a workspace that is not cleared first, so no
value may be one that ordinary data leaves there."""

import ctypes
import subprocess
import sys

import pytest
import torch

from tests.conftest import ROOT, SEED


def _tickets(n):
    from torch_spyre_amd import _lib

    fn = _lib.lib()._ZN9spyre_hip16next_call_ticketEv  # spyre_hip::next_call_ticket()
    fn.restype, fn.argtypes = ctypes.c_uint32, []
    return [fn() for _ in range(n)]


def test_values_are_new_and_scattered():
    """20000 values: none twice, none 0, and small ones (below 2^20, as
    lengths, positions and page numbers are) no more often than chance: 4.9
    expected, 40 is 16 standard deviations away."""
    t = _tickets(20000)
    assert len(set(t)) == len(t) and 0 not in t
    assert sum(x < 1 << 20 for x in t) <= 40


def test_processes_differ():
    """Another process' flags, left in memory this one is given, match none of
    this one's values: of 1000 against 1000, by chance one in 4300 runs."""
    code = "from tests.test_call_tickets import _tickets; print(*_tickets(1000))"
    run = [subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, check=True).stdout
           for _ in range(2)]
    a, b = (set(map(int, r.split())) for r in run)
    assert not a & b


@pytest.mark.gpu
@pytest.mark.parametrize("fill", [*range(1, 9), 64, 700, 0x3c003c00])
def test_spread_call_in_a_used_workspace(cuda, fill):
    """The spread paged call and the split short decode in workspaces full of
    one small whole number (or fp16 ones): the results of a cleared one."""
    import torch_spyre_amd as tsa
    from tests.test_attention_gpu import make_case
    from torch_spyre_amd import _lib

    L = _lib.lib()
    cache, table, lens, q = make_case(cuda, 1, 32, 8, 128, [700], SEED + 570)
    table, lens = table.to(cuda), lens.to(cuda)
    need = L.spyre_paged_decode_attn_call_workspace_bytes(1, 32, 8, 128, 700, 512)
    assert need > L.spyre_paged_decode_attn_workspace_bytes(1, 32, 8, 128, 700, 512)
    g = torch.Generator(device=cuda).manual_seed(SEED + 571)
    qd, k, v = (torch.randn((1, h, n, 128), generator=g, device=cuda).half() for h, n in ((32, 1), (8, 2048), (8, 2048)))
    room = L.spyre_sdpa_fwd_call_workspace_bytes(None, 0, None, 1, 32, 8, 1, 2048, 128)
    assert room > 0
    results = []
    for value in (0, fill):
        ws = torch.full((need // 4,), value, dtype=torch.int32, device=cuda)
        out = torch.full_like(q, float("nan"))
        _lib.check("spread", L.spyre_paged_decode_attn_call_f16(
            q.data_ptr(), cache.k.data_ptr(), cache.v.data_ptr(), table.data_ptr(), table.stride(0), lens.data_ptr(),
            out.data_ptr(), None, ws.data_ptr(), need, 1, 32, 8, 128, 64, cache.k.shape[0], 700, 512, 128 ** -0.5,
            torch.cuda.current_stream().cuda_stream))
        wd = torch.full((room // 4,), value, dtype=torch.int32, device=cuda)
        dense = tsa.scaled_dot_product_attention(qd, k, v, enable_gqa=True, workspace=wd)
        torch.cuda.synchronize()
        results.append((out.view(torch.int16), dense.view(torch.int16)))
    assert all(torch.equal(x, y) for x, y in zip(*results))
