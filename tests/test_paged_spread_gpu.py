"""Paged decode calls of few (sequence, KV head) pairs: a chunk spread over
several workgroups gives the bits of the one-workgroup form."""

import pytest
import torch

from tests.conftest import SEED
from tests.test_attention_gpu import make_case

pytestmark = pytest.mark.gpu
PAGE = 64


def _run(fn, cache, table, lens, q, max_ctx, split, ws):
    from torch_spyre_amd import _lib

    B, Hq, D = q.shape
    out = torch.full_like(q, float("nan"))
    lse = torch.full((B, Hq), float("nan"), dtype=torch.float32, device=q.device)
    rc = fn(q.data_ptr(), cache.k.data_ptr(), cache.v.data_ptr(), table.data_ptr(), table.stride(0), lens.data_ptr(),
            out.data_ptr(), lse.data_ptr(), ws.data_ptr(), ws.numel(), B, Hq, cache.k.shape[1], D, PAGE,
            cache.k.shape[0], max_ctx, split, D ** -0.5, torch.cuda.current_stream().cuda_stream)
    _lib.check(fn.__name__, rc)
    torch.cuda.synchronize()
    return out.view(torch.int16), lse.view(torch.int32)


# Pages of a one-chunk context from which it is spread over workgroups of
# 1, 2 and 4 streaming wavefronts, the least that leave each of 256 units at
# most one workgroup.
FROM = {128: (4, 5, 7), 64: (7, 8, 14)}


def _spreads(pairs, D, max_ctx, split):
    chunks = -(-max_ctx // (8 * split))
    for S, pages in zip((1, 2, 4), FROM[D]):
        if pairs * chunks * (8 // S) <= 256:
            return chunks > 1 or -(-max_ctx // PAGE) >= pages
    return False


# Sequences around one to nine pages, empty ones, one and several chunks
# (split 64: 512 tokens each, split 512: 4096), 1 / 2 / 4 streaming
# wavefronts per workgroup (by the number of pairs), 1 to 16 q heads per KV
# head, a context past max_context_len, and grids too large to spread.
@pytest.mark.parametrize("lens,Hq,Hkv,D,split,max_ctx", [
    ([700], 32, 8, 128, 512, 700),
    ([0, 1, 64, 65, 128, 129], 8, 2, 128, 512, 1024),
    ([193, 256, 257, 512, 575, 577], 32, 4, 64, 512, 4096),
    ([4096, 17], 16, 16, 128, 512, 4096),
    ([1999, 0, 640, 2000, 64, 321, 1300], 16, 8, 128, 512, 2000),
    ([2048, 100, 300, 511, 512, 513, 1025, 2047], 32, 1, 64, 64, 2048),
    ([8000, 200, 4097], 64, 4, 128, 512, 8192),
    ([7000], 8, 8, 64, 64, 8192),
    ([300, 290, 64, 10] * 4, 32, 8, 128, 512, 300),
    ([900, 700, 10], 32, 8, 128, 512, 800),
    ([300] * 20, 32, 8, 128, 512, 300),
    # both sides of each line: pairs that fit the device, pages that pay
    ([192, 150], 32, 8, 128, 512, 192),
    ([256, 193, 130, 64], 32, 8, 128, 512, 256),
    ([256, 240] * 4, 32, 8, 128, 512, 256),
    ([320, 257, 256, 129, 64, 1, 0, 300], 32, 8, 128, 512, 320),
    ([384, 370] * 8, 32, 8, 128, 512, 384),
    ([448, 385, 320, 257] * 4, 32, 8, 128, 512, 448),
    ([448, 440] * 8 + [448], 32, 8, 128, 512, 448),
    ([384, 350], 16, 16, 64, 512, 384),
    ([448, 385], 16, 16, 64, 512, 448),
    ([448, 400, 257], 16, 16, 64, 512, 448),
    ([512, 449, 257, 200], 16, 16, 64, 512, 512),
    ([832, 800] * 4, 16, 16, 64, 512, 832),
    ([896, 833, 513, 257, 256, 129, 64, 0], 16, 16, 64, 512, 896),
    ([700, 520, 130, 70] * 2, 16, 16, 64, 64, 832),
], ids=str)
def test_spread_equals_one_workgroup(cuda, lens, Hq, Hkv, D, split, max_ctx):
    from torch_spyre_amd import _lib

    L = _lib.lib()
    if Hq // Hkv > 16:
        Hq = 16 * Hkv
    B = len(lens)
    cache, table, lens_t, q = make_case(cuda, B, Hq, Hkv, D, [max(x, max_ctx) for x in lens], SEED + 7 * B + D)
    table = table.to(cuda)
    l = torch.tensor(lens, dtype=torch.int32, device=cuda)
    base = L.spyre_paged_decode_attn_workspace_bytes(B, Hq, Hkv, D, max_ctx, split)
    need = L.spyre_paged_decode_attn_call_workspace_bytes(B, Hq, Hkv, D, max_ctx, split)
    assert base > 0
    spread = _spreads(B * Hkv, D, max_ctx, split)
    assert (need > base) == spread
    ws = torch.full((need,), 0xff, dtype=torch.uint8, device=cuda)
    want = _run(L.spyre_paged_decode_attn_f16, cache, table, l, q, max_ctx, split, ws)
    for size in (need, need, base):  # the second meets the first one's workspace; too small: not spread
        got = _run(L.spyre_paged_decode_attn_call_f16, cache, table, l, q, max_ctx, split, ws[:size])
        assert all(torch.equal(x, y) for x, y in zip(got, want))
    if spread:  # an unaligned workspace is not spread either
        buf = torch.empty(need + 4, dtype=torch.uint8, device=cuda)[4:]
        got = _run(L.spyre_paged_decode_attn_call_f16, cache, table, l, q, max_ctx, split, buf)
        assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_spread_under_capture_replays(cuda):
    """A captured call replayed over changing contexts (between one page and
    two chunks), with other work between the replays."""
    import torch_spyre_amd as tsa
    from torch_spyre_amd import _lib

    cache, table, lens_t, q = make_case(cuda, 2, 16, 4, 128, [1100, 1100], SEED + 61)
    table, l = table.to(cuda), lens_t.to(cuda)
    call = tsa.PagedDecode(q, cache.k, cache.v, table, l, split_tokens=64, max_context_len=1100,
                           lse=torch.empty((2, 16), dtype=torch.float32, device=cuda))
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    L = _lib.lib()
    ws = torch.empty(L.spyre_paged_decode_attn_workspace_bytes(2, 16, 4, 128, 1100, 64), dtype=torch.uint8, device=cuda)
    for a, b in [(1100, 64), (65, 1), (0, 513), (1100, 1100), (448, 320), (1, 1024)]:
        l.copy_(torch.tensor([a, b], dtype=torch.int32))
        call.out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        want = _run(L.spyre_paged_decode_attn_f16, cache, table, l, q, 1100, 64, ws)
        assert torch.equal(call.out.view(torch.int16), want[0]) and torch.equal(call.lse.view(torch.int32), want[1])
