"""One prepared call launched on several streams, with launches in flight
together and in graphs: each has a workspace of its own."""

import threading

import pytest
import torch

from tests.conftest import SEED
from tests.test_attention_gpu import make_case

pytestmark = pytest.mark.gpu


def _paged(cuda, lens, split):
    import torch_spyre_amd as tsa

    cache, table, lens_t, q = make_case(cuda, len(lens), 32, 8, 128, lens, SEED + 590)
    return tsa.PagedDecode(q, cache.k, cache.v, table.to(cuda), lens_t.to(cuda), split_tokens=split,
                           max_context_len=max(lens))


def _dense(cuda, Sq, Skv, masked):
    import torch_spyre_amd as tsa

    g = torch.Generator(device=cuda).manual_seed(SEED + 591)
    q, k, v = (torch.randn((1, h, n, 128), generator=g, device=cuda).half() for h, n in ((32, Sq), (8, Skv), (8, Skv)))
    mask = torch.ones((Sq, Skv), dtype=torch.bool, device=cuda).tril(Skv - Sq) if masked else None
    return tsa.SdpaCall(q, k, v, attn_mask=mask, enable_gqa=True)


# Spread, and chunks merged in the kernel; short decode, half steps and a merge
# pass, each over split keys.
CALLS = {"spread": lambda c: _paged(c, [700], 512), "chunks": lambda c: _paged(c, [2000, 900], 64),
         "short": lambda c: _dense(c, 1, 2048, False), "short masked": lambda c: _dense(c, 1, 2048, True),
         "split masked": lambda c: _dense(c, 128, 4096, True)}


@pytest.mark.parametrize("name", CALLS)
def test_launches_on_streams_share_no_workspace(cuda, name):
    """Every workspace pointer handed to the library is a stream's or a
    capture's own: 3 streams, a capture of two launches, threads."""
    call = CALLS[name](cuda)
    call()
    torch.cuda.synchronize()
    want = call.out.clone()
    at = len(call._spaces._before)  # the workspace's place
    attr = "_call_fn" if hasattr(call, "_call_fn") else "_fn"
    fn, seen = getattr(call, attr), []
    setattr(call, attr, lambda *a: (seen.append((a[-1], a[at])), fn(*a))[1])
    streams = [torch.cuda.Stream(device=cuda) for _ in range(3)]

    def on(s):
        with torch.cuda.stream(s):
            for _ in range(5):
                call()

    workers = [threading.Thread(target=on, args=(s,)) for s in streams]
    for w in workers:
        w.start()
    for w in workers:
        w.join()
    torch.cuda.synchronize()
    assert torch.equal(call.out, want)
    assert len(seen) == 15 and len(set(seen)) == len({p for _, p in seen}) == 3
    eager = {p for _, p in seen}
    seen.clear()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=streams[0]):
        call()
        call()
    assert len({p for _, p in seen}) == 2 and not eager & {p for _, p in seen}
    for _ in range(3):
        call.out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        on(streams[0])  # an eager launch on the captured launches' stream
        torch.cuda.synchronize()
        assert torch.equal(call.out, want)


def test_workspaces_of_streams_are_bounded(cuda):
    from torch_spyre_amd._workspace import StreamWorkspaces

    first = torch.empty(64, dtype=torch.uint8, device=cuda)
    spaces = StreamWorkspaces((), first, (), 0)
    assert spaces.on(0)[1] is first
    for s in range(1, 200):  # (any numbers: no launch)
        assert spaces.on(s) is spaces.on(s) and len(spaces._by_stream) <= StreamWorkspaces.STREAMS
