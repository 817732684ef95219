"""Dense SDPA calls and the workspace they are given: a masked call whose
mask is staged as it lies leaves a caller's workspace alone, so such calls
may be in flight at once on one workspace; calls that bring none allocate
what their kernels use."""

import pytest
import torch

from oracle import attention as OA
from tests.conftest import SEED
from tests.test_sdpa_gpu import assert_close, randn
from tests.test_sdpa_nan_gpu import as_mask

pytestmark = pytest.mark.gpu


# Short decode over split keys, decode in chunks, half and full steps over
# split keys.
CASES = [(1, 32, 8, 1, 2048, 128), (2, 16, 8, 1, 20048, 128), (1, 8, 2, 40, 2048, 128), (4, 32, 8, 128, 4096, 128),
         (2, 16, 16, 300, 2048, 64)]


@pytest.mark.parametrize("kind", ["bool", "f16"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_staged_mask_leaves_a_callers_workspace_alone(cuda, case, kind):
    import torch_spyre_amd as tsa
    from torch_spyre_amd import _lib

    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 580)
    k, v = randn((B, Hkv, Skv, D), SEED + 581), randn((B, Hkv, Skv, D), SEED + 582)
    keep = torch.ones((Sq, Skv), dtype=torch.bool).tril(Skv - Sq)
    keep[:, 100:140] = False
    mask = as_mask(kind, keep)
    md = mask.to(cuda)
    m = (md.view(torch.uint8) if kind == "bool" else md).expand(B, Hq, Sq, Skv)
    room = _lib.lib().spyre_sdpa_fwd_call_workspace_bytes(m.data_ptr(), 3 if kind == "bool" else 1,
                                                          _lib.i64_array(m.stride()), B, Hq, Hkv, Sq, Skv, D)
    assert room > 0
    ws = torch.full((room,), 0xa5, dtype=torch.uint8, device=cuda)
    args = (q.to(cuda), k.to(cuda), v.to(cuda), md)
    ref = OA.sdpa_cpu_fp32(q, k, v, attn_mask=mask)
    out = tsa.scaled_dot_product_attention(*args, enable_gqa=True, workspace=ws)
    prepared = tsa.SdpaCall(*args, enable_gqa=True, workspace=ws)()
    torch.cuda.synchronize()
    assert bool((ws == 0xa5).all())
    assert_close(out, ref)
    assert torch.equal(out.view(torch.int16), prepared.view(torch.int16))
    # with a workspace of its own the call splits its keys
    own = tsa.SdpaCall(*args, enable_gqa=True)
    eager = tsa.scaled_dot_product_attention(*args, enable_gqa=True)
    assert_close(own(), ref)
    assert torch.equal(own.out.view(torch.int16), eager.view(torch.int16))


@pytest.mark.parametrize("case", [(2, 16, 16, 300, 301, 64), (1, 32, 8, 1, 255, 128), (16, 32, 8, 1, 2048, 128),
                                  (2, 8, 8, 1, 600, 64)], ids=str)
def test_fp32_mask_allocates_no_copy_of_v(cuda, case):
    import torch_spyre_amd as tsa
    from torch_spyre_amd import _lib

    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 585)
    k, v = randn((B, Hkv, Skv, D), SEED + 586), randn((B, Hkv, Skv, D), SEED + 587)
    mask = torch.randn((1, Hq, Sq, Skv), generator=torch.Generator().manual_seed(SEED + 588))
    args = (q.to(cuda), k.to(cuda), v.to(cuda), mask.to(cuda))
    m = args[3].expand(B, Hq, Sq, Skv)
    part = _lib.lib().spyre_sdpa_fwd_own_workspace_bytes(m.data_ptr(), 2, _lib.i64_array(m.stride()), B, Hq, Hkv, Sq,
                                                         Skv, D)
    assert part < _lib.lib().spyre_sdpa_fwd_workspace_bytes(B, Hkv, Skv, D)
    tsa.scaled_dot_product_attention(*args, enable_gqa=True)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = tsa.scaled_dot_product_attention(*args, enable_gqa=True)
    peak = torch.cuda.max_memory_allocated() - before
    assert peak <= part + 2 * out.numel() + 4 * 512  # (the allocator rounds to 512 bytes)
    assert_close(out, OA.sdpa_cpu_fp32(q, k, v, attn_mask=mask))
