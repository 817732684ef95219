"""Dense K / V into cache pages (spyre_dense_to_pages_f16), bit-exact against
the closed forms of the page layouts: K pages keep their sticks on D, V
pages are the transpose of each 64-token block, tokens past S are zero."""

import pytest
import torch

from tests.conftest import SEED

pytestmark = pytest.mark.gpu

PAGE = 64


def closed_form(k, v):
    """Pages [B P, Hkv, D/64, 64, 64] and [B P, Hkv, D, 64] by torch on the CPU."""
    B, Hkv, S, D = k.shape
    P = max(1, -(-S // PAGE))
    out = []
    for t in (k, v):
        pad = torch.zeros((B, Hkv, P * PAGE, D), dtype=t.dtype)
        pad[:, :, :S] = t
        out.append(pad.view(B, Hkv, P, PAGE, D).permute(0, 2, 1, 3, 4).reshape(B * P, Hkv, PAGE, D))
    kp, vp = out
    return (kp.view(B * P, Hkv, PAGE, D // 64, 64).transpose(2, 3).contiguous(), vp.transpose(2, 3).contiguous())


# One token, a page less one, a page, one over, several ragged; head counts
# and batches whose units are no multiple of a workgroup's four; D 64 to 192.
CASES = [(1, 1, 1, 64), (2, 3, 63, 128), (1, 8, 64, 128), (3, 2, 65, 64), (2, 5, 1000, 128), (1, 1, 130, 192),
         (2, 2, 0, 64)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form", ["bhsd", "bshd", "padded", "offset"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_dense_to_pages(cuda, case, form, dtype):
    """Contiguous, a transposed [B, S, H, D] view, rows wider than D (read as
    they lie) and a storage offset that is not 16-byte aligned (copied)."""
    import torch_spyre_amd as tsa

    B, Hkv, S, D = case
    g = torch.Generator().manual_seed(SEED + 400 + S)
    k, v = (torch.randn((B, Hkv, S, D), generator=g).to(dtype) for _ in range(2))

    def place(t):
        if form == "bshd":
            return t.transpose(1, 2).contiguous().to(cuda).transpose(1, 2)
        if form == "padded":
            wide = torch.full((B, Hkv, S, D + 8), float("nan"), dtype=dtype, device=cuda)
            wide[..., :D] = t.to(cuda)
            return wide[..., :D]
        if form == "offset":
            flat = torch.empty(t.numel() + 1, dtype=dtype, device=cuda)
            flat[1:] = t.flatten().to(cuda)
            return flat[1:].view(t.shape)
        return t.to(cuda)

    cache, table = tsa.dense_to_pages(place(k), place(v))
    kp, vp = closed_form(k, v)
    assert torch.equal(cache.k.view(torch.int16).cpu(), kp.view(torch.int16))
    assert torch.equal(cache.v.view(torch.int16).cpu(), vp.view(torch.int16))
    P = max(1, -(-S // PAGE))
    assert torch.equal(table.cpu(), torch.arange(B * P, dtype=torch.int32).view(B, P))
    assert (cache.num_pages, cache.Hkv, cache.D) == (B * P, Hkv, D)


@pytest.mark.parametrize("S", [0, 100])
def test_empty_batch(cuda, S):
    """No sequences: empty pages and an empty table."""
    import torch_spyre_amd as tsa

    k = torch.empty((0, 8, S, 128), dtype=torch.float16, device=cuda)
    cache, table = tsa.dense_to_pages(k, k)
    assert cache.k.shape == (0, 8, 2, PAGE, 64) and cache.v.shape == (0, 8, 128, PAGE)
    assert cache.num_pages == 0 and table.shape == (0, max(1, -(-S // PAGE)))
