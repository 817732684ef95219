"""Masked SDPA calls on the grids of unmasked ones -- the q heads of a KV
head packed into one block's rows, keys split over blocks, blocks of at most
128 rows in half steps -- and the workgroup shapes of the SDPA forward kernel
(64, 128 or 256 rows), against torch's CPU SDPA in fp32 and the fp64
logsumexp.

Bars: out within 2e-3 + 1e-2 |ref| (tests/test_sdpa_gpu.py); LSE within 2e-3
of fp64 (scores of fp16 products of a prescaled fp16 q).
"""

import numpy as np
import pytest
import torch

from oracle import attention as OA
from tests.conftest import SEED
from tests.test_sdpa_gpu import LSE_ATOL, assert_close, randn

pytestmark = pytest.mark.gpu

DTYPE = {"f16": torch.float16, "f32": torch.float32}
# fp32 masks keep q unscaled: fp32 scores and row sums
LSE_BAR = {"f32": 1e-4}


def make_mask(kind, shape, B, Hq, Sq, Skv, seed):
    """tail: query i sees keys up to Skv - Sq + i; pad: each sequence's own
    number of keys; the other shapes: random, key 0 kept."""
    g = torch.Generator().manual_seed(seed)
    if shape == "tail":
        keep = torch.ones((Sq, Skv), dtype=torch.bool).tril(Skv - Sq)
    elif shape == "pad":
        lens = torch.randint(1, Skv + 1, (B, 1, 1, 1), generator=g)
        keep = torch.arange(Skv)[None, None, None, :] < lens
    else:
        dims = {"qk": (Sq, Skv), "bhqk": (B, Hq, Sq, Skv), "1h1k": (1, Hq, 1, Skv)}[shape]
        keep = torch.rand(dims, generator=g) > 0.3
        keep[..., 0] = True
        if kind != "bool":
            return (torch.randn(dims, generator=g) * 2).to(DTYPE[kind]).masked_fill(~keep, -float("inf"))
    if kind == "bool":
        return keep
    low = torch.finfo(DTYPE[kind]).min if shape == "pad" else -float("inf")
    return torch.zeros(keep.shape, dtype=DTYPE[kind]).masked_fill_(~keep, low)


# Rows per block: 4 (decode), 60, 128 (a whole half-step block), 132 (just
# past it: full steps), 512 (two packed blocks); keys: one step, a step and
# one key, splits of 256 and of 512 with a ragged last one, copied masks
# (odd rows) with a split's partials behind the copy.
CASES = [(3, 8, 2, 1, 64, 128), (2, 32, 8, 1, 1000, 128), (1, 8, 8, 1, 2048, 64), (2, 8, 2, 15, 65, 64),
         (1, 32, 8, 32, 1040, 128), (2, 16, 4, 33, 784, 128), (1, 32, 8, 128, 1536, 128), (1, 16, 16, 130, 640, 64),
         (1, 8, 8, 300, 1100, 128)]


@pytest.mark.parametrize("shape", ["tail", "pad", "bhqk", "1h1k"])
@pytest.mark.parametrize("kind", ["bool", "f16", "f32"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_masked_grids(cuda, case, kind, shape):
    import torch_spyre_amd as tsa

    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 300)
    k, v = randn((B, Hkv, Skv, D), SEED + 301), randn((B, Hkv, Skv, D), SEED + 302)
    mask = make_mask(kind, shape, B, Hq, Sq, Skv, SEED + 303 + Sq + Skv)
    out, lse = tsa.scaled_dot_product_attention(q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=mask.to(cuda),
                                                enable_gqa=True, return_lse=True)
    assert_close(out, OA.sdpa_cpu_fp32(q, k, v, attn_mask=mask))
    _, lse64 = OA.sdpa_decomposition_fp64(q, k, v, attn_mask=mask.numpy(), return_lse=True)
    assert np.allclose(lse.cpu().numpy(), lse64, atol=LSE_BAR.get(kind, LSE_ATOL), rtol=0)


@pytest.mark.parametrize("kind", ["bool", "f16", "f32"])
@pytest.mark.parametrize("Sq,Skv", [(1, 2048), (40, 1536)])
def test_masked_rows_and_splits(cuda, kind, Sq, Skv):
    """Rows with every key masked give zeros and LSE -inf beside live rows of
    the same block, and a split in which some rows see no key adds nothing to
    them: head 0's rows keep only the last 7 keys, head 1's none."""
    import torch_spyre_amd as tsa

    B, Hq, Hkv, D = 2, 8, 2, 128
    q = randn((B, Hq, Sq, D), SEED + 310)
    k, v = randn((B, Hkv, Skv, D), SEED + 311), randn((B, Hkv, Skv, D), SEED + 312)
    keep = torch.ones((1, Hq, Sq, Skv), dtype=torch.bool)
    keep[:, 0, :, :-7] = False
    keep[:, 1] = False
    mask = keep if kind == "bool" else torch.zeros(keep.shape, dtype=DTYPE[kind]).masked_fill_(~keep, -float("inf"))
    out, lse = tsa.scaled_dot_product_attention(q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=mask.to(cuda),
                                                enable_gqa=True, return_lse=True)
    assert not out[:, 1].float().abs().sum() and bool(torch.isneginf(lse[:, 1]).all())
    live = [h for h in range(Hq) if h != 1]
    ref = OA.sdpa_cpu_fp32(q, k, v, attn_mask=mask)
    assert_close(out[:, live], ref[:, live])
    _, lse64 = OA.sdpa_decomposition_fp64(q, k, v, attn_mask=mask.numpy(), return_lse=True)
    assert np.allclose(lse[:, live].cpu().numpy(), lse64[:, live], atol=LSE_BAR.get(kind, LSE_ATOL), rtol=0)


def test_masked_call_with_less_workspace(cuda):
    """A masked call whose workspace holds no split's partials (staged mask:
    16 bytes; copied mask: its copy alone) runs unsplit, within the bar."""
    import torch_spyre_amd as tsa
    from torch_spyre_amd import _lib

    B, Hq, Hkv, Sq, D = 1, 8, 2, 16, 128
    for Skv, room in ((1600, 16), (1603, Sq * 1616)):
        q = randn((B, Hq, Sq, D), SEED + 320).to(cuda)
        k, v = randn((B, Hkv, Skv, D), SEED + 321).to(cuda), randn((B, Hkv, Skv, D), SEED + 322).to(cuda)
        mask = make_mask("bool", "tail", B, Hq, Sq, Skv, 0).to(cuda)
        m = mask.view(torch.uint8).expand(B, Hq, Sq, Skv)
        args = (m.data_ptr(), 3, _lib.i64_array(m.stride()), B, Hq, Hkv, Sq, Skv, D)
        assert _lib.lib().spyre_sdpa_fwd_call_workspace_bytes(*args) > room
        assert _lib.lib().spyre_sdpa_fwd_min_workspace_bytes(*args) <= room
        out = tsa.scaled_dot_product_attention(q, k, v, attn_mask=mask, enable_gqa=True,
                                               workspace=torch.empty(room, dtype=torch.uint8, device=cuda))
        assert_close(out, OA.sdpa_cpu_fp32(q.cpu(), k.cpu(), v.cpu(), attn_mask=mask.cpu()))


# Grids on both sides of the workgroup shapes' lines, for a 256-unit device
# (the numbers of 64-, 128- and 256-row blocks decide): one step of keys; 64
# and 65 rows; 256 and 260 64-row blocks (2 x 32 heads x 256 / 257 queries);
# the same for causal at twice that; whole and partial rounds of 256-row
# blocks; ragged last blocks and steps throughout.
SHAPES = [(1, 8, 8, 64, 64, False), (1, 8, 8, 64, 65, False), (1, 8, 8, 65, 200, False), (2, 32, 8, 256, 130, False),
          (2, 32, 8, 257, 130, False), (2, 32, 32, 512, 512, True), (2, 32, 8, 513, 513, True),
          (4, 32, 8, 500, 90, False), (5, 32, 8, 300, 190, False), (1, 4, 4, 3400, 3400, True)]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("kind", [None, "bool", "f16", "f32"])
@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_workgroup_shapes(cuda, case, kind, D):
    import torch_spyre_amd as tsa

    B, Hq, Hkv, Sq, Skv, causal = case
    if causal and kind is not None:
        pytest.skip("causal calls take no mask")
    q = randn((B, Hq, Sq, D), SEED + 330)
    k, v = randn((B, Hkv, Skv, D), SEED + 331), randn((B, Hkv, Skv, D), SEED + 332)
    mask = None if kind is None else make_mask(kind, "qk", B, Hq, Sq, Skv, SEED + 333)
    out, lse = tsa.scaled_dot_product_attention(
        q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=None if mask is None else mask.to(cuda), is_causal=causal,
        enable_gqa=True, return_lse=True)
    heads = sorted({0, Hq // 2, Hq - 1})  # sampled heads: the reference runs on the CPU
    qs, ks, vs = q[:, heads], k[:, [h // (Hq // Hkv) for h in heads]], v[:, [h // (Hq // Hkv) for h in heads]]
    assert_close(out[:, heads], OA.sdpa_cpu_fp32(qs, ks, vs, attn_mask=mask, is_causal=causal))
    _, lse64 = OA.sdpa_decomposition_fp64(qs, ks, vs, attn_mask=None if mask is None else mask.numpy(),
                                          is_causal=causal, return_lse=True)
    assert np.allclose(lse[:, heads].cpu().numpy(), lse64, atol=LSE_BAR.get(kind, LSE_ATOL), rtol=0)
    assert not torch.isnan(out).any()


@pytest.mark.parametrize("layout", ["rows", "odd_rows", "offset", "transposed", "key_broadcast"])
@pytest.mark.parametrize("case", [(2, 8, 2, 20, 130, 64), (1, 4, 4, 97, 333, 128)], ids=str)
def test_f32_mask_layouts(cuda, case, layout):
    """An fp32 bias as rows of whole 16-byte units (loaded as such), as rows of
    an odd number of floats and from an odd offset (loaded 4 bytes a lane, the
    last row ending with the allocation), and with key strides other than 1
    (the per-wavefront kernel): one answer."""
    import torch_spyre_amd as tsa

    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 340)
    k, v = randn((B, Hkv, Skv, D), SEED + 341), randn((B, Hkv, Skv, D), SEED + 342)
    bias = torch.randn((Hq, Sq, Skv), generator=torch.Generator().manual_seed(SEED + 343))
    if layout == "key_broadcast":
        bias = bias[..., :1].expand(Hq, Sq, Skv)
    n = bias.numel()
    if layout == "rows":
        wide = torch.zeros((Hq, Sq, (Skv + 7) // 4 * 4), device=cuda)
        dev = wide[..., :Skv]
        dev.copy_(bias)
    elif layout == "odd_rows":
        wide = torch.full((Hq, Sq, Skv + 1 + Skv % 2), float("nan"), device=cuda)
        dev = wide[..., :Skv]
        dev.copy_(bias)
    elif layout == "offset":
        flat = torch.empty(n + 1, device=cuda)
        dev = flat[1:].view(Hq, Sq, Skv)
        dev.copy_(bias)
    elif layout == "transposed":
        dev = bias.transpose(1, 2).contiguous().to(cuda).transpose(1, 2)
    else:
        dev = bias[..., :1].contiguous().to(cuda).expand(Hq, Sq, Skv)
    out, lse = tsa.scaled_dot_product_attention(q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=dev[None],
                                                enable_gqa=True, return_lse=True)
    assert_close(out, OA.sdpa_cpu_fp32(q, k, v, attn_mask=bias[None]))
    _, lse64 = OA.sdpa_decomposition_fp64(q, k, v, attn_mask=bias[None].numpy(), return_lse=True)
    assert np.allclose(lse.cpu().numpy(), lse64, atol=1e-4, rtol=0)


# Decode that reads its mask as it lies.  Short-decode kernel: one block with
# ragged and empty slices (1, 31, 33, 300 keys), splits of eight- and of
# four-wavefront blocks, several queries per head.  Split-KV decode kernels:
# one run and several, a ragged last run read as a window, one chunk and
# chunks merged in the kernel and by the merge pass, four-wavefront items.
DECODE = [(2, 8, 2, 1, 1, 128), (3, 4, 4, 1, 31, 64), (1, 8, 2, 3, 33, 128), (1, 8, 8, 4, 300, 64),
          (1, 32, 8, 1, 1500, 128), (2, 16, 2, 2, 2100, 64), (40, 32, 8, 1, 64, 128), (40, 8, 8, 1, 200, 64),
          (16, 32, 8, 1, 2047, 128), (4, 64, 8, 1, 9000, 128), (24, 32, 8, 1, 5000, 128), (8, 32, 8, 1, 1111, 64)]


@pytest.mark.parametrize("shape", ["tail", "pad", "bhqk", "1h1k", "holes"])
@pytest.mark.parametrize("kind", ["bool", "f16", "f32"])
@pytest.mark.parametrize("case", DECODE, ids=str)
def test_masked_decode(cuda, case, kind, shape):
    """holes: whole 64-key runs masked (skipped) in the middle and at both
    ends of a sequence, and one sequence masked altogether (zeros, LSE -inf)."""
    import torch_spyre_amd as tsa

    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 350)
    k, v = randn((B, Hkv, Skv, D), SEED + 351), randn((B, Hkv, Skv, D), SEED + 352)
    dead = []
    if shape == "holes":
        keep = torch.rand((B, 1, 1, (Skv + 63) // 64), generator=torch.Generator().manual_seed(SEED + 353)) > 0.5
        keep = keep.repeat_interleave(64, dim=3)[..., :Skv].clone()
        keep[:, :, :, Skv // 2] = True
        keep[B - 1] = False
        dead = [B - 1]
        mask = keep if kind == "bool" else torch.zeros(keep.shape, dtype=DTYPE[kind]).masked_fill_(~keep, -float("inf"))
    else:
        mask = make_mask(kind, shape, B, Hq, Sq, Skv, SEED + 354 + Skv)
    out, lse = tsa.scaled_dot_product_attention(q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=mask.to(cuda),
                                                enable_gqa=True, return_lse=True)
    live = [b for b in range(B) if b not in dead]
    for b in dead:
        assert not out[b].float().abs().sum() and bool(torch.isneginf(lse[b]).all())
    if not live:
        return
    m = mask[live] if mask.dim() == 4 and mask.shape[0] == B else mask
    ref = OA.sdpa_cpu_fp32(q[live], k[live], v[live], attn_mask=m)
    assert_close(out[live], ref)
    some = live[:3]  # fp64 on a few sequences
    m = mask[some] if mask.dim() == 4 and mask.shape[0] == B else mask
    _, lse64 = OA.sdpa_decomposition_fp64(q[some], k[some], v[some], attn_mask=m.numpy(), return_lse=True)
    assert np.allclose(lse[some].cpu().numpy(), lse64, atol=1e-4, rtol=0)


@pytest.mark.parametrize("case", [(1, 8, 2, 1, 300, 128), (16, 32, 8, 1, 1000, 128)], ids=str)
def test_masked_decode_reads_inside_the_mask(cuda, case):
    """The mask ends with its allocation's last bytes, at an odd address, and
    K / V rows past a padded sequence's end hold NaN: neither is read past."""
    import torch_spyre_amd as tsa

    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 360)
    k, v = randn((B, Hkv, Skv, D), SEED + 361), randn((B, Hkv, Skv, D), SEED + 362)
    lens = torch.linspace(70, Skv, B).long() if B > 1 else torch.tensor([Skv])
    keep = (torch.arange(Skv)[None] < lens[:, None])[:, None, None]
    flat = torch.empty(B * Skv + 3, dtype=torch.bool, device=cuda)
    mask = flat[3:].view(keep.shape)
    mask.copy_(keep.to(cuda))
    kn, vn = k.clone(), v.clone()
    for b in range(B):  # whole 64-key runs past the end
        first = (int(lens[b]) + 127) // 64 * 64
        kn[b, :, first:], vn[b, :, first:] = float("nan"), float("nan")
    if B == 1:
        kn, vn = k, v
    last = Skv % 64  # a ragged last run is read as the 64 keys ending with the last one
    if B > 1 and last:
        kn[:, :, Skv - 64 - 64:], vn[:, :, Skv - 64 - 64:] = k[:, :, Skv - 64 - 64:], v[:, :, Skv - 64 - 64:]
    out = tsa.scaled_dot_product_attention(q.to(cuda), kn.to(cuda), vn.to(cuda), attn_mask=mask, enable_gqa=True)
    assert_close(out, OA.sdpa_cpu_fp32(q, k, v, attn_mask=keep))


@pytest.mark.parametrize("key", [20, -3])
@pytest.mark.parametrize("kind", ["f16", "f32"])
@pytest.mark.parametrize("Sq,Skv,Hkv", [(1, 200, 2), (1, 4100, 8), (1, 20000, 8), (15, 65, 2), (40, 1040, 2),
                                        (128, 4096, 2), (300, 777, 8), (1100, 1100, 8)])
def test_nan_bias_reaches_its_row(cuda, Sq, Skv, Hkv, kind, key):
    """A NaN in a bias makes its row NaN, also where every other score of its
    keys' split or (fp32, or one query) step is -inf, and no other row.  fp16
    biases of several queries skip steps by their largest number, so that NaN
    keys under -inf do not count: their NaN lies among kept keys."""
    import torch_spyre_amd as tsa

    B, Hq, D = 2, 8, 128
    q, k, v = (randn((B, h, s, D), SEED + 330 + i).to(cuda) for i, (h, s) in enumerate([(Hq, Sq), (Hkv, Skv), (Hkv, Skv)]))
    mask = torch.full((B, Hq, Sq, Skv), -float("inf"), dtype=DTYPE[kind], device=cuda)
    mask[..., :40] = 0
    bad = torch.zeros((B, Hq, Sq), dtype=torch.bool, device=cuda)
    bad[0, 1, 0] = bad[1, 7, Sq - 1] = True
    if kind == "f16" and Sq > 1:
        key = 20 if key > 0 else Skv - 20
        mask[..., Skv - 30:] = 0
    mask[..., key][bad] = float("nan")
    got = torch.isnan(tsa.scaled_dot_product_attention(q, k, v, attn_mask=mask, enable_gqa=True))
    assert torch.equal(got.all(-1), bad) and torch.equal(got.any(-1), bad)


@pytest.mark.parametrize("kind", ["none", "bool"])
@pytest.mark.parametrize("Sq,Skv", [(40, 1040), (128, 4096)])
def test_nan_key_reaches_every_row_that_sees_it(cuda, kind, Sq, Skv):
    """Key splits carry a NaN key of one split into the result."""
    import torch_spyre_amd as tsa

    B, Hq, Hkv, D = 2, 8, 2, 128
    q, k, v = (randn((B, h, s, D), SEED + 340 + i).to(cuda) for i, (h, s) in enumerate([(Hq, Sq), (Hkv, Skv), (Hkv, Skv)]))
    k[0, 0, Skv - 2, 5] = float("nan")
    mask = torch.ones((Sq, Skv), dtype=torch.bool, device=cuda) if kind == "bool" else None
    got = torch.isnan(tsa.scaled_dot_product_attention(q, k, v, attn_mask=mask, enable_gqa=True)).all(-1)
    want = torch.zeros((B, Hq, Sq), dtype=torch.bool, device=cuda)
    want[0, :Hq // Hkv] = True
    assert torch.equal(got, want)


@pytest.mark.parametrize("kind", ["bool", "f16"])
@pytest.mark.parametrize("shape", ["qk", "bhqk", "1h1k"])
@pytest.mark.parametrize("Sq,Skv,D", [(40, 7, 64), (40, 9, 128), (130, 16, 64), (70, 17, 128), (33, 63, 64), (130, 65, 128),
                                      (65, 95, 64), (40, 97, 128), (300, 129, 64), (20, 1023, 128), (333, 333, 128)])
def test_mask_rows_of_any_alignment(cuda, Sq, Skv, D, shape, kind):
    """Half steps read mask rows that start anywhere and end inside a 16-byte
    unit as they lie: views into a buffer whose other elements are NaN (or
    True), the last row ending with the buffer."""
    import torch_spyre_amd as tsa

    B, Hq, Hkv = 2, 8, 4
    q = randn((B, Hq, Sq, D), SEED + 350)
    k, v = randn((B, Hkv, Skv, D), SEED + 351), randn((B, Hkv, Skv, D), SEED + 352)
    mask = make_mask(kind, shape, B, Hq, Sq, Skv, SEED + 353 + Sq + Skv)
    wide = torch.full((*mask.shape[:-1], Skv + 3), True if kind == "bool" else float("nan"), dtype=mask.dtype, device=cuda)
    view = wide[..., 3:]
    view.copy_(mask)
    out, lse = tsa.scaled_dot_product_attention(q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=view, enable_gqa=True,
                                                return_lse=True)
    assert_close(out, OA.sdpa_cpu_fp32(q, k, v, attn_mask=mask))
    _, lse64 = OA.sdpa_decomposition_fp64(q, k, v, attn_mask=mask.numpy(), return_lse=True)
    assert np.allclose(lse.cpu().numpy(), lse64, atol=LSE_ATOL, rtol=0)
