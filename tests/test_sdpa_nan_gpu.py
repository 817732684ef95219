"""NaN in masked SDPA calls: one in a key or a bias that a row keeps makes
that row NaN, wherever its key lies; what a row's mask drops does not."""

import pytest
import torch

from oracle import attention as OA
from tests.conftest import SEED
from tests.test_sdpa_gpu import assert_close, randn

pytestmark = pytest.mark.gpu

DTYPE = {"f16": torch.float16, "f32": torch.float32}


def as_mask(kind, keep):
    if kind == "bool":
        return keep
    return torch.zeros(keep.shape, dtype=DTYPE[kind]).masked_fill_(~keep, -float("inf"))


def nan_rows(cuda, q, k, v, mask, scale=None):
    """Rows of the result that are NaN; a row is NaN in every feature or in none."""
    import torch_spyre_amd as tsa

    out = tsa.scaled_dot_product_attention(q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=mask.to(cuda), scale=scale,
                                           enable_gqa=True)
    got = torch.isnan(out)
    assert torch.equal(got.any(-1), got.all(-1))
    return got.all(-1).cpu()


# Short decode with its keys split over blocks (16 splits of four-wavefront
# blocks, 8 of eight-wavefront ones), every kept key in one split.
@pytest.mark.parametrize("kind", ["bool", "f16", "f32"])
@pytest.mark.parametrize("first,kept", [(0, 100), (20, 1), (1000, 20)])
@pytest.mark.parametrize("case", [(1, 32, 8, 1, 2048, 128), (2, 32, 8, 1, 2048, 128), (1, 8, 8, 3, 4096, 64),
                                  (3, 32, 8, 2, 2000, 128)], ids=str)
def test_nan_in_the_only_split_with_kept_keys(cuda, case, first, kept, kind):
    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 500)
    k, v = randn((B, Hkv, Skv, D), SEED + 501), randn((B, Hkv, Skv, D), SEED + 502)
    keep = torch.zeros((B, 1, Sq, Skv), dtype=torch.bool)
    keep[..., first:first + kept] = True
    mask = as_mask(kind, keep)
    k[B - 1, Hkv - 1, first, 3] = float("nan")
    want = torch.zeros((B, Hq, Sq), dtype=torch.bool)
    want[B - 1, Hq - Hq // Hkv:] = True
    assert torch.equal(nan_rows(cuda, q, k, v, mask), want)
    if kind != "bool":
        mask = mask.expand(B, Hq, Sq, Skv).clone()
        mask[0, 1, Sq - 1, first] = float("nan")
        want[0, 1, Sq - 1] = True
        assert torch.equal(nan_rows(cuda, q, k, v, mask), want)


# Half steps of 32 keys (Sq 40; 128 packed rows), with and without a key
# split, and full steps of 64 (300, 1000).
SQ = [(40, 300, 2), (40, 2048, 2), (128, 1000, 8), (128, 4096, 2), (300, 2048, 8), (1000, 1000, 8)]


@pytest.mark.parametrize("scale", [None, 2.0])
@pytest.mark.parametrize("kind", ["bool", "f16", "f32"])
@pytest.mark.parametrize("Sq,Skv,Hkv", SQ)
def test_nan_alone_in_its_step(cuda, Sq, Skv, Hkv, kind, scale):
    """The one kept key of its step is NaN (keys 0 .. 64 are kept), then the
    one number that is no -inf of its step is a NaN bias; q prescaled in fp16
    and (scale 2) not."""
    B, Hq, D = 2, 8, 128
    q = randn((B, Hq, Sq, D), SEED + 510)
    k, v = randn((B, Hkv, Skv, D), SEED + 511), randn((B, Hkv, Skv, D), SEED + 512)
    keep = torch.zeros((Sq, Skv), dtype=torch.bool)
    keep[:, :65] = True
    bad = k.clone()
    bad[1, 0, 64, 9] = float("nan")
    want = torch.zeros((B, Hq, Sq), dtype=torch.bool)
    want[1, :Hq // Hkv] = True
    assert torch.equal(nan_rows(cuda, q, bad, v, as_mask(kind, keep), scale), want)
    if kind != "bool":
        mask = as_mask(kind, keep).expand(B, Hq, Sq, Skv).clone()
        mask[0, 2, Sq // 2, 200] = float("nan")
        want = torch.zeros((B, Hq, Sq), dtype=torch.bool)
        want[0, 2, Sq // 2] = True
        assert torch.equal(nan_rows(cuda, q, k, v, mask, scale), want)


@pytest.mark.parametrize("low", [-float("inf"), torch.finfo(torch.float16).min])
@pytest.mark.parametrize("Sq,Skv,Hkv", [(128, 1000, 8), (300, 2048, 8), (1000, 1000, 8)])
def test_steps_of_dropped_keys_stay_skipped(cuda, Sq, Skv, Hkv, low):
    """fp16 biases: NaN keys of whole steps that a bias drops (-inf or the
    type's lowest number) after kept ones do not reach a row."""
    import torch_spyre_amd as tsa

    B, Hq, D = 1, 8, 128
    q = randn((B, Hq, Sq, D), SEED + 520)
    k, v = randn((B, Hkv, Skv, D), SEED + 521), randn((B, Hkv, Skv, D), SEED + 522)
    mask = torch.zeros((Sq, Skv), dtype=torch.float16)
    mask[:, 128:] = low
    kn = k.clone()
    kn[:, :, 192:] = float("nan")
    out = tsa.scaled_dot_product_attention(q.to(cuda), kn.to(cuda), v.to(cuda), attn_mask=mask.to(cuda), enable_gqa=True)
    assert_close(out, OA.sdpa_cpu_fp32(q, k, v, attn_mask=mask))


@pytest.mark.parametrize("kind", ["bool", "f16", "f32"])
@pytest.mark.parametrize("case", [(1, 32, 8, 1, 200, 128), (1, 32, 8, 1, 2048, 128), (2, 8, 2, 3, 500, 64),
                                  (1, 8, 8, 1, 4000, 64), (16, 32, 8, 1, 2048, 128)], ids=str)
def test_decode_ignores_unused_cache(cuda, case, kind):
    """A padded decode over a cache never written past its 64-token run of
    real keys: NaN in K and V there does not reach the result."""
    import torch_spyre_amd as tsa

    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 530)
    k, v = randn((B, Hkv, Skv, D), SEED + 531), randn((B, Hkv, Skv, D), SEED + 532)
    lens = [70 + 7 * b for b in range(B)]
    keep = torch.zeros((B, 1, 1, Skv), dtype=torch.bool)
    kn, vn = k.clone(), v.clone()
    for b, n in enumerate(lens):
        keep[b, ..., :n] = True
        end = (n + 63) // 64 * 64
        kn[b, :, end:], vn[b, :, end:] = float("nan"), float("nan")
    mask = as_mask(kind, keep)
    out = tsa.scaled_dot_product_attention(q.to(cuda), kn.to(cuda), vn.to(cuda), attn_mask=mask.to(cuda), enable_gqa=True)
    assert_close(out, OA.sdpa_cpu_fp32(q, k, v, attn_mask=mask))
