"""NaN in masked SDPA calls: one in a key or a bias that a row keeps makes
that row NaN, wherever its key lies."""

import pytest
import torch

from tests.conftest import SEED
from tests.test_sdpa_gpu import randn

pytestmark = pytest.mark.gpu

DTYPE = {"f16": torch.float16, "f32": torch.float32}


def as_mask(kind, keep):
    if kind == "bool":
        return keep
    return torch.zeros(keep.shape, dtype=DTYPE[kind]).masked_fill_(~keep, -float("inf"))


def nan_rows(cuda, q, k, v, mask):
    """Rows of the result that are NaN; a row is NaN in every feature or in none."""
    import torch_spyre_amd as tsa

    out = tsa.scaled_dot_product_attention(q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=mask.to(cuda), enable_gqa=True)
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
