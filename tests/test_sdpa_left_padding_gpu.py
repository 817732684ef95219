"""fp16 additive masks whose dropped keys hold the type's lowest number and
come first (sequences padded on the left): the kept keys' scores keep the
precision they have without the padding."""

import pytest
import torch

from oracle import attention as OA
from tests.conftest import SEED
from tests.test_sdpa_gpu import randn

pytestmark = pytest.mark.gpu

LOW = torch.finfo(torch.float16).min


def _attend(cuda, q, k, v, mask):
    """The result and the fp64 attention."""
    import torch_spyre_amd as tsa

    out = tsa.scaled_dot_product_attention(q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=mask.to(cuda), enable_gqa=True)
    return out.double().cpu(), torch.as_tensor(OA.sdpa_decomposition_fp64(q, k, v, attn_mask=mask.numpy()))


def _error(cuda, q, k, v, mask):
    """Relative 2-norm distance from the fp64 attention."""
    out, ref = _attend(cuda, q, k, v, mask)
    return float((out - ref).norm() / ref.norm())


# Half steps (Sq 40, 128), half steps over split keys (Skv 2048), full steps
# (300 and 1000 queries, the latter over split keys at D 64), short decode.
@pytest.mark.parametrize("real", [20, 40, 130])
@pytest.mark.parametrize("case", [(2, 8, 2, 40, 300, 128), (1, 16, 16, 128, 512, 64), (1, 32, 8, 40, 2048, 128),
                                  (4, 32, 8, 300, 512, 128), (2, 16, 16, 1000, 1001, 64), (2, 8, 2, 1, 900, 128)],
                         ids=str)
def test_left_padding_keeps_precision(cuda, case, real):
    """No less precise than the same call on the kept keys alone (1.3: both
    errors are dominated by the roundings of q, P and out to fp16, in another
    order)."""
    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 540) * 2
    k, v = randn((B, Hkv, Skv, D), SEED + 541), randn((B, Hkv, Skv, D), SEED + 542)
    mask = torch.zeros((1, 1, Sq, Skv), dtype=torch.float16)
    mask[..., :Skv - real] = LOW
    padded = _error(cuda, q, k, v, mask)
    alone = _error(cuda, q, k[:, :, -real:], v[:, :, -real:], mask[..., -real:])
    print(f"{case} {real} kept: {padded:.3e} padded, {alone:.3e} alone", flush=True)
    assert padded <= 1.3 * alone


@pytest.mark.parametrize("case", [(2, 8, 2, 40, 300, 128), (1, 32, 8, 40, 2048, 128), (2, 16, 16, 1000, 1001, 64),
                                  (4, 32, 8, 300, 512, 128)], ids=str)
def test_rows_of_dropped_keys_alone(cuda, case):
    """Causal on top of the padding: the first rows see dropped keys alone,
    all at the lowest number, and weigh them by their scores as other rows
    do.  At 65504 log2(e) fp32 steps by 2^-7, so a score is off by up to 2^-8
    and a weight by 2^-8 ln 2 = 0.27 %: with weights that sum to 1 and |v| < 6
    at most 0.017 before the rounding of P and out."""
    B, Hq, Hkv, Sq, Skv, D = case
    q = randn((B, Hq, Sq, D), SEED + 550)
    k, v = randn((B, Hkv, Skv, D), SEED + 551), randn((B, Hkv, Skv, D), SEED + 552)
    keep = torch.ones((Sq, Skv), dtype=torch.bool).tril(Skv - Sq)
    keep[:, :Skv - Sq + 35] = False
    mask = torch.zeros((1, 1, Sq, Skv), dtype=torch.float16).masked_fill_(~keep, LOW)
    out, ref = _attend(cuda, q, k, v, mask)
    err = (out - ref).abs()
    assert float(err[:, :, :35].max()) <= 0.017 + 2e-3
    assert bool((err[:, :, 35:] <= 2e-3 + 1e-2 * ref[:, :, 35:].abs()).all())
