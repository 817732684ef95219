"""Relayouts of odd sizes and alignments, bit-exact: rows that start anywhere
are moved in 16-byte items, and the nests of one description that write
apart from each other share a launch (others keep their order)."""

import numpy as np
import pytest
import torch

from oracle import layout as OL
from tests.conftest import SEED

pytestmark = pytest.mark.gpu

# Odd row lengths (rows on odd elements), remainders of 1 to 63 elements, one
# row, fewer elements than an item, batches beside the stick, 64 and 32
# element sticks, aligned rows whose sticks a tile kernel could take too.
SIZES = [[2, 77, 501], [33, 65], [1, 63], [5, 1], [3, 41, 100], [8, 33, 1000], [130, 4097], [7, 3, 9, 67],
         [64, 2056], [2, 40, 129]]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("size", SIZES, ids=str)
def test_odd_sizes_and_offsets_vs_oracle(cuda, size, off, dtype):
    """Host order at an element offset -> the default layout -> host order at
    another; what lies around the host tensors stays as it was."""
    import torch_spyre_amd as tsa

    n = int(np.prod(size))
    it, npt, name = ((torch.int16, np.uint16, "float16") if dtype == torch.float16 else
                     (torch.int32, np.uint32, "float32"))
    raw = torch.randint(-(2 ** 15), 2 ** 15 - 1, (n + 2 * off,), generator=torch.Generator().manual_seed(SEED + n)).to(it)
    st = OL.contiguous_strides(size)
    lay = tsa.SpyreTensorLayout(size, dtype)
    src = raw.to(cuda).view(dtype)
    dev = tsa.device_buffer(tsa.spyre_empty_with_layout(size, st, dtype, lay, cuda))
    tsa.DmaCopy(src, dev, tsa.dma_plan(size, st, st, off, lay, True))()
    want = OL.h2d(raw[off:off + n].numpy().view(npt), size, st, 0, OL.stl_default(size, name))
    got = dev.contiguous().view(it).cpu().numpy().view(npt).reshape(-1)
    assert np.array_equal(got[:want.size], want)
    back = torch.full((n + 7,), -1, dtype=it, device=cuda)
    tsa.DmaCopy(dev, back.view(dtype), tsa.dma_plan(size, st, st, 5, lay, False))()
    torch.cuda.synchronize()
    back = back.cpu()
    assert torch.equal(back[5:5 + n], raw[off:off + n])
    assert bool((back[:5] == -1).all()) and bool((back[5 + n:] == -1).all())


@pytest.mark.parametrize("rows,cols", [(9, 33), (64, 1001), (300, 5001)])
def test_overwrite_of_odd_rows(cuda, rows, cols):
    """A block of odd-length rows into a wider tensor (both sides' runs
    contiguous, neither side's rows aligned)."""
    import torch_spyre_amd as tsa

    g = torch.Generator().manual_seed(SEED + rows)
    x = torch.randn((rows, cols), generator=g).half()
    y = torch.randn((rows + 2, cols + 4), generator=g).half()
    out = y.to(cuda)
    tsa.overwrite(x.to(cuda), out, [0, 1], [1, 3])
    y[1:1 + rows, 3:3 + cols] = x
    assert torch.equal(out.cpu().view(torch.int16), y.view(torch.int16))


def _nest(loops, off_s, off_d):
    from torch_spyre_amd import _lib

    info = _lib.StrideInfo()
    info.rank = len(loops)
    for q, (n, ss, sd) in enumerate(loops):
        info.size[q], info.stride_src[q], info.stride_dst[q] = n, ss, sd
    info.offset_src, info.offset_dst = off_s, off_d
    return info


def test_nests_that_overlap_keep_their_order(cuda):
    """Nests writing the same elements: the last one's values stay, whichever
    strides they are stated with; ten disjoint ones (two launches) all land."""
    import torch_spyre_amd as tsa

    src = torch.arange(40000, dtype=torch.int32).to(torch.int16).to(cuda).view(torch.float16)

    def run(nests, n=20000):
        dst = torch.full((n,), -1, dtype=torch.int16, device=cuda)
        tsa.DmaCopy(src, dst.view(torch.float16), nests)()
        torch.cuda.synchronize()
        want = np.full(n, -1, dtype=np.int16)
        s = src.view(torch.int16).cpu().numpy()
        for info in nests:
            idx_s, idx_d = np.array([info.offset_src]), np.array([info.offset_dst])
            for q in range(info.rank):
                k = np.arange(info.size[q])
                idx_s = (idx_s[:, None] + k * info.stride_src[q]).reshape(-1)
                idx_d = (idx_d[:, None] + k * info.stride_dst[q]).reshape(-1)
            want[idx_d] = s[idx_s]
        assert np.array_equal(dst.cpu().numpy(), want)

    run([_nest([(9000, 1, 1)], 0, 0), _nest([(9000, 1, 1)], 20000, 4500)])          # overlapping halves
    run([_nest([(64, 1, 1), (100, 70, 80)], 0, 0), _nest([(40, 1, 1), (90, 50, 75)], 9000, 30)])  # other strides
    run([_nest([(64, 1, 1), (50, 64, 100)], 0, 0), _nest([(36, 1, 1), (50, 64, 100)], 7000, 64)])  # apart
    run([_nest([(17 + i, 1, 1), (20, 40, 1000)], 900 * i, 50 * i) for i in range(10)])


@pytest.mark.parametrize("rows", [8730, 8760])
def test_items_to_a_lane(cuda, rows):
    """Both sides of one or four items to a lane (rows of 120 items and a
    remainder; 256 units x 16 blocks of 256 items are 8738.1 rows)."""
    test_odd_sizes_and_offsets_vs_oracle(cuda, [rows, 1001], 1, torch.float16)
