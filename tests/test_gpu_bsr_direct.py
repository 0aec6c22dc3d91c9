"""BSR SpMM by wavefronts that take the steps in turn or alone, each case in the kernel that it names: none to six steps for a
wavefront, ragged and single feature tiles, blocks of several slices, arrays that start at an odd element.  Checked against the
fp64 oracle as in test_gpu_bsr.py."""
import numpy as np
import pytest
import torch

from helpers import bsr_form
from sparsetir_amd import datasets, ops
from test_gpu_bsr import _check

pytestmark = pytest.mark.gpu


def _edges(dev, mb, nb, blk, feat, at_most, form, dtype, out_start=None):
    rng = np.random.default_rng(mb + feat)
    cfg = datasets.config4(seed=mb, mb=mb, nb=nb, blk=blk, density=0.0, feat=feat)
    counts = rng.integers(at_most // 2, at_most + 1, mb)
    few = min(6, at_most + 1, mb - 1)
    counts[:few], counts[-1] = np.arange(few), at_most
    rows = [rng.permutation(nb)[:k].astype(np.int32) for k in counts]
    cfg["indptr"] = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    cfg["indices"] = np.concatenate(rows).astype(np.int32)
    nnzb = len(cfg["indices"])
    cfg["data"] = rng.standard_normal((nnzb, blk, blk)).astype(np.float32) * 0.1
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    out, start = out_start or ((torch.float32, 1) if (mb & 1) == (dtype is torch.float16) else (dtype, 0))
    assert bsr_form(mb, nb, blk, feat, nnzb, cus, out is torch.float32) == form

    def place(values):
        t = torch.empty(values.size + start, dtype=dtype, device=dev)[start:]
        t.copy_(torch.from_numpy(values.reshape(-1)))
        return t

    a, x = place(cfg["data"]), place(cfg["x"])
    y = torch.full((mb * blk * feat + start,), float("nan"), dtype=out, device=dev)[start:]
    ops.build_bsrmm(mb, nb, nnzb, blk, feat, dtype, out)(a, x, y, torch.from_numpy(cfg["indptr"]).to(dev),
                                                         torch.from_numpy(cfg["indices"]).to(dev))
    torch.cuda.synchronize()
    _check(y.float().cpu().numpy().reshape(mb * blk, feat), cfg, a.float().cpu().numpy().reshape(-1, blk, blk),
           x.float().cpu().numpy().reshape(nb * blk, feat), out is not torch.float32, f"{mb}x{nb} blk {blk} feat {feat} {dtype}")


@pytest.mark.parametrize("mb,nb,blk,feat,at_most,form", [
    (40, 70, 32, 96, 50, "128 by 8"),         # up to seven steps a wavefront
    (24, 40, 64, 416, 26, "128 by 8"),        # two slices, two steps a block
    (150, 25, 32, 352, 12, "128 by 4"),       # up to three steps a wavefront, and none for some
    (6, 9, 96, 224, 9, "128 by 4"),           # three slices, three steps a block
    (9, 40, 32, 64, 24, "128 by 4"),
    (240, 40, 32, 288, 20, "128 by 2"),       # more steps than tiles side by side are good for
    (100, 40, 32, 800, 12, "128 by 2"),
    (40, 12, 64, 992, 6, "128 by 2"),
    (230, 33, 32, 416, 6, "128 by 2"),        # the last of 32 features
    (331, 20, 32, 160, 7, "128 by 2"),        # two tiles to a slice
    (300, 40, 32, 544, 7, "128 by 1"),
    (160, 9, 96, 160, 3, "128 by 2"),
    (230, 9, 96, 160, 3, "128 by 1"),
    (70, 200, 32, 2336, 30, "128 by 1, one step"),     # nothing to one step for some
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_direct_edges(dev, mb, nb, blk, feat, at_most, form, dtype):
    _edges(dev, mb, nb, blk, feat, at_most, form, dtype)


# 16-row slices, two chunks of 16 columns to a step: odd numbers of chunks, none, and features that end inside a tile
@pytest.mark.parametrize("mb,nb,blk,feat,at_most,form", [
    (40, 90, 16, 96, 85, "128 by 8"),         # up to six steps a wavefront
    (21, 40, 48, 224, 40, "128 by 8"),        # three chunks a block
    (150, 60, 16, 352, 30, "128 by 4"),       # up to four steps a wavefront, and none for some
    (64, 30, 80, 160, 9, "128 by 4"),         # five chunks
    (300, 30, 16, 1184, 21, "128 by 2, two tiles"),
    (640, 25, 16, 608, 17, "128 by 2, two tiles"),       # ... of five
    (160, 9, 112, 288, 3, "128 by 2, two tiles"),
    (420, 45, 16, 480, 7, "128 by 1"),
    (96, 750, 16, 2176, 61, "128 by 1, one step"),     # nothing to one step for some
    (1050, 20, 16, 480, 16, "256 by 1"),
    (205, 20, 80, 480, 4, "128 by 2, two tiles"),
    (180, 60, 48, 992, 24, "256 by 4"),
    (180, 140, 48, 992, 40, "256 by 4 ranked"),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_direct16_edges(dev, mb, nb, blk, feat, at_most, form, dtype):
    _edges(dev, mb, nb, blk, feat, at_most, form, dtype)


# 64 features by eight wavefronts, X through LDS: slices beyond the first, several steps or odd numbers of chunks a block, more
# blocks in a row than lanes, and rows with none
@pytest.mark.parametrize("mb,nb,blk,feat,at_most,form", [
    (260, 90, 16, 64, 85, "LDS 64 by 8"),
    (92, 40, 48, 64, 19, "LDS 64 by 8"),    # three chunks a block
    (55, 20, 80, 32, 13, "LDS 64 by 8"),    # five, half of the features
    (40, 90, 32, 96, 89, "LDS 64 by 8"),
    (40, 40, 64, 64, 26, "LDS 64 by 8"),    # two slices, two steps a block
    (40, 24, 96, 32, 23, "LDS 64 by 8"),    # three
    (20, 20, 128, 192, 19, "LDS 64 by 8"),  # four
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_lds_split_edges(dev, mb, nb, blk, feat, at_most, form, dtype):
    _edges(dev, mb, nb, blk, feat, at_most, form, dtype)


# results of 16 bits leave 16 bytes at a time, wherever the array starts
@pytest.mark.parametrize("mb,nb,blk,feat,at_most,form", [
    (150, 25, 32, 352, 12, "128 by 4"),
    (70, 200, 32, 2336, 30, "128 by 1, one step"),
    (301, 17, 32, 608, 9, "256 by 1"),
    (64, 30, 80, 160, 9, "128 by 4"),
    (640, 25, 16, 608, 17, "128 by 2, two tiles"),
    (1050, 20, 16, 480, 16, "256 by 1"),
    (180, 60, 48, 992, 24, "256 by 4"),
    (260, 90, 16, 64, 85, "LDS 64 by 8"),
    (147, 13, 64, 2400, 8, "LDS 64 x 256"),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_sixteen_bit_results_at_an_odd_element(dev, mb, nb, blk, feat, at_most, form, dtype):
    _edges(dev, mb, nb, blk, feat, at_most, form, dtype, (dtype, 1))
