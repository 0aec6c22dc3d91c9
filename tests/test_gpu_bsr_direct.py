"""BSR SpMM by wavefronts that make their operands in registers: none to five steps for a wavefront, ragged and single feature
tiles, blocks of several slices, arrays that start at an odd element.  Checked against the fp64 oracle as in
test_gpu_bsr.py."""
import ctypes

import numpy as np
import pytest
import torch

from sparsetir_amd import _lib, datasets, ops
from test_gpu_bsr import _check

pytestmark = pytest.mark.gpu


def _edges(dev, mb, nb, blk, feat, at_most, waves, dtype):
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
    code = _lib.lib().stir_bsr_form(cus, mb, nb, blk, feat, ctypes.c_int64(nnzb))
    assert code // 32 == waves  # 16 + 1: one wavefront with one step on its way
    out, start = (torch.float32, 1) if (mb & 1) == (dtype is torch.float16) else (dtype, 0)

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


@pytest.mark.parametrize("mb,nb,blk,feat,at_most,waves", [
    (40, 70, 32, 96, 50, 8),         # up to seven steps a wavefront
    (24, 40, 64, 416, 26, 8),        # two slices, two steps a block
    (150, 25, 32, 352, 12, 4),       # up to three steps a wavefront, and none for some
    (6, 9, 96, 224, 9, 4),           # three slices, three steps a block
    (9, 40, 32, 64, 24, 4),
    (240, 40, 32, 288, 20, 2),       # more steps than tiles side by side are good for
    (100, 40, 32, 800, 12, 2),
    (40, 12, 64, 992, 6, 2),
    (230, 33, 32, 416, 6, 1),        # four tiles to a workgroup, the last of 32 features
    (331, 20, 32, 160, 5, 1),        # two tiles to a slice: two slices in a workgroup
    (300, 40, 32, 544, 7, 1),
    (160, 9, 96, 160, 3, 1),
    (70, 200, 32, 2336, 30, 17),     # one step on its way; nothing to one step for some
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_direct_edges(dev, mb, nb, blk, feat, at_most, waves, dtype):
    _edges(dev, mb, nb, blk, feat, at_most, waves, dtype)


# 16-row slices, two chunks of 16 columns to a step: odd numbers of chunks, none, and features that end inside a tile
@pytest.mark.parametrize("mb,nb,blk,feat,at_most,waves", [
    (40, 90, 16, 96, 85, 8),         # up to six steps a wavefront
    (21, 40, 48, 224, 40, 8),        # three chunks a block
    (150, 60, 16, 352, 30, 4),       # up to four steps a wavefront, and none for some
    (64, 30, 80, 160, 9, 4),         # five chunks
    (300, 30, 16, 1184, 21, 2),      # two tiles to a workgroup
    (640, 25, 16, 608, 17, 2),       # ... of five
    (160, 9, 112, 288, 3, 2),
    (420, 45, 16, 480, 7, 1),        # 128 features by one wavefront
    (96, 750, 16, 2176, 61, 17),     # one step on its way; nothing to one step for some
    (1050, 20, 16, 480, 16, 1),      # 256
    (205, 20, 80, 480, 4, 1),
    (230, 140, 48, 992, 12, 4),      # 256 by four
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_direct16_edges(dev, mb, nb, blk, feat, at_most, waves, dtype):
    _edges(dev, mb, nb, blk, feat, at_most, waves, dtype)
