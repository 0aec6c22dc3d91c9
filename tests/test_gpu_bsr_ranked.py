"""BSR SpMM where X does not fit an L2: slices taken in order of their length or as they come, by a wavefront each or not.
Empty block rows, a few with more blocks than a wavefront has lanes, block columns in any order, ragged feature
tiles, arrays that start at an odd element.  Checked against the fp64 oracle as in test_gpu_bsr.py."""
import numpy as np
import pytest
import torch

from sparsetir_amd import datasets, ops
from helpers import bsr_form
from test_gpu_bsr import RTOL, _check

pytestmark = pytest.mark.gpu


def _config(mb, nb, blk, density, feat, seed):
    """config4 with two long block rows and the columns of every row shuffled."""
    cfg = datasets.config4(seed=seed, mb=mb, nb=nb, blk=blk, density=density, feat=feat)
    rng = np.random.default_rng(seed)
    rows = [rng.permutation(cfg["indices"][cfg["indptr"][i]:cfg["indptr"][i + 1]]) for i in range(mb)]
    for i in (1, mb - 2):
        rows[i] = rng.permutation(nb)[:max(nb // 2, 1)].astype(np.int32)
    cfg["indptr"] = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    cfg["indices"] = np.concatenate(rows).astype(np.int32)
    cfg["data"] = rng.standard_normal((len(cfg["indices"]), blk, blk)).astype(np.float32) * 0.1
    return cfg


@pytest.mark.parametrize("mb,nb,blk,density,feat", [
    (1024, 193, 32, 0.004, 224),
    (1030, 200, 32, 0.004, 256),   # 32-row slices by a wavefront each
    (430, 200, 32, 0.004, 288),    # the last of three tiles with 32
    (220, 200, 32, 0.01, 672),
    (150, 200, 32, 0.02, 1056),
    (150, 70, 96, 0.04, 352),
    (170, 260, 32, 0.02, 992),
    (650, 200, 32, 0.005, 512),    # two full tiles of 256
    (70, 70, 96, 0.04, 1440),      # three slices per block row, 5.6 feature tiles
    (257, 250, 32, 0.01, 832),
    (343, 200, 32, 0.01, 736),
    (20, 200, 64, 0.03, 96),       # steps in turn by eight, four and two wavefronts
    (12, 100, 128, 0.05, 160),
    (14, 100, 128, 0.05, 160),
    (60, 200, 64, 0.03, 416),
    (33, 100, 128, 0.05, 544),
    (36, 100, 128, 0.05, 544),
    (40, 20, 64, 0.1, 1056),
    (83, 20, 64, 0.1, 1056),       # 64 rows by four wavefronts, 256 features each, the last with 32
    (1, 6200, 32, 0.001, 64),
    (1030, 90, 16, 0.02, 224),     # 16-row slices by a wavefront each: plain order
    (1024, 400, 16, 0.004, 512),   # 256 features
    (512, 520, 16, 0.004, 1024),
    (700, 400, 16, 0.004, 320),    # 128 features, an odd number of blocks
    (410, 1000, 16, 0.004, 544),
    (230, 50, 48, 0.05, 352),      # chunks of two blocks in one step
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("start", [0, 1])
def test_bsr_ranked_edges(dev, mb, nb, blk, density, feat, dtype, start):
    cfg = _config(mb, nb, blk, density, feat, seed=mb + feat) if mb > 2 else datasets.config4(
        seed=1, mb=mb, nb=nb, blk=blk, density=density, feat=feat)
    out = torch.float32 if start and dtype is torch.float16 else dtype

    def place(values, dt):
        t = torch.empty(values.size + start, dtype=dt, device=dev)[start:]
        t.copy_(torch.from_numpy(values.reshape(-1)))
        return t

    a, x = place(cfg["data"], dtype), place(cfg["x"], dtype)
    y = torch.full((mb * blk * feat + start,), float("nan"), dtype=out, device=dev)[start:]
    f = ops.build_bsrmm(mb, nb, len(cfg["indices"]), blk, feat, dtype, out)
    f(a, x, y, torch.from_numpy(cfg["indptr"]).to(dev), torch.from_numpy(cfg["indices"]).to(dev))
    torch.cuda.synchronize()
    a32 = a.float().cpu().numpy().reshape(-1, blk, blk)
    x32 = x.float().cpu().numpy().reshape(nb * blk, feat)
    _check(y.float().cpu().numpy().reshape(mb * blk, feat), cfg, a32, x32, out is not torch.float32,
           f"{mb}x{nb} blk {blk} feat {feat} {dtype} start {start}")


def _cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize("mb,nb,blk,density,feat,form", [
    (430, 200, 32, 0.004, 288, "128 by 1"),
    (650, 200, 32, 0.005, 512, "256 by 1"),
    (83, 20, 64, 0.1, 1056, "LDS 64 x 256"),
    (1030, 90, 16, 0.02, 224, "128 by 1"),
    (1024, 400, 16, 0.004, 512, "256 by 1"),
    # 32-row slices by a wavefront each, in order of their length: the last of six feature tiles with 32
    (257, 250, 32, 0.07, 1312, "256 by 1 ranked"),
    (1024, 250, 32, 0.07, 512, "256 by 1 ranked"),    # as many block rows as a wavefront ranks
    (1025, 250, 32, 0.07, 448, "256 by 1 ranked"),    # two groups, of 513 and 512
    (2051, 200, 32, 0.15, 256, "256 by 1 ranked"),    # three, one feature tile for all XCDs, X in an L2 but long rows
    (72, 90, 96, 0.07, 1440, "256 by 1 ranked"),      # six tiles over eight XCDs: the slices of a block row on one of them
    (40, 60, 160, 0.07, 1760, "256 by 1 ranked"),
    (220, 100, 96, 0.02, 1024, "256 by 1"),
    # 64 rows by four wavefronts
    (200, 250, 64, 0.05, 416, "LDS 64 x 128 ranked"),
    (100, 130, 64, 0.08, 2048, "LDS 64 x 256 ranked"),
    (1030, 100, 64, 0.15, 256, "LDS 64 x 128 ranked"),
    (33, 100, 128, 0.06, 3072, "LDS 64 x 256 ranked"),   # too few block rows to deal them to XCDs
    (44, 100, 128, 0.06, 2304, "LDS 64 x 256 ranked by rows"),
    (16, 60, 128, 0.05, 2080, "LDS 64 x 128 by rows"),
    (16, 30, 192, 0.1, 1056, "LDS 64 x 128 by rows"),
    # 16-row slices
    (1030, 490, 16, 0.07, 512, "256 by 1 ranked"),
    (430, 1000, 16, 0.04, 672, "128 by 1 ranked"),
    (171, 120, 48, 0.1, 1024, "256 by 4"),
    (171, 170, 48, 0.16, 1024, "256 by 4 ranked"),     # the slices of a block row on one XCD
    (200, 330, 48, 0.05, 608, "128 by 4"),
    (200, 330, 48, 0.08, 608, "128 by 1 ranked"),
    (230, 140, 48, 0.03, 1024, "128 by 2, two tiles"),
    (110, 40, 80, 0.2, 1024, "256 by 4"),             # little X, long rows
    (400, 140, 48, 0.03, 288, "128 by 4"),
])
def test_bsr_forms(dev, mb, nb, blk, density, feat, form):
    """Every form of a launch, with long and empty block rows and columns in any order, against the same sums in fp64 by
    torch, block by block."""
    cfg = _config(mb, nb, blk, density, feat, seed=mb + feat)
    nnzb = len(cfg["indices"])
    dtype, out = ((torch.float16, torch.float32), (torch.bfloat16, torch.bfloat16))[mb & 1]
    assert bsr_form(mb, nb, blk, feat, nnzb, _cus(), out is torch.float32) == form
    a, x = (torch.from_numpy(cfg[k]).to(dev).to(dtype) for k in ("data", "x"))
    y = torch.full((mb * blk * feat,), float("nan"), dtype=out, device=dev)
    d_ptr, d_idx = torch.from_numpy(cfg["indptr"]).to(dev), torch.from_numpy(cfg["indices"]).to(dev)
    ops.build_bsrmm(mb, nb, nnzb, blk, feat, dtype, out)(a.reshape(-1), x.reshape(-1), y, d_ptr, d_idx)
    torch.cuda.synchronize()
    rows_of = torch.repeat_interleave(torch.arange(mb, device=dev), torch.from_numpy(np.diff(cfg["indptr"])).to(dev))
    want = torch.zeros(mb, blk, feat, dtype=torch.float64, device=dev)
    scale = torch.zeros_like(want)
    a64, x64 = a.double(), x.view(nb, blk, feat).double()
    for lo in range(0, nnzb, 2048):
        xb = x64[d_idx[lo:lo + 2048].long()]
        want.index_add_(0, rows_of[lo:lo + 2048], torch.bmm(a64[lo:lo + 2048], xb))
        scale.index_add_(0, rows_of[lo:lo + 2048], torch.bmm(a64[lo:lo + 2048].abs(), xb.abs()))
    # the bound of test_gpu_bsr.py: fp32 sums of exact products, and a rounding of the result
    bound = 1e-5 * scale + (0.0 if out is torch.float32 else RTOL * want.abs()) + 1e-30
    assert bool(((y.view(mb, blk, feat).double() - want).abs() <= bound).all())
