"""BSR SpMM where X does not fit an L2: slices taken in order of their length or as they come, by a wavefront each or not.
Empty block rows, a few with more blocks than a wavefront has lanes, block columns in any order, ragged feature
tiles, arrays that start at an odd element.  Checked against the fp64 oracle as in test_gpu_bsr.py."""
import numpy as np
import pytest
import torch

from sparsetir_amd import datasets, ops
from test_gpu_bsr import _check

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
    (1024, 193, 32, 0.004, 224),   # 32-row slices by a wavefront each, 128 features: as they come
    (1030, 200, 32, 0.004, 256),
    (430, 200, 32, 0.004, 288),    # the last of three tiles with 32
    (220, 200, 32, 0.01, 672),
    (150, 200, 32, 0.02, 1056),    # five tiles of 256 would be
    (150, 70, 96, 0.04, 352),
    (170, 260, 32, 0.02, 992),     # too few for 256 features each
    (650, 200, 32, 0.005, 512),    # two full tiles of 256
    (70, 70, 96, 0.04, 1440),      # three slices per block row, 5.6 feature tiles; few steps: as they come
    (72, 90, 96, 0.07, 1440),      # ranked, six feature tiles over eight XCDs: the slices of a block row on one of them
    (257, 250, 32, 0.01, 832),     # ranked, the last of four feature tiles with 64
    (257, 200, 32, 0.08, 832),     # less of X, 16 steps a slice
    (343, 200, 32, 0.01, 736),
    (20, 200, 64, 0.03, 96),       # eight wavefronts
    (12, 100, 128, 0.05, 160),
    (14, 100, 128, 0.05, 160),
    (60, 200, 64, 0.03, 416),      # four wavefronts per 64 rows, ranked
    (33, 100, 128, 0.05, 544),     # too few block rows to deal them to XCDs
    (36, 100, 128, 0.05, 544),     # block rows dealt to XCDs
    (40, 20, 64, 0.1, 1056),       # few workgroups: 128 features each
    (83, 20, 64, 0.1, 1056),       # as many as take 256 features each, the last with 32
    (1, 6200, 32, 0.001, 64),
    (1030, 90, 16, 0.02, 224),     # 16-row slices by a wavefront each: plain order
    (1024, 400, 16, 0.004, 512),   # 256 features
    (512, 520, 16, 0.004, 1024),   # ranked, 256 features
    (700, 400, 16, 0.004, 320),    # 128 features, an odd number of blocks
    (410, 1000, 16, 0.004, 544),   # ranked, 128 features
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


def test_bsr_ranked_blocks_of_three(dev):
    """16-row slices of blocks of 48 in the ranked order, more than 64 blocks in a row, an odd number of chunks in most."""
    test_bsr_ranked_edges(dev, 171, 170, 48, 0.07, 1024, torch.float16, 1)
