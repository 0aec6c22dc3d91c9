"""BSR SpMM with infinities and NaN in X: rows of X that no block names take no part in the result, in any of the kernels
and for odd numbers of 16-column chunks (whose second half of a step is not there); values that are named reach the
features they belong to and no others.  Checked against the fp64 oracle as in test_gpu_bsr.py."""
import numpy as np
import pytest
import torch

from helpers import bsr_f64, bsr_form
from sparsetir_amd import datasets, ops

pytestmark = pytest.mark.gpu

SHAPES = [
    (1024, 60, 16, 0.1, 224, "128 by 1"),     # 16-row slices by a wavefront each
    (1024, 400, 16, 0.01, 512, "256 by 1"),
    (230, 50, 48, 0.05, 352, "128 by 1"),     # three chunks a block
    (230, 140, 48, 0.03, 1024, "128 by 2, two tiles"),
    (180, 50, 48, 0.35, 1024, "256 by 4"),
    (150, 40, 16, 0.2, 1184, "128 by 2, two tiles"),
    (61, 23, 80, 0.3, 480, "128 by 2, two tiles"),
    (3, 200, 16, 0.5, 64, "128 by 8"),
    (260, 60, 16, 0.75, 64, "LDS 64 by 8"),   # 64 features by eight, through LDS
    (9, 90, 32, 0.6, 96, "LDS 64 by 8"),
    (343, 200, 32, 0.01, 736, "128 by 1"),    # 32-row slices by a wavefront each
    (520, 200, 32, 0.01, 800, "128 by 1"),
    (650, 200, 32, 0.005, 512, "256 by 1"),
    (397, 30, 32, 0.2, 416, "128 by 1"),
    (147, 13, 64, 0.3, 2400, "LDS 64 x 256"),  # 64 rows by four wavefronts
    (14, 100, 128, 0.05, 160, "128 by 4"),
]


def _without(cfg, cols):
    """The configuration without the blocks of these block columns, every other block row of an odd length."""
    rows = [r[~np.isin(r, cols)] for r in np.split(cfg["indices"], cfg["indptr"][1:-1])]
    rows = [r[:len(r) - 1] if len(r) and (len(r) + i) % 2 == 0 else r for i, r in enumerate(rows)]
    cfg["indptr"] = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    cfg["indices"] = np.concatenate(rows).astype(np.int32)
    rng = np.random.default_rng(len(rows))
    cfg["data"] = (rng.choice([-1.0, 1.0], (len(cfg["indices"]), cfg["blk"], cfg["blk"])) *
                   rng.uniform(0.01, 0.03, (len(cfg["indices"]), cfg["blk"], cfg["blk"]))).astype(np.float32)
    return cfg


@pytest.mark.parametrize("mb,nb,blk,density,feat,form", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_non_finite_x(dev, mb, nb, blk, density, feat, form, dtype):
    unnamed = np.array([0, 1, nb - 1])
    cfg = _without(datasets.config4(seed=mb + feat, mb=mb, nb=nb, blk=blk, density=density, feat=feat), unnamed)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert bsr_form(mb, nb, blk, feat, len(cfg["indices"]), cus, floats=True) == form
    x = cfg["x"].reshape(nb, blk, feat)
    x[unnamed[0]], x[unnamed[1]], x[unnamed[2]] = np.inf, np.nan, -np.inf
    named = int(cfg["indices"][len(cfg["indices"]) // 2])
    f_inf, f_nan = feat - 1, feat // 2
    x[named, blk // 2, f_inf], x[named, 3, f_nan] = np.inf, np.nan
    a = torch.from_numpy(cfg["data"]).to(dev).to(dtype)
    t = torch.from_numpy(cfg["x"]).to(dev).to(dtype)
    y = torch.zeros(mb * blk * feat, dtype=torch.float32, device=dev)
    ops.build_bsrmm(mb, nb, len(cfg["indices"]), blk, feat, dtype, torch.float32)(
        a.reshape(-1), t.reshape(-1), y, torch.from_numpy(cfg["indptr"]).to(dev), torch.from_numpy(cfg["indices"]).to(dev))
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(mb, blk, feat)
    a32, x32 = a.float().cpu().numpy(), t.float().cpu().numpy()
    has = np.array([named in r for r in np.split(cfg["indices"], cfg["indptr"][1:-1])])
    assert has.any() and not has.all()
    assert np.isinf(got[has][:, :, f_inf]).all() and np.isnan(got[has][:, :, f_nan]).all()
    got[np.ix_(has, np.arange(blk), [f_inf, f_nan])] = 0.0
    assert np.isfinite(got).all()
    # the finite rest: the same with zeros where the values are not finite
    x32 = np.where(np.isfinite(x32), x32, 0.0).astype(np.float32)
    want = bsr_f64(cfg["indptr"], cfg["indices"], a32, x32, mb, nb, blk).reshape(mb, blk, feat)
    scale = bsr_f64(cfg["indptr"], cfg["indices"], np.abs(a32), np.abs(x32), mb, nb, blk).reshape(mb, blk, feat)
    want[np.ix_(has, np.arange(blk), [f_inf, f_nan])] = 0.0
    assert np.all(np.abs(got - want) <= 1e-5 * scale + 1e-30)  # fp32 sums of exact products, as in test_gpu_bsr.py
