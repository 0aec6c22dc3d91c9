"""BSR SpMM at the edges of its launch rules: few workgroups (steps of a block row taken in turn by the wavefronts of a
workgroup, more than 64 blocks in a row, rows with fewer steps than wavefronts and empty ones), blocks of an odd
multiple of 16 with an odd number of column chunks, and feature-tile counts that are not multiples of the
eight XCDs.  Checked against the fp64 oracle as in test_gpu_bsr.py."""
import pytest
import torch

from sparsetir_amd import datasets
from test_gpu_bsr import _check, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mb,nb,blk,density,feat", [
    (1, 1, 16, 1.0, 32),          # one workgroup, one step, half of its features
    (5, 90, 32, 0.95, 96),        # more blocks in a row than lanes
    (7, 9, 48, 0.4, 224),         # odd numbers of chunks, 16-row slices
    (3, 200, 16, 0.5, 64),
    (4, 3, 128, 0.6, 352),
    (160, 60, 32, 0.6, 256),      # more workgroups than are resident at once, long block rows
    (300, 120, 16, 0.5, 256),
    (150, 40, 16, 0.2, 1184),     # 16-row slices: large launches, ragged feature tiles
    (61, 23, 80, 0.3, 480),
    (400, 20, 16, 0.3, 224),
    (397, 30, 32, 0.2, 416),      # 32-row slices, feature tiles 4, 5, 9 and 3
    (301, 17, 32, 0.3, 608),
    (143, 11, 32, 0.4, 1120),
    (147, 13, 64, 0.3, 2400),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_bsr_launch_edges(dev, mb, nb, blk, density, feat, dtype):
    cfg = datasets.config4(seed=mb + feat, mb=mb, nb=nb, blk=blk, density=density, feat=feat)
    out = torch.float32 if (mb & 1) == (dtype is torch.float16) else None
    got, a32, x32 = _run(dev, cfg, dtype, out)
    _check(got, cfg, a32, x32, out is None, f"{mb}x{nb} blk {blk} feat {feat} {dtype}")
