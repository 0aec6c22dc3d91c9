"""Condensed SpMM with a plan: row tiles around the length that is cut into pieces (32 steps of 32 columns),
tiles with fewer steps than wavefronts and without any, an output that does not begin on a 16-byte boundary, and
launches with enough tiles for wide units (128 features) and for two wavefronts a unit."""
import numpy as np
import pytest
import torch

import sparsetir_amd as st
from sparsetir_amd import ops
from test_gpu_tcspmm import _run

pytestmark = pytest.mark.gpu


def _rows(rng, n, deg):
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    return indptr, np.concatenate([np.sort(rng.choice(n, d, replace=False)) for d in deg]).astype(np.int32)


@pytest.mark.parametrize("t", [8, 16, 32])
@pytest.mark.parametrize("feat", [32, 64, 96, 160, 256])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_tile_lengths(dev, t, feat, out_dtype):
    rng = np.random.default_rng(feat + t)
    n = 3001
    cols = [1, 16, 17, 0, 32, 33, 128, 129, 1008, 1024, 1025, 1041, 2048, 2049, 0, 3001, 160]
    deg = np.zeros(len(cols) * t - 3, np.int64)
    deg[np.arange(len(cols)) * t + rng.integers(0, t - 3, len(cols))] = cols
    indptr, indices = _rows(rng, n, deg)
    _run(dev, indptr, indices, n, feat, False, out_dtype, t=t)


@pytest.mark.parametrize("t,tiles,feat", [(8, 8200, 32), (8, 8200, 64), (16, 3100, 128), (16, 8200, 96), (32, 2700, 192), (16, 5100, 128)])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_many_tiles(dev, t, tiles, feat, out_dtype):
    rng = np.random.default_rng(feat)
    deg = rng.integers(0, 5, tiles * t)
    deg[[3, tiles * t - 1]] = 1500
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    n = 12000
    indices = ((np.arange(indptr[-1]) * 7 + rng.integers(0, 7, indptr[-1])) % n).astype(np.int32)  # distinct in a row
    _run(dev, indptr, indices, n, feat, False, out_dtype, t=t)


@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_output_between_boundaries(dev, out_dtype):
    rng = np.random.default_rng(5)
    n, feat, t = 1500, 64, 16
    indptr, indices = _rows(rng, n, np.array([3, 0, 1400, 20] * 20))
    gptr, tiles, mask = st.condense(indptr, indices, t, 16)
    td = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev)
    mb = len(gptr) - 1
    args = [td(mask.astype(np.float16).ravel()), td(rng.standard_normal(n * feat).astype(np.float16))]
    tail = [td(gptr), td(tiles.ravel())]
    f = ops.build_tcspmm(mb, tiles.shape[0], feat, t, 16, n, out_dtype)
    c = torch.full((mb * t * feat,), float("nan"), dtype=out_dtype, device=dev)
    shifted = torch.full((mb * t * feat + 1,), float("nan"), dtype=out_dtype, device=dev)
    f(*args, c, *tail)
    f(*args, shifted[1:], *tail)
    torch.cuda.synchronize()
    assert torch.equal(c, shifted[1:])


@pytest.mark.parametrize("t,feat,out_dtype", [(8, 32, torch.float32), (16, 96, torch.float16), (32, 64, torch.float16)])
def test_long_tiles_left_whole(dev, t, feat, out_dtype):
    """Enough steps in all for tiles of more than 32 to stay whole: around that length and around the one from which
    they are cut, the 2048th part of all steps."""
    rng = np.random.default_rng(t)
    steps = np.array([32, 33, 40, 51, 52, 102, 103, 66, 129, 200, 1, 0] * 130)
    assert steps.sum() // 2048 == 51
    rng.shuffle(steps)
    deg = np.zeros(len(steps) * t, np.int64)
    deg[np.arange(len(steps)) * t + rng.integers(0, t, len(steps))] = steps * 32 - rng.integers(0, 16, len(steps)) * (steps > 0)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    n = 9001
    indices = ((np.arange(indptr[-1]) * 7 + 3) % n).astype(np.int32)  # distinct in a row: 7 * 6400 steps, n is no multiple of 7
    _run(dev, indptr, indices, n, feat, False, out_dtype, t=t)
