"""The CSR product without a workspace: one launch below a size, a second one for long rows above it."""
import ctypes

import numpy as np
import pytest
import torch

import test_gpu_odd_widths
import test_gpu_spmm
from sparsetir_amd import _lib
from test_gpu_spmm import _check

pytestmark = pytest.mark.gpu

FEW = 1 << 18  # nonzeros; below, two launches from 20 M products on, from there on from 6 M


def _run(dev, m, n, feat, indptr, indices, vals, x):
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    p = lambda a: ctypes.c_void_p(a.data_ptr())
    arrays = [t(vals), t(x.ravel()), torch.full((m * feat,), float("nan"), device=dev), t(indptr), t(indices)]
    _lib.check(_lib.lib().stir_csr_spmm_f32(m, n, feat, len(indices), *[p(a) for a in arrays],
                                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    return arrays[2].cpu().numpy().reshape(m, feat)


@pytest.mark.parametrize("feat,nnz", [(77, 20_000_000 // 77), (77, 20_000_000 // 77 + 1), (100, 199_999), (100, 200_000),
                                      (512, 39_063), (24, FEW - 1), (24, FEW), (23, FEW), (128, FEW)])
@pytest.mark.parametrize("m", [90, 3000, 60000])
def test_both_sides_of_the_lines(dev, m, feat, nnz):
    """Row lengths around the longest that stays with a wavefront (64 to 256, by the average row), empty rows and
    rows of many pieces, at sizes next to where the second launch begins."""
    n = 5000
    rng = np.random.default_rng(feat + nnz + m)
    average = nnz // m
    ordinary = min(256, max(64, 4 * average)) if nnz < FEW else 64
    deg = np.zeros(m, np.int64)
    for k, d in enumerate([ordinary, ordinary + 1, 64, 65, 0, 128, 129, 4000, 257, 0, 2049]):
        deg[m - 1 - 2 * k] = d
    free = np.flatnonzero(deg == 0)[:-3]
    deg += np.bincount(rng.choice(free, nnz - deg.sum()), minlength=m)
    assert deg.sum() == nnz
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    indices = rng.integers(0, n, nnz).astype(np.int32)
    vals = rng.random(nnz, dtype=np.float32) - np.float32(0.4)
    x = rng.standard_normal((n, feat), dtype=np.float32)
    got = _run(dev, m, n, feat, indptr, indices, vals, x)
    assert np.all(got[deg == 0] == 0.0)
    _check(got, indptr, indices, vals, x, f"m={m} feat={feat} nnz={nnz}")


@pytest.mark.parametrize("feat", [3, 4, 16, 47, 64, 128, 200, 512, 600])
@pytest.mark.parametrize("m", [1, 9, 1003, 20001])
def test_one_launch(dev, feat, m):
    """Every lane group width with a wavefront per row and (above 20000 rows) a lane group per row; hub rows that the
    workgroup shares, several of them in one workgroup, at lengths around the limit of 128 and far above it."""
    n = 3000
    rng = np.random.default_rng(feat + m)
    deg = rng.integers(0, 3, m) if m * feat < 2_000_000 else (rng.random(m) < 0.1).astype(np.int64)
    for k, d in enumerate([129, 128, 0, 2049, 127, 256, 135, 1, 700]):
        deg[m - 1 - k if k < m else 0] = d
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    assert indptr[-1] * feat < 20_000_000 and indptr[-1] < FEW
    indices = np.concatenate([np.sort(rng.choice(n, d, replace=False)) for d in deg]).astype(np.int32)
    vals = rng.random(len(indices), dtype=np.float32) - np.float32(0.4)
    x = rng.standard_normal((n, feat), dtype=np.float32)
    got = _run(dev, m, n, feat, indptr, indices, vals, x)
    assert np.all(got[deg == 0] == 0.0)
    _check(got, indptr, indices, vals, x, f"m={m} feat={feat}")


# The operator takes the products of these tests through its workspace: here they go the way without one that they
# were written for.
@pytest.fixture
def stateless(monkeypatch):
    def run_csr(dev, indptr, indices, vals, x, feat):
        return _run(dev, len(indptr) - 1, x.shape[0], feat, indptr, indices, vals, x)

    monkeypatch.setattr(test_gpu_spmm, "_run_csr", run_csr)
    monkeypatch.setattr(test_gpu_odd_widths, "_run_csr", run_csr)


@pytest.mark.parametrize("feat", [32, 128, 512, 96])
def test_hub_rows_in_pieces(dev, stateless, feat):
    test_gpu_spmm.test_csr_spmm_hub_rows_are_split(dev, feat)


@pytest.mark.parametrize("feat", [4, 8, 12, 32, 40, 64, 128])
@pytest.mark.parametrize("split", [False, True])
def test_lane_group_per_row(dev, stateless, feat, split):
    test_gpu_spmm.test_csr_spmm_lane_group_per_row(dev, feat, split)


@pytest.mark.parametrize("feat", test_gpu_odd_widths.WIDTHS)
@pytest.mark.parametrize("hubs", [False, True])
def test_odd_widths(dev, stateless, feat, hubs):
    test_gpu_odd_widths.test_csr_odd_width(dev, feat, hubs)
