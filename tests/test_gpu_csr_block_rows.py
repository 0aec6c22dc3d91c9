"""CSR products small enough for one launch: rows above 128 nonzeros are shared by a workgroup."""
import numpy as np
import pytest

from test_gpu_spmm import _check, _run_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("feat", [4, 16, 47, 64, 128, 200, 512])
@pytest.mark.parametrize("m", [1, 9, 1003, 20001])
def test_hub_rows_in_one_launch(dev, feat, m):
    """Row lengths around the limit and around what a wavefront's stretch of a row is rounded to, several
    long rows in one workgroup, the last row long; m above 20000: a lane group per row."""
    n = 3000
    rng = np.random.default_rng(feat + m)
    nnz_most = 5_900_000 // feat
    deg = rng.integers(0, 3, m) if m * feat < 2_000_000 else (rng.random(m) < 0.1).astype(np.int64)
    for k, d in enumerate([129, 128, 0, 2049, 127, 256, 135, 1, 700]):
        deg[m - 1 - k if k < m else 0] = d if deg.sum() + d < nnz_most else 2
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    assert indptr[-1] * feat < 6_000_000
    indices = np.concatenate([np.sort(rng.choice(n, d, replace=False)) for d in deg]).astype(np.int32)
    vals = rng.random(len(indices), dtype=np.float32) - 0.4
    x = rng.standard_normal((n, feat), dtype=np.float32)
    got = _run_csr(dev, indptr, indices, vals, x, feat)
    assert np.all(got[deg == 0] == 0.0)
    _check(got, indptr, indices, vals, x, f"m={m} feat={feat}")
