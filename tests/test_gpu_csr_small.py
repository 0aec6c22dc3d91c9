"""CSR products of few rows in one launch: a wavefront's own row and its shares of the workgroup's long rows are one
sequence of up to 64 nonzeros at a time."""
import numpy as np
import pytest

from test_gpu_spmm import _check, _run_csr

pytestmark = pytest.mark.gpu

# eight rows a workgroup: none, some or all of them above 128 nonzeros, of lengths around 64 at a time and around what
# the shares are rounded to (129: the last wavefront has none), in several rounds where the rows are wide
GROUPS = [[0] * 8, [64, 65, 63, 1, 128, 127, 0, 2], [129] * 8, [0, 0, 0, 0, 0, 0, 0, 1025], [513, 0, 160, 64, 161, 0, 1000, 65],
          [128] * 8, [512, 511, 256, 257, 288, 289, 33, 130], [900, 16, 16]]


@pytest.mark.parametrize("feat", [4, 16, 20, 32, 47, 64, 100, 128, 256, 300, 340])
@pytest.mark.parametrize("groups", [GROUPS, GROUPS[-1:], GROUPS[2:3]], ids=["all", "last", "even"])
def test_own_and_shared_rows(dev, feat, groups):
    n = 2500
    rng = np.random.default_rng(feat + len(groups))
    deg = [d for g in groups for d in g]
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    assert indptr[-1] * feat < 3_000_000  # in one launch
    indices = np.concatenate([np.sort(rng.choice(n, d, replace=False)) for d in deg]).astype(np.int32)
    vals = rng.random(len(indices), dtype=np.float32) - 0.4
    x = rng.standard_normal((n, feat), dtype=np.float32)
    got = _run_csr(dev, indptr, indices, vals, x, feat)
    assert np.all(got[np.asarray(deg) == 0] == 0.0)
    _check(got, indptr, indices, vals, x, f"feat={feat}")
    assert np.array_equal(got, _run_csr(dev, indptr, indices, vals, x, feat))  # no atomics: the same bits


@pytest.mark.parametrize("feat", [257, 260, 384, 509, 512])
def test_wide_rows_end_in_two_four_or_eight(dev, feat):
    """Above 256 features the rows of B are in flight eight at a time, and the last ones of up to 64 nonzeros in steps of
    four or two: own rows and shares of long ones that end in each."""
    deg = list(range(0, 19)) + [61, 62, 63, 64, 65, 66, 68, 71, 128, 129, 136, 137, 160, 200, 250, 264]
    n = 700
    rng = np.random.default_rng(feat)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    assert indptr[-1] * feat < 3_000_000
    indices = np.concatenate([np.sort(rng.choice(n, d, replace=False)) for d in deg]).astype(np.int32)
    vals = rng.random(len(indices), dtype=np.float32) - 0.4
    x = rng.standard_normal((n, feat), dtype=np.float32)
    got = _run_csr(dev, indptr, indices, vals, x, feat)
    assert got[0].max() == 0.0 == got[0].min()
    _check(got, indptr, indices, vals, x, f"feat={feat}")
    assert np.array_equal(got, _run_csr(dev, indptr, indices, vals, x, feat))
