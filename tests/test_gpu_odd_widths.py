"""Feature widths that are no multiple of four: the last lane of a row loads four features that end
at the row's end, some of them its neighbour's (CSR, hyb and SDDMM kernels).  Widths around every
lane-group size; the dense operands end with the array, so a load past a row's end would leave it."""
import numpy as np
import pytest

from helpers import random_csr, sddmm_f64
from test_gpu_sddmm import _run as run_sddmm
from test_gpu_spmm import RTOL, _check, _hyb_as_coo, _hyb_setup, _run_csr, _run_hyb

pytestmark = pytest.mark.gpu
WIDTHS = [5, 6, 7, 15, 17, 31, 33, 47, 63, 65, 127, 129, 255, 257, 259, 510, 511, 513]


@pytest.mark.parametrize("feat", WIDTHS)
@pytest.mark.parametrize("hubs", [False, True])
def test_csr_odd_width(dev, feat, hubs):
    """hubs: enough nonzeros for the launch that adds up long rows with atomics."""
    m, n = 1501, 6000
    rng = np.random.default_rng(feat)
    deg = rng.integers(0, 40, m)
    deg[[0, 7, m - 1]] = [700, 65, 3]
    if hubs:
        deg[10:70] = 5000
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    assert (indptr[-1] >= 1 << 18) == hubs
    indices = np.concatenate([np.sort(rng.choice(n, d, replace=False)) for d in deg]).astype(np.int32)
    indices[-1] = n - 1  # the last row of X
    vals = rng.random(len(indices), dtype=np.float32) - 0.3
    x = rng.standard_normal((n, feat), dtype=np.float32)
    got = _run_csr(dev, indptr, indices, vals, x, feat)
    assert np.all(got[deg == 0] == 0.0)
    _check(got, indptr, indices, vals, x, f"feat={feat}")


@pytest.mark.parametrize("feat", WIDTHS)
@pytest.mark.parametrize("parts,buckets", [(1, [1, 2, 4, 8, 16, 32, 64, 128]), (2, [1, 3, 8, 300]), (6, [1, 4, 16])])
def test_hyb_odd_width(dev, feat, parts, buckets):
    """One partition stores, two add in phases without atomics, six run as merged rows."""
    m = n = 1003
    indptr, indices = random_csr(m, n, 20000, feat, skew=1.2)
    triples = _hyb_setup(dev, indptr, indices, m, n, parts, buckets, weighted=True, seed=feat)
    x = np.random.default_rng(feat).standard_normal((n, feat), dtype=np.float32)
    got, _ = _run_hyb(dev, m, n, feat, parts, buckets, triples, x)
    import scipy.sparse as sp
    r, c, v = _hyb_as_coo(triples)
    a = sp.csr_matrix((v.astype(np.float64), (r, c)), shape=(m, n))
    assert np.all(np.abs(got - a @ x.astype(np.float64)) <= RTOL * (a @ np.abs(x).astype(np.float64)) + 1e-30)


@pytest.mark.parametrize("feat", WIDTHS)
def test_sddmm_odd_width(dev, feat):
    m, n = 300, 401
    indptr, indices = random_csr(m, n, 5003, feat, skew=1.1)
    indices[-1] = n - 1
    rng = np.random.default_rng(feat)
    a = rng.standard_normal((m, feat), dtype=np.float32)
    b = rng.standard_normal((n, feat), dtype=np.float32)
    got, _ = run_sddmm(dev, indptr, indices, a, b, feat)
    rows = np.repeat(np.arange(m), np.diff(indptr))
    scale = np.einsum("ek,ek->e", np.abs(a).astype(np.float64)[rows], np.abs(b).astype(np.float64)[indices])
    assert np.all(np.abs(got - sddmm_f64(indptr, indices, a, b)) <= RTOL * scale + 1e-30)
