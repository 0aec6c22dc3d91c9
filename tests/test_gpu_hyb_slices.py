"""hyb SpMM in feature slices: launches with few wavefronts (slices of 32 features) and with enough of them (64, or
one piece), widths whose last slice is ragged, narrower than a chunk of four features, or that are not cut.
Checked against the fp64 product as in test_gpu_spmm.py; one partition stores, two add."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from helpers import random_csr
from test_gpu_spmm import RTOL, _hyb_as_coo, _hyb_setup, _run_hyb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz,feat", [
    (9000, 34), (9000, 66), (9000, 98), (9000, 131), (9000, 160), (9000, 196), (9000, 255),
    (400000, 68), (400000, 96), (400000, 128), (400000, 160), (400000, 224), (400000, 256), (400000, 257),
])
@pytest.mark.parametrize("parts,buckets", [(1, [1, 2, 4, 8, 16, 32, 64, 128]), (2, [1, 4, 32, 100])])
def test_hyb_feature_slices(dev, nnz, feat, parts, buckets):
    m, n = 2999, 3001
    indptr, indices = random_csr(m, n, nnz, feat, skew=1.1)
    triples = _hyb_setup(dev, indptr, indices, m, n, parts, buckets, weighted=True, seed=feat)
    x = np.random.default_rng(feat).standard_normal((n, feat), dtype=np.float32)
    got, _ = _run_hyb(dev, m, n, feat, parts, buckets, triples, x)
    r, c, v = _hyb_as_coo(triples)
    a = sp.csr_matrix((v.astype(np.float64), (r, c)), shape=(m, n))
    assert np.all(np.abs(got - a @ x.astype(np.float64)) <= RTOL * (a @ np.abs(x).astype(np.float64)) + 1e-30)


@pytest.mark.parametrize("feat", [8, 31, 67, 129, 192, 255, 300])
@pytest.mark.parametrize("parts", [2, 5])
def test_hyb_merged_rows_of_equal_work(dev, feat, parts):
    """Column partitions whose rows run merged, a row over many workgroups among them; the product is added."""
    m, n = 8500, 4000
    rng = np.random.default_rng(feat + parts)
    deg = rng.integers(0, 30, m)
    deg[[0, 77, m - 1]] = [3900, 129, 700]
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    indices = np.concatenate([np.sort(rng.choice(n, d, replace=False)) for d in deg]).astype(np.int32)
    buckets = [1, 2, 4, 8, 16, 32]
    triples = _hyb_setup(dev, indptr, indices, m, n, parts, buckets, weighted=True, seed=feat)
    x = rng.standard_normal((n, feat), dtype=np.float32)
    got, (f, args) = _run_hyb(dev, m, n, feat, parts, buckets, triples, x)
    r, c, v = _hyb_as_coo(triples)
    a = sp.csr_matrix((v.astype(np.float64), (r, c)), shape=(m, n))
    want, bound = a @ x.astype(np.float64), RTOL * (a @ np.abs(x).astype(np.float64)) + 1e-30
    assert np.all(np.abs(got - want) <= bound)
    y = torch.from_numpy(got.ravel().copy()).to(dev)
    f(torch.from_numpy(x.ravel()).to(dev), y, *args)  # the operator adds to what is there
    torch.cuda.synchronize()
    assert np.all(np.abs(y.cpu().numpy().reshape(m, feat) - 2 * want) <= 3 * bound)


@pytest.mark.parametrize("m,nnz,feat", [
    (70000, 900000, 96), (70000, 900000, 128), (70000, 900000, 132), (30000, 900000, 132), (70000, 900000, 192),
    (60000, 900000, 192), (100000, 1500000, 80)])
def test_hyb_between_phases_and_merged_rows(dev, m, nnz, feat):
    """Two partitions above a million slots: merged rows up to 127 features (not with more slots) and, above 128, with
    short rows unless the phases run in slices; phases else."""
    indptr, indices = random_csr(m, m, nnz, feat, skew=1.0)
    buckets = [1, 2, 4, 8, 16, 32]
    triples = _hyb_setup(dev, indptr, indices, m, m, 2, buckets, weighted=True, seed=feat)
    x = np.random.default_rng(feat).standard_normal((m, feat), dtype=np.float32)
    got, (f, args) = _run_hyb(dev, m, m, feat, 2, buckets, triples, x)
    r, c, v = _hyb_as_coo(triples)
    a = sp.csr_matrix((v.astype(np.float64), (r, c)), shape=(m, m))
    want, bound = a @ x.astype(np.float64), RTOL * (a @ np.abs(x).astype(np.float64)) + 1e-30
    assert np.all(np.abs(got - want) <= bound)
    y = torch.from_numpy(got.ravel().copy()).to(dev)
    f(torch.from_numpy(x.ravel()).to(dev), y, *args)  # the operator adds to what is there
    torch.cuda.synchronize()
    assert np.all(np.abs(y.cpu().numpy().reshape(m, feat) - 2 * want) <= 3 * bound)
