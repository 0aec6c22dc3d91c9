"""hyb SpMM in feature slices: launches with few wavefronts (slices of 32 features) and with enough of them (64, or
one piece), widths whose last slice is ragged, narrower than a chunk of four features, or that are not cut.
Checked against the fp64 product as in test_gpu_spmm.py; one partition stores, two add."""
import numpy as np
import pytest
import scipy.sparse as sp

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
