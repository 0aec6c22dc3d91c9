"""CSR products by workgroups of equal work: one launch, rows cut between workgroups and lane groups."""
import ctypes

import numpy as np
import pytest
import torch

from sparsetir_amd import _lib, ops
from test_gpu_spmm import _check

pytestmark = pytest.mark.gpu


def _matrix(rng, m, n, lengths, most):
    """Row degrees 0 to `most` with the given lengths at the front, in the middle and at the end."""
    deg = rng.integers(0, most + 1, m)
    deg[m // 4:m // 3] = 0  # a run of empty rows
    for k, d in enumerate(lengths):
        deg[k] = deg[m // 2 + 3 * k] = deg[m - 1 - 2 * k] = d
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    return deg, indptr, rng.integers(0, n, indptr[-1]).astype(np.int32)


@pytest.mark.parametrize("feat", [4, 13, 16, 32, 47, 64, 100, 128, 256, 300, 512])
@pytest.mark.parametrize("m,most", [(8192, 3), (9001, 24), (40003, 14)])
def test_rows_across_workgroups(dev, feat, m, most):
    """Rows around the length that is never cut, rows over many workgroups next to each other, empty
    rows, arrays longer than the last row pointer; the same bits again, on another stream and recorded."""
    rng = np.random.default_rng(feat + m)
    n = 5000
    deg, indptr, indices = _matrix(rng, m, n, [0, 128, 129, 127, 1, 4000, 3000, 512, 640, 0, 257, 130], most)
    spare = 7
    indices = np.concatenate([indices, np.zeros(spare, np.int32)])
    vals = rng.random(len(indices), dtype=np.float32) - 0.4
    x = rng.standard_normal((n, feat), dtype=np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    args = (t(vals), t(x.ravel()))
    tail = (t(indptr), t(indices))
    f = ops.build_csrmm(m, n, feat, len(indices))
    c = [torch.full((m * feat,), float("nan"), device=dev) for _ in range(3)]
    f(*args, c[0], *tail)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        f(*args, c[1], *tail)
        f(*args, c[1], *tail)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        f(*args, c[2], *tail)
    for _ in range(3):
        c[2].fill_(float("nan"))
        graph.replay()
        f(*args, c[1], *tail)
        torch.cuda.synchronize()
        assert torch.equal(c[0], c[1]) and torch.equal(c[0], c[2])
    got = c[0].cpu().numpy().reshape(m, feat)
    assert np.all(got[deg == 0] == 0.0)
    _check(got, indptr, indices[:-spare], vals[:-spare], x, f"m={m} feat={feat}")


@pytest.mark.parametrize("feat,m,most", [(128, 9001, 300), (192, 9001, 200), (256, 40003, 34), (320, 9001, 120),
                                         (512, 9001, 80)])
def test_feature_slices(dev, feat, m, most):
    """Products large enough for slices of 64 features, two to eight of them."""
    test_rows_across_workgroups(dev, feat, m, most)


@pytest.mark.parametrize("feat,m,most", [(8, 25001, 40), (13, 60003, 62), (8, 120001, 64), (300, 60003, 35),
                                         (260, 60003, 58), (32, 60003, 75), (47, 60003, 75), (100, 60003, 75)])
def test_workgroups_by_size(dev, feat, m, most):
    """Hundreds of entries a workgroup, as many as it holds, and several turns of fewer."""
    test_rows_across_workgroups(dev, feat, m, most)


@pytest.mark.parametrize("feat", [4, 47, 64, 256])
def test_only_the_counters_are_cleared(dev, feat):
    """What is in the workspace behind the counters does not matter, and the counters are zero again afterwards."""
    rng = np.random.default_rng(feat)
    m, n = 9001, 3000
    deg, indptr, indices = _matrix(rng, m, n, [129, 4000, 1000], 30)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    p = lambda a: ctypes.c_void_p(a.data_ptr())
    vals = rng.random(len(indices), dtype=np.float32) - np.float32(0.4)
    x = rng.standard_normal((n, feat), dtype=np.float32)
    lib = _lib.lib()
    size = (m, n, feat, len(indices))
    clear = lib.stir_csr_spmm_workspace_clear_bytes(*size)
    ws = torch.full((lib.stir_csr_spmm_workspace_bytes(*size),), 255, dtype=torch.uint8, device=dev)
    ws[:clear] = 0
    args = [t(vals), t(x.ravel()), torch.full((m * feat,), float("nan"), device=dev), t(indptr), t(indices), ws]
    for _ in range(2):
        _lib.check(lib.stir_csr_spmm_f32_workspace(*size, *[p(a) for a in args],
                                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        assert not ws[:clear].any()
        _check(args[2].cpu().numpy().reshape(m, feat), indptr, indices, vals, x, f"feat={feat}")


@pytest.mark.parametrize("feat,hub", [(4, 1_200_000), (16, 1_000_003), (256, 400_001), (300, 300_000)])
def test_a_row_over_thousands_of_workgroups(dev, feat, hub):
    """The workgroup that finishes last adds hundreds of partial rows per lane group, a number that is no multiple of
    those it requests at a time; the same bits again."""
    rng = np.random.default_rng(feat)
    m, n = 12000, 20000
    deg = rng.integers(0, 4, m)
    deg[m // 3] = hub
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    indices = rng.integers(0, n, indptr[-1]).astype(np.int32)
    vals = rng.random(len(indices), dtype=np.float32) - np.float32(0.4)
    x = rng.standard_normal((n, feat), dtype=np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    f = ops.build_csrmm(m, n, feat, len(indices))
    c = [torch.full((m * feat,), float("nan"), device=dev) for _ in range(2)]
    args = [t(vals), t(x.ravel())], [t(indptr), t(indices)]
    for y in c:
        f(*args[0], y, *args[1])
    torch.cuda.synchronize()
    assert torch.equal(*c)
    _check(c[0].cpu().numpy().reshape(m, feat), indptr, indices, vals, x, f"feat={feat} hub={hub}")


def test_more_streams_than_workspaces(dev):
    """An operator keeps workspaces for four streams: a fifth takes the place of the one used longest ago, whose
    kernels may still be running."""
    rng = np.random.default_rng(6)
    m, n, feat = 20000, 5000, 64
    deg, indptr, indices = _matrix(rng, m, n, [3000, 700, 129], 20)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    args = [t(rng.random(len(indices), dtype=np.float32)), t(rng.standard_normal(n * feat).astype(np.float32))]
    tail = [t(indptr), t(indices)]
    f = ops.build_csrmm(m, n, feat, len(indices))
    want = torch.empty(m * feat, device=dev)
    f(*args, want, *tail)
    streams = [torch.cuda.Stream() for _ in range(6)]
    out = [torch.full((m * feat,), float("nan"), device=dev) for _ in range(60)]
    torch.cuda.synchronize()
    for k, c in enumerate(out):
        with torch.cuda.stream(streams[(k * 5 + k // 7) % 6]):
            f(*args, c, *tail)
    torch.cuda.synchronize()
    assert all(torch.equal(c, want) for c in out)
