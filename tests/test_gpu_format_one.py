"""column_part_hyb for one column partition on the device: the short path with its own sizing, scan and
placement kernels, against the host routine (which is pinned to the oracle)."""
import ctypes

import numpy as np
import pytest
import torch

import sparsetir_amd as st
from sparsetir_amd import _lib
from sparsetir_amd._lib import SparseTIRError

pytestmark = pytest.mark.gpu


def _csr(m, n, degrees, seed):
    rng = np.random.default_rng(seed)
    indptr = np.concatenate([[0], np.cumsum(degrees)]).astype(np.int32)
    return indptr, rng.integers(0, n, indptr[-1]).astype(np.int32)


def _compare(dev, m, n, indptr, indices, buckets):
    t = lambda a: torch.from_numpy(a).to(dev)
    vals = np.random.default_rng(1).random(len(indices), dtype=np.float32) + 0.5
    rows, cols, mask, avals = st.column_part_hyb(m, n, t(indptr), t(indices), 1, buckets, t(vals))
    rows0, cols0, mask0 = st.column_part_hyb(m, n, t(indptr), t(indices), 1, buckets)
    h_rows, h_cols, h_mask = st.column_part_hyb(m, n, indptr, indices, 1, buckets)
    # where a nonzero lies: its row's slots in order, so the values follow from a walk over the host result
    at = indptr[:-1].astype(np.int64).copy()
    for b in range(len(buckets)):
        for got, got0, want in ((rows, rows0, h_rows), (cols, cols0, h_cols), (mask, mask0, h_mask)):
            assert got[0][b].shape == want[0][b].shape and got[0][b].dtype == torch.int32
            assert np.array_equal(got[0][b].cpu().numpy(), want[0][b]), (b, buckets)
            assert np.array_equal(got0[0][b].cpu().numpy(), want[0][b]), (b, buckets)
        want_a = np.zeros(h_mask[0][b].shape, np.float32)
        for r, row in enumerate(h_rows[0][b]):
            k = int(h_mask[0][b][r].sum())
            want_a[r, :k] = vals[at[row]:at[row] + k]
            at[row] += k
        assert np.array_equal(avals[0][b].cpu().numpy(), want_a)


@pytest.mark.parametrize("m", [1, 63, 64, 65, 255, 257, 1025])
@pytest.mark.parametrize("buckets", [[1], [1, 2, 4, 8, 16, 32], [3, 7], list(range(1, 33))])
def test_matches_host(dev, m, buckets):
    rng = np.random.default_rng(m)
    deg = rng.integers(0, 12, m)
    deg[m // 2] = 1500  # more than a tile of nonzeros in one row
    deg[m - 1] = 0
    _compare(dev, m, 900, *_csr(m, 900, deg, m), buckets)


@pytest.mark.parametrize("m", [64 * 256, 64 * 256 + 1, 1 << 20, (1 << 20) + 1])
def test_around_the_changes_of_kernel(dev, m):
    """The most rows whose counts the counting kernel scans itself, the most whose ids are written with the columns,
    and one more; rows of many ELL rows and runs of empty ones."""
    rng = np.random.default_rng(m)
    deg = rng.integers(0, 9 if m < 1 << 20 else 3, m)
    deg[[0, m // 3, m - 1]] = [700, 20000, 40]
    deg[m // 2:m // 2 + 300] = 0
    _compare(dev, m, 5000, *_csr(m, 5000, deg, m), [1, 2, 4, 8, 16, 32])


def test_long_runs_of_empty_rows(dev):
    """More rows around a tile's nonzeros than the row window holds: the per-nonzero search."""
    deg = np.zeros(5000, np.int64)
    deg[[0, 700, 2999, 4999]] = [3, 1, 40, 2]
    _compare(dev, 5000, 64, *_csr(5000, 64, deg, 0), [1, 2, 4])


def test_more_rows_than_one_scan(dev):
    """Above a million rows the counts are scanned by three kernels."""
    m = 64 * 16384 + 65
    deg = np.zeros(m, np.int64)
    deg[::97] = 2
    deg[[5, m - 1]] = [9, 4]
    indptr, indices = _csr(m, 50, deg, 3)
    t = lambda a: torch.from_numpy(a).to(dev)
    got = st.column_part_hyb(m, 50, t(indptr), t(indices), 1, [1, 2, 4])
    want = st.column_part_hyb(m, 50, indptr, indices, 1, [1, 2, 4])
    for g, w in zip(got, want):
        for b in range(3):
            assert np.array_equal(g[0][b].cpu().numpy(), w[0][b])


def test_refuses_what_the_arrays_cannot_mean(dev):
    t = lambda a: torch.tensor(a, dtype=torch.int32, device=dev)
    ok = st.column_part_hyb(3, 4, t([0, 1, 1, 2]), t([3, 0]), 1, [1, 2])
    assert ok[0][0][0].tolist() == [0, 2]
    for indptr, indices, msg in (([0, 1, 1, 3], [3, 0], "row pointer"), ([0, 2, 1, 2], [3, 0], "row pointer"),
                                 ([-1, 1, 1, 2], [3, 0], "row pointer"), ([0, 1, 1, 2], [4, 0], "outside"),
                                 ([0, 1, 1, 2], [3, -1], "outside")):
        with pytest.raises(SparseTIRError, match=msg):
            st.column_part_hyb(3, 4, t(indptr), t(indices), 1, [1, 2])
    m = 9000  # what is wrong lies with a later group of rows, a later workgroup of the check
    indptr = torch.arange(0, 10 * m + 1, 10, dtype=torch.int32, device=dev)
    indices = torch.zeros(10 * m, dtype=torch.int32, device=dev)
    indices[70001] = 4
    with pytest.raises(SparseTIRError, match="outside"):
        st.column_part_hyb(m, 4, indptr, indices, 1, [1, 2])
    indices[70001] = 0
    indptr[8500] = 0
    with pytest.raises(SparseTIRError, match="row pointer"):
        st.column_part_hyb(m, 4, indptr, indices, 1, [1, 2])
    empty = st.column_part_hyb(2, 4, t([0, 0, 0]), t([]), 1, [1, 2])
    assert [x.numel() for x in empty[0][0]] == [0, 0]


@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("parts,buckets", [(1, [1, 2, 4]), (2, [1, 2, 4]), (1, list(range(1, 41)))])
def test_buckets_that_can_be_read_once(dev, strided, parts, buckets):
    """Widths from an iterator, for arrays that the native path takes and for those that it hands on."""
    rng = np.random.default_rng(parts)
    indptr, indices = _csr(200, 60, rng.integers(0, 9, 200), parts)
    d_idx = torch.from_numpy(np.repeat(indices, 2) if strided else indices).to(dev)
    got = st.column_part_hyb(200, 60, torch.from_numpy(indptr).to(dev), d_idx[::2] if strided else d_idx, parts, iter(buckets))
    want = st.column_part_hyb(200, 60, indptr, indices, parts, iter(buckets))
    for g, w in zip(got, want):
        for p in range(parts):
            for b in range(len(buckets)):
                assert np.array_equal(g[p][b].cpu().numpy(), w[p][b])


@pytest.mark.parametrize("m", [300, 64 * 256, 64 * 256 + 1])
def test_sizes_of_the_c_entry_leave_nothing_running(dev, m):
    """The C entry for the sizes waits for its kernels, whether it takes the matrix or refuses it: another stream may
    fill, and use the workspace again, at once."""
    L, buckets = _lib.lib(), [1, 2, 4, 8]
    deg = np.random.default_rng(m).integers(0, 11, m)
    indptr, indices = _csr(m, 700, deg, m)
    want = st.column_part_hyb(m, 700, indptr, indices, 1, buckets)
    d_ptr, d_idx = torch.from_numpy(indptr).to(dev), torch.from_numpy(indices).to(dev)
    nnz = len(indices)
    ws = torch.zeros(L.stir_column_part_hyb_device_workspace_bytes(m, 1, len(buckets), nnz), dtype=torch.uint8, device=dev)
    out = [[torch.zeros(w[0][b].shape, dtype=torch.int32, device=dev) for b in range(len(buckets))] for w in want]
    sizing, filling = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    w32 = np.array(buckets, np.int32)
    nrows = np.zeros(len(buckets), np.int64)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    host = lambda a: ctypes.c_void_p(a.ctypes.data)
    sizes = lambda p: L.stir_column_part_hyb_one_sizes(m, 700, ptr(p), ptr(d_idx), nnz, host(w32), len(buckets), ptr(ws),
                                                       host(nrows), ctypes.c_void_p(sizing.cuda_stream))
    wrong = d_ptr.clone()
    wrong[m // 2] = nnz + 1
    torch.cuda.synchronize()
    for _ in range(8):
        assert sizes(wrong) == -1
        assert sizing.query()
        assert sizes(d_ptr) == 0
        assert sizing.query()
    assert nrows.tolist() == [len(r) for r in want[0][0]]
    tables = [(ctypes.c_void_p * len(buckets))(*[t.data_ptr() for t in o]) for o in out]
    assert L.stir_column_part_hyb_one_fill(m, 700, ptr(d_ptr), ptr(d_idx), nnz, None, len(buckets), ptr(ws), *tables, None,
                                           ctypes.c_void_p(filling.cuda_stream)) == 0
    filling.synchronize()
    for got, w in zip(out, want):
        for b in range(len(buckets)):
            assert np.array_equal(got[b].cpu().numpy(), w[0][b])
