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


def _hub_case(dev, rng, feat, longest, t=16, out_dtype=torch.float32):
    """A product whose long tiles are cut, its arguments without the output, and the output's length."""
    n = 9001
    deg = rng.integers(0, 6, 3000)
    deg[::300] = longest
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    indices = ((np.arange(indptr[-1]) * 7 + 3) % n).astype(np.int32)
    gptr, tiles, mask = st.condense(indptr, indices, t, 16)
    td = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev)
    mb = len(gptr) - 1
    args = [td(mask.astype(np.float16).ravel()), td(rng.standard_normal(n * feat).astype(np.float16))]
    return args, [td(gptr), td(tiles.ravel())], mb, tiles.shape[0], n, mb * t * feat


def test_streams_share_an_operator(dev):
    """Calls of one operator on two streams, and replays of its recorded call, run at the same time: each stream, and
    the graph, has counters and partial tiles of its own."""
    rng = np.random.default_rng(11)
    feat, t = 128, 16
    args, tail, mb, nnzb, n, length = _hub_case(dev, rng, feat, 8000)
    f = ops.build_tcspmm(mb, nnzb, feat, t, 16, n, torch.float32)
    want = torch.full((length,), float("nan"), device=dev)
    f(*args, want, *tail)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    recorded = torch.full((length,), float("nan"), device=dev)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        f(*args, recorded, *tail)
    out = [torch.full((length,), float("nan"), device=dev) for _ in range(40)]
    torch.cuda.synchronize()
    for k, c in enumerate(out):
        with torch.cuda.stream(streams[k % 2]):
            f(*args, c, *tail)
        if k % 10 == 0:
            graph.replay()
    torch.cuda.synchronize()
    assert all(torch.equal(c, want) for c in out) and torch.equal(recorded, want)
    assert f.plan_builds == 1


def test_first_calls_on_one_stream_with_other_row_pointers(dev):
    """One operator, two arrays of group counts of the same length and sum: the second has a longer tile, so that the
    memory of the stream grows between calls of the first."""
    rng = np.random.default_rng(13)
    feat, t, n, mb = 64, 16, 5000, 40
    base = np.full(mb, 4, np.int64)
    short, long = base.copy(), base.copy()
    short[3], short[7] = 404, 400     # 202 and 200 steps
    long[3] = 804 - 4
    long[7] = short.sum() - (long.sum() - long[7])
    assert short.sum() == long.sum()
    td = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev)
    nnzb = int(short.sum())
    a = torch.rand(nnzb * t * 16, device=dev).half()
    b = torch.randn(n * feat, device=dev).half()
    idx = torch.randint(n, (nnzb * 16,), dtype=torch.int32, device=dev)
    f = ops.build_tcspmm(mb, nnzb, feat, t, 16, n, torch.float32)
    blocks = torch.bmm(a.view(nnzb, t, 16).float(), b.view(n, feat).float()[idx.long()].view(nnzb, 16, feat).contiguous())
    ptrs = [td(np.concatenate([[0], np.cumsum(v)]).astype(np.int32)) for v in (short, long)]
    wants = [torch.zeros(mb, t, feat, device=dev, dtype=torch.float64).index_add_(
        0, torch.repeat_interleave(torch.arange(mb, device=dev), td(v)), blocks.double()) for v in (short, long)]
    for k in (0, 1, 0, 1, 1, 0):
        c = torch.full((mb * t * feat,), float("nan"), device=dev)
        f(a, b, c, ptrs[k], idx)
        # sums of up to 12 800 products, magnitudes 0.5: 2^-24 of their sum each
        assert (c.view(mb, t, feat).double() - wants[k]).abs().max() < 2e-3
    assert f.plan_builds == 2
