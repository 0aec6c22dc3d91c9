"""Condensed SpMM of more than 64 features with a plan: tiles of an odd number of groups, whose last step has one group only --
an infinity among the rows of B that it gathers stays an infinity where every row of the tile has an entry, and reaches no
other feature -- ragged feature tiles, and arrays that start at an odd element."""
import numpy as np
import pytest
import torch

import sparsetir_amd as st
from helpers import tc_form
from sparsetir_amd import ops
from test_gpu_tcspmm import _run

pytestmark = pytest.mark.gpu


def _odd_groups(dev, t, feat, out_dtype, start, empty=0, form=None):
    rng = np.random.default_rng(feat + t)
    n, counts = 900, [16, 48, 80, 32, 144, 0, 688] + [0] * empty  # columns of a tile: 1, 3, 5, 2, 9, 0 and 43 groups
    cols = [np.sort(rng.choice(np.arange(1, n), c, replace=False)) for c in counts]
    rows = [c for c in cols for _ in range(t)]
    indptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    gptr, tiles, mask = st.condense(indptr, np.concatenate(rows).astype(np.int32), t, 16)
    mb = len(gptr) - 1
    # no tile is long: the longest has 43 groups, 22 steps
    assert form is None or tc_form(t, out_dtype, mb, feat, tiles.shape[0]) == form
    a = (mask * rng.uniform(0.1, 1.0, mask.shape)).astype(np.float16)
    b = rng.standard_normal((n, feat)).astype(np.float16)
    named = int(cols[1][-1])  # in the last group of the second tile
    b[named, feat - 1] = np.inf

    def place(v):
        x = torch.empty(v.size + start, dtype=torch.float16, device=dev)[start:]
        x.copy_(torch.from_numpy(v.reshape(-1)))
        return x

    td = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev)
    c = torch.full((mb * t * feat + start,), float("nan"), dtype=out_dtype, device=dev)[start:]
    f = ops.build_tcspmm(mb, tiles.shape[0], feat, t, 16, n, out_dtype)
    f(place(a), place(b), c, td(gptr), td(tiles.ravel()))
    got = c.float().cpu().numpy().reshape(mb, t, feat)
    has = np.array([named in k for k in cols])
    assert np.isposinf(got[has, :, feat - 1]).all()
    b[named, feat - 1] = 0.0
    got[has, :, feat - 1] = 0.0
    for io in range(mb):
        lo, hi = gptr[io], gptr[io + 1]
        at = np.concatenate(list(a[lo:hi].astype(np.float64)), axis=1) if hi > lo else np.zeros((t, 0))
        bt = b[tiles[lo:hi].reshape(-1)].astype(np.float64)
        want, scale = at @ bt, np.abs(at) @ np.abs(bt)
        if has[io]:
            want[:, feat - 1], scale[:, feat - 1] = 0.0, 0.0
        # fp32 sums of up to 688 exact products: 688 roundings of 2^-24 of the terms; one more of an fp16 result
        bound = 688 * 2.0 ** -24 * scale + (2.0 ** -11 * np.abs(want) if out_dtype is torch.float16 else 0.0) + 1e-7
        assert np.all(np.abs(got[io] - want) <= bound)


@pytest.mark.parametrize("t", [8, 16, 32])
@pytest.mark.parametrize("feat", [96, 128, 224, 288])
@pytest.mark.parametrize("out_dtype,start", [(torch.float16, 1), (torch.float32, 1), (torch.float32, 0)])
def test_odd_groups(dev, t, feat, out_dtype, start):
    _odd_groups(dev, t, feat, out_dtype, start)


@pytest.mark.parametrize("t", [8, 16, 32])
@pytest.mark.parametrize("feat", [160, 288])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_a_unit_of_32_features(dev, t, feat, out_dtype):
    """32 features with a unit of 128 to themselves, in a launch of many units."""
    _odd_groups(dev, t, feat, out_dtype, 1, 13_000_000 // (2 * feat * t) + 1)


# the forms of launches of many units, by empty tiles: two wavefronts to a unit, one step of a wavefront on its way
@pytest.mark.parametrize("t,feat,out_dtype,empty,form", [
    (8, 192, torch.float16, 2600, "128 by 2"),
    (8, 192, torch.float32, 2600, "128 by 2"),
    (8, 224, torch.float16, 10000, "128 by 2, one step"),
    (8, 224, torch.float32, 10000, "128 by 2, one step"),
    (16, 192, torch.float16, 2600, "128 by 2, one step"),
    (16, 224, torch.float16, 2600, "128 by 2"),
    (16, 192, torch.float32, 2600, "128 by 2, one step"),
    (16, 256, torch.float32, 2600, "128 by 2"),
    (32, 96, torch.float16, 1300, "128 by 4, one step"),
    (32, 160, torch.float32, 650, "128 by 4, one step"),
    (32, 160, torch.float32, 600, "64 by 4"),
    (8, 160, torch.float16, 1500, "64 by 4"),
    (32, 192, torch.float16, 2600, "128 by 2, one step"),
    (32, 192, torch.float32, 2600, "128 by 2, one step"),
    (32, 256, torch.float16, 2600, "128 by 2"),
])
def test_forms(dev, t, feat, out_dtype, empty, form):
    _odd_groups(dev, t, feat, out_dtype, 1, empty, form)


@pytest.mark.parametrize("t,feat,tiles,deg,out_dtype,form", [
    (8, 128, 6000, 18, torch.float16, "64 by 2"),             # two units of 64 to a tile of several steps
    (32, 96, 1400, 1, torch.float32, "128 by 4, one step"),   # with tiles that are cut into pieces
    (32, 192, 2600, 1, torch.float16, "128 by 2, one step"),
])
def test_forms_of_whole_graphs(dev, t, feat, tiles, deg, out_dtype, form):
    rng = np.random.default_rng(tiles)
    counts = np.full(tiles * t, deg)
    if deg == 1:
        counts[[t + 1, 5 * t]] = 1500
    indptr = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n = 12000
    indices = ((np.arange(indptr[-1]) * 7 + rng.integers(0, 7, indptr[-1])) % n).astype(np.int32)  # distinct in a row
    gptr = st.condense(indptr, indices, t, 16)[0]
    assert tc_form(t, out_dtype, tiles, feat, int(gptr[-1])) == form
    _run(dev, indptr, indices, n, feat, False, out_dtype, t=t)
