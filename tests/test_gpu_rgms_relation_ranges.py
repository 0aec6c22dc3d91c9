"""The destination-tiled fp16 RGMS with more relations than the LDS holds: two ranges of relations with a launch each
need 1.3 M slots (0.85 M where a relation's W is large), fewer are one launch that reads W from memory."""
import pytest
import torch

import sparsetir_amd as st
from sparsetir_amd import ops

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 4, 8, 16]
ROWS = [256 // w for w in WIDTHS]


def _csf(dev, n, R, edges, empty):
    """CSF arrays on the device: relation sizes 1, 1/2, 1/3, ... in a shuffled order, some relations empty."""
    g = torch.Generator(device=dev).manual_seed(R)
    size = 1.0 / torch.arange(1, R + 1, device=dev, dtype=torch.float64)
    size[torch.randperm(R, generator=g, device=dev)[:empty]] = 0
    size = size[torch.randperm(R, generator=g, device=dev)]
    rel = torch.multinomial(size, edges, replacement=True, generator=g)
    dst = torch.randint(n, (edges,), generator=g, device=dev)
    src = torch.randint(n, (edges,), generator=g, device=dev)
    key = torch.unique((rel * n + dst) * n + src)
    rel, dst, src = key // n // n, key // n % n, key % n
    pair, counts = torch.unique_consecutive(key // n, return_counts=True)
    ptr = lambda c: torch.cat([c.new_zeros(1), torch.cumsum(c, 0)]).int()
    csf = (ptr(torch.bincount(pair // n, minlength=R)), (pair % n).int(), ptr(counts), src.int())
    return csf, (rel, dst, src), g


@pytest.mark.parametrize("R,fin,fout,edges,ranges", [
    (80, 32, 32, 1_400_000, 2), (80, 32, 32, 900_000, 1), (130, 32, 32, 1_400_000, 2), (24, 64, 64, 950_000, 2),
    (24, 64, 64, 600_000, 1), (200, 32, 32, 1_400_000, 3)])
@pytest.mark.parametrize("static,dtype", [(False, torch.float16), (True, torch.float16), (True, torch.bfloat16)])
def test_ranges_of_relations(dev, R, fin, fout, edges, ranges, static, dtype):
    n = 30000
    csf, (rel, dst, src), g = _csf(dev, n, R, edges, 3)
    ptr, rows, cols, mask = st.csf_to_ell3d(*csf, ROWS, WIDTHS)
    slots = sum(c.numel() for c in cols)
    enough = slots >= (850_000 if fin * fout >= 2048 else 1_300_000)
    assert enough == (ranges > 1)  # the figures of the rule; three ranges are never taken
    x = torch.randn(n, fin, generator=g, device=dev).to(dtype)
    w = (torch.randn(R, fin, fout, generator=g, device=dev) * 0.1).to(dtype)
    flat, mids = [], []
    for p, r, c, k in zip(ptr, rows, cols, mask):
        flat += [k.reshape(-1).to(dtype), r.reshape(-1), c.reshape(-1)]
        mids.append(torch.repeat_interleave(torch.arange(R, dtype=torch.int32, device=dev), (p[1:] - p[:-1]).long()))
    f = ops.build_rgms(n, n, R, fin, fout, ROWS, WIDTHS, [c.shape[0] for c in cols], dtype, static_weights=static)
    want = torch.zeros(n, fout, dtype=torch.float64, device=dev)
    scale = torch.zeros_like(want)
    for r in range(R):
        e = rel == r
        want.index_add_(0, dst[e], x[src[e]].double() @ w[r].double())
        scale.index_add_(0, dst[e], x[src[e]].double().abs() @ w[r].double().abs())
    for _ in range(2):  # the call that makes the indices, and one more
        y = torch.full((n * fout,), 0.5, device=dev)
        f(w.reshape(-1), x.reshape(-1), y, *flat, *mids)
        # 16-bit factors, products and sums in fp32, 21 bits of the products and 24 of the sums kept
        err = (y.view(n, fout).double() - 0.5 - want).abs()
        assert bool((err <= 1e-5 * scale + 1e-6).all()), float((err / (scale + 1e-6)).max())
