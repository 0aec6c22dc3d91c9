"""The destination-tiled fp16 RGMS over an even number of 32-feature tiles, two to a pass: W in the LDS and W read from
memory, one and two passes, units that begin and end tiles, and the odd number of tiles beside them."""
import ctypes

import pytest
import torch

import sparsetir_amd as st
from sparsetir_amd import _lib, ops
from test_gpu_rgms_relation_ranges import ROWS, WIDTHS, _csf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,fin,fout", [
    (8, 16, 64), (9, 32, 64), (7, 48, 64), (5, 64, 64), (6, 32, 128), (6, 32, 96),  # W in the LDS
    (90, 16, 64), (50, 32, 64), (30, 48, 64), (25, 64, 64), (40, 32, 128), (40, 32, 96), (20, 80, 64)])
@pytest.mark.parametrize("static,dtype,out", [(False, torch.float16, torch.float32), (True, torch.float16, torch.float32),
                                              (True, torch.bfloat16, torch.float32), (True, torch.float16, torch.float16)])
@pytest.mark.parametrize("n", [130, 2500])  # a few tiles, all cut; about two for each workgroup of a share
def test_two_tiles_of_features(dev, R, fin, fout, static, dtype, out, n):
    csf, (rel, dst, src), g = _csf(dev, n, R, 20_000 if n == 130 else 60_000, 1)
    ptr, rows, cols, mask = st.csf_to_ell3d(*csf, ROWS, WIDTHS)
    assert sum(c.numel() for c in cols) >= 8192  # else the kernel without an index
    x = torch.randn(n, fin, generator=g, device=dev).to(dtype)
    w = (torch.randn(R, fin, fout, generator=g, device=dev) * 0.1).to(dtype)
    flat, mids = [], []
    for p, r, c, k in zip(ptr, rows, cols, mask):
        flat += [k.reshape(-1).to(dtype), r.reshape(-1), c.reshape(-1)]
        mids.append(torch.repeat_interleave(torch.arange(R, dtype=torch.int32, device=dev), (p[1:] - p[:-1]).long()))
    f = ops.build_rgms(n, n, R, fin, fout, ROWS, WIDTHS, [c.shape[0] for c in cols], dtype, static_weights=static,
                       out_dtype=out)
    want = torch.zeros(n, fout, dtype=torch.float64, device=dev)
    scale = torch.zeros_like(want)
    for r in range(R):
        e = rel == r
        want.index_add_(0, dst[e], x[src[e]].double() @ w[r].double())
        scale.index_add_(0, dst[e], x[src[e]].double().abs() @ w[r].double().abs())
    for _ in range(2):  # the call that makes the index, and one more
        y = torch.full((n * fout,), 0.5, device=dev, dtype=out)
        f(w.reshape(-1), x.reshape(-1), y, *flat, *mids)
        err = (y.view(n, fout).double() - 0.5 - want).abs()
        if out == torch.float32:  # 21 bits of the products and 24 of the sums are kept
            bound = 1e-5 * scale + 1e-6
        else:  # products rounded to 11 bits, sums by each piece of a tile: a few, two for each team where n is small
            bound = 2.0 ** -11 * (scale + (64 if n == 130 else 4) * (want.abs() + scale.sqrt() + 0.5))
        assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("warm,captured", [(32, 64), (64, 32)])
def test_captured_with_another_number_of_tiles(dev, warm, captured):
    """A plan launched with one workgroup size and recorded with sizes that would take the other."""
    n, R, fin = 2500, 8, 32
    csf, _, g = _csf(dev, n, R, 60_000, 1)
    ptr, rows, cols, mask = st.csf_to_ell3d(*csf, ROWS, WIDTHS)
    arrays = [[k.reshape(-1).half() for k in mask], [r.reshape(-1) for r in rows], [c.reshape(-1) for c in cols],
              [torch.repeat_interleave(torch.arange(R, dtype=torch.int32, device=dev), (p[1:] - p[:-1]).long())
               for p in ptr]]
    nb = len(WIDTHS)
    L = _lib.lib()
    ints = lambda v: (ctypes.c_int32 * nb)(*v)
    pointers = [(ctypes.c_void_p * nb)(*[t.data_ptr() for t in a]) for a in arrays]
    x = torch.randn(n * fin, generator=g, device=dev).half()
    w = {f: (torch.randn(R * fin * f, generator=g, device=dev) * 0.1).half() for f in (32, 64)}

    def plan():
        p = ctypes.c_void_p()
        _lib.check(L.stir_rgms_plan_create(ctypes.byref(p), nb, ints(ROWS), ints(WIDTHS),
                                           (ctypes.c_int64 * nb)(*[c.shape[0] for c in cols]), *pointers))
        return p

    def run(p, fout, y):
        _lib.check(L.stir_rgms_f16(p, n, n, R, fin, fout, w[fout].data_ptr(), x.data_ptr(), y.data_ptr(),
                                   torch.cuda.current_stream().cuda_stream))

    want = torch.zeros(n * captured, device=dev)
    other = plan()
    run(other, captured, want)
    p = plan()
    y0, y = torch.zeros(n * warm, device=dev), torch.zeros(n * captured, device=dev)
    run(p, warm, y0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y.zero_()
        run(p, captured, y)
    for _ in range(3):
        y.fill_(5.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        # the cuts between shares lie elsewhere, so sums of 16-bit products differ in the order of fp32 additions
        assert torch.allclose(y, want, rtol=1e-5, atol=1e-4)
    y.zero_()
    run(p, captured, y)
    assert torch.allclose(y, want, rtol=1e-5, atol=1e-4)
    del graph
    for q in (p, other):
        L.stir_rgms_plan_destroy(q)
