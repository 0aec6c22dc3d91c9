"""The native host path of the operators: which plan a call uses, and when it leaves a call to Python."""
import sys
import threading

import numpy as np
import pytest
import torch

from sparsetir_amd import ops
from sparsetir_amd._lib import SparseTIRError

pytestmark = pytest.mark.gpu


def _graphs(dev, count, m=200, w=4, feat=32):
    """Matrices of one hyb bucket that differ in their columns only, and their products with x."""
    g = torch.Generator(device=dev).manual_seed(count)
    x = torch.randn(m, feat, device=dev, generator=g)
    rows = torch.arange(m, dtype=torch.int32, device=dev)
    out = []
    for _ in range(count):
        cols = torch.randint(m, (m, w), dtype=torch.int32, device=dev, generator=g)
        a = torch.rand(m, w, device=dev, generator=g)
        want = (a.double()[:, :, None] * x.double()[cols.long()]).sum(1)
        out.append((a.reshape(-1), rows.clone(), cols.reshape(-1), want))
    return x, out, ops.build_hyb_csrmm(m, m, feat, 1, [w, 2 * w], [m, 0])


@pytest.mark.parametrize("count", [1, 2, 8, 9])
def test_plans_of_several_matrices(dev, count):
    """Up to eight matrices in turn keep their plans; a ninth evicts the one used longest ago, and a
    call with that one makes it anew instead of using what was destroyed."""
    x, mats, f = _graphs(dev, count)
    z = torch.zeros(0, device=dev)
    zi = torch.zeros(0, dtype=torch.int32, device=dev)
    for _ in range(3):
        for a, r, c, want in mats:
            y = torch.zeros_like(x)
            f(x.reshape(-1), y.reshape(-1), a, r, c, z, zi, zi)
            assert torch.allclose(y.double(), want, rtol=1e-5, atol=1e-5)
    assert f.plan_builds == (count if count <= 8 else 3 * count)


def test_falls_back_to_python(dev):
    """Arguments the launcher does not take get the same answer, or the same error, as before."""
    x, mats, f = _graphs(dev, 1)
    a, r, c, want = mats[0]
    z, zi = torch.zeros(0, device=dev), torch.zeros(0, dtype=torch.int32, device=dev)
    y = torch.zeros(x.numel(), device=dev)
    args = [x.reshape(-1), y, a, r, c, z, zi, zi]
    f(*args)
    builds = f.plan_builds
    with pytest.raises(SparseTIRError, match="shape"):
        f(x.reshape(-1)[:-1], *args[1:])
    with pytest.raises(SparseTIRError, match="dtype"):
        f(args[0].double(), *args[1:])
    with pytest.raises(SparseTIRError, match="compact"):
        f(torch.zeros(2 * x.numel(), device=dev)[::2], *args[1:])
    with pytest.raises(SparseTIRError, match="num_args"):
        f(*args[:-1])
    f.invalidate()
    y.zero_()
    f(*args)
    assert f.plan_builds == builds + 1
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # the stream that is current when the call is made
        y2 = torch.zeros_like(y)
        f(args[0], y2, *args[2:])
    side.synchronize()
    for got in (y, y2):
        assert np.allclose(got.cpu().numpy().reshape(want.shape), want.cpu().numpy(), rtol=1e-5, atol=1e-5)


def test_threads_share_an_operator(dev):
    """Four threads with three matrices each use one operator, more matrices than it keeps plans: every product is
    that of the arrays handed in, during the calls and afterwards (a plan filed under another thread's arrays would
    multiply the wrong matrix from then on)."""
    x, mats, f = _graphs(dev, 12)
    z, zi = torch.zeros(0, device=dev), torch.zeros(0, dtype=torch.int32, device=dev)

    def product(k):
        a, r, c, want = mats[k]
        y = torch.zeros_like(x)
        f(x.reshape(-1), y.reshape(-1), a, r, c, z, zi, zi)
        assert torch.allclose(y.double(), want, rtol=1e-5, atol=1e-5), f"matrix {k}"

    failed = []

    def work(first):
        try:
            for _ in range(25):
                for k in range(first, 12, 4):
                    product(k)
        except BaseException as e:  # noqa: B036 (reported by the test)
            failed.append(e)

    before = sys.getswitchinterval()
    sys.setswitchinterval(1e-5)
    try:
        threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(before)
    assert not failed, failed[0]
    assert len(f._plans) == f._plans.capacity
    for k in range(12):
        product(k)


def test_inference_tensors_get_the_same_bits(dev):
    """Tensors made under inference_mode count no versions, which only what a plan depends on has to: a CSR product
    and the features of a planned operator take the same way as under no_grad, to the same bits."""
    rng = np.random.default_rng(3)
    m, n, feat = 9001, 3000, 64
    deg = rng.integers(0, 12, m)
    deg[[0, 5, m // 2, m - 1]] = [3000, 129, 1000, 400]
    indptr = torch.from_numpy(np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)).to(dev)
    nnz = int(deg.sum())
    indices = torch.from_numpy(rng.integers(0, n, nnz).astype(np.int32)).to(dev)
    a, x = torch.rand(nnz, device=dev), torch.randn(n * feat, device=dev)
    f = ops.build_csrmm(m, n, feat, nnz)
    want = torch.empty(m * feat, device=dev)
    f(a, x, want, indptr, indices)
    with torch.inference_mode():
        args = [t.clone() for t in (a, x, want, indptr, indices)]
        assert all(t.is_inference() for t in args)
        args[2].fill_(float("nan"))
        f(*args)
        assert torch.equal(args[2], want)
    args = [a, x, torch.empty_like(want), indptr, indices]
    f._call(*args)  # the way of a call that the launcher did not take, on another device than the current one say
    assert torch.equal(args[2], want)

    x, mats, f = _graphs(dev, 1)
    a, r, c, want = mats[0]
    z, zi = torch.zeros(0, device=dev), torch.zeros(0, dtype=torch.int32, device=dev)
    y = torch.zeros_like(x)
    f(x.reshape(-1), y.reshape(-1), a, r, c, z, zi, zi)
    builds, slow = f.plan_builds, f._call
    f._call = None  # not needed
    with torch.inference_mode():
        x2, y2 = x.clone().reshape(-1), torch.zeros_like(x).reshape(-1)
        f(x2, y2, a, r, c, z, zi, zi)
        assert torch.equal(y2, y.reshape(-1)) and f.plan_builds == builds
    f._call = slow
