"""The tile form of the fp32 RGMS multiplies with three bf16 terms per factor and must give what fp32 products give:
very small and very large factors, infinities, and both kinds side by side."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from sparsetir_amd import ops

pytestmark = pytest.mark.gpu

N, R = 700, 5
SIZES = [(32, 16), (32, 32), (16, 64), (64, 16), (36, 32), (64, 64)]  # one per kernel


def _graph(rng, counts):
    """CSF arrays: rows of so many edges in every relation, and rows of none."""
    p0, i0, p1, i1 = [0], [], [0], []
    for _ in range(R):
        for row in np.sort(rng.choice(N, N - 50, replace=False)):
            count = int(rng.choice(counts))
            i0.append(row)
            i1.append(np.sort(rng.choice(N, count, replace=False)))
            p1.append(p1[-1] + count)
        p0.append(len(i0))
    csf = [np.asarray(v, np.int32) for v in (p0, i0, p1)] + [np.concatenate(i1).astype(np.int32)]
    assert len(csf[3]) >= 8192
    return csf


def _sums(csf, a, x):
    """A_r @ X of every relation in float64 (infinities multiply the stored edges only)."""
    p0, i0, p1, i1 = csf
    for r in range(R):
        e0, e1 = p1[p0[r]], p1[p0[r + 1]]
        rows = np.repeat(i0[p0[r]:p0[r + 1]], np.diff(p1[p0[r]:p0[r + 1] + 1]))
        yield sp.csr_matrix((a[e0:e1].astype(np.float64), (rows, i1[e0:e1])), shape=(N, N)) @ x.astype(np.float64)


def _reference(csf, a, x, w):
    """Y, and the sum of the magnitudes of all terms, in float64; rows a relation does not store add nothing."""
    y, scale = np.zeros((N, w.shape[1])), np.zeros((N, w.shape[1]))
    with np.errstate(invalid="ignore"):
        for r, (s, t) in enumerate(zip(_sums(csf, a, x), _sums(csf, np.abs(a), np.abs(x)))):
            stored = csf[1][csf[0][r]:csf[0][r + 1]]
            y[stored] += s[stored] @ w[r].T.astype(np.float64)
            scale[stored] += t[stored] @ np.abs(w[r].T.astype(np.float64))
    return y, scale


def _run(dev, csf, a, x, w):
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev)
    y = torch.zeros(N * w.shape[1], device=dev)
    f = ops.build_rgms_csf(N, N, R, w.shape[2], w.shape[1], len(csf[1]), len(csf[3]))
    f(t(a), t(w.ravel()), t(x.ravel()), y, *[t(c) for c in csf])
    return y.cpu().numpy().reshape(N, -1)


def _inputs(fin, fout, counts=(1, 2, 3, 5, 9, 40)):  # up to several chains and batches
    rng = np.random.default_rng(fin * 100 + fout)
    csf = _graph(rng, counts)
    return (csf, rng.random(len(csf[3]), dtype=np.float32) + np.float32(0.1),
            rng.standard_normal((N, fin), dtype=np.float32), rng.standard_normal((R, fout, fin), dtype=np.float32))


def _close(got, want, scale, w, what):
    # sums of up to 200 edges and 64 inputs: 200 + 64 + 5 additions and the products, 2^-24 of the terms each.  Where
    # fp32 numbers are subnormal a rounding is 2^-150: of 200 edges, which the weights of the inputs then multiply,
    # and of the 64 products and 5 sums themselves.
    err = np.abs(got - want)
    tiny = 2.0 ** -150 * (2 * 200 * w.shape[2] * float(np.abs(w).max()) + 140)
    assert np.all(err <= 280 * 2.0 ** -24 * scale + tiny), f"{what}: worst {(err / scale).max():.2e}"
    assert np.linalg.norm(err) <= 1e-6 * np.linalg.norm(want) + tiny * want.size ** 0.5, what


@pytest.mark.parametrize("fin,fout", SIZES)
@pytest.mark.parametrize("xs,ws", [(1, 1), (1e-36, 1), (1e-20, 1e-16), (1, 1e-36), (1e-41, 1), (1e30, 1),
                                   (1e10, 1e20), (1e-30, 1e30), (1e-42, 1e33)])
def test_magnitudes(dev, fin, fout, xs, ws):
    csf, a, x, w = _inputs(fin, fout)
    x, w = x * np.float32(xs), w * np.float32(ws)
    _close(_run(dev, csf, a, x, w), *_reference(csf, a, x, w), w, f"{xs} {ws}")


@pytest.mark.parametrize("fin,fout", SIZES)
def test_small_inputs_beside_large_ones(dev, fin, fout):
    """Half of the inputs are tiny, and half of the outputs depend on those alone."""
    csf, a, x, w = _inputs(fin, fout)
    x[:, :fin // 2] *= np.float32(1e-36)
    w[:, :fout // 2, fin // 2:] = 0
    got, (want, scale) = _run(dev, csf, a, x, w), _reference(csf, a, x, w)
    half = fout // 2
    _close(got[:, :half], want[:, :half], scale[:, :half], w, "tiny")
    _close(got[:, half:], want[:, half:], scale[:, half:], w, "ordinary")


@pytest.mark.parametrize("where", ["x", "w", "a", "large"])
@pytest.mark.parametrize("fin,fout", SIZES)
def test_infinities(dev, fin, fout, where):
    """An infinity in X, W or the edge weights reaches the outputs as it does in fp32: with its sign, NaN only where
    two of opposite signs meet, and no other output; finite values next to the largest stay finite."""
    # (the pieces of a pair longer than a batch meet the weights one by one: an infinite weight may meet sums of both signs)
    csf, a, x, w = _inputs(fin, fout, (2, 3, 5, 9, 16)) if where == "w" else _inputs(fin, fout)
    if where == "x":
        x[5, 3], x[17, fin - 1] = np.inf, -np.inf
    elif where == "w":
        w[2, fout - 1, 1] = np.inf
    elif where == "a":
        a[1234] = np.inf
    else:
        x[5], a = np.float32(3.39e38), a * np.float32(0.01)
    got, (want, scale) = _run(dev, csf, a, x, w), _reference(csf, a, x, w)
    bad = ~np.isfinite(want)
    if where == "large":
        fits = scale < 3e38
        assert np.all(np.abs(got - want)[fits] <= 280 * 2.0 ** -24 * scale[fits]) and (scale[fits] > 1e36).any()
        return
    assert bad.any() and not bad.all()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    assert np.all(np.abs(got[~bad] - want[~bad]) <= 280 * 2.0 ** -24 * scale[~bad])
