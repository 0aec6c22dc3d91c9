"""The tile form of the fp32 RGMS at the edges of its batches: chains of four edges, pairs longer than a
batch, sixteen pairs and one more, tiles of 128 rows and the rows beyond, whole and cut tiles."""
import numpy as np
import pytest
import torch

from sparsetir_amd import ops
from helpers import rgms_f64

pytestmark = pytest.mark.gpu


def _csf(rng, n, R, lengths_of):
    """CSF arrays whose relation r has the (row, edge count) list lengths_of(r)."""
    p0, i0, p1, i1 = [0], [], [0], []
    for r in range(R):
        for row, count in sorted(lengths_of(r).items()):
            i0.append(row)
            i1.append(np.sort(rng.choice(n, count, replace=False)))
            p1.append(p1[-1] + count)
        p0.append(len(i0))
    return [np.asarray(v, np.int32) for v in (p0, i0, p1)] + [np.concatenate(i1).astype(np.int32)]


@pytest.mark.parametrize("fin,fout", [(4, 1), (16, 64), (32, 8), (32, 16), (32, 17), (32, 32), (36, 16), (48, 32), (64, 64), (64, 33)])
@pytest.mark.parametrize("n", [129, 1000])
def test_chains_and_batches(dev, fin, fout, n):
    rng = np.random.default_rng(fin * 100 + fout + n)
    R = 7

    def lengths_of(r):
        rows = rng.choice(n, n - 3, replace=False)
        pick = {int(v): int(rng.choice([1, 1, 2, 3, 4, 5])) for v in rows[:[n - 3, 16, 17, 15, 1, 0, n // 2][r]]}
        if r in (0, 6):  # pairs of every length around a column, a batch and twice a batch
            for k, c in enumerate([4, 5, 8, 9, 15, 16, 17, 31, 32, 33, 64, 65, 100, n - 1]):
                pick[int(rows[k])] = min(c, n - 1)
        if r == 0:
            pick[n - 1] = 3
        return pick

    csf = _csf(rng, n, R, lengths_of)
    # enough edges for the tile form: relation 0 again and again under other numbers
    reps = 1 + 9000 // len(csf[3])
    p0 = np.concatenate([[0]] + [csf[0][1:] + k * len(csf[1]) for k in range(reps)]).astype(np.int32)
    p1 = np.concatenate([[0]] + [csf[2][1:] + k * len(csf[3]) for k in range(reps)]).astype(np.int32)
    csf = [p0, np.tile(csf[1], reps), p1, np.tile(csf[3], reps)]
    R *= reps
    assert len(csf[3]) >= 8192
    a = rng.random(len(csf[3]), dtype=np.float32) - 0.3
    x = rng.standard_normal((n, fin), dtype=np.float32)
    w = rng.standard_normal((R, fout, fin), dtype=np.float32) * 0.1
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev)
    f = ops.build_rgms_csf(n, n, R, fin, fout, len(csf[1]), len(csf[3]))
    args = [t(a), t(w.ravel()), t(x.ravel())]
    rest = [t(c) for c in csf]
    ys = []
    for _ in range(2):
        y = torch.full((n * fout,), 0.5, dtype=torch.float32, device=dev)
        f(*args, y, *rest)
        ys.append(y)
    torch.cuda.synchronize()
    assert torch.equal(*ys)
    got = ys[0].cpu().numpy().reshape(n, fout) - np.float32(0.5)
    wt = np.ascontiguousarray(w.transpose(0, 2, 1))
    want = rgms_f64(*csf, a, x, wt, n)
    scale = rgms_f64(*csf, np.abs(a), np.abs(x), np.abs(wt), n)
    err = np.abs(got - want)
    assert np.all(err <= 1e-5 * np.abs(want) + 1e-5 * scale + 1e-6), f"worst {err.max():.3e}"
    assert np.linalg.norm(err) <= 1e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("fin,fout", [(32, 32), (32, 64), (64, 32), (64, 64)])
def test_stretches_of_batches(dev, fin, fout):
    """Tiles of 1 to 20 batches, each of another relation or with two in a row of one, for workgroups of 4 and 8
    wavefronts: fewer batches than wavefronts, as many, and every remainder."""
    rng = np.random.default_rng(fin + fout)
    tiles, R = 20, 20
    n = 128 * (tiles + 1)

    def lengths_of(r):
        pick = {}
        for t in range(r, tiles):  # tile t: relations 0 ... t
            if t % 2 == 0 and r == t:
                continue  # instead of the last relation a second batch of the one before
            pairs = 17 if t % 2 == 0 and r == t - 1 else 1 + (r + t) % 16
            for k in rng.choice(128, pairs, replace=False):
                pick[128 * t + int(k)] = 1
        if r < 10:  # a tile of many batches, and edges enough for the tile form
            for k in range(128):
                pick[128 * tiles + k] = 7
        return pick

    csf = _csf(rng, n, R, lengths_of)
    assert len(csf[3]) >= 8192
    a = rng.random(len(csf[3]), dtype=np.float32) - 0.3
    x = rng.standard_normal((n, fin), dtype=np.float32)
    w = rng.standard_normal((R, fout, fin), dtype=np.float32) * 0.1
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev)
    f = ops.build_rgms_csf(n, n, R, fin, fout, len(csf[1]), len(csf[3]))
    y = torch.full((n * fout,), 0.5, dtype=torch.float32, device=dev)
    f(t(a), t(w.ravel()), t(x.ravel()), y, *[t(c) for c in csf])
    got = y.cpu().numpy().reshape(n, fout) - np.float32(0.5)
    wt = np.ascontiguousarray(w.transpose(0, 2, 1))
    want = rgms_f64(*csf, a, x, wt, n)
    scale = rgms_f64(*csf, np.abs(a), np.abs(x), np.abs(wt), n)
    err = np.abs(got - want)
    assert np.all(err <= 1e-5 * np.abs(want) + 1e-5 * scale + 1e-6), f"worst {err.max():.3e}"
