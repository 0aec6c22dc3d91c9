"""What this library is measured on: the sparse kernels as a program calls them, on synthetic
graphs, pruned weights and relational graphs of the sizes this repository's configurations use.

A case is a dict; its ``kind`` names the path:

  csr        C = A X, CSR row-split                    full-graph GNN layer, any feature width
  hyb        C += A X over a kept hyb decomposition    full-graph GNN layer, the tuned format
  train      Y = A X, dX = A^T dY, dA = <dY[i], X[j]>  one layer's forward and backward pass
  sddmm      E = A * <X[i], Y[j]> per edge             attention scores, decoder scores
  minibatch  decompose a sampled block and multiply    neighbour-sampled training: every batch has
                                                       a matrix of its own, nothing can be kept
  bsr        Y = W X, W in dense blocks                pruned linear layer, activations X
  tc         C = A X over condensed row tiles, fp16    full-graph GNN layer in half precision
  rgms       Y += sum_r A_r X W_r, 16-bit              relational GCN layer, inference
  rgms_f32   the same in fp32 over the CSF arrays      relational GCN layer, training precision

Graphs have power-law row degrees; ``columns`` says whether the column ids are uniform or skewed
like the rows.  Everything random comes from the seed.  Outputs that an operator accumulates into
are cleared in ``run``, as its callers have to.
"""
import math

import torch

import sparsetir_amd as st
from sparsetir_amd import ops

DEV = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
ELL3D_WIDTHS = [1, 2, 4, 8, 16]
ELL3D_GROUP = 256  # slots per ELL3D group

LARGE_EDGES, LARGE_FEAT = 61_859_140, 128  # the work no drawn graph case may exceed


# ---------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: a citation-sized graph with narrow features, launch latency
        dict(name="csr_small", kind="csr", nodes=4096, edges=65536, feat=32, alpha=1.2, max_deg=1024,
             columns="uniform"),
        # the last layer of a node classifier: as many features as classes, here an odd number
        dict(name="csr_classes", kind="csr", nodes=169343, edges=1166243, feat=47, alpha=1.1, max_deg=13000,
             columns="skewed"),
        # an ordinary full-graph layer
        dict(name="hyb_medium", kind="hyb", nodes=169343, edges=1166243, feat=128, alpha=1.1, max_deg=13000,
             columns="uniform", parts=1),
        # the headline workload
        dict(name="hyb_large", kind="hyb", nodes=2449029, edges=LARGE_EDGES, feat=LARGE_FEAT, alpha=1.0,
             max_deg=17500, columns="uniform", parts=1),
        # one training step of an ordinary layer on a graph with hubs on both sides
        dict(name="train_step", kind="train", nodes=169343, edges=1166243, feat=64, alpha=1.1, max_deg=13000,
             columns="skewed"),
        # edge scores of the large graph, scaled by edge weights
        dict(name="sddmm_large", kind="sddmm", nodes=2449029, edges=LARGE_EDGES, feat=64, alpha=1.0,
             max_deg=17500, columns="uniform", scaled=True),
        # one sampled block of a mini-batch: its own matrix, decomposed and used once
        dict(name="minibatch", kind="minibatch", rows=4096, cols=45000, fanout=15, feat=100),
        # a pruned linear layer at a modest batch
        dict(name="bsr_layer", kind="bsr", mb=128, nb=128, blk=32, density=0.10, feat=512, dtype="f16"),
        # a large pruned layer over many tokens
        dict(name="bsr_large", kind="bsr", mb=512, nb=512, blk=32, density=0.10, feat=4096, dtype="bf16"),
        # half-precision aggregation on the matrix cores
        dict(name="tc_medium", kind="tc", nodes=169343, edges=1166243, feat=128, alpha=1.1, max_deg=13000,
             columns="uniform", tile=16, out="f16"),
        # a relational layer; the 0/1 edge mask is promised not to change
        dict(name="rgms_layer", kind="rgms", nodes=100000, rels=65, edges=2000000, fin=32, fout=32, dtype="f16",
             out="f32", static=True),
        # the same layer in single precision
        dict(name="rgms_f32_layer", kind="rgms_f32", nodes=100000, rels=65, edges=2000000, fin=32, fout=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _feat(rng, lo, hi):
    """Hidden sizes are round, input and class counts are not."""
    f = _log(rng, lo, hi)
    step = rng.choice([32, 16, 4, 1])
    return max(lo, f // step * step)


def _graph(rng, lo, hi, feat_lo, feat_hi):
    nodes = _log(rng, lo, hi)
    edges = int(nodes * rng.uniform(4, 26))
    feat = _feat(rng, feat_lo, feat_hi)
    edges = min(edges, LARGE_EDGES * LARGE_FEAT // feat // 2)
    return dict(nodes=nodes, edges=edges, feat=feat, alpha=round(rng.uniform(0.8, 1.2), 2),
                max_deg=min(nodes // 4, rng.choice([500, 2000, 8000, 17500])),
                columns=rng.choice(["uniform", "skewed"]))


def draw(rng):
    kind = rng.choice(["csr", "hyb", "train", "sddmm", "minibatch", "bsr", "tc", "rgms", "rgms_f32"])
    if kind == "csr":
        return dict(kind=kind, **_graph(rng, 3000, 300000, 8, 256))
    if kind == "hyb":
        return dict(kind=kind, parts=rng.choice([1, 1, 2]), **_graph(rng, 10000, 2000000, 16, 256))
    if kind == "train":
        return dict(kind=kind, **_graph(rng, 10000, 300000, 16, 256))
    if kind == "sddmm":
        return dict(kind=kind, scaled=rng.random() < 0.5, **_graph(rng, 10000, 2000000, 16, 128))
    if kind == "minibatch":
        rows = _log(rng, 500, 60000)
        return dict(kind=kind, rows=rows, cols=rows * rng.randint(4, 12) + rng.randint(0, 99),
                    fanout=rng.choice([5, 10, 15, 25]), feat=_feat(rng, 32, 256))
    if kind == "bsr":
        blk = rng.choice([16, 32, 32, 64, 128])
        rows, cols = _log(rng, 1024, 16384) // blk, _log(rng, 1024, 16384) // blk
        feat = 32 * _log(rng, 2, 128)
        density = round(rng.uniform(0.04, 0.25), 3)
        most = 0.1 * 512 * 512 * 32 * 32 * 4096 / (4 if blk == 16 else 1)  # narrow blocks: less reuse per byte
        density = min(density, most / (rows * blk * cols * blk * feat))
        return dict(kind=kind, mb=rows, nb=cols, blk=blk, density=density, feat=feat,
                    dtype=rng.choice(["f16", "bf16"]))
    if kind == "tc":
        g = _graph(rng, 10000, 200000, 32, 256)
        g["feat"] = max(32, g["feat"] // 32 * 32)
        return dict(kind=kind, tile=rng.choice([8, 16, 32]), out=rng.choice(["f16", "f32"]), **g)
    nodes = _log(rng, 10000, 120000)
    edges = int(nodes * rng.uniform(5, 20))
    rels = rng.choice([8, 24, 50, 65, 90, 130])
    if kind == "rgms":
        dtype = rng.choice(["f16", "f16", "bf16"])
        out = rng.choice(["f32", "f16"]) if dtype == "f16" else "f32"
        return dict(kind=kind, nodes=nodes, rels=rels, edges=edges, fin=rng.choice([16, 32, 64]),
                    fout=rng.choice([32, 64]), dtype=dtype, out=out, static=rng.random() < 0.7)
    return dict(kind=kind, nodes=nodes, rels=rels, edges=edges, fin=rng.choice([16, 32, 32, 48, 64]),
                fout=rng.choice([8, 16, 32, 32, 64]))


# ---------------------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _skew_cdf(nodes, edges, alpha, max_deg, g):
    """Cumulative distribution over the nodes of weights (rank + shift)^-alpha; the shift keeps the
    expected degree of the heaviest node near ``max_deg``."""
    rank = torch.arange(1, nodes + 1, device=DEV, dtype=torch.float64)
    lo, hi = 0.0, float(nodes)
    for _ in range(40):
        mid = 0.5 * (lo + hi)
        w = (rank + mid).pow(-alpha)
        lo, hi = (mid, hi) if float(edges * w[0] / w.sum()) > max_deg else (lo, mid)
    w = (rank + hi).pow(-alpha)[torch.randperm(nodes, generator=g, device=DEV)]
    cdf = torch.cumsum(w / w.sum(), 0)
    cdf[-1] = 1.0
    return cdf


def _pick(cdf, count, g):
    u = torch.rand(count, generator=g, device=DEV, dtype=torch.float64)
    return torch.searchsorted(cdf, u, right=True).clamp_(max=cdf.numel() - 1)


def _csr(rows, cols, m):
    indptr = torch.zeros(m + 1, dtype=torch.int32, device=DEV)
    indptr[1:] = torch.cumsum(torch.bincount(rows, minlength=m), 0)
    return indptr, cols.to(torch.int32)


def _graph_csr(case, g):
    """(rows, cols) of a graph with exactly ``edges`` distinct edges, sorted by row, then column."""
    n, nnz = case["nodes"], case["edges"]
    cdf = _skew_cdf(n, nnz, case["alpha"], case["max_deg"], g)
    key = torch.empty(0, dtype=torch.int64, device=DEV)
    more = nnz + nnz // 50 + 64
    while True:
        rows = _pick(cdf, more, g)
        cols = (torch.randint(n, (more,), generator=g, device=DEV) if case["columns"] == "uniform"
                else _pick(cdf, more, g))
        key = torch.unique(torch.cat([key, rows.mul_(n).add_(cols)]))
        if key.numel() >= nnz:
            break
        more = 2 * (nnz - key.numel()) + 64
    extra = key.numel() - nnz
    if extra:  # leave out as many edges as there are too many, anywhere
        keep = torch.ones(key.numel(), dtype=torch.bool, device=DEV)
        keep[torch.randperm(key.numel(), generator=g, device=DEV)[:extra]] = False
        key = key[keep]
    return key // n, key % n


def _csf(case, g):
    """CSF arrays of a relational graph: edges split over the relations by Zipf(1)."""
    n, R, E = case["nodes"], case["rels"], case["edges"]
    w = 1.0 / torch.arange(1, R + 1, device=DEV, dtype=torch.float64)
    cdf = torch.cumsum(w / w.sum(), 0)
    rel = _pick(cdf, E, g)
    dst = torch.randint(n, (E,), generator=g, device=DEV)
    src = torch.randint(n, (E,), generator=g, device=DEV)
    key = torch.unique((rel * n + dst) * n + src)
    pair, src = key // n, key % n
    pair, counts = torch.unique_consecutive(pair, return_counts=True)
    indptr0, _ = _csr(pair // n, pair, R)
    indptr1 = torch.zeros(pair.numel() + 1, dtype=torch.int32, device=DEV)
    indptr1[1:] = torch.cumsum(counts, 0)
    i32 = lambda a: a.to(torch.int32)
    return indptr0, i32(pair % n), indptr1, i32(src)


def prepare(case, seed):
    g = _generator(seed)
    return globals()["_prepare_" + case["kind"]](case, g)


def _prepare_csr(case, g):
    n, f, nnz = case["nodes"], case["feat"], case["edges"]
    rows, cols = _graph_csr(case, g)
    indptr, indices = _csr(rows, cols, n)
    return dict(run=_run_csr, f=ops.build_csrmm(n, n, f, nnz), a=_rand(g, nnz), x=_randn(g, n * f),
                c=torch.empty(n * f, device=DEV), indptr=indptr, indices=indices)


def _hyb_arguments(rows, cols, values):
    """Flat (A_k, rows_k, cols_k) arguments of the hyb operator and the ELL rows per bucket."""
    flat, nrows = [], []
    for row_p, col_p, val_p in zip(rows, cols, values):
        for r, c, v in zip(row_p, col_p, val_p):
            flat += [v.reshape(-1), r, c.reshape(-1)]
            nrows.append(r.shape[0])
    return flat, nrows


def _prepare_hyb(case, g):
    n, f, nnz = case["nodes"], case["feat"], case["edges"]
    indptr, indices = _csr(*_graph_csr(case, g), n)
    _, widths = st.suggest_decomposition(n, n, nnz, f)
    rows, cols, _, values = st.column_part_hyb(n, n, indptr, indices, case["parts"], widths, _rand(g, nnz))
    flat, nrows = _hyb_arguments(rows, cols, values)
    return dict(run=_run_hyb, f=ops.build_hyb_csrmm(n, n, f, case["parts"], widths, nrows), flat=flat,
                x=_randn(g, n * f), c=torch.zeros(n * f, device=DEV))


def _prepare_train(case, g):
    n, f, nnz = case["nodes"], case["feat"], case["edges"]
    rows, cols = _graph_csr(case, g)
    indptr, indices = _csr(rows, cols, n)
    order = torch.argsort(cols, stable=True)  # the transposed matrix, made once per graph
    t_indptr, t_indices = _csr(cols[order], rows[order], n)
    a = _rand(g, nnz)
    mid = torch.empty(nnz, dtype=torch.int32, device=DEV)
    da = torch.empty(nnz, device=DEV)
    x, dy = _randn(g, n * f), _randn(g, n * f)
    ops.build_sddmm_preproc(n, n, f, nnz)(dy, x, da, indptr, indices, mid)
    return dict(run=_run_train, spmm=ops.build_csrmm(n, n, f, nnz), sddmm=ops.build_sddmm(n, n, f, nnz), a=a,
                a_t=a[order].contiguous(), indptr=indptr, indices=indices, t_indptr=t_indptr, t_indices=t_indices,
                mid=mid, x=x, dy=dy, y=torch.empty(n * f, device=DEV), dx=torch.empty(n * f, device=DEV), da=da)


def _prepare_sddmm(case, g):
    n, f, nnz = case["nodes"], case["feat"], case["edges"]
    indptr, indices = _csr(*_graph_csr(case, g), n)
    x, y = _randn(g, n * f), _randn(g, n * f)
    mid = torch.empty(nnz, dtype=torch.int32, device=DEV)
    c = torch.empty(nnz, device=DEV)
    ops.build_sddmm_preproc(n, n, f, nnz)(x, y, c, indptr, indices, mid)
    build = ops.build_sddmm_scaled if case["scaled"] else ops.build_sddmm
    args = [x, y, c, indptr, indices, mid] + ([_rand(g, nnz)] if case["scaled"] else [])
    return dict(run=_run_sddmm, f=build(n, n, f, nnz), args=args, c=c)


def _prepare_minibatch(case, g):
    m, n, f = case["rows"], case["cols"], case["feat"]
    deg = torch.randint(1, case["fanout"] + 1, (m,), generator=g, device=DEV)
    rows = torch.repeat_interleave(torch.arange(m, device=DEV), deg)
    cols = torch.randint(n, (rows.numel(),), generator=g, device=DEV)
    key = torch.unique(rows * n + cols)
    indptr, indices = _csr(key // n, key % n, m)
    return dict(run=_run_minibatch, m=m, n=n, feat=f, indptr=indptr, indices=indices, a=_rand(g, indices.numel()),
                x=_randn(g, n * f))


def _prepare_bsr(case, g):
    mb, nb, blk, f, dt = case["mb"], case["nb"], case["blk"], case["feat"], DTYPES[case["dtype"]]
    rows, cols = (_rand(g, mb, nb) < case["density"]).nonzero(as_tuple=True)
    indptr, indices = _csr(rows, cols, mb)
    nnzb = indices.numel()
    return dict(run=_run_bsr, f=ops.build_bsrmm(mb, nb, nnzb, blk, f, dt),
                a=(_randn(g, nnzb * blk * blk) * 0.02).to(dt), x=_randn(g, nb * blk * f).to(dt),
                y=torch.empty(mb * blk * f, dtype=dt, device=DEV), indptr=indptr, indices=indices)


def _prepare_tc(case, g):
    n, f, t, out = case["nodes"], case["feat"], case["tile"], DTYPES[case["out"]]
    indptr, indices = _csr(*_graph_csr(case, g), n)
    gptr, tiles, mask = st.condense(indptr, indices, t, 16)
    mb = gptr.numel() - 1
    return dict(run=_run_tc, f=ops.build_tcspmm(mb, tiles.shape[0], f, t, 16, n, out),
                a=(mask * _rand(g, *mask.shape)).reshape(-1).half(), b=_randn(g, n * f).half(),
                c=torch.empty(mb * t * f, dtype=out, device=DEV), indptr=gptr, indices=tiles.reshape(-1))


def _prepare_rgms(case, g):
    n, R, fin, fout, dt = case["nodes"], case["rels"], case["fin"], case["fout"], DTYPES[case["dtype"]]
    rows_bkt = [ELL3D_GROUP // w for w in ELL3D_WIDTHS]
    ptr, rows, cols, mask = st.csf_to_ell3d(*_csf(case, g), rows_bkt, ELL3D_WIDTHS)
    rel = torch.arange(R, dtype=torch.int32, device=DEV)
    flat, mids = [], []
    for p, r, c, k in zip(ptr, rows, cols, mask):
        flat += [k.reshape(-1).to(dt), r.reshape(-1), c.reshape(-1)]
        mids.append(torch.repeat_interleave(rel, (p[1:] - p[:-1]).long()))
    f = ops.build_rgms(n, n, R, fin, fout, rows_bkt, ELL3D_WIDTHS, [c.shape[0] for c in cols], dt,
                       static_weights=case["static"], out_dtype=DTYPES[case["out"]])
    return dict(run=_run_rgms, f=f, w=(_randn(g, R * fin * fout) * 0.1).to(dt), x=_randn(g, n * fin).to(dt),
                y=torch.zeros(n * fout, dtype=DTYPES[case["out"]], device=DEV), rest=flat + mids)


def _prepare_rgms_f32(case, g):
    n, R, fin, fout = case["nodes"], case["rels"], case["fin"], case["fout"]
    csf = _csf(case, g)
    stored, nnz = csf[1].numel(), csf[3].numel()
    return dict(run=_run_rgms_f32, f=ops.build_rgms_csf(n, n, R, fin, fout, stored, nnz), a=_rand(g, nnz),
                w=_randn(g, R * fout * fin) * 0.1, x=_randn(g, n * fin), y=torch.zeros(n * fout, device=DEV), csf=csf)


# ---------------------------------------------------------------------------------- one pass
def run(state):
    return state["run"](state)


def _run_csr(s):
    s["f"](s["a"], s["x"], s["c"], s["indptr"], s["indices"])
    return s["c"]


def _run_hyb(s):
    s["c"].zero_()
    s["f"](s["x"], s["c"], *s["flat"])
    return s["c"]


def _run_train(s):
    s["spmm"](s["a"], s["x"], s["y"], s["indptr"], s["indices"])
    s["spmm"](s["a_t"], s["dy"], s["dx"], s["t_indptr"], s["t_indices"])
    s["sddmm"](s["dy"], s["x"], s["da"], s["indptr"], s["indices"], s["mid"])
    return s["y"], s["dx"], s["da"]


def _run_sddmm(s):
    s["f"](*s["args"])
    return s["c"]


def _run_minibatch(s):
    m, n, f = s["m"], s["n"], s["feat"]
    parts, widths = st.suggest_decomposition(m, n, s["indices"].numel(), f)
    rows, cols, _, values = st.column_part_hyb(m, n, s["indptr"], s["indices"], parts, widths, s["a"])
    flat, nrows = _hyb_arguments(rows, cols, values)
    c = torch.zeros(m * f, device=DEV)
    ops.build_hyb_csrmm(m, n, f, parts, widths, nrows)(s["x"], c, *flat)
    return c


def _run_bsr(s):
    s["f"](s["a"], s["x"], s["y"], s["indptr"], s["indices"])
    return s["y"]


def _run_tc(s):
    s["f"](s["a"], s["b"], s["c"], s["indptr"], s["indices"])
    return s["c"]


def _run_rgms(s):
    s["y"].zero_()
    s["f"](s["w"], s["x"], s["y"], *s["rest"])
    return s["y"]


def _run_rgms_f32(s):
    s["y"].zero_()
    s["f"](s["a"], s["w"], s["x"], s["y"], *s["csf"])
    return s["y"]


# ---------------------------------------------------------------------------------- what a pass needs
def work(case):
    """Each input read once, each output written once; padding and gathered repeats not counted."""
    kind = case["kind"]
    if kind in ("csr", "hyb"):
        n, e, f = case["nodes"], case["edges"], case["feat"]
        return {"bytes": 8 * e + 4 * (n + 1) + 8 * n * f, "flops": 2 * e * f}
    if kind == "train":
        n, e, f = case["nodes"], case["edges"], case["feat"]
        return {"bytes": 28 * e + 8 * (n + 1) + 4 * 4 * n * f, "flops": 6 * e * f}
    if kind == "sddmm":
        n, e, f = case["nodes"], case["edges"], case["feat"]
        return {"bytes": (16 if case["scaled"] else 12) * e + 8 * n * f, "flops": 2 * e * f}
    if kind == "minibatch":
        m, n, f = case["rows"], case["cols"], case["feat"]
        e = m * (case["fanout"] + 1) // 2
        reached = n * (1 - math.exp(-e / n))  # rows of X that some edge reads
        return {"bytes": 8 * e + 4 * (m + 1) + 4 * f * (reached + m), "flops": 2 * e * f}
    if kind == "bsr":
        mb, nb, blk, f = case["mb"], case["nb"], case["blk"], case["feat"]
        nnzb = mb * nb * case["density"]
        return {"bytes": 2 * nnzb * blk * blk + 4 * nnzb + 4 * (mb + 1) + 2 * (nb + mb) * blk * f,
                "flops": 2 * nnzb * blk * blk * f}
    if kind == "tc":
        n, e, f = case["nodes"], case["edges"], case["feat"]
        return {"bytes": 6 * e + 2 * n * f + (2 if case["out"] == "f16" else 4) * n * f, "flops": 2 * e * f}
    n, R, e, fin, fout = case["nodes"], case["rels"], case["edges"], case["fin"], case["fout"]
    size = 4 if kind == "rgms_f32" else 2
    y = 2 if case.get("out") == "f16" else 4
    return {"bytes": 8 * e + size * (n * fin + R * fin * fout) + y * n * fout, "flops": 2 * e * fin * fout + 2 * e * fout}


def tolerance(case):
    if case["kind"] == "bsr":
        return {"rel": 8e-3} if case["dtype"] == "bf16" else {"rel": 1e-3}
    if case.get("out") == "f16":
        # one rounding of fp32 sums; the relational layer may round once per part of a row
        return {"rel": 4e-3 if case["kind"] == "rgms" else 1e-3}
    return {"rel": 1e-5}
