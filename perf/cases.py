"""The work that users of this library have it do, as cases that can be timed and compared.

A case is a dict of plain values: `kind` names the entry point and the other fields the sizes and
options it is called with.

  kind      entry point (public Python API)                         what it stands for
  dropin    networkit_amd.centrality.PageRank(G).run(), scores()    a script that ranks one small
                                                                    NetworKit graph: export, upload,
                                                                    solve, result, all in the call
  solve     capi.DeviceGraph.run on a resident handle               PageRank again and again on one
                                                                    graph (other options, other
                                                                    starts), scores kept on the GPU
  first     capi.DeviceGraph(...) and its first run                 one PageRank of lists that some
                                                                    other GPU code produced
  ppr       capi.DeviceGraph.ppr_batch                              personalised PageRank of many
                                                                    users (seed sets) at once
  batch     capi.DeviceGraph.run_batch                              features of many small graphs
  grad      autograd.PageRankOperator, forward and backward         a training step on edge weights
  power     capi.DeviceGraph.power_run                              eigenvector and Katz centrality
  csr       capi.DeviceCSR.pagerank_step / spmv                     products with NetworKit's CSR
                                                                    matrix (AlgebraicPageRank)
  apr       capi.DeviceAPR.run                                      local clustering around a seed

Graphs: `rmat` is the benchmark's generator (power-law degrees, sinks; a node count that is not a
power of two takes the arcs among the first n nodes), `rhg` the random hyperbolic graph
(undirected, clustered, slowly mixing), `er` Erdos-Renyi with multi-edges removed (undirected, near
regular) and `ba` Barabasi-Albert (undirected).
"""
import math

import numpy as np
import torch

import networkit_amd as nk
from networkit_amd import autograd, capi, generators

DEV = "cuda"
PRECISION = {"fp64": capi.NKPR_FP64, "mixed": capi.NKPR_MIXED}


# ---- the cases --------------------------------------------------------------------------------

def listed():
    return [
        # a small graph through the drop-in API: everything a script pays for, every call
        dict(name="dropin_small", kind="dropin", n=1500, deg=6, weighted=True, directed=True),
        # a small resident graph with the library's defaults (FP64, L2 step): launches and latency
        dict(name="solve_small", kind="solve", graph="rmat", n=20011, deg=8, weighted=False,
             precision="fp64", norm=1, sinks=0, normalized=False, tol=1e-8),
        # an ordinary weighted graph, FP64, Google-matrix sinks; 1.4e7 arcs (odd node count)
        dict(name="solve_medium", kind="solve", graph="rmat", n=900001, deg=16, weighted=True,
             precision="fp64", norm=0, sinks=1, normalized=False, tol=1e-8),
        # an unweighted clustered graph to a certified error
        dict(name="solve_rhg", kind="solve", graph="rhg", n=1500007, deg=20, weighted=False,
             precision="mixed", norm=1, sinks=0, normalized=False, tol=1e-8),
        # the largest: the benchmark's generator at scale 25, 5.3e8 weighted arcs, certified
        dict(name="solve_large", kind="solve", graph="rmat", n=1 << 25, deg=16, weighted=True,
             precision="mixed", norm=1, sinks=0, normalized=False, tol=1e-8),
        # one certified PageRank of lists on the GPU, with the handle built for it
        dict(name="first_solve", kind="first", graph="rmat", n=1 << 20, deg=16, weighted=True,
             precision="mixed", tol=1e-8),
        # 96 users' seed sets on a Barabasi-Albert graph
        dict(name="ppr_users", kind="ppr", n=150000, k=96, seeds=100, precision="mixed", tol=1e-8),
        # 160 small graphs in one handle with the reference's rule
        dict(name="batch_graphs", kind="batch", graphs=160, lo=500, hi=16000, deg=12,
             weighted=False, precision="fp64", tol=1e-8),
        # a training step: scores forward, gradients of weights and teleport backward
        dict(name="train_step", kind="grad", n=300007, deg=16, tol=1e-8, teleport=True),
        # eigenvector centrality of a large weighted graph, 1.3e8 arcs
        dict(name="eigenvector_large", kind="power", n=1 << 23, deg=16, weighted=True,
             centrality="eigenvector", tol=1e-9),
        # one AlgebraicPageRank iteration on a CSR matrix of 1e6 rows
        dict(name="csr_step", kind="csr", n=1000003, deg=16, op="step"),
        # one seed's approximate PageRank vector on a graph of 2e6 nodes
        dict(name="apr_seed", kind="apr", n=2000003, deg=20, seeds=1, alpha=0.1, eps=1e-8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin", "solve", "solve", "solve", "first", "ppr", "batch", "grad",
                       "power", "csr", "apr"])
    if kind == "dropin":
        return dict(kind=kind, n=_log(rng, 200, 20000), deg=rng.randint(2, 16),
                    weighted=rng.random() < 0.5, directed=rng.random() < 0.5)
    if kind == "solve":
        graph = rng.choice(["rmat", "rmat", "er", "rhg"])
        precision = rng.choice(["fp64", "mixed"])
        n = _log(rng, 1 << 11, 1 << (22 if precision == "fp64" else 23))
        if rng.random() < 0.2:
            n = 1 << max(11, n.bit_length() - 1)
        return dict(kind=kind, graph=graph, n=max(n, 20000) if graph == "rhg" else n,
                    deg=rng.randint(4, 24), weighted=graph == "rmat" and rng.random() < 0.6,
                    precision=precision, norm=rng.randint(0, 1),
                    sinks=int(rng.random() < 0.3), normalized=rng.random() < 0.3,
                    tol=rng.choice([1e-6, 1e-8, 1e-9]))
    if kind == "first":
        graph = rng.choice(["rmat", "rhg"])
        return dict(kind=kind, graph=graph, n=_log(rng, 1 << 15, 1 << 22), deg=rng.randint(4, 20),
                    weighted=graph == "rmat", precision=rng.choice(["fp64", "mixed"]), tol=1e-8)
    if kind == "ppr":
        k = _log(rng, 1, 160)
        return dict(kind=kind, n=min(_log(rng, 5000, 250000), 24000000 // k), k=k,
                    seeds=_log(rng, 1, 500), precision=rng.choice(["fp64", "mixed"]), tol=1e-8)
    if kind == "batch":
        hi = _log(rng, 500, 60000)
        return dict(kind=kind, graphs=min(_log(rng, 8, 400), 8000000 // hi), lo=max(2, hi // 20),
                    hi=hi, deg=rng.randint(3, 16), weighted=rng.random() < 0.4,
                    precision=rng.choice(["fp64", "mixed"]), tol=1e-8)
    if kind == "grad":
        return dict(kind=kind, n=_log(rng, 1 << 12, 1 << 20), deg=rng.randint(6, 16), tol=1e-8,
                    teleport=rng.random() < 0.5)
    if kind == "power":
        return dict(kind=kind, n=_log(rng, 1 << 13, 1 << 22), deg=rng.randint(6, 16),
                    weighted=rng.random() < 0.6, centrality=rng.choice(["eigenvector", "katz"]),
                    tol=rng.choice([1e-8, 1e-9]))
    if kind == "csr":
        return dict(kind=kind, n=_log(rng, 1 << 11, 1 << 22), deg=rng.randint(3, 40),
                    op=rng.choice(["step", "spmv"]))
    return dict(kind="apr", n=_log(rng, 20000, 1 << 21), deg=rng.randint(8, 24),
                seeds=rng.randint(1, 8), alpha=rng.choice([0.05, 0.1, 0.2]),
                eps=rng.choice([1e-6, 1e-7, 1e-8]))


# ---- inputs (plain lists on the GPU, made from the seed alone) ---------------------------------

def _csc(n, row, src, weight=None):
    """In-lists (rows ascending, sources ascending) of distinct arcs src -> row."""
    key = torch.sort(row * n + src)[0]
    row = torch.div(key, n, rounding_mode="floor")
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    return dict(z=n, colptr=ptr, src=(key - row * n).to(torch.int32), weight=weight)


def _undirected(n, u, v):
    """In-lists of the undirected graph with edges {u, v}: loops and repeats removed."""
    keep = u != v
    u, v = torch.minimum(u, v)[keep], torch.maximum(u, v)[keep]
    key = torch.unique(u * n + v)
    u = torch.div(key, n, rounding_mode="floor")
    v = key - u * n
    return _csc(n, torch.cat([u, v]), torch.cat([v, u]))


def _graph(case, seed):
    kind, n, deg = case.get("graph", "rmat"), case["n"], case["deg"]
    gseed = 1000003 * (seed % 100003) + 17
    if kind == "rhg":
        return generators.rhg(n, float(deg), 3.0, gseed)
    if kind == "er":
        g = torch.Generator(device=DEV).manual_seed(gseed)
        e = torch.randint(n, (2, n * deg // 2), generator=g, device=DEV)
        return _undirected(n, e[0], e[1])
    scale = max(1, (n - 1).bit_length())
    g = generators.rmat(scale, deg, gseed, weighted=case.get("weighted", True), device=DEV)
    if g["z"] != n:
        ends = int(g["colptr"][n])
        keep = g["src"][:ends] < n
        rows = _rows(g)[:ends][keep]
        ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
        ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
        g = dict(z=n, colptr=ptr, src=g["src"][:ends][keep].contiguous(),
                 weight=None if g["weight"] is None else g["weight"][:ends][keep].contiguous())
    return g


def _rows(g):
    return torch.repeat_interleave(torch.arange(g["z"], device=DEV), torch.diff(g["colptr"]))


def _host_edges(case, seed):
    """A host edge list: power-law-ish sources, distinct arcs, a few sinks."""
    rng = np.random.default_rng(seed)
    n, m = case["n"], case["n"] * case["deg"]
    u = np.minimum((n * rng.random(m) ** 1.7).astype(np.int64), n - 1)
    v = rng.integers(0, n, m)
    key = np.unique((u * n + v)[u != v])
    w = rng.uniform(0.5, 1.5, len(key)) if case["weighted"] else None
    order = rng.permutation(len(key))
    key = key[order]
    return key // n, key % n, w


def _ppr_inputs(case, seed):
    n = case["n"]
    u, v = generators.barabasi_albert(n, 8, seed % 100003 + 1)
    g = _undirected(n, torch.from_numpy(u).to(DEV), torch.from_numpy(v).to(DEV))
    rng = np.random.default_rng(seed)
    most = min(2 * case["seeds"], n)
    seeds = [rng.choice(n, int(rng.integers(1, most + 1)), replace=False)
             for _ in range(case["k"])]
    return g, seeds


def _batch_inputs(case, seed):
    # the sizes are the case's, so that every seed's union has as many nodes
    sizes = np.random.default_rng(case["hi"]).integers(case["lo"], case["hi"] + 1, case["graphs"])
    offs = np.zeros(case["graphs"] + 1, dtype=np.int64)
    offs[1:] = np.cumsum(sizes)
    n = int(offs[-1])
    size = torch.from_numpy(sizes).to(DEV)
    base = torch.from_numpy(offs[:-1]).to(DEV)
    which = torch.repeat_interleave(torch.arange(case["graphs"], device=DEV),
                                    size * case["deg"] // 2)
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = torch.rand(2, which.numel(), generator=g, device=DEV, dtype=torch.float64)
    e = torch.minimum((r * size[which]).long(), size[which] - 1) + base[which]
    out = _undirected(n, e[0], e[1])
    if case["weighted"]:
        # a weight per edge, the same in both directions
        a, b = _rows(out), out["src"].long()
        h = (torch.minimum(a, b) * 40503 + torch.maximum(a, b) * 2654435761) % 65521
        out["weight"] = (0.5 + h.double() / 65521).float()
    return out, offs


def _grad_inputs(case, seed):
    g = _graph(dict(case, weighted=True), seed)
    # every seed has as many arcs: evenly spread ones of those the generator made
    rows, m = _rows(g), int(0.6 * case["n"] * case["deg"])
    if rows.numel() < m:
        raise ValueError("the generator made only %d arcs" % rows.numel())
    keep = torch.div(torch.arange(m, device=DEV) * rows.numel(), m, rounding_mode="floor")
    g["colptr"] = torch.zeros_like(g["colptr"])
    g["colptr"][1:] = torch.cumsum(torch.bincount(rows[keep], minlength=case["n"]), 0)
    g["src"], g["weight"] = g["src"][keep], g["weight"][keep]
    gen = torch.Generator(device=DEV).manual_seed(seed + 1)
    # the loss is a linear functional of the scores (a ranking target), as a learner sends back
    c = torch.randn(case["n"], generator=gen, device=DEV)
    t = None
    if case["teleport"]:
        t = torch.rand(case["n"], generator=gen, device=DEV, dtype=torch.float64) + 0.1
        t /= t.sum()
    return g, c, t


def _csr_inputs(case, seed):
    g = _graph(dict(case, weighted=True), seed)
    n = case["n"]
    deg = torch.zeros(n, dtype=torch.float64, device=DEV)
    src = g["src"].long()
    w = g["weight"].double()
    deg.index_add_(0, src, w)
    gen = torch.Generator(device=DEV).manual_seed(seed + 1)
    x = torch.rand(n, generator=gen, device=DEV, dtype=torch.float64)
    return g["colptr"], src, 0.85 * w / deg[src], x / x.sum()


def _apr_inputs(case, seed):
    g = generators.rhg(case["n"], float(case["deg"]), 3.0, 1000003 * (seed % 100003) + 17)
    deg = torch.diff(g["colptr"])
    rng = np.random.default_rng(seed)
    ids = torch.nonzero(deg > 0).flatten()
    at = rng.choice(int(ids.numel()), case["seeds"], replace=False)
    return g, ids[torch.from_numpy(at).to(DEV)].cpu().numpy()


def _power_alpha(g):
    """Katz: 1 / (1 + the largest out-degree), the reference's default."""
    return 1.0 / (1 + int(torch.bincount(g["src"].long(), minlength=g["z"]).max()))


# ---- prepare and run ---------------------------------------------------------------------------

def _solve_params(case):
    mixed = case["precision"] == "mixed"
    return capi.default_params(
        tol=case["tol"], norm=case.get("norm", 1), sink_handling=case.get("sinks", 0),
        normalized=int(case.get("normalized", False)), precision=PRECISION[case["precision"]],
        stop=capi.NKPR_STOP_L1_ERROR if mixed else capi.NKPR_STOP_STEP, scores_on_device=1)


def _handle(g, **kw):
    torch.cuda.synchronize()
    return capi.DeviceGraph(g["z"], g["colptr"], g["src"], g["weight"], device=True, **kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dropin":
        u, v, w = _host_edges(case, seed)
        G = nk.Graph(case["n"], case["weighted"], case["directed"])
        G.addEdges(u, v, w)
        return dict(kind=kind, G=G)
    if kind == "solve":
        h = _handle(_graph(case, seed))
        return dict(kind=kind, h=h, p=_solve_params(case),
                    x=torch.empty(case["n"], dtype=torch.float64, device=DEV))
    if kind == "first":
        g = _graph(case, seed)
        torch.cuda.synchronize()
        return dict(kind=kind, g=g, p=_solve_params(case),
                    x=torch.empty(case["n"], dtype=torch.float64, device=DEV))
    if kind == "ppr":
        g, seeds = _ppr_inputs(case, seed)
        return dict(kind=kind, h=_handle(g), seeds=seeds, p=_solve_params(case),
                    x=torch.empty((case["k"], case["n"]), dtype=torch.float64, device=DEV))
    if kind == "batch":
        g, offs = _batch_inputs(case, seed)
        size = torch.from_numpy(np.diff(offs)).to(DEV)
        start = torch.repeat_interleave(1.0 / size.double(), size)
        h = _handle(g, graph_offsets=offs.astype(np.uint64))
        return dict(kind=kind, h=h, p=_solve_params(case), start=start,
                    x=torch.empty_like(start))
    if kind == "grad":
        g, c, t = _grad_inputs(case, seed)
        op = autograd.PageRankOperator(g["colptr"], g["src"], tol=case["tol"])
        return dict(kind=kind, op=op, c=c, w=g["weight"].requires_grad_(),
                    t=None if t is None else t.requires_grad_())
    if kind == "power":
        g = _graph(case, seed)
        katz = case["centrality"] == "katz"
        h = _handle(g, out_wdeg=torch.ones(case["n"], dtype=torch.float64, device=DEV))
        p = capi.default_power_params(kind=capi.NKPR_KATZ if katz else capi.NKPR_EIGENVECTOR,
                                      alpha=_power_alpha(g) if katz else 0.0, tol=case["tol"],
                                      scores_on_device=1)
        return dict(kind=kind, h=h, p=p,
                    x=torch.empty(case["n"], dtype=torch.float64, device=DEV))
    if kind == "csr":
        ptr, col, val, x = _csr_inputs(case, seed)
        n = case["n"]
        return dict(kind=kind, op=case["op"], m=capi.DeviceCSR(n, n, ptr, col, val), x=x,
                    shift=0.15 / n, y=torch.empty_like(x),
                    sq=torch.empty(1, dtype=torch.float64, device=DEV))
    g, seeds = _apr_inputs(case, seed)
    torch.cuda.synchronize()
    h = capi.DeviceAPR(case["n"], g["colptr"], g["src"], None, device=True)
    return dict(kind="apr", h=h, seeds=seeds, alpha=case["alpha"], eps=case["eps"])


def run(s):
    kind = s["kind"]
    if kind == "dropin":
        pr = nk.centrality.PageRank(s["G"])
        pr.run()
        return np.array(pr.scores())
    if kind == "solve":
        s["x"].fill_(1.0 / s["x"].numel())
        torch.cuda.current_stream().synchronize()
        s["h"].run(s["x"], s["p"])
        return s["x"]
    if kind == "first":
        g = s["g"]
        h = capi.DeviceGraph(g["z"], g["colptr"], g["src"], g["weight"], device=True)
        s["x"].fill_(1.0 / s["x"].numel())
        torch.cuda.current_stream().synchronize()
        h.run(s["x"], s["p"])
        return s["x"]
    if kind == "ppr":
        s["x"].fill_(1.0 / s["x"].shape[1])
        torch.cuda.current_stream().synchronize()
        s["h"].ppr_batch(s["seeds"], scores=s["x"], params=s["p"])
        return s["x"]
    if kind == "batch":
        s["x"].copy_(s["start"])
        torch.cuda.current_stream().synchronize()
        s["h"].run_batch(s["x"], s["p"])
        return s["x"]
    if kind == "grad":
        x = s["op"](s["w"], s["t"])
        loss = torch.dot(x, s["c"].to(x.dtype))
        wanted = [s["w"]] if s["t"] is None else [s["w"], s["t"]]
        return [x.detach()] + list(torch.autograd.grad(loss, wanted))
    if kind == "power":
        s["h"].power_run(s["x"], s["p"])
        return s["x"]
    if kind == "csr":
        if s["op"] == "spmv":
            return s["m"].spmv(s["x"], y=s["y"])
        return s["m"].pagerank_step(s["x"], s["shift"], y=s["y"], step_sq=s["sq"])
    # the touched nodes' scores and residuals, as vectors over all nodes
    ids, p, r, _ = s["h"].run(s["seeds"], s["alpha"], s["eps"])
    out = np.zeros((2, s["h"].z))
    out[0, ids], out[1, ids] = p, r
    return out


# ---- what a pass cannot do without -------------------------------------------------------------

def work(case):
    """Bytes and operations of one pass.  An iterative solve reads the arcs (a 4-byte id, a 4-byte
    weight where there is one) and the vector once per product; the products are those of the
    method the case asks for: FP64 steps to the tolerance, or the fewer of a certified solve."""
    kind = case["kind"]
    if kind == "batch":
        n = case["graphs"] * (case["lo"] + case["hi"]) // 2
    else:
        n = case["n"]
    weighted = case.get("weighted", kind in ("grad", "csr"))
    undirected = case.get("graph") in ("er", "rhg") or kind == "batch"
    m = int(n * (16 if kind == "ppr" else case["deg"] *
                 (0.6 if kind == "grad" else 0.97 if undirected else 0.9)))
    mixed = case.get("precision") == "mixed" or kind == "grad"
    per_arc = 8 if weighted else 4
    sweep = m * per_arc + n * (8 if mixed else 16)
    flops = 2.0 * m
    if kind in ("dropin", "solve", "batch", "first"):
        steps = 14 if mixed else 30
        extra = 16 * n + (m * per_arc if kind == "first" else 0)
        return dict(bytes=steps * sweep + extra, flops=steps * flops)
    if kind == "ppr":
        steps, width = 20, 4 if mixed else 8
        return dict(bytes=steps * (4 * m + 2 * width * n * case["k"]) + 16 * n * case["k"],
                    flops=steps * flops * case["k"])
    if kind == "grad":
        # a solve forward and one backward, the gradient of every weight
        return dict(bytes=2 * 14 * sweep + 12 * m, flops=2 * 14 * flops)
    if kind == "power":
        steps = 18 if case["centrality"] == "eigenvector" else 6
        return dict(bytes=steps * sweep, flops=steps * flops)
    if kind == "csr":
        return dict(bytes=16 * m + 24 * n, flops=flops)
    # about 1 / (eps alpha) degree-weighted pushes at most, each arc pushed over at least once in
    # the ball that the seeds reach
    edges = min(1.0 / (case["eps"] * case["alpha"]) / 50, 2.0 * m)
    return dict(bytes=28 * edges, flops=2 * edges)


def tolerance(case):
    """Largest differences that another correct implementation would show, about four times those
    seen against `exact` and between two orders of the sums."""
    kind = case["kind"]
    if kind == "grad":
        # float32 scores and weight gradients (2.5e-8), solved to a relative residual of 1e-8
        return {"rel": 1e-7, "max": 2e-5}
    if kind == "apr":
        # residuals in 2^-62 units, rounded at every push: 9e-13 seen on the final residuals
        return {"rel": 4e-12, "max": 2e-10}
    if case.get("precision") == "mixed":
        # certified to an L1 error of tol; how far below it a solver ends depends on its steps
        return {"rel": 10 * case["tol"], "max": 1e3 * case["tol"]}
    return {"rel": 1e-13, "max": 4e-12}


# ---- the same in plain FP64 --------------------------------------------------------------------

PIECE = 256  # arcs of a row that are added one after another


class _Product:
    """x -> the sums over every row of coef * x[src], in FP64; `ptr` are the rows' offsets.  Rows
    are added in pieces and the pieces then, so that a long row does not hold the others up."""

    def __init__(self, ptr, src, coef):
        self.src, self.coef = src, coef
        count = torch.div(torch.diff(ptr) + PIECE - 1, PIECE, rounding_mode="floor")
        rows = torch.zeros_like(ptr)
        rows[1:] = torch.cumsum(count, 0)
        row = torch.repeat_interleave(torch.arange(count.numel(), device=DEV), count)
        at = torch.arange(row.numel(), device=DEV) - rows[row]
        pieces = torch.cat([ptr[row] + PIECE * at, ptr[-1:]])
        # a part of the offsets for each call of segment_reduce, which takes so many at most
        self.parts = []
        for offsets in (pieces, rows):
            cut = list(range(0, max(1, offsets.numel() - 1), 1 << 22)) + [offsets.numel() - 1]
            ends = offsets[torch.tensor(cut, device=DEV)].tolist()
            self.parts.append([(offsets[a:b + 1] - x, x, y) for a, b, x, y in
                               zip(cut, cut[1:], ends, ends[1:])])

    def __call__(self, x):
        v = x[self.src]
        if self.coef is not None:
            v = v * (self.coef if x.dim() == 1 else self.coef[:, None])
        for parts in self.parts:
            v = torch.cat([torch.segment_reduce(v[x:y], "sum", offsets=offsets, axis=0, initial=0,
                                                unsafe=True) for offsets, x, y in parts])
        return v


def _by_source(g):
    """The out-lists: offsets per source, the rows they go to and the weights."""
    order = torch.sort(g["src"], stable=True)[1]
    ptr = torch.zeros_like(g["colptr"])
    ptr[1:] = torch.cumsum(torch.bincount(g["src"], minlength=g["z"]), 0)
    w = torch.ones(order.numel(), dtype=torch.float64, device=DEV) if g["weight"] is None \
        else g["weight"].double()[order]
    return ptr, _rows(g)[order].to(torch.int32), w


def _degrees(g):
    """The weighted out-degrees and the nodes without out-arcs."""
    ptr, row, w = _by_source(g)
    count = torch.diff(ptr)
    deg = _Product(ptr, row, w)(torch.ones(g["z"], dtype=torch.float64, device=DEV))
    return deg, count == 0


def _coef(g, deg):
    w = 1.0 if g["weight"] is None else g["weight"].double()
    return w / deg[g["src"]]


def _pagerank(g, case, d=0.85, offsets=None):
    """The reference's iteration to its rule (fp64) or to 1e-14 (mixed), for every graph of a
    block-diagonal union whose nodes start at `offsets`."""
    n = g["z"]
    deg, sink = _degrees(g)
    product = _Product(g["colptr"], g["src"], _coef(g, deg))
    mixed = case["precision"] == "mixed"
    if offsets is None:
        offsets = torch.tensor([0, n], device=DEV)
    groups = offsets.numel() - 1
    size = torch.diff(offsets).double()
    group = torch.repeat_interleave(torch.arange(groups, device=DEV), torch.diff(offsets))
    total = _Product(offsets, torch.arange(n, device=DEV), None)
    x = (1.0 / size)[group]
    tele = ((1 - d) / size)[group]
    done = torch.zeros(groups, dtype=torch.bool, device=DEV)
    for it in range(400):
        y = d * product(x) + tele
        if case.get("sinks", 0):
            y += (d * total(x * sink) / size)[group]
        if groups > 1:
            y = torch.where(done[group], x, y)
        diff = y - x
        x = y
        if mixed:
            if it % 8 == 7 and float(diff.abs().sum()) <= 1e-14 * groups:
                break
        else:
            step = total(diff * diff).sqrt() if case.get("norm", 1) else total(diff.abs())
            done |= step <= case["tol"]
            if bool(done.all()):
                break
    if case.get("normalized"):
        factor = (1.0 / size) * ((1 - d) + d * total(x * sink))
    else:
        factor = total(x)
    return x / factor[group]


def _exact_grad(case, seed):
    g, c, t = _grad_inputs(case, seed)
    d, n, src = 0.85, case["n"], g["src"].long()
    deg, _ = _degrees(g)
    product = _Product(g["colptr"], g["src"], _coef(g, deg))
    ptr, to, w = _by_source(g)
    back = _Product(ptr, to, w / torch.repeat_interleave(deg, torch.diff(ptr)))
    base = torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV) if t is None else t
    y = base
    for _ in range(230):
        y = d * product(y) + (1 - d) * base
    s = y.sum()
    x = y / s
    gf = (c.double() - (c.double() * x).sum()) / s
    lam = gf
    for _ in range(230):
        lam = d * back(lam) + gf
    mu = back(lam)
    gw = d * y[src] / deg[src] * (lam[_rows(g)] - mu[src])
    return [x, gw] + ([] if t is None else [(1 - d) * lam])


def _exact_power(case, seed):
    g = _graph(case, seed)
    katz = case["centrality"] == "katz"
    alpha = _power_alpha(g) if katz else 1.0
    product = _Product(g["colptr"], g["src"],
                       None if g["weight"] is None else g["weight"].double())
    x = torch.ones(g["z"], dtype=torch.float64, device=DEV)
    old = 0.0
    for _ in range(2000):
        y = alpha * product(x + 1.0) + 0.1 if katz else product(x)
        length = float(y.norm())
        x = y if katz else y / length
        if abs(length - old) <= case["tol"]:
            break
        old = length
    return x / length if katz else (x.abs() if float(x[0]) < 0 else x)


def _exact_apr(case, seed):
    """The pushes a frontier at a time: every node at or above its threshold pushes the residual
    it holds at the start of the round."""
    g, seeds = _apr_inputs(case, seed)
    n, ptr, dst = case["n"], g["colptr"], g["src"].long()
    deg = torch.diff(ptr)
    vol = deg.double()
    alpha, eps = case["alpha"], case["eps"]
    r = torch.zeros(n, dtype=torch.float64, device=DEV)
    p = torch.zeros_like(r)
    front = torch.from_numpy(np.sort(seeds)).to(DEV)
    r[front] = 1.0 / front.numel()
    while front.numel():
        res = r[front]
        p[front] += alpha * res
        r[front] = (1 - alpha) * res / 2
        cnt = deg[front]
        first = torch.cumsum(cnt, 0) - cnt
        each = torch.repeat_interleave(torch.arange(front.numel(), device=DEV), cnt)
        arc = ptr[front][each] + torch.arange(each.numel(), device=DEV) - first[each]
        to = dst[arc]
        keep = to != front[each]
        to, each = to[keep], each[keep]
        r.index_add_(0, to, ((1 - alpha) * res / (2 * vol[front]))[each])
        near = torch.unique(torch.cat([to, front]))
        front = near[r[near] >= eps * vol[near]]
    return torch.stack([p, r])


def exact(case, seed):
    kind = case["kind"]
    if kind == "dropin":
        u, v, w = _host_edges(case, seed)
        n = case["n"]
        if not case["directed"]:
            u, v = np.concatenate([u, v]), np.concatenate([v, u])
            w = None if w is None else np.concatenate([w, w])
        w = np.ones(len(u)) if w is None else w
        deg = np.bincount(u, weights=w, minlength=n)
        x = np.full(n, 1.0 / n)
        while True:
            y = 0.85 * np.bincount(v, weights=w / deg[u] * x[u], minlength=n) + 0.15 / n
            step = float(np.sqrt(((y - x) ** 2).sum()))
            x = y
            if step <= 1e-8:
                return x / x.sum()
    if kind in ("solve", "first"):
        return _pagerank(_graph(case, seed), case)
    if kind == "ppr":
        g, seeds = _ppr_inputs(case, seed)
        n = case["n"]
        product = _Product(g["colptr"], g["src"], _coef(g, _degrees(g)[0]))
        out = []
        for a in range(0, case["k"], 32):
            part = seeds[a:a + 32]
            t = torch.zeros(n, len(part), dtype=torch.float64, device=DEV)
            for j, s in enumerate(part):
                t[torch.from_numpy(s).to(DEV), j] = 1.0 / len(s)
            x = torch.full_like(t, 1.0 / n)
            done = torch.zeros(len(part), dtype=torch.bool, device=DEV)
            for _ in range(300):
                y = torch.where(done, x, 0.85 * product(x) + 0.15 * t)
                diff = y - x
                x = y
                if case["precision"] == "mixed":
                    done = diff.abs().sum(0) <= 1e-14
                else:
                    done |= diff.square().sum(0).sqrt() <= case["tol"]
                if bool(done.all()):
                    break
            out.append((x / x.sum(0)).T)
        return torch.cat(out)
    if kind == "batch":
        g, offs = _batch_inputs(case, seed)
        return _pagerank(g, case, offsets=torch.from_numpy(offs).to(DEV))
    if kind == "grad":
        return _exact_grad(case, seed)
    if kind == "power":
        return _exact_power(case, seed)
    if kind == "csr":
        ptr, col, val, x = _csr_inputs(case, seed)
        y = _Product(ptr, col, val)(x)
        if case["op"] == "spmv":
            return y
        y += 0.15 / case["n"]
        return y, (y - x).square().sum().reshape(1)
    return _exact_apr(case, seed)
