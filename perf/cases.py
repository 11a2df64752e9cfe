"""The work a program built on pyglass_amd has it do, as cases to be timed.

Each case is one call (or one short sequence of calls) through the package's
public entry points:

  search   one host query per call (Searcher.search)
  host     a host batch (Searcher.batch_search)
  device   a device-resident batch (Searcher.search_batch_dev)
  efk      a device batch with per-query ef and k (Searcher.search_batch_efk_dev)
  served   queued requests through the Server (Server.replay, all queued at once)
  load     an index taken into service (Graph.from_arrays + Searcher)
  fit      k-means training (Clustering.fit)
  predict  nearest centroids (Clustering.predict)

Base rows and graphs come from fixed seeds (an index is built once and then
searched), queries and training rows from the case's seed.  The graphs are
built here in a second on the GPU, in the shape the index builders give: rows
of near neighbours, nearest first, with some long links and -1 padding, under
an HNSW hierarchy or a single entry point (NSG).
"""

from __future__ import annotations

import math
from collections import OrderedDict

import numpy as np
import torch

import pyglass_amd as pg

INT_QUANTS = ("SQ8U", "SQ4U", "SQ2U")
BITS = {"FP32": 32, "FP16": 16, "BF16": 16, "E5M2": 8, "SQ8U": 8, "SQ8": 8, "SQ6": 6, "SQ4U": 4, "SQ4": 4, "SQ2U": 2,
        "PQ8": 2}
REFINE_FACTOR = {"SQ8U": 1.5, "SQ8": 1.5, "SQ4U": 1.5, "PQ8": 1.5, "SQ2U": 3.0}
DEV = "cuda"


# ---- the cases --------------------------------------------------------------


def _search(name, call, n, dim, data, graph, degree, metric, quant, refine, factor, nq, ef, k, **more):
    return dict(name=name, kind="search", call=call, n=n, dim=dim, data=data, graph=graph, degree=degree,
                metric=metric, quant=quant, refine=refine, factor=float(factor), nq=nq, ef=ef, k=k, **more)


def listed():
    return [
        # The first call of every user: one query at the default ef, on the
        # host; all latency (copies, launch, one query's chain of expansions).
        _search("one_query", "search", 100_000, 128, "mixture", "hnsw", 32, "L2", "SQ8U", "", 0, 1, 32, 10),
        # A retrieval step of an application: a handful of 768-d embeddings.
        _search("few_embeddings", "host", 100_000, 768, "unit", "nsg", 48, "IP", "SQ8", "FP32", 0, 16, 64, 10),
        # Word-vector-like rows whose dimension is no multiple of 16, half
        # precision codes, an evaluation-sized host batch.
        _search("word_vectors", "host", 200_000, 100, "unit", "hnsw", 32, "IP", "FP16", "", 0, 1_000, 96, 10),
        # The headline benchmark: 10,000 queries on 1M x 128, SQ4U codes and
        # FP32 re-rank, in the launch shape optimize() settles on there.
        _search("headline_batch", "device", 1_000_000, 128, "mixture", "hnsw", 32, "L2", "SQ4U", "FP32", 8, 10_000,
                64, 10, team=8, waves=1, visited=2048),
        # Every query with its own ef (16-512) and k (1-100) over wide rows,
        # as a mixed request stream gives them.
        _search("mixed_ef_k", "efk", 100_000, 960, "gamma", "nsg", 64, "L2", "SQ8U", "", 0, 1_000, 512, 100),
        # Two-bit codes, deep search and a large batch: bulk offline lookup.
        _search("bulk_two_bit", "device", 1_000_000, 128, "mixture", "hnsw", 32, "L2", "SQ2U", "FP32", 4, 20_000,
                128, 10),
        # Embedding search in bulk: 768-d unit rows by inner product.
        _search("bulk_embeddings", "device", 100_000, 768, "unit", "nsg", 48, "IP", "SQ8", "FP32", 0, 4_000, 128, 10),
        # Six-bit codes of an uneven dimension, a mid-sized batch.
        _search("six_bit", "device", 300_000, 200, "mixture", "hnsw", 24, "L2", "SQ6", "", 0, 3_000, 64, 20),
        # A service under a backlog: requests of 1-32 queries, queued at once.
        _search("served_backlog", "served", 100_000, 128, "mixture", "hnsw", 32, "L2", "SQ4U", "FP32", 4, 16_000, 64,
                10),
        # Start-up of a service: graph and rows into device memory, rows encoded.
        dict(name="load_index", kind="load", n=500_000, dim=128, data="mixture", degree=32, metric="L2", quant="SQ4U",
             refine="FP32"),
        # Training of a coarse quantizer, and assigning rows to it.
        dict(name="kmeans_fit", kind="fit", n=200_000, dim=128, data="mixture", clusters=1024, epochs=10,
             init="random"),
        dict(name="kmeans_assign", kind="predict", n=200_000, dim=96, data="mixture", clusters=1000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["search"] * 9 + ["load", "fit", "predict"])
    data = rng.choice(["mixture", "mixture", "gamma", "unit"])
    if kind == "fit":
        dim, clusters = _log(rng, 16, 300), _log(rng, 16, 1024)
        n = max(4 * clusters, _log(rng, 5_000, 200_000))
        epochs = rng.randint(3, 10)
        while epochs * min(n, 100_000) * clusters * dim > 10 * 100_000 * 1024 * 128:
            clusters //= 2
        return dict(kind="fit", n=n, dim=dim, data=data, clusters=clusters, epochs=epochs,
                    init=rng.choice(["random", "random", "kmeans++"]) if clusters <= 256 else "random")
    if kind == "predict":
        dim = _log(rng, 16, 300)
        return dict(kind="predict", n=_log(rng, 1_000, 200_000), dim=dim, data=data, clusters=_log(rng, 16, 1024))
    quant = rng.choice(["SQ8U", "SQ8U", "SQ4U", "SQ4U", "SQ2U", "SQ8", "SQ8", "FP16", "FP32", "BF16", "E5M2", "SQ6", "SQ4",
                        "PQ8"])
    refine = rng.choice(["", "FP32", "FP16"]) if quant in REFINE_FACTOR else ""
    metric = rng.choice(["L2", "IP"]) if data == "unit" else "L2"
    dim = _log(rng, 24, 960)
    n = _log(rng, 10_000, min(1_000_000, 60_000_000 // dim))
    if quant == "PQ8":  # its codebooks are trained on the host
        dim = 4 * _log(rng, 8, 32)
        n = _log(rng, 10_000, 20_000)
    degree = rng.choice([16, 24, 32, 32, 48, 64])
    if kind == "load":
        return dict(kind="load", n=n, dim=dim, data=data, degree=degree, metric=metric, quant=quant, refine=refine)
    call = rng.choice(["search", "host", "host", "device", "device", "device", "efk", "served"])
    ef = _log(rng, 16, 512 if call in ("search", "efk") else 256)
    k = min(_log(rng, 1, 100), ef)
    nq = 1 if call == "search" else _log(rng, 2, max(4, min(20_000, 1_000_000 // ef, 50_000_000 // (ef * dim))))
    case = _search("", call, n, dim, data, rng.choice(["hnsw", "nsg"]), degree, metric, quant, refine,
                   rng.choice([0, 2, 4, 8]) if refine else 0, nq, ef, k)
    del case["name"]
    return case


# ---- rows and graphs --------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _rows(data, n, dim, seed):
    """n rows on the GPU; the mixture's centers are the same for every seed."""
    g = _gen(1_000_003 * dim + 17 * seed + 1)
    if data == "mixture":  # integer-valued, as byte descriptors are
        centers = torch.rand(1024, dim, device=DEV, generator=_gen(dim)) * 255
        x = centers[torch.randint(0, 1024, (n,), device=DEV, generator=g)]
        x += 20 * torch.randn(n, dim, device=DEV, generator=g)
        return x.clamp_(0, 255).round_()
    if data == "gamma":  # non-negative, of norm 10: the sum of two exponentials is Gamma(2)
        x = -torch.log1p(-torch.rand(n, dim, device=DEV, generator=g))
        x -= torch.log1p(-torch.rand(n, dim, device=DEV, generator=g))
        return x * (10 / x.norm(dim=1, keepdim=True))
    x = torch.randn(n, dim, device=DEV, generator=g)
    return x / x.norm(dim=1, keepdim=True)


def _nearest(x, nodes, deg):
    """For each of `nodes`, the deg nearest others among them (all pairs)."""
    y = x[nodes]
    sq = (y * y).sum(1)
    deg = min(deg, len(nodes) - 1)
    out = torch.empty(len(nodes), deg, dtype=torch.int64, device=DEV)
    step = max(1, (1 << 28) // len(nodes))
    for s in range(0, len(nodes), step):
        d = sq[None, :] - 2 * (y[s:s + step] @ y.T)
        d.diagonal(s).fill_(math.inf)
        out[s:s + step] = nodes[d.topk(deg, largest=False, sorted=True).indices]
    return out


def _adjacency(x, degree, g):
    """Rows of up to `degree` ids, nearest first, -1 padded: near neighbours
    found within groups of rows around random pivots (two groupings), then
    long links."""
    n, group = x.shape[0], 512
    near = degree * 3 // 8
    sq = (x * x).sum(1)
    ids, dist = [], []
    for _ in range(2):
        piv = x[torch.randint(0, n, (max(1, n // 256),), device=DEV, generator=g)]
        psq = (piv * piv).sum(1)
        home = torch.empty(n, dtype=torch.int64, device=DEV)
        step = max(1, (1 << 28) // len(piv))
        for s in range(0, n, step):
            home[s:s + step] = (psq[None, :] - 2 * (x[s:s + step] @ piv.T)).argmin(1)
        order = torch.sort(home, stable=True).indices
        order = torch.cat([order, order[: -n % group]]).view(-1, group)
        got = torch.empty(n, near, dtype=torch.int64, device=DEV)
        far = torch.empty(n, near, device=DEV)
        step = max(1, (1 << 27) // (group * max(group, x.shape[1])))
        for s in range(0, len(order), step):
            o = order[s:s + step]
            y = x[o]
            d = sq[o][:, None, :] + sq[o][:, :, None] - 2 * torch.bmm(y, y.transpose(1, 2).contiguous())
            d.masked_fill_(o[:, None, :] == o[:, :, None], math.inf)
            v, i = d.topk(near, largest=False, sorted=True)
            # the rows that fill up the last group have a place of their own
            at = o.reshape(-1)[: n - s * group]
            got[at] = o.gather(1, i.view(len(o), -1)).view(-1, near)[: len(at)]
            far[at] = v.view(-1, near)[: len(at)]
        ids.append(got)
        dist.append(far)
    longs = degree - 2 * near
    ids.append(torch.randint(0, n, (n, longs), device=DEV, generator=g))
    dist.append(torch.full((n, longs), 1e30, device=DEV))
    ids, dist = torch.cat(ids, 1), torch.cat(dist, 1)
    by_id = ids.argsort(dim=1, stable=True)
    ids, dist = ids.gather(1, by_id), dist.gather(1, by_id)
    bad = ids == torch.arange(n, device=DEV)[:, None]
    bad[:, 1:] |= ids[:, 1:] == ids[:, :-1]
    dist.masked_fill_(bad, math.inf)
    by_dist = dist.argsort(dim=1, stable=True)
    ids, dist = ids.gather(1, by_dist), dist.gather(1, by_dist)
    return ids.masked_fill_(dist.isinf(), -1).to(torch.int32).cpu().numpy()


def _hierarchy(x, up_k, g):
    """HNSW upper layers: 1 node in 32 on each level above the one below."""
    n = x.shape[0]
    levels = torch.zeros(n, dtype=torch.int32, device=DEV)
    nodes = torch.randperm(n, device=DEV, generator=g)
    per_level = []
    while len(nodes) // 32 >= 2:
        nodes = nodes[: len(nodes) // 32]
        levels[nodes] += 1
        per_level.append(nodes)
    lv = levels.cpu().numpy()
    first = np.concatenate([[0], np.cumsum(lv[:-1], dtype=np.int64)])
    lists = np.full((int(lv.sum()), up_k), -1, np.int32)
    for level, at in enumerate(per_level):
        nn = _nearest(x, at, up_k).to(torch.int32).cpu().numpy()
        lists[first[at.cpu().numpy()] + level, : nn.shape[1]] = nn
    return up_k, int(nodes[0]), lv, lists


_indexes = OrderedDict()  # base rows and graph arrays last used, on the host


def _index(n, dim, data, graph, degree):
    key = (n, dim, data, graph, degree)
    if key not in _indexes:
        x = _rows(data, n, dim, 1234)
        g = _gen(n + degree)
        adj = _adjacency(x, degree, g)
        if graph == "hnsw":
            upper, eps = _hierarchy(x, degree // 2, g), ()
        else:
            upper, eps = None, (int(((x - x.mean(0)) ** 2).sum(1).argmin()),)
        while len(_indexes) >= 2:
            _indexes.popitem(last=False)
        _indexes[key] = x.cpu().numpy(), adj, eps, upper
    _indexes.move_to_end(key)
    return _indexes[key]


# ---- preparing and running a case -------------------------------------------


def prepare(case, seed):
    if case["kind"] == "load":
        adj = _index(case["n"], case["dim"], case["data"], "hnsw", case["degree"])
        rows = _rows(case["data"], case["n"], case["dim"], seed + 2).cpu().numpy()
        return dict(case=case, rows=rows, adj=adj[1], upper=adj[3])
    if case["kind"] in ("fit", "predict"):
        rows = _rows(case["data"], case["n"], case["dim"], seed + 2).cpu().numpy()
        st = dict(case=case, rows=rows)
        if case["kind"] == "predict":  # a codebook fitted once, on other rows
            st["model"] = pg.Clustering(case["clusters"], 2)
            st["model"].fit(_rows(case["data"], 8 * case["clusters"], case["dim"], 1).cpu().numpy())
        return st
    rows, adj, eps, upper = _index(case["n"], case["dim"], case["data"], case["graph"], case["degree"])
    s = pg.Searcher(pg.Graph.from_arrays(adj, eps, upper), rows, case["metric"], case["quant"], case["refine"])
    s.set_ef(case["ef"])
    if case["factor"]:
        s.set_refine_factor(case["factor"])
    if "team" in case:  # a launch shape tuned once
        s.set_launch(case["team"], case["waves"])
        s.set_visited_capacity(case["visited"])
    nq, k = case["nq"], case["k"]
    q = _rows(case["data"], nq, case["dim"], seed + 100_000)
    st = dict(case=case, searcher=s)
    if case["call"] in ("search", "host", "served"):
        st["q"] = q.cpu().numpy()
        if case["call"] == "served":
            rng = np.random.default_rng(seed)
            sizes = []
            while sum(sizes) < nq:
                sizes.append(min(int(rng.integers(1, 33)), nq - sum(sizes)))
            st["sizes"] = np.array(sizes, np.int32)
            st["server"] = pg.Server(s, 4096, max(k, 10), 4)
        return st
    st["q"], total = q, nq * k
    if case["call"] == "efk":
        rng = np.random.default_rng(seed)
        ef = np.rint(np.exp(rng.uniform(math.log(min(16, case["ef"])), math.log(case["ef"]), nq))).astype(np.int32)
        kk = rng.permutation(np.linspace(1, k, nq).round().astype(np.int32))
        total = int(kk.sum())
        st["ef"], st["k"] = torch.from_numpy(ef).to(DEV), torch.from_numpy(kk).to(DEV)
        st["off"] = torch.from_numpy(np.cumsum(kk, dtype=np.int64) - kk).to(DEV)
    st["ids"] = torch.empty(total, dtype=torch.int32, device=DEV)
    st["dists"] = torch.empty(total, dtype=torch.float32, device=DEV)
    return st


def run(state):
    case = state["case"]
    if case["kind"] == "load":
        g = pg.Graph.from_arrays(state["adj"], (), state["upper"])
        s = pg.Searcher(g, state["rows"], case["metric"], case["quant"], case["refine"])
        return s.codes(), s.calibration()
    if case["kind"] == "fit":
        model = pg.Clustering(case["clusters"], case["epochs"], case["init"])
        model.fit(state["rows"])
        return model.centroids()
    if case["kind"] == "predict":
        return state["model"].predict(state["rows"])
    s, q = state["searcher"], state["q"]
    if case["call"] == "search":
        return s.search(q[0], case["k"])
    if case["call"] == "host":
        return s.batch_search(q, case["k"])
    if case["call"] == "served":
        sizes = state["sizes"]
        return state["server"].replay(q, sizes, case["ef"], case["k"], np.zeros(len(sizes), np.int64))[1:]
    stream = torch.cuda.current_stream().cuda_stream
    if case["call"] == "efk":
        s.search_batch_efk_dev(q.data_ptr(), case["nq"], state["ef"].data_ptr(), state["k"].data_ptr(),
                               state["off"].data_ptr(), state["ids"].data_ptr(), case["ef"], case["k"],
                               state["dists"].data_ptr(), stream=stream)
    else:
        s.search_batch_dev(q.data_ptr(), case["nq"], case["k"], state["ids"].data_ptr(), state["dists"].data_ptr(),
                           stream=stream)
    return state["ids"], state["dists"]


# ---- what a case cannot do without, and what it computes in 64 bits ----------


def work(case):
    n, dim = case["n"], case["dim"]
    if case["kind"] == "load":  # rows and graph in, codes and re-rank rows out
        out = n * dim * (BITS[case["quant"]] + {"": 0, "FP32": 32, "FP16": 16}[case["refine"]]) / 8
        return {"bytes": n * (4 * dim + 4 * case["degree"]) + out, "flops": 6 * n * dim}
    if case["kind"] in ("fit", "predict"):
        k = case["clusters"]
        m, sweeps = (min(n - 1, 100_000), case["epochs"]) if case["kind"] == "fit" else (n, 1)
        return {"bytes": sweeps * 4 * (m * dim + k * dim + m), "flops": 3 * sweeps * m * k * dim}
    # Graph search: an expansion reads its row of the graph, and about a third
    # of a row's neighbours are new and have their codes read; the re-rank
    # reads its rows.  The mean ef of a log-uniform mix from 16 lies near a
    # third of the largest, the mean k at half.
    ef, k = case["ef"], case["k"]
    if case["call"] == "efk":
        ef, k = max(1, ef / 3), k / 2
    evals = ef * case["degree"] / 3
    b = evals * dim * BITS[case["quant"]] / 8 + ef * 4 * case["degree"] + 4 * dim + 8 * k
    f = 3 * evals * dim
    if case["refine"]:
        m = k * (case["factor"] or REFINE_FACTOR[case["quant"]])
        b += m * dim * (4 if case["refine"] == "FP32" else 2)
        f += 3 * m * dim
    return {"bytes": case["nq"] * b, "flops": case["nq"] * f}


def _raw_draws(count):
    """The first outputs of a 32-bit Mersenne twister with its default seed."""
    return np.random.RandomState(5489).randint(0, 1 << 32, count, dtype=np.uint32).astype(np.int64)


def _sample(size, n, raw):
    """`size` distinct ids of n: sorted draws, made distinct, rotated."""
    at = np.sort(raw[:size] % (n - size))
    at = np.maximum.accumulate(at - np.arange(size)) + np.arange(size)
    return (at + raw[size] % n) % n


def exact(case, seed):
    """The values that exist in 64 bits: calibrations and k-means centroids.
    A graph search's answers depend on the path that its codes lead it along,
    and codes and ids are whole numbers: no 64-bit value."""
    if case["kind"] == "fit" and case["init"] == "random":
        rows = _rows(case["data"], case["n"], case["dim"], seed + 2)
        m = min(case["n"] - 1, 100_000)
        raw = _raw_draws(m + 1)
        x = rows[torch.from_numpy(_sample(m, case["n"], raw)).to(DEV)].double()
        c = x[torch.from_numpy(_sample(case["clusters"], m, raw)).to(DEV)].clone()
        for _ in range(case["epochs"]):
            near = torch.cat([((c * c).sum(1)[None, :] - 2 * (y @ c.T)).argmin(1) for y in x.split(1 << 14)])
            count = torch.bincount(near, minlength=len(c))
            c = torch.zeros_like(c).index_add_(0, near, x) / count.clamp(min=1)[:, None]
        return c.cpu().numpy()
    if case["kind"] == "load" and case["quant"] in ("SQ8U", "SQ4U", "SQ2U", "SQ8", "SQ6", "SQ4"):
        x = _rows(case["data"], case["n"], case["dim"], seed + 2).view(-1)
        quant, n, dim = case["quant"], case["n"], case["dim"]
        if quant == "SQ8U" and case["metric"] == "IP":
            return None, np.array([float(x.abs().max())])
        if quant in INT_QUANTS:
            items = len(x) if quant == "SQ8U" else int(np.float32(len(x)) * np.float32(0.1))
            ratio = {"SQ8U": 0.0, "SQ4U": 0.01, "SQ2U": 0.05}[quant]
            v = x[:items].sort().values
            top = int(np.float32(items) * np.float32(ratio)) + 1
            lo, hi = float(v[top - 1]), float(v[items - top])
            return None, np.array([lo, hi - lo])
        # per "dimension" j: the flattened items [j * n, (j + 1) * n)
        top = 1 if quant == "SQ8" else int(np.float32(n) * np.float32(0.01)) + 1
        v = x.view(dim, n).sort(1).values.double().cpu().numpy()
        width = 8 if quant == "SQ6" else 16
        out = np.zeros((2, -(-dim // width) * width))
        out[0, :dim], out[1, :dim] = v[:, top - 1], v[:, n - top] - v[:, top - 1]
        return None, out.reshape(-1)
    return None
