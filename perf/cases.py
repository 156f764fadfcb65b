"""What a user of ibfs_amd has it do, as cases that can be timed.

Every form of the framework appears: one group through the engine, a source
set in groups (the reference's form), the batched launcher, closeness without
depth arrays, the query server, the allocation-free call, depth arrays on the
host, and GroupBy.  Graphs are R-MAT (edge factor 16), Chung-Lu power law and
grid graphs from a thousand to four million vertices; source sets run from
one source to every vertex.

A small graph is made from the seed.  A large one is one fixed graph that stays
resident on the device while source sets of different seeds are run against it,
as a program that serves or analyses one graph keeps it.  Depth arrays go to a
torch tensor, which a program that works on them has.
"""
from functools import lru_cache

import numpy as np
import torch

import ibfs_amd

SMALL = 100_000  # vertices: graphs up to this size are made from the seed


def listed():
    return [
        # the smallest call: one BFS on a small graph, latency alone
        dict(name="one_source", form="engine", graph="rmat", scale=16, n=1, lanes=128),
        # one full group of the reference's concurrent count on a small graph
        dict(name="group_small", form="engine", graph="rmat", scale=16, n=128, lanes=128),
        # the headline workload: 1,024 GroupBy-ordered sources in 8 groups of 128
        dict(name="groups_large", form="engine", graph="rmat", scale=22, n=1024, lanes=128),
        # the same 1,024 sources through the batched launcher as it is tuned for this graph
        dict(name="batch_large", form="batch", graph="rmat", scale=22, n=1024, tuned="rmat_s22"),
        # batched run on a social-network degree distribution; odd vertex count,
        # so depth rows are unaligned; a partial last group
        dict(name="batch_power_law", form="batch", graph="chung_lu", verts=1_000_003, mean=76,
             n=500, lanes=256, contexts=2, burst=4),
        # closeness centrality of every vertex
        dict(name="closeness_all", form="closeness", graph="rmat", scale=18, n=262_144, lanes=256,
             contexts=2, burst=4),
        # a burst of 32 queries of 1..256 sources at a query server
        dict(name="served_burst", form="served", graph="rmat", scale=20, n=32, lanes=256),
        # a mesh: about a thousand levels with small frontiers
        dict(name="mesh", form="engine", graph="grid", rows=512, cols=512, n=128, lanes=128),
        # the reference's own schedule (fixed switch level, its degree classes)
        # on an odd-sized power-law graph, with a last group of one source
        dict(name="fixed_switch", form="engine", graph="chung_lu", verts=300_007, mean=40, n=257,
             lanes=128, switch=2),
        # depth arrays wanted in host memory
        dict(name="host_arrays", form="host", graph="rmat", scale=18, n=64, lanes=64),
        # a caller that must not allocate
        dict(name="noalloc", form="noalloc", graph="rmat", scale=16, n=100),
        # ordering a source set before it is run in groups
        dict(name="groupby", form="groupby", graph="rmat", scale=22, n=1024),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    form = rng.choice(["engine"] * 6 + ["batch"] * 5 + ["closeness"] * 2 + ["served"] * 2
                      + ["noalloc"] * 2 + ["host", "groupby"])
    kinds = ["rmat", "rmat", "chung_lu"] + (["grid"] if form in ("engine", "batch") else [])
    kind = rng.choice(kinds)
    case = dict(form=form, graph=kind)
    if kind == "rmat":
        case["scale"] = rng.randint(11, 17 if form == "noalloc" else 18 if form == "host" else 21)
        verts = 1 << case["scale"]
    elif kind == "chung_lu":
        verts = _log(rng, 3_000, 120_000 if form in ("noalloc", "host") else 800_000) | 1
        case.update(verts=verts, mean=_log(rng, 8, 76))
    else:
        case.update(rows=_log(rng, 24, 400), cols=_log(rng, 24, 400))
        verts = case["rows"] * case["cols"]
    if form in ("noalloc", "host"):
        case["n"] = _log(rng, 1, 128)
    elif form == "served":
        case["n"] = _log(rng, 1, 32)
    elif form == "closeness":
        case["n"] = _log(rng, 16, max(16, min(verts // 4, 20_000)))
    elif form == "groupby":
        case["n"] = _log(rng, 16, max(16, min(verts // 4, 100_000)))
    else:
        case["n"] = _log(rng, 1, 256 if kind == "grid" else min(1024, verts // 4))
    if form == "engine":
        case["lanes"] = rng.choice([64, 128, 128, 128, 256, 512])
        if rng.random() < 0.2 and kind != "grid":
            case["switch"] = rng.choice([1, 2, 3])
    elif form == "host":
        case["lanes"] = 128
    elif form in ("batch", "closeness", "served"):
        case["lanes"] = rng.choice([64, 128, 256, 256, 512])
        if form != "served":
            case.update(contexts=rng.choice([1, 2, 2, 3]), burst=rng.choice([4, 8]))
    return case


def _verts(case):
    if case["graph"] == "rmat":
        return 1 << case["scale"]
    return case["verts"] if case["graph"] == "chung_lu" else case["rows"] * case["cols"]


def _entries(case):
    """Directed adjacency entries, about (duplicates are removed)."""
    v = _verts(case)
    if case["graph"] == "rmat":
        return 2 * 16 * v * 0.95
    return v * case["mean"] if case["graph"] == "chung_lu" else 4 * v


def _grid(rows, cols):
    v = np.arange(rows * cols).reshape(rows, cols)
    a = np.concatenate([v[:, :-1].ravel(), v[:, 1:].ravel(), v[:-1].ravel(), v[1:].ravel()])
    b = np.concatenate([v[:, 1:].ravel(), v[:, :-1].ravel(), v[1:].ravel(), v[:-1].ravel()])
    order = np.lexsort((b, a))
    beg = np.concatenate([[0], np.cumsum(np.bincount(a, minlength=rows * cols))])
    return ibfs_amd.HostCsr.from_arrays(beg, b[order])


def _host_graph(kind, size, mean, seed):
    if kind == "rmat":
        return ibfs_amd.HostCsr.rmat(size[0], 16, seed=seed)
    if kind == "chung_lu":
        return ibfs_amd.HostCsr.chung_lu(size[0], 2.2, float(mean), min(33_000.0, size[0] / 10),
                                         seed=seed)
    return _grid(*size)


def _graph(kind, size, mean, seed):
    host = _host_graph(kind, size, mean, seed)
    return host, ibfs_amd.DeviceGraph(host)


_resident = lru_cache(maxsize=None)(_graph)


def _graph_key(case, seed):
    kind = case["graph"]
    size = {"rmat": lambda: (case["scale"],), "chung_lu": lambda: (case["verts"],),
            "grid": lambda: (case["rows"], case["cols"])}[kind]()
    return kind, size, case.get("mean", 0), seed + 1 if _verts(case) <= SMALL else 1


def _sources(case, seed, host):
    """The case's sources: one array, or one per query."""
    rng = np.random.default_rng(seed)
    if case["form"] == "closeness" and case["n"] >= host.vert_count:
        return rng.permutation(host.vert_count).astype(np.int32)
    if case["form"] == "served":
        pool = host.gen_sources(min(4096, host.vert_count // 4), seed=seed + 2)
        # log-uniform sizes: the same multiset for every seed, in the seed's order
        sizes = np.exp((np.arange(case["n"]) + 0.5) / case["n"] * np.log(256)).astype(int)
        return [rng.choice(pool, size=k) for k in rng.permutation(sizes)]
    return host.gen_sources(case["n"], seed=seed + 2)


class Rows:
    """n depth rows in a torch tensor, as the framework's device outputs take them."""

    def __init__(self, n, verts, depth=None):
        self.depth = torch.empty((n, verts), dtype=torch.int32, device="cuda") if depth is None else depth
        self.ptr = self.depth.data_ptr()
        self.nbytes = self.depth.numel() * 4


def prepare(case, seed):
    key = _graph_key(case, seed)
    host, g = (_graph if _verts(case) <= SMALL else _resident)(*key)
    src = _sources(case, seed, host)
    form, verts = case["form"], host.vert_count
    s = {"form": form, "graph": g, "src": src}
    if form in ("engine", "host"):
        opts = dict(lane_bits=case["lanes"])
        if "switch" in case:
            opts.update(policy=ibfs_amd.POLICY_FIXED, sw_level=case["switch"], sml_shed=32)
        s["engine"] = ibfs_amd.Engine(g, **opts)
        if case["n"] > case["lanes"]:
            s["src"] = src = g.groupby(src)
    elif form in ("batch", "closeness"):
        if "tuned" in case:
            opts, contexts, burst, _ = ibfs_amd.tuned_batch_settings(case["tuned"])
        else:
            opts, contexts, burst = dict(lane_bits=case["lanes"]), case["contexts"], case["burst"]
        s["batch"] = ibfs_amd.Batch(g, contexts=contexts, burst=burst, **opts)
    elif form == "served":
        s["server"] = ibfs_amd.Server(g, lane_bits=case["lanes"])
        all_rows = Rows(sum(len(q) for q in src), verts)
        ends = np.cumsum([len(q) for q in src])
        s["views"] = [Rows(0, 0, all_rows.depth[e - len(q):e]) for q, e in zip(src, ends)]
        s["out"] = all_rows
        return s
    if form in ("engine", "batch", "noalloc"):
        s["out"] = Rows(len(src), verts)
    return s


def run(s):
    form, src = s["form"], s["src"]
    if form == "engine":
        eng = s["engine"]
        (eng.traversal if len(src) <= eng.lane_bits else eng.run_groups)(src, out=s["out"])
        return {"depth": s["out"].depth, "edges": eng.last_stats.traversed_edges}
    if form == "host":
        return {"depth": s["engine"].traversal(src), "edges": s["engine"].last_stats.traversed_edges}
    if form == "batch":
        s["batch"].run(src, out=s["out"])
        return {"depth": s["out"].depth, "edges": s["batch"].last_stats.traversed_edges}
    if form == "closeness":
        total, reach = s["batch"].closeness(src)
        return {"sum": total, "reach": reach}
    if form == "served":
        srv = s["server"]
        ids = [srv.submit(q, v) for q, v in zip(src, s["views"])]
        for i in ids:
            srv.wait(i)
        for i in ids:
            srv.release(i)
        return {"depth": s["out"].depth}
    if form == "noalloc":
        return {"edges": s["graph"].traversal_noalloc(src, s["out"]), "depth": s["out"].depth}
    return {"order": s["graph"].groupby(src)}


def work(case):
    """The graph read once, the sources read and the results written once."""
    v, e, n = _verts(case), _entries(case), case["n"]
    graph = 8 * v + 4 * e
    if case["form"] == "groupby":  # the sources' lists and their neighbours' degrees
        return {"bytes": 8 * n + n * (16 + 8 * e / v), "flops": 0}
    if case["form"] == "closeness":
        return {"bytes": graph + 20 * n, "flops": 0}
    if case["form"] == "served":
        n *= 46  # mean of the query sizes
    return {"bytes": graph + 4 * n + 4 * n * v, "flops": 0}


def _depths(beg, adj, src, most_levels=64):
    """Depth arrays of the sources, all lanes at once as bits of 64-bit words
    per vertex; None when the graph is too deep for that to be quick."""
    v, n = len(beg) - 1, len(src)
    words = np.zeros((v, (n + 63) // 64), dtype=np.uint64)
    lane = np.arange(n)
    bit = np.uint64(1) << (lane % 64).astype(np.uint64)
    np.bitwise_or.at(words, (src, lane // 64), bit)
    depth = np.full((n, v), -1, dtype=np.int32)
    depth[lane, src] = 0
    some = np.flatnonzero(np.diff(beg))  # vertices with neighbours
    for level in range(1, most_levels):
        near = np.zeros_like(words)
        near[some] = np.bitwise_or.reduceat(words[adj], beg[:-1][some], axis=0)
        new = near & ~words
        at = np.flatnonzero(new.any(axis=1))
        if not len(at):
            return depth
        words[at] |= new[at]
        for k in range(n):
            depth[k, at[(new[at, k // 64] & bit[k]) != 0]] = level
    return None


def exact(case, seed):
    kind, size, mean, graph_seed = _graph_key(case, seed)
    form = case["form"]
    n = case["n"] * (46 if form == "served" else 1)
    if kind == "grid" or n * _entries(case) > 1e9:
        return None
    host = _host_graph(kind, size, mean, graph_seed)
    beg, adj = host.arrays()
    deg = np.diff(beg)
    src = _sources(case, seed, host)

    def ordered(order):
        """GroupBy: sources of degree <= 128 by their first neighbour of
        degree > 128, in input order among equals; then the others."""
        key = []
        for s in order:
            near = adj[beg[s]:beg[s + 1]]
            hubs = near[deg[near] > 128]
            key.append(int(hubs[0]) if deg[s] <= 128 and len(hubs) else len(deg))
        return order[np.argsort(key, kind="stable")]

    if form == "groupby":
        return {"order": ordered(src)}
    if form == "served":
        src = np.concatenate(src)
    elif form in ("engine", "host") and len(src) > case["lanes"]:
        src = ordered(src)
    depth = _depths(beg, adj, src)
    if depth is None:
        return None
    if form == "closeness":
        return {"sum": np.where(depth > 0, depth, 0).sum(axis=1, dtype=np.int64),
                "reach": (depth >= 0).sum(axis=1, dtype=np.int64)}
    if form == "served":
        return {"depth": depth}
    return {"depth": depth, "edges": int(sum(deg[d >= 0].sum() for d in depth))}
