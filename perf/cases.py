"""The work that a user of this framework has it do, as cases to time.

Every case goes through the public Python entry points of par-cd_amd/parcd
(each a thin call of include/parcd.h): refinement of one graph from labels on
the host to labels on the host, merging, the triangle counts behind WCC, the
contraction to the community graph, the evaluation of a given partition, the
allocation-free label compression, and a batch of independent graphs.

Sizes are those of the repository's benchmark and tests: the 10,000-vertex
stochastic block model, R-MAT graphs up to scale 22 (a/b/c/d =
0.57/0.19/0.19/0.05, 16 draws per vertex), the 1,000,000-vertex Chung-Lu graph
with 32 planted communities, batches of block-model graphs of 50-20,000
vertices, and the small graphs of the tests.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "par-cd_amd"))

import parcd  # noqa: E402

RULES = {"mod": parcd.RULE_MODULARITY, "cpm": parcd.RULE_CPM, "wcc": parcd.RULE_WCC}


def _refine(name, graph, rule, lam=0.0, strategy=0, rounds=1, passes=-1, tie=0, init="singleton"):
    """pcd_refine of one graph; passes -1: until the score stops rising."""
    return {"name": name, "do": "refine", "rule": rule, "lam": lam, "strategy": strategy, "rounds": rounds,
            "passes": passes, "tie": tie, "init": init, **graph}


def _sbm(blocks, size, p_in, p_out, topology=1):
    return {"graph": "sbm", "topology": topology, "blocks": blocks, "size": size, "p_in": p_in, "p_out": p_out}


def _rmat(scale, draws_per=16.0, topology=2):
    return {"graph": "rmat", "topology": topology, "scale": scale, "draws_per": draws_per}


def _chung_lu(n, dmax, comms, cmax, topology=3):
    return {"graph": "chung_lu", "topology": topology, "n": n, "dmax": dmax, "comms": comms, "cmax": cmax}


def listed():
    return [
        # a label compression inside a caller's own device loop (no allocation, no copy): latency
        {"name": "compress-20011", "do": "compress", "n": 20011, "communities": 2900, "new_share": 0.15},
        # one small graph of a stream of requests, to convergence: latency of the whole loop
        _refine("refine-sbm210-mod", _sbm(21, 10, 0.5, 0.02), "mod"),
        # the 10,000-vertex block model of the benchmark, to convergence
        _refine("refine-sbm10000-mod", _sbm(100, 100, 0.08, 0.0005), "mod"),
        # an ordinary graph under CPM with alternating propagation and merging
        _refine("refine-rmat16-cpm-s2", _rmat(16), "cpm", lam=0.01, strategy=2, passes=16),
        # the headline graph: propagation passes from singletons under modularity
        _refine("refine-rmat22-mod", _rmat(22), "mod", passes=20),
        # a large graph under CPM in the deterministic mode (lowest-label ties)
        _refine("refine-rmat20-cpm-lowest", _rmat(20), "cpm", lam=0.01, passes=20, tie=1),
        # parallel merging (-s 1) of a large graph
        _refine("merge-rmat20-mod", _rmat(20), "mod", strategy=1, passes=10),
        # WCC from the triangle-based initial partition, triangles counted before
        _refine("refine-chunglu-wcc", _chung_lu(1000000, 5000, 32, 50000), "wcc", passes=8, init="clustering"),
        # triangle counts and clustering coefficient of a power-law graph
        {"name": "triangles-rmat18", "do": "triangles", **_rmat(18)},
        # the community graph of a partition: one level of a multilevel method
        {"name": "contract-rmat18", "do": "contract", **_rmat(18)},
        # sizes, volumes and the scores of a partition that came from elsewhere
        {"name": "evaluate-rmat20", "do": "evaluate", "lam": 0.01, **_rmat(20)},
        # many independent graphs at once, host arrays to host labels
        {"name": "batch-256", "do": "batch", "topology": 4, "count": 256, "nmin": 50, "nmax": 20000},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _draw_sbm(rng, nmin, nmax, topology):
    n = _log(rng, nmin, nmax)
    size = max(5, int(_log(rng, 8, min(400, n / 3))))
    blocks = max(2, int(n / size))
    p_in = min(0.6, rng.uniform(4, 16) / size)
    p_out = min(0.05, rng.uniform(1, 6) / (blocks * size))
    return _sbm(blocks, size, round(p_in, 5), round(p_out, 7), topology)


def _draw_rule(rng):
    if rng.random() < 0.6:
        return "mod", 0.0
    return "cpm", round(_log(rng, 0.005, 0.05), 5)


def draw(rng):
    do = rng.choice(["compress", "refine-sbm", "refine-sbm", "refine-rmat", "refine-rmat", "merge", "wcc", "triangles",
                     "contract", "evaluate", "batch"])
    draws_per = round(rng.uniform(8, 20), 2)
    topology = rng.randint(1, 1 << 30)
    if do == "compress":
        n = int(_log(rng, 500, parcd.NOALLOC_MAX_VERTICES))
        return {"do": do, "n": n, "communities": max(1, int(n * rng.uniform(0.002, 1.0))),
                "new_share": round(rng.uniform(0, 0.3), 3)}
    if do == "triangles":
        return {"do": do, **_rmat(rng.randint(9, 18), draws_per, topology)}
    if do == "contract":
        return {"do": do, **_rmat(rng.randint(9, 18), draws_per, topology)}
    if do == "evaluate":
        return {"do": do, "lam": round(_log(rng, 0.005, 0.05), 5), **_rmat(rng.randint(9, 20), draws_per, topology)}
    if do == "batch":
        return {"do": do, "topology": topology, "count": int(_log(rng, 8, 256)), "nmin": 50, "nmax": int(_log(rng, 500, 20000))}
    if do == "wcc":
        n = int(_log(rng, 3000, 1000000))
        g = _chung_lu(n, max(20, min(5000, n // 20)), 32, max(200, n // 20), topology)
        c = _refine("", g, "wcc", passes=rng.randint(3, 8), init="clustering")
    else:
        rule, lam = _draw_rule(rng)
        tie = rng.randint(0, 1)
        if do == "refine-sbm":
            c = _refine("", _draw_sbm(rng, 50, 40000, topology), rule, lam, strategy=rng.choice([0, 0, 2]),
                        rounds=rng.choice([1, 1, 3]), passes=rng.randint(10, 60), tie=tie)
        elif do == "refine-rmat":
            c = _refine("", _rmat(rng.randint(8, 21), draws_per, topology), rule, lam, strategy=rng.choice([0, 0, 0, 2]),
                        passes=rng.randint(8, 20), tie=tie)
        else:
            c = _refine("", _rmat(rng.randint(9, 20), draws_per, topology), rule, lam, strategy=1, rounds=rng.choice([1, 1, 2]),
                        passes=rng.randint(4, 10), tie=tie)
    del c["name"]
    return c


# ------------------------------------------------------------ inputs
# A case names its graph's topology; the seed decides the vertex ids (a random
# order among vertices of equal degree), the initial labels and the seed of
# the job, so that inputs of another seed are another file of the same size.
def _csr(u, v, n, owner, seed):
    """Degree-sorted CSR (as `convert` writes it) of the edges (u, v), loops,
    duplicates and isolated vertices dropped.  owner[x] is the graph that
    vertex x belongs to (ascending; None: one graph).  Returns the owners of
    the kept vertices, the row offsets, the neighbour ids and, per vertex,
    its neighbour of the largest degree if larger than its own (a partition
    that does not depend on the seed but for the names)."""
    keep = u != v
    u, v = u[keep], v[keep]
    key = torch.unique(torch.cat([u * n + v, v * n + u]))
    u, v = key // n, key % n
    deg = torch.bincount(u, minlength=n)
    own = torch.zeros_like(deg) if owner is None else owner
    top = int(deg.max()) + 1
    nv = int((deg > 0).sum())
    # kept vertices by owner, then by degree, descending
    order = torch.argsort((deg == 0).long() * (int(own.max()) + 1) * top + own * top + (top - 1 - deg), stable=True)[:nv]
    rank = torch.zeros_like(deg)
    rank[order] = torch.arange(nv, device=deg.device)
    deg, own = deg[order], own[order]
    key = torch.sort(rank[u] * nv + rank[v])[0]
    u, v = key // nv, key % nv
    start = torch.cumsum(deg, 0) - deg
    hub = torch.minimum(v[start], torch.arange(nv, device=deg.device))
    # the seed's order among equal degrees
    g = torch.Generator(device=deg.device).manual_seed(seed)
    mix = torch.randperm(nv, generator=g, device=deg.device)
    order = mix[torch.argsort((own * top + (top - 1 - deg))[mix], stable=True)]
    sigma = torch.empty_like(order)
    sigma[order] = torch.arange(nv, device=deg.device)
    v = torch.sort(sigma[u] * nv + sigma[v])[0] % nv
    labels = torch.empty_like(hub)
    labels[sigma] = sigma[hub]
    ind = torch.zeros(nv + 1, dtype=torch.int64, device=deg.device)
    ind[1:] = torch.cumsum(deg, 0)
    return own, ind, v, labels


def _edges(case):
    """The endpoints of the case's edges on the device, and the vertices."""
    if case["graph"] == "rmat":
        scale = case["scale"]
        draws = int(case["draws_per"] * (1 << scale))
        g = torch.Generator(device="cuda").manual_seed(case["topology"])
        u = torch.zeros(draws, dtype=torch.int64, device="cuda")
        v = torch.zeros(draws, dtype=torch.int64, device="cuda")
        for _ in range(scale):
            r = torch.rand(draws, generator=g, device="cuda")
            u = 2 * u + (r >= 0.76)
            v = 2 * v + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        return u, v, 1 << scale
    if case["graph"] == "sbm":
        a, b, n = parcd.gen_sbm(case["topology"], [case["size"]] * case["blocks"], case["p_in"], case["p_out"])
    else:
        a, b, n = parcd.gen_chung_lu(case["topology"], case["n"], 2.3, 4, case["dmax"], case["comms"], 100,
                                     case["cmax"], 20.0)
    return torch.from_numpy(a).cuda().long(), torch.from_numpy(b).cuda().long(), n


def _make_graph(case, seed):
    """(n, m, indices, adj) on the host, and the neighbour labels."""
    u, v, n = _edges(case)
    _, ind, adj, labels = _csr(u, v, n, None, seed)
    ind, adj, labels = (x.to(torch.int32).cpu().numpy() for x in (ind, adj, labels))
    return (ind.size - 1, adj.size // 2, ind, adj), labels


def _make_batch(case, seed):
    """Block-model graphs in page-locked memory, and their rules: n
    log-uniform, 2-64 blocks, p_in 0.05-0.3, p_out 0.001-0.01, modularity or
    CPM at 0.005-0.05."""
    graphs, params = parcd.gen_sbm_batch(case["topology"], case["count"], nmin=case["nmin"], nmax=case["nmax"])
    keep = [i for i, x in enumerate(graphs) if x[1] > 0]
    graphs, params = [graphs[i] for i in keep], params[keep]
    n = torch.tensor([x[0] for x in graphs], device="cuda")
    off = torch.cumsum(n, 0) - n
    owner = torch.repeat_interleave(torch.arange(len(graphs), device="cuda"), n)
    us, vs = [], []
    for i, (_, _, ind, adj) in enumerate(graphs):
        deg = torch.from_numpy(np.diff(ind)).cuda()
        at = int(off[i])
        us.append(torch.repeat_interleave(torch.arange(at, at + deg.numel(), device="cuda"), deg))
        vs.append(torch.from_numpy(adj).cuda().long() + at)
    u, v = torch.cat(us), torch.cat(vs)
    del us, vs
    own, ind, adj, _ = _csr(u[u < v], v[u < v], int(n.sum()), owner, seed)
    del u, v
    n = torch.bincount(own, minlength=len(graphs))
    off = torch.cumsum(n, 0) - n
    adj = adj - torch.repeat_interleave(off[own], ind[1:] - ind[:-1])
    n, off, ind = n.tolist(), off.tolist(), ind.tolist()
    flat = parcd.pinned_empty(adj.numel())
    flat[:] = adj.to(torch.int32).cpu().numpy()
    rows = parcd.pinned_empty(len(ind) + len(n))
    out = []
    for i, k in enumerate(n):
        lo, hi = ind[off[i]], ind[off[i] + k]
        r = rows[off[i] + i: off[i] + i + k + 1]
        r[:] = ind[off[i]: off[i] + k + 1]
        r -= lo
        out.append((k, (hi - lo) // 2, r, flat[lo:hi]))
    return out, params


def _singletons(n, seed):
    """framework.cpp:14-24: every vertex its own label, in a random order."""
    return np.random.default_rng(seed).permutation(n).astype(np.int32)


def prepare(case, seed):
    do = case["do"]
    st = {"do": do, "case": case}
    if do == "compress":
        g = torch.Generator(device="cuda").manual_seed(seed)
        n = case["n"]
        ids = torch.randperm(n, generator=g, device="cuda")[: case["communities"]]
        lab = ids[torch.randint(0, ids.numel(), (n,), generator=g, device="cuda")].to(torch.int32)
        lab[torch.rand(n, generator=g, device="cuda") < case["new_share"]] = parcd.NEW_LABEL
        st.update(n=n, labels=lab, out=torch.empty_like(lab), k=torch.zeros(1, dtype=torch.int32, device="cuda"))
        torch.cuda.synchronize()
        return st
    if do == "batch":
        graphs, params = _make_batch(case, seed)
        labels = parcd.pinned_empty(sum(x[0] for x in graphs))
        at, labs, jobs = 0, [], []
        for i, x in enumerate(graphs):
            labels[at: at + x[0]] = _singletons(x[0], seed + i)
            labs.append(labels[at: at + x[0]])
            at += x[0]
            jobs.append(parcd.job(kind=int(params[i][4]), lam=float(params[i][5]), seed=seed + i, iter_cap=100))
        arena = sum(parcd.batch_footprint(x[0], x[1]) for x in graphs) + (64 << 20)
        st.update(graphs=graphs, labels=labs, jobs=jobs,
                  batch=parcd.Batch(0, max_graphs=len(graphs), arena_bytes=arena))
        return st
    graph, hubs = _make_graph(case, seed)
    ctx = parcd.Context(0)
    ctx.upload_graph(*graph)
    st["ctx"] = ctx
    if do == "refine":
        st["job"] = parcd.job(kind=RULES[case["rule"]], lam=case["lam"], max_iter=case["passes"], tie=case["tie"],
                              seed=seed)
        if case["init"] == "clustering":
            ctx.triangles()
        else:
            st["labels"] = _singletons(graph[0], seed)
    else:
        st["labels"] = hubs
    return st


# ------------------------------------------------------------ the calls
def run(st):
    do, case = st["do"], st["case"]
    if do == "compress":
        parcd.compress_labels_noalloc(st["n"], st["labels"].data_ptr(), st["out"].data_ptr(), st["k"].data_ptr())
        return {"labels": st["out"], "k": st["k"]}
    if do == "batch":
        b = st["batch"]
        slots = b.add_many(st["graphs"], st["labels"], st["jobs"], wait=False)
        while b.step(1):
            pass
        labels = b.labels_many(slots)
        status = [b.status(s) for s in slots]
        for s in slots:
            b.release(s)
        return {"labels": np.concatenate(labels), "iterations": np.array([x[1] for x in status], np.int64),
                "k": np.array([x[2] for x in status], np.int64), "score": np.array([x[3] for x in status])}
    ctx = st["ctx"]
    if do == "triangles":
        tri, tdeg, cc = ctx.triangles()
        return {"tri": tri, "tri_deg": tdeg, "cc": cc}
    if do == "refine":
        if case["init"] == "clustering":
            ctx.clustering()
        else:
            ctx.upload_labels(st["labels"])
        score, it, k = ctx.refine(st["job"], strategy=case["strategy"], rounds=case["rounds"])
        return {"labels": ctx.labels(), "score": score, "iterations": it, "k": k}
    ctx.upload_labels(st["labels"])
    ctx.compress()
    k = ctx.statistics()
    if do == "contract":
        a, b, w = ctx.contract()
        return {"labels": ctx.labels(), "l": a, "k": b, "links": w}
    size, iv, ev = ctx.stats(k)
    return {"labels": ctx.labels(), "sizes": size, "int_volume": iv, "ext_volume": ev,
            "mod": ctx.metric(parcd.RULE_MODULARITY), "cpm": ctx.metric(parcd.RULE_CPM, case["lam"]),
            "conductance": ctx.metric(parcd.RULE_CONDUCTANCE)}


# ------------------------------------------------------------ what a pass cannot do without
def _size(case):
    """Vertices and adjacency entries of the case's graph, nearly."""
    if case["graph"] == "rmat":
        # isolated vertices and duplicate draws are dropped
        e = 2 * case["draws_per"] * (1 << case["scale"]) * min(0.96, 0.58 + 0.0175 * case["scale"])
        return 0.9 * (1 << case["scale"]) * max(0.5, 1.2 - 0.026 * case["scale"]), e
    if case["graph"] == "sbm":
        n = case["blocks"] * case["size"]
        return n, n * (case["size"] * case["p_in"] + n * case["p_out"])
    return case["n"], 14.8 * case["n"]


def work(case):
    if case["do"] == "compress":
        return {"bytes": 8.0 * case["n"], "flops": 0}  # labels in, labels out
    if case["do"] == "batch":
        # n log-uniform, 2-64 blocks, p_in 0.05-0.3, p_out 0.001-0.01; about
        # 20 passes a graph, half of the vertices active in each
        lo, hi = case["nmin"], case["nmax"]
        span = math.log(hi / lo)
        n = (hi - lo) / span
        n2 = (hi * hi - lo * lo) / 2 / span
        e = n2 * (0.175 * 0.055 + 0.0055)
        return {"bytes": case["count"] * (4 * e + 8 * n + 20 * (0.5 * 8 * e + 8 * n)), "flops": 0}
    n, e = _size(case)
    if case["do"] == "triangles":
        # the rows once, and an ordered-row intersection per edge
        return {"bytes": 4 * e + 12 * n, "flops": e / 2 * math.sqrt(e / max(n, 1))}
    if case["do"] == "contract":
        # each entry's neighbour and its label, the pairs out
        return {"bytes": 8 * e + 8 * n + 12 * 0.15 * e, "flops": 0}
    if case["do"] == "evaluate":
        return {"bytes": 8 * e + 12 * n + 12 * 0.3 * n, "flops": 0}
    # per pass the active vertices' entries (neighbour and label), labels in and out
    passes = case["passes"] if case["passes"] >= 0 else 45
    share = 0.5 if case["strategy"] == 0 else 1.0 if case["strategy"] == 1 else 0.75
    return {"bytes": passes * (share * 8 * e + 8 * n) + 8 * n, "flops": 0}


# ------------------------------------------------------------ the same in 64 bits, without the framework
def exact(case, seed):
    do = case["do"]
    if do == "evaluate":
        (n, m, ind, adj), lab = _make_graph(case, seed)
        deg = np.diff(ind).astype(np.int64)
        same = lab[np.repeat(np.arange(n), deg)] == lab[adj]
        cnt = np.bincount(np.repeat(np.arange(n), deg)[same], minlength=n)
        ids, dense = np.unique(lab, return_inverse=True)
        size = np.bincount(dense)
        iv = np.bincount(dense, weights=cnt)
        vol = np.bincount(dense, weights=deg)
        two_m = 2.0 * m
        return {"labels": None, "sizes": None, "int_volume": None, "ext_volume": None,
                "mod": float(iv.sum() / two_m - np.dot(vol, vol) / (two_m * two_m)),
                "cpm": float((iv.sum() - case["lam"] * np.dot(size, size - 1.0)) / two_m),
                "conductance": float((size * (iv / vol)).sum() / n)}
    if do == "triangles" and case["scale"] <= 18:
        (n, _, ind, adj), _ = _make_graph(case, seed)
        deg = torch.from_numpy(np.diff(ind).astype(np.int64)).cuda()
        row = torch.repeat_interleave(torch.arange(n, device="cuda"), deg)
        col = torch.from_numpy(adj).cuda().long()
        low = col < row
        row, col = row[low], col[low]  # every edge once, from its higher id; rows ascending
        key = row * n + col
        cnt = torch.bincount(row, minlength=n)
        start = torch.cumsum(cnt, 0) - cnt
        tri = torch.zeros(n, dtype=torch.int64, device="cuda")
        wedges = torch.cumsum(cnt[col], 0)
        at, edges = 0, row.numel()
        while at < edges:
            base = int(wedges[at - 1]) if at else 0
            end = max(at + 1, int(torch.searchsorted(wedges, base + (1 << 26))))
            v, u = row[at:end], col[at:end]
            rep = torch.repeat_interleave(torch.arange(end - at, device="cuda"), cnt[u])
            off = torch.arange(rep.numel(), device="cuda") - (wedges[at:end] - cnt[u] - base)[rep]
            w = col[start[u][rep] + off]
            want = v[rep] * n + w
            pos = torch.searchsorted(key, want).clamp_(max=edges - 1)
            hit = key[pos] == want
            for x in (v[rep][hit], u[rep][hit], w[hit]):
                tri += torch.bincount(x, minlength=n)
            at = end
        d = deg.double()
        cc = torch.where(deg > 1, 2.0 * tri.double() / (d * (d - 1.0)).clamp(min=1.0), torch.zeros_like(d)).sum() / n
        return {"tri": None, "tri_deg": None, "cc": float(cc)}
    return None
