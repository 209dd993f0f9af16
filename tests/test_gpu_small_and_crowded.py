"""GPU parity where kernels share an address or a workgroup: partitions with
a few large communities (every member's update falls on the same records),
and sizes at the edges of tiles, tables and launch forms."""
import time

import numpy as np
import pytest

import oracle_lib as O
import gpu_graphs as GG
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

parcd = pytest.importorskip("parcd")


@pytest.fixture(scope="module")
def ctx():
    if parcd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP runtime")
    c = parcd.Context(0)
    yield c
    c.close()


def crowded(kind, n):
    """Labels whose communities are few and large, or both large and many."""
    rng = np.random.default_rng(11)
    v = np.arange(n)
    if kind == "one":
        return np.full(n, n - 1, np.int32)
    if kind == "singletons":  # hardly two members of a wave share one
        return rng.permutation(n).astype(np.int32)
    if kind == "half":  # one community of half the vertices among singletons
        return np.where(rng.random(n) < 0.5, n // 2, v).astype(np.int32)
    if kind == "table":  # more communities than a workgroup's accumulators, some of them large
        return np.where(rng.random(n) < 0.7, rng.integers(0, 3, n), rng.integers(0, 900, n)).astype(np.int32)
    return np.where(rng.random(n) < 0.1, -1, v % 7).astype(np.int32)  # seven communities and NEW_LABEL vertices


@pytest.mark.parametrize("kind", ["one", "half", "table", "seven_new", "singletons"])
@pytest.mark.parametrize("graph", ["bin_zoo", "unsorted", "rmat12", "rmat14", "star"])
def test_statistics_of_crowded_partitions(ctx, graph, kind):
    """Compression, the full count, and the statistics updated from the moved
    rows over four steps equal the oracle's full count, for both tie orders:
    crowded communities lose and gain many members at once, or none does, on
    graphs on both sides of the entries from which the two kinds of step have
    a kernel each."""
    g = {"bin_zoo": GG.bin_zoo, "rmat14": lambda: GG.rmat(14), "unsorted": lambda: GG.unsorted_copy(GG.bin_zoo()), "rmat12": lambda: GG.rmat(12),
         "star": lambda: GG.csr_direct(700, [(0, i) for i in range(1, 700)])}[graph]()
    n, m, ind, adj = g[:4]
    ctx.upload_graph(n, m, ind, adj)
    lab_in = crowded(kind, n)
    ctx.upload_labels(lab_in)
    for step, (rule, lam, tie) in enumerate([(O.MOD, 0.0, 1), (O.CPM, 0.01, 1), (O.CPM, 0.2, 0), (O.MOD, 0.0, 0)]):
        k = ctx.compress()
        want, k_o = O.compress_labels(lab_in)
        assert k == k_o
        lab = ctx.labels()
        assert np.array_equal(lab, want)
        assert ctx.statistics() == k
        _, so, ivo, evo = O.collect_statistics(n, ind, adj, lab)
        for got, w in zip(ctx.stats(k), (so, ivo, evo)):
            assert np.array_equal(got, w), (graph, kind, step)
        ctx.propagate(rule, lam, frac=0.9, seed=21, step=step, tie=tie)
        lab_in = ctx.labels()


@pytest.mark.parametrize("n", [2, 3, 64, 65, 66, 130, 1025, 1026, 2051])
def test_triangles_of_cliques(ctx, n):
    """Prefixes at the edges of the wave table (64), of a workgroup table's
    chunk (1024) and over several chunks: in a clique of n with one pendant
    vertex every vertex is on C(n-1, 2) triangles and every edge but the
    pendant's on one."""
    i, j = np.triu_indices(n, 1)
    g = GG.csr_from_edges(np.append(i, 0), np.append(j, n))
    ctx.upload_graph(*g[:4])
    tri, tdeg, cc = ctx.triangles()
    deg = np.diff(g[2])
    inside = deg > 1 if n > 2 else np.zeros(n + 1, bool)
    assert np.array_equal(tri, np.where(inside, (n - 1) * (n - 2), 0))
    assert np.array_equal(tdeg, np.where(inside, n - 1, 0))
    want = (tri / np.maximum(deg * (deg - 1.0), 1.0)).sum() / (n + 1)
    assert cc == pytest.approx(want, rel=1e-12, abs=1e-300)


@pytest.mark.parametrize("labels", [1, 2, 7])
@pytest.mark.parametrize("graph", ["bin_zoo", "dense", "unsorted"])
def test_internal_triangles(ctx, graph, labels):
    """WCC of partitions with long and short prefixes inside and across
    communities, over several passes that reuse the flags."""
    g = {"bin_zoo": GG.bin_zoo, "dense": GG.dense_blocks, "unsorted": lambda: GG.unsorted_copy(GG.bin_zoo())}[graph]()
    n, m, ind, adj = g[:4]
    ctx.upload_graph(n, m, ind, adj)
    tri, tdeg, _ = ctx.triangles()
    _, t_o, td_o, _ = O.count_triangles(n, ind, adj)
    assert np.array_equal(tri, t_o) and np.array_equal(tdeg, td_o)
    for seed in (1, 2):
        lab, _ = O.compress_labels(np.random.default_rng(seed).integers(0, labels, n).astype(np.int32))
        ctx.upload_labels(lab)
        ctx.compress()
        ctx.statistics()
        s, _, _ = O.collect_statistics(n, ind, adj, lab)[1:]
        want = O.wcc_calculate(n, ind, adj, lab, s, t_o, td_o)[0]
        assert ctx.metric(O.WCC) == pytest.approx(want, rel=1e-9, abs=1e-12)


def renamed(g, name):
    """The graph with vertex v as name[v]."""
    n, _, ind, adj = g[:4]
    v = np.repeat(np.arange(n), np.diff(ind))
    low = adj < v
    return GG.csr_direct(n, list(zip(name[v[low]].tolist(), name[adj[low]].tolist())))


def late_hubs(kind):
    """Graphs whose hubs come after their neighbours: prefixes of several
    table chunks, met by rows below and above one step of a wave, with gaps."""
    rng = np.random.default_rng(17)
    if kind == "reversed":
        g = GG.rmat(12, factor=24)
        return renamed(g, np.arange(g[0])[::-1])
    if kind == "shuffled":
        g = GG.rmat(13)
        return renamed(g, rng.permutation(g[0]))
    n = 4200  # three hubs over a random graph whose rows reach 60 or 500 entries
    a, b = np.triu_indices(n - 3, 1)
    pick = rng.random(a.size) < np.where(a % 2 == 1, 0.014, np.where(b < 2400, 0.2, 0.001))
    e = [np.stack([a[pick], b[pick]], 1)]
    for h in (n - 3, n - 2, n - 1):
        v = np.flatnonzero(rng.random(h) < 0.9)
        e.append(np.stack([v, np.full(v.size, h)], 1))
    return GG.csr_direct(n, np.concatenate(e).tolist())


@pytest.mark.parametrize("kind", ["reversed", "shuffled", "random"])
def test_triangles_of_late_hubs(ctx, kind):
    n, m, ind, adj = late_hubs(kind)[:4]
    low = np.array([np.searchsorted(adj[ind[v]:ind[v + 1]], v) for v in range(n)])
    assert low.max() > 1024  # several chunks
    ctx.upload_graph(n, m, ind, adj)
    tri, tdeg, _ = ctx.triangles()
    _, t_o, td_o, _ = O.count_triangles(n, ind, adj)
    assert np.array_equal(tri, t_o) and np.array_equal(tdeg, td_o)
    lab, _ = O.compress_labels(np.random.default_rng(2).integers(0, 3, n).astype(np.int32))
    ctx.upload_labels(lab)
    ctx.compress()
    ctx.statistics()
    s, _, _ = O.collect_statistics(n, ind, adj, lab)[1:]
    want = O.wcc_calculate(n, ind, adj, lab, s, t_o, td_o)[0]
    assert ctx.metric(O.WCC) == pytest.approx(want, rel=1e-9, abs=1e-12)


@pytest.mark.parametrize("n", [1023, 1025, 20480, 20481])
def test_triangles_of_listed_vertices(ctx, n):
    """The list of long prefixes at the edges of its scans' tiles: wheels whose
    hubs lie there, and at the last id."""
    v = np.arange(100, 200)  # the rim, below every hub
    e = [np.stack([v, np.where(v == 199, 100, v + 1)], 1)]
    hubs = [h for h in (200, 1022, 1023, 1024, 4095, 4096, 20479, n - 1) if h < n]
    for i, h in enumerate(hubs):
        k = (64, 65, 100)[i % 3]  # a wave's prefix, and two longer ones
        e.append(np.stack([v[:k], np.full(k, h)], 1))
    n, m, ind, adj = GG.csr_direct(n, np.concatenate(e).tolist())[:4]
    ctx.upload_graph(n, m, ind, adj)
    tri, tdeg, cc = ctx.triangles()
    _, t_o, td_o, cc_o = O.count_triangles(n, ind, adj)
    assert np.array_equal(tri, t_o) and np.array_equal(tdeg, td_o)
    assert cc == pytest.approx(cc_o, rel=1e-9)


def test_a_late_hub_costs_what_its_rows_hold(ctx):
    """A hub after its 200,000 neighbours: their rows are looked up in the
    chunks of the hub's prefix that they can meet (in all 196, the wheel took
    57 times what the star takes, whose rows hold nothing to look up)."""
    n = 200001
    v = np.arange(n - 1)

    def best(u, w):
        key = np.sort(np.concatenate([u * n + w, w * n + u]))
        ind = np.zeros(n + 1, np.int32)
        ind[1:] = np.cumsum(np.bincount(key // n, minlength=n))
        ctx.upload_graph(n, key.size // 2, ind, (key % n).astype(np.int32))
        times = []
        for _ in range(4):
            t = time.perf_counter()
            tri = ctx.triangles()[0]
            times.append(time.perf_counter() - t)
        return min(times), tri

    hub = np.full(n - 1, n - 1)
    star, tri = best(v, hub)
    assert not tri.any()
    wheel, tri = best(np.concatenate([v, v]), np.concatenate([hub, (v + 1) % (n - 1)]))
    assert tri[n - 1] == 2 * (n - 1) and (tri[:n - 1] == 4).all()
    assert wheel < 15 * star


@pytest.mark.parametrize("hub", [0, 200])
@pytest.mark.parametrize("n", [2047, 2048, 6000])
def test_clustering_of_rows_of_every_length(ctx, n, hub):
    """Rows at the edges of the eight-lane and the whole-wave reader (8, 32, 33,
    64, 65 entries), the rounds' vertices consecutive (no row of n / 64
    entries) and spread over the waves (one hub)."""
    rng = np.random.default_rng(n)
    v = np.arange(n)
    e = [np.stack([v, (v + 1) % n], 1)]
    for size in (7, 8, 9, 31, 32, 33) + ((63, 64, 65) if n == 6000 else ()):
        for _ in range(4 if hub or n == 6000 else 0):
            m = rng.choice(n, size, replace=False)
            e.append(np.stack([np.repeat(m[:1], size - 1), m[1:]], 1))
            i, j = np.triu_indices(min(size, 9), 1)
            e.append(np.stack([m[i], m[j]], 1))
    if hub:
        e.append(np.stack([np.full(hub, 5), rng.choice(np.arange(6, n), hub, replace=False)], 1))
    n, m, ind, adj = GG.csr_direct(n, np.concatenate(e).tolist())[:4]
    assert (64 * int(np.diff(ind).max()) >= n) == bool(hub)
    ctx.upload_graph(n, m, ind, adj)
    tri = ctx.triangles()[0]
    want = O.clustering_partition(n, ind, adj, tri)
    for rounds in (1, 128):
        ctx.set_tuning("cluster_rounds", rounds)
        ctx.clustering()
        ctx.set_tuning("cluster_rounds", 128)
        assert np.array_equal(ctx.labels(), want), rounds


def small_graphs():
    """Sizes at the edges of the one-workgroup loop: degrees in every table
    class, isolated vertices, unsorted ids, the largest vertex and entry
    counts it takes and the first it does not."""
    rng = np.random.default_rng(3)
    out = {"tiny_" + name: GG.csr_direct(*g) for name, g in GG.TINY.items()}
    out["sbm"] = GG.sbm(21, 10, 0.5, 0.02)
    out["rmat9"] = GG.rmat(9)
    out["rmat10_unsorted"] = GG.unsorted_copy(GG.rmat(10, factor=8))
    star = [(0, i) for i in range(1, 4096)]
    out["hub_4095"] = GG.csr_direct(4096, star + [(i, i + 1) for i in range(1, 1200)])
    for name, n, m in (("n4096", 4096, 12000), ("n4097", 4097, 12000), ("e32768", 3000, 16384), ("e32770", 3000, 16385),
                       ("degree_70_300", 500, 15000)):
        a, b = rng.integers(0, n, (2, 4 * m))
        if name.startswith("degree"):
            a = np.where(rng.random(a.size) < 0.5, a % 60, a)
        keep = a < b
        e = np.unique(np.stack([a[keep], b[keep]], 1), axis=0)
        e = e[rng.permutation(len(e))[:m]]
        assert len(e) == m
        out[name] = GG.csr_direct(n, [tuple(x) for x in e.tolist()])
    return out


SMALL = small_graphs()


@pytest.mark.parametrize("name", sorted(SMALL))
def test_small_graph_loop(ctx, name):
    """Refinement and ranges of passes equal the pass-by-pass loop: labels,
    score, passes, communities and statistics, from labels of outside (with
    NEW_LABEL) and from where another range stopped."""
    n, m, ind, adj = SMALL[name][:4]
    rng = np.random.default_rng(n + m)
    starts = [rng.permutation(n).astype(np.int32), np.where(rng.random(n) < 0.3, -1, rng.integers(0, max(1, n // 9), n))]
    ctx.upload_graph(n, m, ind, adj)
    for i, (kind, lam, tie, frac) in enumerate([(O.MOD, 0.0, 0, 0.5), (O.CPM, 0.05, 1, 0.5), (O.CPM, 0.3, 0, 1.0),
                                                (O.MOD, 0.0, 1, 0.8)]):
        lab = starts[i % 2].astype(np.int32)
        got = []
        for solo, fused, graph in ((2, 1, 1), (1, 1, 1), (0, 1, 1), (0, 0, 1), (0, 0, 0)):
            ctx.set_tuning("solo_loop", solo)
            ctx.set_tuning("fused_pass", fused)
            ctx.set_tuning("graph_loop", graph)
            one = []
            for job in (parcd.job(kind=kind, lam=lam, frac=frac, tie=tie, seed=5, iter_cap=40),
                        parcd.job(kind=kind, lam=lam, frac=frac, tie=tie, seed=6, max_iter=7)):
                ctx.upload_labels(lab)
                score, it, k = ctx.refine(job)
                one += [score, it, k, ctx.labels()] + list(ctx.stats(k))
            job = parcd.job(kind=kind, lam=lam, frac=frac, tie=tie, seed=5, iter_cap=1000, max_iter=900)
            ctx.upload_labels(lab)
            at, prev = 0, 0.0
            for count in (1, 3, 2):
                p, prev, k, done = ctx.iterate_many(job, at, count, prev)
                assert p == count and not done
                at += p
                one += [prev, k]
            one += [ctx.iterate(job, at, prev)[0], ctx.compress(), ctx.labels()]
            got.append(one)
        for key in ("solo_loop", "fused_pass", "graph_loop"):
            ctx.set_tuning(key, 1)
        for other in got[1:]:
            assert len(other) == len(got[0])
            for x, y in zip(got[0], other):
                assert np.array_equal(x, y, equal_nan=True) if isinstance(x, float) else np.array_equal(x, y), (name, i)


@pytest.mark.parametrize("hubs,degree", [(60, 265), (30, 530), (0, 0)])
def test_small_graph_loop_is_not_the_slower_way(hubs, degree):
    """Small graphs whose passes one workgroup runs two to four times slower
    than the whole chip (many rows that it takes one by one; 32,000 entries)
    take the whole chip."""
    rng = np.random.default_rng(hubs)
    a, b = [rng.integers(hubs, 4000, 300 if hubs else 16300)], [rng.integers(hubs, 4000, 300 if hubs else 16300)]
    for h in range(hubs):
        a.append(np.full(degree, h))
        b.append(hubs + rng.choice(4000 - hubs, degree, replace=False))
    g = GG.csr_from_edges(np.concatenate(a), np.concatenate(b))
    lab = rng.permutation(g[0]).astype(np.int32)
    with parcd.Context(0) as c:
        c.upload_graph(*g[:4])

        def best(solo):
            c.set_tuning("solo_loop", solo)
            times = []
            for _ in range(8):
                c.upload_labels(lab)
                t = time.perf_counter()
                c.refine(parcd.job(kind=O.CPM, lam=0.005, seed=3, max_iter=20))
                times.append(time.perf_counter() - t)
            return min(times)

        assert best(1) < 1.4 * best(0)


@pytest.mark.parametrize("n", [1023, 1024, 1025, 20480, 20481, 65536, 65537])
def test_fused_pass_sizes(ctx, n):
    """Sizes at the edges of the numbering's tiles and of the direct forms:
    every vertex on a ring with chords (degrees 2-40 and one hub), modularity
    and CPM with leaving vertices, equal pass by pass."""
    rng = np.random.default_rng(n)
    a = np.arange(n)
    u, v = np.concatenate([a, rng.integers(0, n, 3 * n), np.zeros(min(n - 1, 6000), int)]), \
        np.concatenate([(a + 1) % n, rng.integers(0, n, 3 * n), np.arange(1, min(n, 6001))])
    g = GG.csr_from_edges(u, v)
    assert g[0] == n
    ctx.upload_graph(*g[:4])
    lab = rng.integers(0, n, n).astype(np.int32)
    for kind, lam, tie in ((O.MOD, 0.0, 0), (O.CPM, 0.4, 1)):
        got = []
        for fused, graph in ((1, 1), (0, 1), (0, 0)):
            ctx.set_tuning("solo_loop", 0)
            ctx.set_tuning("fused_pass", fused)
            ctx.set_tuning("graph_loop", graph)
            ctx.upload_labels(lab)
            one = list(ctx.refine(parcd.job(kind=kind, lam=lam, tie=tie, seed=3, max_iter=9)))
            one += [ctx.labels()] + list(ctx.stats(one[2]))
            ctx.upload_labels(lab)  # the captured pass again, stopped by its range
            at, prev = 0, 0.0
            for count in (4, 3):
                p, prev, k, done = ctx.iterate_many(parcd.job(kind=kind, lam=lam, tie=tie, seed=3, max_iter=90), at,
                                                    count, prev)
                at += p
                one += [prev, k]
            got.append(one + [ctx.compress(), ctx.labels()])
        for key in ("solo_loop", "fused_pass", "graph_loop"):
            ctx.set_tuning(key, 1)
        for other in got[1:]:
            assert all(np.array_equal(x, y) for x, y in zip(got[0], other)), (n, kind)


@pytest.mark.parametrize("kind", ["one", "half", "table", "singletons"])
@pytest.mark.parametrize("graph", ["bin_zoo", "rmat12", "star", "no_edges"])
def test_merging_of_crowded_partitions(ctx, graph, kind):
    """Rows laid out by counters that many vertices ask at once: partners and
    statistics of a merging step equal the sorted-pair form's and the oracle's
    full count, with one round and three."""
    g = {"bin_zoo": GG.bin_zoo, "rmat12": lambda: GG.rmat(12), "no_edges": lambda: GG.csr_direct(6, []),
         "star": lambda: GG.csr_direct(2049, [(0, i) for i in range(1, 2049)])}[graph]()
    n, m, ind, adj = g[:4]
    lab = crowded(kind, n)
    ctx.upload_graph(n, m, ind, adj)
    for rule, lam, rounds, tie in ((O.MOD, 0.0, 1, 0), (O.CPM, 0.001, 3, 1)):
        got = []
        for sort in (0, 1):
            ctx.set_tuning("merge_sort", sort)
            ctx.upload_labels(lab)
            ctx.compress()
            ctx.statistics()
            ctx.merge(rule, lam, rounds=rounds, seed=4, step=1, tie=tie)
            got.append(ctx.labels())
            k = ctx.compress()
            ctx.statistics()
            _, so, ivo, evo = O.collect_statistics(n, ind, adj, ctx.labels())
            for x, y in zip(ctx.stats(k), (so, ivo, evo)):
                assert np.array_equal(x, y), (sort, rule)
        ctx.set_tuning("merge_sort", 0)
        assert np.array_equal(got[0], got[1]), rule


@pytest.mark.parametrize("n", [0, 1, 63, 64, 1023, 1025, 4096, 4097, 8193, 12289, 20481, 28673, 36864, 36865, 262144,
                               262145, 600001])
def test_noalloc_compression_sizes(ctx, n):
    """The allocation-free compression at the edges of its one-workgroup and
    tiled forms, few and many labels, with NEW_LABEL and
    with a label out of range (k = -1, the flag cleared for the next call)."""
    hip = Hip()
    rng = np.random.default_rng(n + 1)
    d, out, k_dev = hip.alloc(4 * n), hip.alloc(4 * (n + 8)), hip.alloc(4)
    for kinds, new, bad in ((max(1, n // 3), 0.2, False), (3, 0.0, True), (3, 0.0, False), (max(1, n), 0.0, False)):
        lab = (rng.integers(0, kinds, n) * 7 % max(1, n)).astype(np.int32)
        lab[rng.random(n) < new] = -1
        if bad and n:
            lab[n // 2] = n
        if n:
            hip.put(d, lab)
        hip.put(out, np.full(n + 8, -9, np.int32))
        parcd.compress_labels_noalloc(n, d, out, k_dev)
        hip.ok(hip.h.hipStreamSynchronize(None))
        got = hip.get(out, n + 8)
        assert (got[n:] == -9).all()
        if bad and n:
            assert int(hip.get(k_dev, 1)[0]) == -1
            continue
        want, k = O.compress_labels(lab) if n else (lab, 0)
        assert int(hip.get(k_dev, 1)[0]) == k
        assert np.array_equal(got[:n], want)
    for p in (d, out, k_dev):
        hip.ok(hip.h.hipFree(p))


def ring(n):  # 2n entries
    return GG.csr_direct(n, [(i, (i + 1) % n) for i in range(n)])


@pytest.mark.parametrize("kind", ["one", "half", "table", "seven_new", "planted", "sparse_ids", "singletons"])
@pytest.mark.parametrize("graph", ["bin_zoo", "unsorted", "rmat12", "ring", "one_tile", "past_a_tile", "wide"])
def test_contraction_by_rows_and_by_sort(ctx, graph, kind):
    """Pairs counted over community rows in tiles, and sorted entry by entry,
    equal the oracle's: few large rows, rows that cross tiles, empty rows (ids
    in use with gaps), both sides of the row length from which the rows are
    used, and tiles of 2,048 different pairs (half of a tile's table).  The
    limits on entries and labels force each way."""
    g = {"bin_zoo": GG.bin_zoo, "unsorted": lambda: GG.unsorted_copy(GG.bin_zoo()), "rmat12": lambda: GG.rmat(12),
         "ring": lambda: ring(5000), "one_tile": lambda: ring(1024), "past_a_tile": lambda: ring(1025),
         "wide": lambda: ring(33000)}[graph]()  # more communities than one pass of the sums takes
    n, m, ind, adj = g[:4]
    if kind == "planted":
        lab = (np.arange(n) * 40 // n).astype(np.int32)
    elif kind == "sparse_ids":
        lab = (np.arange(n) % 61 * (n // 64)).astype(np.int32)  # not compressed: empty rows between
    else:
        lab = crowded(kind, n)
    ctx.upload_graph(n, m, ind, adj)
    ctx.upload_labels(lab)
    if kind != "sparse_ids":
        ctx.compress()
        lab = ctx.labels()
    k = ctx.statistics()
    want = O.community_pairs(n, ind, adj, lab, k)
    try:
        for least, labels in ((0, 1 << 30), (0, 0), (0, 512), (1 << 30, 512)):  # rows, sort, by the volumes, sort
            ctx.set_tuning("contract_rows_min", least)
            ctx.set_tuning("contract_rows_labels", labels)
            got = ctx.contract()
            for x, y in zip(got, want):
                assert np.array_equal(x, y), (graph, kind, least, labels)
    finally:
        ctx.set_tuning("contract_rows_min", 1 << 22)
        ctx.set_tuning("contract_rows_labels", 512)


@pytest.mark.parametrize("cut", [1, 2, 3])
def test_batch_rows_of_every_width(cut):
    # one graph per row width at the edges of the short-row classes
    graphs, jobs = [], []
    for i, deg in enumerate([2, 4, 6, 8, 10, 16, 18, 32, 34, 64, 66, 130]):
        n = 2 * deg + 3 + 97 * i
        v = np.arange(n)
        nb = np.sort(np.stack([(v + s * d) % n for d in range(1, deg // 2 + 1) for s in (1, -1)], 1), axis=1)
        graphs.append((n, n * deg // 2, (np.arange(n + 1) * deg).astype(np.int32), nb.ravel().astype(np.int32)))
        # graphs end in different rounds, so the lists hold finished ones too
        jobs.append(parcd.job(kind=O.MOD, seed=i, max_iter=1 + (i + cut) % 4))
    graphs.append(GG.rmat(10, seed=5)[:4])  # rows of up to a few hundred
    jobs.append(parcd.job(kind=O.CPM, lam=0.01, seed=5, max_iter=5))
    labels = [np.arange(x[0], dtype=np.int32) for x in graphs]
    if cut == 3:
        labels = [np.where(np.arange(x[0]) % 5 == 0, -1, np.arange(x[0]) % 11).astype(np.int32) for x in graphs]
    with parcd.Batch(0, max_graphs=16, arena_bytes=256 << 20) as b:
        slots = [b.add(*x, lab, jb) for x, lab, jb in zip(graphs, labels, jobs)]
        while b.step(cut):
            pass
        got = [(b.labels(s),) + b.status(s)[1:] for s in slots]
    for x, lab, jb, (bl, it, k, score) in zip(graphs, labels, jobs, got):
        with parcd.Context(0) as c:
            pl, ps, pit, pk = c.run(*x, lab, jb)
        assert np.array_equal(bl, pl) and (it, k, score) == (pit, pk, ps)


@pytest.mark.parametrize("n", [200, 1025, 3001])
def test_wcc_loop_of_a_small_graph(n):
    rng = np.random.default_rng(n)
    deg = 12
    a = np.repeat(np.arange(n), deg)
    g = GG.csr_from_edges(a, (a + rng.integers(1, 24, n * deg)) % n)
    lab = (np.arange(g[0]) // 9).astype(np.int32)
    res = []
    for loop in (1, 0):
        with parcd.Context(0) as c:
            c.set_tuning("graph_loop", loop)
            c.upload_graph(*g[:4])
            c.triangles()
            c.upload_labels(lab)
            res.append(c.refine(parcd.job(kind=O.WCC, seed=3, max_iter=6)) + (c.labels(),))
    assert np.array_equal(res[0][-1], res[1][-1]) and res[0][:-1] == res[1][:-1]
