"""Level kernels at the edges of their tiles and steps: list lengths around
the head array, the gather steps and the degree classes, vertex counts around
the inspector's tiles and the bottom-up tiles, every lane width, against the
oracle.  Needs an MI355X."""
import sys

import numpy as np
import pytest

import ibfs_amd
import oracle

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def _symmetric(V, a, b):
    keep = a != b
    key = np.unique(np.concatenate([a[keep] * V + b[keep], b[keep] * V + a[keep]]))
    beg = np.concatenate([[0], np.cumsum(np.bincount(key // V, minlength=V))]).astype(np.int64)
    return beg, (key % V).astype(np.int32)


def _degrees_graph(V, seed):
    """A path over the first half of the vertices, and one vertex per listed
    degree d joined to d vertices of the path, three apart from its start."""
    half = V // 2
    a, b = [np.arange(half - 1)], [np.arange(1, half)]
    degrees = [1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 13, 63, 64, 65, 71, 72, 73, 135, 136, 137, 511, 512,
               513, 520, 521, 1031, 1032, 1033, 2048, 2049, 4200]
    rng = np.random.default_rng(seed)
    for i, d in enumerate(x for x in degrees for _ in range(3)):
        if d < half and half + i < V:
            a.append(np.full(d, half + i))
            b.append(rng.choice(half, size=d, replace=False))
    return _symmetric(V, np.concatenate(a), np.concatenate(b))


@pytest.mark.parametrize("V", [64, 513, 9000, 70_001])
@pytest.mark.parametrize("hubs", [None, 0, 16])
def test_list_lengths_around_the_gather_steps(V, hubs):
    """Lists of 1 to 4,200 neighbours (lengths around 4, 8, 12, 64 + 8, 128 + 8,
    512 + 8 and 1,024 + 8), with and without a hub cache, under the bottom-up,
    the hybrid and the alpha/beta policy, classes by default and with every
    vertex above degree 9 in the workgroup class."""
    beg, adj = _degrees_graph(V, seed=V)
    g = ibfs_amd.DeviceGraph(ibfs_amd.HostCsr.from_arrays(beg, adj), hub_count=hubs)
    src = np.random.default_rng(1).integers(0, V, size=130).astype(np.int32)
    want = oracle.bfs_many(beg, adj, src, threads=8)
    for lanes in (64, 128, 256, 512):
        for pol in (ibfs_amd.POLICY_BU_ONLY, ibfs_amd.POLICY_HYBRID, ibfs_amd.POLICY_ALPHA_BETA):
            for cls in ({}, dict(sml_shed=5, lrg_shed=9)):
                say(f"[gpu] lists V={V} hubs={hubs} lanes={lanes} policy={pol} {cls}")
                e = ibfs_amd.Engine(g, lane_bits=lanes, policy=pol, hybrid_hubs=40, **cls)
                np.testing.assert_array_equal(e.run_groups(src), want)
                e.close()


@pytest.mark.parametrize("V", [1, 2, 255, 256, 257, 511, 512, 513, 4095, 4097, 8 * 2048 + 1,
                               9 * 2048 - 1, 65_537, 300_001])
def test_vertex_counts_around_the_tiles(V):
    """Ring graphs with chords: every vertex count around the inspector's tiles
    and queue segments, frontiers in every segment, candidates queued and
    scanned, engine and batched form; depths and traversed edges."""
    say(f"[gpu] tiles V={V}")
    v = np.arange(V)
    beg, adj = _symmetric(V, np.concatenate([v, v]), np.concatenate([(v + 1) % V, (v * 7 + 3) % V]))
    g = ibfs_amd.DeviceGraph(ibfs_amd.HostCsr.from_arrays(beg, adj))
    src = np.random.default_rng(V).integers(0, V, size=40).astype(np.int32)
    want = oracle.bfs_many(beg, adj, src, threads=8)
    edges = sum(oracle.traversed_edges(beg, d) for d in want)
    for opts in (dict(), dict(policy=ibfs_amd.POLICY_BU_ONLY), dict(wg_size=256, inspect_vpt=1),
                 dict(wg_size=1024, inspect_vpt=8, policy=ibfs_amd.POLICY_BU_ONLY)):
        for lanes in (64, 256):
            e = ibfs_amd.Engine(g, lane_bits=lanes, **opts)
            np.testing.assert_array_equal(e.traversal(src), want)
            assert e.last_stats.traversed_edges == edges
            e.close()
    b = ibfs_amd.Batch(g, lane_bits=128, contexts=2, burst=4)
    np.testing.assert_array_equal(b.run(src), want)
    b.close()


@pytest.mark.parametrize("V", [1, 2, 3, 9, 10, 18, 65, 300, 2100])
@pytest.mark.parametrize("ring", [4, 9, 10, 32, 255])
def test_closeness_windows(V, ring):
    """Closeness on paths (an extra isolated vertex beside them): windows of
    one snapshot, of 8 and 9, of many, continued windows, lanes started
    later, at every width; sums and reach against closed forms."""
    say(f"[gpu] closeness path V={V} ring={ring}")
    v = np.arange(V - 1)
    beg, adj = _symmetric(V + 1, v, v + 1)
    g = ibfs_amd.DeviceGraph(ibfs_amd.HostCsr.from_arrays(beg, adj))
    src = np.arange(min(V + 1, 700), dtype=np.int32)
    if V > 1:
        src[-1] = V  # the isolated vertex
    s = src.astype(np.int64)
    want_sum = np.where(s < V, s * (s + 1) // 2 + (V - 1 - s) * (V - s) // 2, 0)
    want_reach = np.where(s < V, V, 1)
    for lanes in (64, 128, 256, 512):
        for opts in ({}, dict(phase_offsets=2, tail_div=0)):
            b = ibfs_amd.Batch(g, lane_bits=lanes, contexts=2, burst=4, ring_levels=ring, **opts)
            dsum, reach = b.closeness(src)
            np.testing.assert_array_equal(reach, want_reach)
            np.testing.assert_array_equal(dsum, want_sum)
            b.close()


def test_groupby_sizes_and_threads():
    """GroupBy around the steps of its sort and its small/large limit, sources
    with repeats and isolated ones, and four threads on one graph at once."""
    import threading
    h = ibfs_amd.HostCsr.rmat(15, 16, seed=5)
    beg, adj = h.arrays()
    g = ibfs_amd.DeviceGraph(h)
    rng = np.random.default_rng(3)
    for n in (1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 1000, 1024, 1025, 2049, 4095, 4096, 4097):
        say(f"[gpu] groupby n={n}")
        src = rng.integers(0, h.vert_count, size=n).astype(np.int32)
        np.testing.assert_array_equal(g.groupby(src), oracle.groupby(beg, adj, src))
    lists = [rng.integers(0, h.vert_count, size=700 + i).astype(np.int32) for i in range(4)]
    got = [[] for _ in lists]

    def work(i):
        for _ in range(20):
            got[i].append(g.groupby(lists[i]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    for src, outs in zip(lists, got):
        want = oracle.groupby(beg, adj, src)
        assert len(outs) == 20
        for o in outs:
            np.testing.assert_array_equal(o, want)


@pytest.mark.parametrize("keep", [False, True])
def test_groupby_across_graphs(keep):
    """GroupBy on graphs made and closed in turn, with one of the device kept
    alive or none, and on two graphs from two threads at once."""
    import threading
    say(f"[gpu] groupby across graphs keep={keep}")
    kept = ibfs_amd.DeviceGraph(ibfs_amd.HostCsr.rmat(10, 8, seed=9)) if keep else None
    for seed in range(4):
        hosts = [ibfs_amd.HostCsr.rmat(9 + seed, 16, seed=seed), ibfs_amd.HostCsr.rmat(11, 16, seed=seed)]
        graphs = [ibfs_amd.DeviceGraph(h) for h in hosts]
        lists = [np.random.default_rng(seed).integers(0, h.vert_count, size=900).astype(np.int32)
                 for h in hosts]
        got = [[], []]

        def work(i):
            for _ in range(10):
                got[i].append(graphs[i].groupby(lists[i]))

        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=60)
        for h, src, outs in zip(hosts, lists, got):
            want = oracle.groupby(*h.arrays(), src)
            assert len(outs) == 10
            for o in outs:
                np.testing.assert_array_equal(o, want)
        for g in graphs:
            g.close()
    if kept:
        kept.close()


@pytest.mark.parametrize("rows,cols,n", [(512, 512, 70), (40, 300, 128), (1, 50, 1)])
def test_noalloc_levels_enqueued_in_bursts(rows, cols, n):
    """Grids through the allocation-free call: at the vertex limit its ring
    holds 8 snapshots and is flushed over a hundred times, smaller graphs keep
    up to 32; traversals that end anywhere in a burst of eight levels."""
    say(f"[gpu] noalloc grid {rows}x{cols}")
    v = np.arange(rows * cols).reshape(rows, cols)
    beg, adj = _symmetric(rows * cols, np.concatenate([v[:, :-1].ravel(), v[:-1].ravel()]),
                          np.concatenate([v[:, 1:].ravel(), v[1:].ravel()]))
    g = ibfs_amd.DeviceGraph(ibfs_amd.HostCsr.from_arrays(beg, adj))
    out = ibfs_amd.DeviceBuffer(4 * n * rows * cols)
    src = np.random.default_rng(rows).integers(0, rows * cols, size=n).astype(np.int32)
    want = oracle.bfs_many(beg, adj, src, threads=8)
    edges = g.traversal_noalloc(src, out)
    np.testing.assert_array_equal(out.to_host().reshape(n, -1), want)
    assert edges == sum(oracle.traversed_edges(beg, d) for d in want)
    for k in range(1, min(cols, 20)):  # one source ever closer to the end
        s = np.array([rows * cols - k], dtype=np.int32)
        g.traversal_noalloc(s, out)
        np.testing.assert_array_equal(out.to_host(count=rows * cols),
                                      oracle.bfs_many(beg, adj, s, threads=1)[0])


@pytest.mark.parametrize("V,isolated", [(5, 5), (3, 0), (17, 1), (4097, 100), (70_001, 30_000)])
@pytest.mark.parametrize("lanes", [64, 128, 256, 512])
def test_planned_traversals_start_over(V, isolated, lanes):
    """Groups and cohorts of changing size started over and over on the same
    contexts (set-up block, snapshots, flags and counters of the traversal
    before), with repeated and isolated sources, on a graph without an edge,
    below one workgroup's share, and of many shares."""
    say(f"[gpu] starts V={V} isolated={isolated} lanes={lanes}")
    n = V - isolated
    v = np.arange(max(n, 1))
    beg, adj = _symmetric(V, np.concatenate([v, v]),
                          np.concatenate([(v + 1) % max(n, 1), (v * 7 + 3) % max(n, 1)]))
    g = ibfs_amd.DeviceGraph(ibfs_amd.HostCsr.from_arrays(beg, adj))
    b = ibfs_amd.Batch(g, lane_bits=lanes, contexts=2, burst=3)
    s = ibfs_amd.Server(g, lane_bits=lanes)
    for k in (1, lanes + 3, 2 * lanes + 17, 5):
        src = np.random.default_rng(k).integers(0, V, size=k).astype(np.int32)
        src[k // 2] = src[0]
        src[-1] = V - 1
        want = oracle.bfs_many(beg, adj, src, threads=8)
        np.testing.assert_array_equal(b.run(src), want)
        out = ibfs_amd.DeviceBuffer(4 * k * V)
        s.wait(s.submit(src, out))
        np.testing.assert_array_equal(out.to_host(np.int32, k * V).reshape(k, V), want)
    s.close()
    b.close()


@pytest.mark.parametrize("rows,cols", [(1, 150), (7, 43), (40, 301), (3, 1200)])
@pytest.mark.parametrize("mode", [0, 2, 3])
def test_emission_of_deep_windows(rows, cols, mode):
    """Paths and grids of 47 to 1,200 levels: emission windows of 16 levels and
    more (rings of 32 and 64) and of 64 and more (ring of 255), continued ones
    too, aligned and unaligned rows, a partial second group, in the engine, the
    batched form, the server and the allocation-free call."""
    V = rows * cols
    v = np.arange(V).reshape(rows, cols)
    beg, adj = _symmetric(V, np.concatenate([v[:, :-1].ravel(), v[:-1].ravel()]),
                          np.concatenate([v[:, 1:].ravel(), v[1:].ravel()]))
    g = ibfs_amd.DeviceGraph(ibfs_amd.HostCsr.from_arrays(beg, adj))
    every = np.random.default_rng(V).integers(0, V, size=515).astype(np.int32)
    depths = oracle.bfs_many(beg, adj, every, threads=8)
    for lanes in (64, 128, 256, 512):
        src, want = every[:lanes + 3], depths[:lanes + 3]
        for ring in (32, 64, 255):
            say(f"[gpu] deep windows {rows}x{cols} mode={mode} lanes={lanes} ring={ring}")
            e = ibfs_amd.Engine(g, lane_bits=lanes, emit_mode=mode, ring_levels=ring)
            np.testing.assert_array_equal(e.run_groups(src), want)
            e.close()
            b = ibfs_amd.Batch(g, lane_bits=lanes, contexts=2, burst=8, emit_mode=mode,
                               ring_levels=ring)
            np.testing.assert_array_equal(b.run(src), want)
            b.close()
        s = ibfs_amd.Server(g, lane_bits=lanes, emit_mode=mode)
        out = ibfs_amd.DeviceBuffer(4 * len(src) * V)
        s.wait(s.submit(src, out))
        np.testing.assert_array_equal(out.to_host(np.int32, len(src) * V).reshape(-1, V), want)
        s.close()
    out = ibfs_amd.DeviceBuffer(4 * 128 * V)
    g.traversal_noalloc(every[:128], out, ibfs_amd.default_config(emit_mode=mode))
    np.testing.assert_array_equal(out.to_host().reshape(128, V), depths[:128])


def test_groupby_takes_the_sources_of_its_own_call():
    """Calls of one size with other sources each time, on two graphs in turn
    and with nothing in between: the block that holds the sources is the same."""
    say("[gpu] groupby, other sources each call")
    hosts = [ibfs_amd.HostCsr.rmat(13, 16, seed=s) for s in (1, 2)]
    graphs = [ibfs_amd.DeviceGraph(h) for h in hosts]
    rng = np.random.default_rng(0)
    for n in (1, 16, 700, 4096):
        lists = [rng.integers(0, 1 << 13, size=n).astype(np.int32) for _ in range(12)]
        got = [graphs[i % 2].groupby(s) for i, s in enumerate(lists)]
        for i, s in enumerate(lists):
            np.testing.assert_array_equal(got[i], oracle.groupby(*hosts[i % 2].arrays(), s))


@pytest.mark.parametrize("opts", [dict(policy=ibfs_amd.POLICY_FIXED, sw_level=1),
                                  dict(policy=ibfs_amd.POLICY_FIXED, sw_level=3),
                                  dict(policy=ibfs_amd.POLICY_BU_ONLY),
                                  dict(hybrid_gamma=0), dict(hybrid_gamma=0, alpha=14, beta=24)])
def test_posted_directions_follow_the_rule(opts):
    """The direction of every level is the rule's for the counters posted with
    it, where the host launches the posted direction's kernel (kernel timing)
    and where levels are enqueued ahead; both log the same levels."""
    say(f"[gpu] posted directions {opts}")
    h = ibfs_amd.HostCsr.rmat(14, 16, seed=6)
    g = ibfs_amd.DeviceGraph(h)
    src = h.gen_sources(256, seed=7)
    want = oracle.bfs_many(*h.arrays(), src, threads=8)
    cfg = ibfs_amd.default_config(**opts)

    def rule(level, prev, li, li_before):
        if cfg.policy == ibfs_amd.POLICY_BU_ONLY:
            return 1
        if cfg.policy == ibfs_amd.POLICY_FIXED:
            return 0 if level <= cfg.sw_level else 1
        if prev != 1:
            return 1 if li["m_frontier"] * cfg.alpha > li["m_unvisited"] else 0
        nf = li["n_frontier"]
        return 0 if nf * cfg.beta < h.vert_count and nf < li_before["n_frontier"] else 1

    logs = []
    for timing in (1, 0):
        e = ibfs_amd.Engine(g, lane_bits=128, kernel_timing=timing, **opts)
        for half, depths in ((src[:128], want[:128]), (src[128:], want[128:])):
            np.testing.assert_array_equal(e.traversal(half), depths)
            log = e.level_log()
            for level in range(1, len(log)):
                before = log[level - 2] if level > 1 else dict(n_frontier=1 << 62)
                prev = log[level - 1]["direction"] if level > 1 else -1
                assert log[level]["direction"] == rule(level, prev, log[level - 1], before), level
            logs.append([(x["direction"], x["n_changed"], x["n_frontier"], x["n_unvisited"]) for x in log])
        e.close()
    assert logs[:2] == logs[2:]


def test_groupby_calls_do_not_wait_for_each_other():
    """Two threads, each with its graph: calls overlap on the device, so both
    take well under the time that one thread takes for all of them (half of it
    where they overlap, nearly all of it where a call waits for the other's)."""
    import threading
    import time
    say("[gpu] groupby of two graphs at once")
    hosts = [ibfs_amd.HostCsr.rmat(14, 16, seed=s) for s in (3, 4)]
    graphs = [ibfs_amd.DeviceGraph(h) for h in hosts]
    lists = [np.random.default_rng(s).integers(0, 1 << 14, size=4096).astype(np.int32) for s in (3, 4)]

    def calls(i, out=None):
        for _ in range(300):
            got = graphs[i].groupby(lists[i])
        if out is not None:
            out[i] = got

    def at_once(out):
        threads = [threading.Thread(target=calls, args=(i, out)) for i in (0, 1)]
        t0 = time.perf_counter()
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=60)
        return time.perf_counter() - t0

    def in_turn():
        t0 = time.perf_counter()
        calls(0)
        calls(1)
        return time.perf_counter() - t0

    got = [None, None]
    at_once(got)
    for h, src, o in zip(hosts, lists, got):
        np.testing.assert_array_equal(o, oracle.groupby(*h.arrays(), src))
    ratio = min(at_once(got) for _ in range(5)) / min(in_turn() for _ in range(5))
    say(f"[gpu] at once / in turn: {ratio:.2f}")
    assert ratio < 0.75


def test_groupby_past_the_wait_limit():
    """Calls that give up (the limit set from the host; their kernels end
    normally) from many threads, then closing their graph, and calls of another
    graph before and after it: exact, and no call of the other graph fails."""
    import threading
    say("[gpu] groupby past the wait limit")
    h = ibfs_amd.HostCsr.rmat(14, 16, seed=5)
    src = np.random.default_rng(5).integers(0, 1 << 14, size=4096).astype(np.int32)
    want = oracle.groupby(*h.arrays(), src)
    other = ibfs_amd.DeviceGraph(h)
    for _ in range(3):
        g = ibfs_amd.DeviceGraph(h)
        codes = []

        def work():
            for _ in range(8):
                try:
                    np.testing.assert_array_equal(g.groupby(src), want)
                except ibfs_amd.IbfsError as e:
                    codes.append(e.code)

        old = ibfs_amd.get_wait_timeout()
        ibfs_amd.set_wait_timeout(1e-9)
        try:
            threads = [threading.Thread(target=work) for _ in range(6)]
            for t in threads:
                t.start()
            for t in threads:
                t.join(timeout=60)
        finally:
            ibfs_amd.set_wait_timeout(old)
        assert set(codes) <= {ibfs_amd._lib.IBFS_ERR_STATE}
        np.testing.assert_array_equal(other.groupby(src), want)
        g.close()
        np.testing.assert_array_equal(other.groupby(src), want)


def test_server_launches_two_bursts_after_a_run_of_deep_cohorts():
    """Polls of the host per cohort (four or eight levels each, by the server's
    counter): a query of 12 levels takes fewer once two such cohorts came in a
    row, not before, and one of two levels ends that."""
    say("[gpu] server bursts")
    n = 2000  # a star, and a path of 12 behind it
    a = np.concatenate([np.zeros(n - 1, dtype=np.int64), n + np.arange(11)])
    b = np.concatenate([np.arange(1, n), n + 1 + np.arange(11)])
    beg, adj = _symmetric(n + 12, a, b)
    g = ibfs_amd.DeviceGraph(ibfs_amd.HostCsr.from_arrays(beg, adj))
    s = ibfs_amd.Server(g, lane_bits=64)
    out = ibfs_amd.DeviceBuffer(4 * (n + 12))
    want = {v: oracle.bfs_many(beg, adj, np.array([v], dtype=np.int32), threads=1)[0] for v in (n, 5)}

    def polls(v):
        before = s.counters()["levels"]
        q = s.submit(np.array([v], dtype=np.int32), out)
        s.wait(q)
        s.release(q)
        np.testing.assert_array_equal(out.to_host(), want[v])
        return s.counters()["levels"] - before

    for _ in range(2):
        assert [polls(n) for _ in range(2)] == [3] * 2  # levels 1 to 12, the last changes nothing
        assert polls(n) == 2
        assert polls(5) == 1
        assert polls(n) == 3 and polls(5) == 1
    s.close()
