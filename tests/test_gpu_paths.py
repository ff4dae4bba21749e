"""Kernel variants and dispatch rules at the sizes where they can go wrong
(edges of tiles, remainders, escapes), against the CPU oracle.  Results are
whole numbers: equal, no tolerance."""
import numpy as np
import pytest

from graphs import csc_from_edges, path_graph, random_graph, star_graph, symmetrize
from oracle import cpu

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def some_graph(name):
    """(col_ptr, row_idx, n_rows, symmetric, root)"""
    rng = np.random.default_rng(41)
    if name == "one":
        return np.zeros(2, np.uint32), np.zeros(0, np.uint32), 1, True, 0
    if name == "path2500":
        return (*path_graph(2500), 2500, True, 0)
    if name == "star70001":
        return (*star_graph(70001), 70001, True, 5)
    if name == "directed4099":
        cp, ri = random_graph(rng, 4099, 30000)
        ri = ri[: int(cp[3000])]
        cp = np.minimum(cp, cp[3000]).astype(np.uint64)
        return cp, ri, 3000, False, int(np.flatnonzero(np.diff(cp.astype(np.int64)))[0])
    n = int(name)
    cp, ri = random_graph(rng, n, 3 * n, directed=False)
    return cp, ri, n, True, int(np.argmax(np.diff(cp)))


# a work-group of the histogram takes 4096 vertices, a lane four; tables of
# more than 4096 levels are counted in global memory; degrees of 65535 and
# more are not in the 16-bit array
@pytest.mark.parametrize("name", ["one", "3", "4", "257", "4096", "4099", "20001", "path2500",
                                  "star70001", "directed4099"])
def test_level_histogram_edges(engine, name):
    say("histogram", name)
    cp, ri, n_rows, sym, root = some_graph(name)
    engine.upload_csc(cp, ri, n_rows=n_rows, symmetric=sym)
    want, ec, _ = cpu.bfs_queue(cp, ri, root, n_rows=n_rows)
    deg = np.where(np.arange(len(want)) < n_rows, np.diff(cp.astype(np.int64)), 0)
    hist = np.bincount(want[want >= 0])
    lev, st = engine.run(root, "llb")
    assert (lev == want).all()
    assert [st[k] for k in ("edges_count", "reached", "max_level", "n_levels")] == [
        ec, int(hist.sum()), len(hist) - 1, len(hist)]
    for size in (8, 1024, 4096):
        counts, edges = engine.level_histogram(size)
        assert (counts == hist).all()
        assert (edges == np.bincount(want[want >= 0], weights=deg[want >= 0])).all()


# tiny levels run in one work-group: tiles of 1024 frontier entries, up to
# 2048 edges a level, 4096 levels a launch
@pytest.mark.parametrize("name", ["one", "path2500", "path9001", "star70001", "directed4099",
                                  "hub1023", "hub1025", "hub2045", "hub2048", "hub2049", "hub4097"])
def test_tiny_levels_loop(engine, name):
    say("tiny levels", name)
    if name.startswith("hub"):
        # a hub at the end of a path whose k leaves share one far vertex
        k = int(name[3:])
        src = np.concatenate([[0, 1], np.full(k, 2), np.arange(k) + 3])
        dst = np.concatenate([[1, 2], np.arange(k) + 3, np.full(k, k + 3)])
        cp, ri = csc_from_edges(k + 4, *symmetrize(src, dst))
        n_rows, sym, root = k + 4, True, 0
    elif name == "path9001":
        cp, ri, n_rows, sym, root = *path_graph(9001), 9001, True, 4500
    else:
        cp, ri, n_rows, sym, root = some_graph(name)
    engine.upload_csc(cp, ri, n_rows=n_rows, symmetric=sym)
    want, ec, _ = cpu.bfs_queue(cp, ri, root, n_rows=n_rows)
    engine.load_scheduler()
    try:
        for s, kw in [("llb", {}), ("slb", {}), ("learned", {}), ("llb", {"hub_degree": 512}),
                      ("llb", {"mark_ratio_q10": 0}), ("slb", {"mark_ratio_q10": 0xFFFFFFFF})]:
            before = engine.params
            if kw:
                engine.set_params(**kw)
            lev, st, par = engine.run(root, s, parents=True)
            engine.set_params(**before)
            assert (lev == want).all(), (s, kw)
            assert cpu.check_parents(cp, ri, root, want, par, n_rows=n_rows) == 0
            assert [st[k] for k in ("edges_count", "reached", "max_level", "n_levels")] == [
                ec, int((want >= 0).sum()), int(want.max()), int(want.max()) + 1]
            assert sum(st["steps"].values()) == st["n_levels"]
            if s != "learned":
                assert st["steps"][s] == st["n_levels"]
    finally:
        engine.set_scheduler_weights(None)


# several work-groups share a tile of frontier entries: tiles of one hub, of
# hubs beside empty lists, totals that are no multiple of a round or a part
@pytest.mark.parametrize("leaves", [4096, 4097, 20011, 150001])
@pytest.mark.parametrize("ptr", [np.uint32, np.uint64])
def test_tiles_shared_by_groups(engine, leaves, ptr):
    say("shared tiles", leaves, ptr.__name__)
    rng = np.random.default_rng(leaves)
    k, n = 29, leaves + 400
    # root -> k hubs (far apart), each hub -> a random tenth of the leaves
    hubs = 1 + 13 * np.arange(k)
    src, dst = [np.zeros(k, np.int64)], [hubs]
    for h in hubs:
        to = rng.permutation(np.arange(400, n))[: leaves // 10 + h]
        src.append(np.full(len(to), h))
        dst.append(to)
    src, dst = np.concatenate(src), np.concatenate(dst)
    for sym in (False, True):
        e = symmetrize(src, dst) if sym else (src, dst)
        cp, ri = csc_from_edges(n, *e, dtype=ptr)
        engine.upload_csc(cp, ri, n_rows=n if sym else n - 7, symmetric=sym)
        want, ec, _ = cpu.bfs_queue(cp, ri, 0, n_rows=n if sym else n - 7)
        before = engine.params
        for kw in ({}, {"llb_wg": 64}, {"llb_wg": 1024}, {"hub_degree": 1024},
                   {"hub_degree": 16, "llb_wg": 128},
                   {"mark_ratio_q10": 0}, {"mark_ratio_q10": 0xFFFFFFFF}):
            engine.set_params(**kw)
            for s in ("llb", "slb"):
                for loop in ({}, {"parents": True}, {"graph_loop": True}, {"device_loop": True}):
                    lev, st = engine.run(0, s, **loop)[:2]
                    assert (lev == want).all() and st["edges_count"] == ec, (kw, s, loop)
            engine.set_params(**before)


# the allocation-free search: tiny levels in one work-group (up to 2048 edges),
# exact-once and marking levels, tiles shared by groups, compaction of 8192
# vertices per group, level arrays at any 4-byte alignment
@pytest.mark.parametrize("name", ["one", "3", "257", "8191", "8193", "20001", "path9001",
                                  "star70001", "directed4099", "hub2047", "hub2049", "hub20011",
                                  "rmat15", "wide4194304"])
@pytest.mark.parametrize("ptr", [np.uint32, np.uint64])
@pytest.mark.parametrize("shift", [0, 1])
def test_noalloc_edges(engine, name, ptr, shift):
    import ctypes as C

    import bfsx
    from test_zz_no_alloc import Dev, hip
    say("noalloc", name, ptr.__name__, shift)
    h = hip()
    if name.startswith("hub"):
        k = int(name[3:])
        src = np.concatenate([[0, 1], np.full(k, 2), np.arange(k) + 3])
        dst = np.concatenate([[1, 2], np.arange(k) + 3, np.full(k, k + 3)])
        cp, ri = csc_from_edges(k + 4, *symmetrize(src, dst))
        n_rows, root = k + 4, 0
    elif name.startswith("wide"):
        # one level of nearly every vertex, which fills the queue's buffer up
        # to the marks, then 200000 leaves of which share one more vertex
        n_rows = int(name[4:])
        leaf = np.arange(1, n_rows - 3)
        src = np.concatenate([np.zeros(len(leaf), np.int64), leaf[-200000:], [n_rows - 3]])
        dst = np.concatenate([leaf, np.full(200000, n_rows - 3), [n_rows - 2]])
        cp, ri = csc_from_edges(n_rows, *symmetrize(src, dst))
        root = 7
    elif name == "rmat15":
        engine.generate_rmat(15, 16, 0.57, 0.19, 0.19, 3, 4, 4)
        cp, ri = engine.download_csc()
        n_rows, root = 1 << 15, int(engine.pick_roots(1, 5)[0])
    elif name == "path9001":
        cp, ri, n_rows, root = *path_graph(9001), 9001, 4500
    else:
        cp, ri, n_rows, _, root = some_graph(name)
    cp, n = cp.astype(ptr), len(cp) - 1
    want, _, _ = cpu.bfs_queue(cp, ri, root, n_rows=n_rows)
    d_cp, d_ri, d_lev = Dev.of(h, cp), Dev.of(h, ri), Dev(h, 4 * (n + 2))
    try:
        def run(row_idx, col_ptr):
            nl = C.c_uint32(0)
            rc = bfsx.lib().bfsx_run_noalloc(0, None, col_ptr.p, cp.itemsize, row_idx.p, n, n_rows,
                                             len(ri), root, d_lev.p.value + 4 * shift, C.byref(nl))
            return rc, nl.value, d_lev.get(np.int32, n + 2)[shift:shift + n]
        for _ in range(2):
            rc, nl, lev = run(d_ri, d_cp)
            assert rc == 0 and (lev == want).all() and nl == int(want.max()) + 1
        # entries past the graph are skipped and reported, in lists and offsets
        if len(ri) > 100:
            bad = ri.copy()
            bad[len(ri) // 2] = n + 1000
            used = np.searchsorted(cp.astype(np.int64), len(ri) // 2, side="right") - 1
            d_bad = Dev.of(h, bad)
            rc, _, lev = run(d_bad, d_cp)
            d_bad.free()
            assert rc == (1 if used < n_rows and want[used] >= 0 else 0)
            assert ((lev >= 0) <= (want >= 0)).all() and (lev[lev >= 0] >= want[lev >= 0]).all()
            cut = cp.copy()
            cut[root + 1] = len(ri) + 5  # the root's list runs past the end
            d_cut = Dev.of(h, cut)
            rc, _, lev = run(d_ri, d_cut)
            d_cut.free()
            assert rc == 1 and lev[root] == 0
    finally:
        for d in (d_cp, d_ri, d_lev):
            d.free()


# levels cross as 1, 2 or 4 bytes each (up to 254, 65534 or more levels) in
# pieces of 2 MB through eight pinned buffers, whole pieces by up to four
# threads; graphs cross as bytes the same way
@pytest.mark.parametrize("depth", [254, 255, 256, 65535, 65536])
@pytest.mark.parametrize("n", [70001, 1 << 20, (1 << 20) + 1, 5 * (1 << 20) + 13])
def test_levels_and_graphs_to_pageable_memory(engine, depth, n):
    say("transfer", depth, n)
    # a path of depth + 1 vertices; the other vertices hang off its first one
    # (a third of them) or are isolated
    rng = np.random.default_rng(n)
    other = np.arange(depth + 1, n)
    leaf = other[rng.random(len(other)) < 0.33]
    src = np.concatenate([np.arange(depth), np.zeros(len(leaf), np.int64)])
    dst = np.concatenate([np.arange(depth) + 1, leaf])
    cp, ri = csc_from_edges(n, *symmetrize(src, dst), dtype=np.uint64)
    engine.upload_csc(cp, ri, symmetric=True)
    got_cp, got_ri = engine.download_csc()
    assert (got_cp == cp).all() and (got_ri == ri).all()
    want = np.full(n, -1, np.int32)
    want[: depth + 1] = np.arange(depth + 1)
    want[leaf] = 1
    lev, st, par = engine.run(0, "llb", parents=True)
    assert st["max_level"] == depth and (lev == want).all()
    ok = par[1:depth + 1] == np.arange(depth)
    assert ok.all() and (par[leaf] == 0).all() and par[0] == 0
    assert (par[want < 0] == 0xFFFFFFFF).all()


# a graph is checked on the card beside the resident one: refused graphs leave
# that as it was, wherever the bad entry is
@pytest.mark.parametrize("ptr", [np.uint32, np.uint64])
@pytest.mark.parametrize("nnz", [4, 7, 1023, 400001])
def test_refused_graphs(engine, ptr, nnz):
    import bfsx
    say("refused", ptr.__name__, nnz)
    cp0, ri0 = path_graph(100)
    engine.upload_csc(cp0, ri0, symmetric=True)
    rng = np.random.default_rng(nnz)
    n = max(3, nnz // 5)
    src = np.sort(rng.integers(0, n, nnz))
    cp = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(ptr)
    ri = rng.integers(0, n, nnz).astype(np.uint32)

    def refused(cp, ri, text, n_rows=None):
        with pytest.raises(bfsx.BfsxError) as e:
            engine.upload_csc(cp, ri, n_rows=n_rows)
        assert e.value.status == 1 and text in e.value.msg
        lev, _ = engine.run(99, "llb")
        assert (lev == 99 - np.arange(100)).all()

    for at in sorted({0, 1, nnz // 2, nnz - 1}):
        bad = ri.copy()
        bad[at] = n
        refused(cp, bad, "row_idx entry >= n_cols")
        bad[at] = 0xFFFFFFFF
        refused(cp, bad, "row_idx entry >= n_cols")
    for at in sorted({1, n // 2, n - 1}):
        bad = cp.copy()
        bad[at] = nnz + 9
        refused(bad, ri, "not monotone")
    refused(cp + ptr(1), ri, "col_ptr[0] != 0")
    refused(cp, ri[:-1], "end does not match")
    engine.upload_csc(cp, ri)
    got_cp, got_ri = engine.download_csc()
    assert (got_cp == cp).all() and (got_ri == ri).all()


# runs of 4096 edges find their columns: a list longer than a run, more than
# 4096 empty columns inside one, lists behind n_rows; chunks of 2048 vertices
@pytest.mark.parametrize("shape", ["hub", "gaps", "tail", "small"])
@pytest.mark.parametrize("order", ["hub_first", "id", "pull_hub_first"])
def test_order_adjacency_runs(engine, shape, order):
    say("order", shape, order)
    rng = np.random.default_rng(len(shape))
    n = {"hub": 30011, "gaps": 70001, "tail": 5000, "small": 3}[shape]
    if shape == "hub":
        src = np.concatenate([np.full(20000, 7), rng.integers(0, n, 30000)])
    elif shape == "gaps":
        src = np.concatenate([rng.integers(0, 50, 9000), np.full(3, 20000), np.full(9000, n - 2)])
    else:
        src = rng.integers(0, n, 4 * n)
    dst = rng.integers(0, n, len(src))
    sym = shape != "tail"
    e = symmetrize(src, dst) if sym else (src, dst)
    cp, ri = csc_from_edges(n, *e)
    ri = ri.copy()
    for v in range(n):  # any order: the lists are sorted by the engine
        rng.shuffle(ri[cp[v]:cp[v + 1]])
    n_rows = n if sym else n - 1000
    engine.upload_csc(cp, ri, n_rows=n_rows, symmetric=sym)
    engine.order_adjacency(order)
    got_cp, got = engine.download_csc()
    deg = np.diff(cp.astype(np.int64)) * (np.arange(n) < n_rows)
    rank = np.empty(n, np.int64)
    rank[np.lexsort((np.arange(n), -deg))] = np.arange(n)
    col = np.repeat(np.arange(n), np.diff(cp.astype(np.int64)))
    assert (got_cp == cp).all()
    if order == "pull_hub_first":
        assert (got == ri).all()
    else:
        key = ri.astype(np.int64) if order == "id" else rank[ri]
        want = ri[np.lexsort((key, col))]
        rows = slice(0, int(cp[n_rows]))
        assert (got[rows] == want[rows]).all()
    for root in rng.integers(0, n_rows, 3):
        want, _, _ = cpu.bfs_queue(cp, ri, int(root), n_rows=n_rows)
        for s in ["llb", "glb"] + (["pull"] if sym else []):
            assert (engine.run(int(root), s)[0] == want).all(), (s, root)


# bottom-up with the hub-first copy: candidates of one to six neighbours (the
# first four beside the list), degrees that the 16-bit array does not hold,
# chunks of 2048 vertices, no hubs below 64 vertices
@pytest.mark.parametrize("n", [5, 63, 64, 2047, 2048, 2049, 6000, 140001])
@pytest.mark.parametrize("ptr", [np.uint32, np.uint64])
def test_bottom_up_short_lists(engine, n, ptr):
    say("bottom-up", n, ptr.__name__)
    rng = np.random.default_rng(n)
    # vertex v picks v % 4 earlier neighbours; the largest graph's vertex 0 is
    # next to every second vertex (degree 70000)
    src = np.repeat(np.arange(n), np.arange(n) % 4)
    dst = (rng.random(len(src)) * np.maximum(src, 1)).astype(np.int64)
    if n > 100000:
        even = np.arange(2, n, 2)
        src, dst = np.concatenate([src, even]), np.concatenate([dst, np.zeros(len(even), np.int64)])
    keep = src != dst
    cp, ri = csc_from_edges(n, *symmetrize(src[keep], dst[keep]), dtype=ptr)
    engine.upload_csc(cp, ri, symmetric=True)
    engine.order_adjacency("pull_hub_first")
    deg = np.diff(cp.astype(np.int64))
    for root in {0, int(np.flatnonzero(deg)[-1]), int(np.argmin(np.where(deg > 0, deg, 9999999)))}:
        want, ec, _ = cpu.bfs_queue(cp, ri, root)
        lev, st, par = engine.run(root, "pull", parents=True)
        assert (lev == want).all() and st["edges_count"] == ec
        assert cpu.check_parents(cp, ri, root, want, par) == 0
        engine.run(root, "pull", levels=False, step_times=True)
        later = lambda k: (want > k) | (want < 0)
        for t in engine.last_trace():
            lo = int(deg[later(t["level"] + 1)].sum()) + int((want == t["level"] + 1).sum())
            assert lo <= t["pull_scanned"] <= int(deg[later(t["level"])].sum())


# batches: level rows of any length (128 vertices per group, four per word),
# every bitset width, lists beyond 256 edges shared by waves, active vertices
# listed again after bottom-up levels, more vertices than the totals have parts
@pytest.mark.parametrize("n", [1, 2, 5, 127, 128, 129, 4099, 70002])
@pytest.mark.parametrize("n_bits", [1, 33, 128, 250])
def test_batch_edges(engine, n, n_bits):
    say("batch", n, n_bits)
    rng = np.random.default_rng(n + n_bits)
    m = 3 * n
    src = (rng.random(m) ** 3 * n).astype(np.int64)
    dst = rng.integers(0, n, m)
    for sym in (True, False):
        cp, ri = csc_from_edges(n, *(symmetrize(src, dst) if sym else (src, dst)))
        n_rows = n if sym else n - n // 10
        engine.upload_csc(cp, ri, n_rows=n_rows, symmetric=sym)
        sources = rng.integers(0, n, n_bits + 3)
        bits = np.concatenate([np.arange(n_bits), rng.integers(0, n_bits, 3)])
        want = cpu.msbfs_u8(cp, ri, sources, bits, n_bits, n_rows=n_rows)
        deg = np.diff(cp.astype(np.int64))[:n_rows]
        ec = int(((want[:, :n_rows] != 0xFF) * deg).sum())
        before = engine.params
        for kw in ({}, {"ms_relabel": 0, "ms_push_divisor": 1}, {"ms_push_divisor": 1024}):
            engine.set_params(**kw)
            lev, st = engine.run_multi(sources, bits, n_bits)
            engine.set_params(**before)
            assert (lev == want).all() and st["edges_count"] == ec, kw


# small graphs: waves of the bottom-up step take down to two bitmap words of a
# chunk, with and without the hub-first copy; GLB marks up to 2^22 vertices and
# buckets beyond or when asked to
@pytest.mark.parametrize("n", [40, 65, 2050, 33000, 300001])
@pytest.mark.parametrize("order", ["", "pull_hub_first"])
def test_small_graph_steps(engine, n, order):
    say("small graphs", n, order)
    rng = np.random.default_rng(n)
    src = (rng.random(4 * n) ** 2 * n).astype(np.int64)
    dst = rng.integers(0, n - n // 8, 4 * n)
    cp, ri = csc_from_edges(n, *symmetrize(src, dst))
    engine.upload_csc(cp, ri, symmetric=True)
    if order:
        engine.order_adjacency(order)
    engine.load_scheduler()
    before = engine.params
    try:
        for root in rng.choice(src, 3):
            want, ec, _ = cpu.bfs_queue(cp, ri, int(root))
            for wg in (64, 512):
                engine.set_params(pull_wg=wg)
                lev, st, par = engine.run(int(root), "pull", parents=True)
                assert (lev == want).all() and st["edges_count"] == ec
                assert cpu.check_parents(cp, ri, int(root), want, par) == 0
                assert (engine.run(int(root), "learned")[0] == want).all()
            for ratio in (0, 512):
                engine.set_params(bucket_ratio_q10=ratio)
                assert (engine.run(int(root), "glb")[0] == want).all()
            engine.set_params(**before)
    finally:
        engine.set_params(**before)
        engine.set_scheduler_weights(None)


# the last of a speculative step's groups ends the level: frontiers of one
# group, of whole and ragged tiles, of more tiles than the grid has groups
@pytest.mark.parametrize("width", [700, 4096, 4097, 20011, 140003])
@pytest.mark.parametrize("kind", [0, 2])  # LLB, SLB
@pytest.mark.parametrize("ptr", [np.uint32, np.uint64])
def test_level_end_by_last_group(engine, width, kind, ptr):
    say("last group", width, kind, ptr.__name__)
    rng = np.random.default_rng(width)
    depth, n = 6, 1 + 6 * width
    lay = 1 + width * np.arange(depth)
    src, dst = [np.zeros(width, np.int64)], [lay[0] + np.arange(width)]
    for i in range(depth - 1):
        for _ in range(4):
            src.append(lay[i] + rng.integers(0, width, width))
            dst.append(lay[i + 1] + np.arange(width))
    cp, ri = csc_from_edges(n, *symmetrize(np.concatenate(src), np.concatenate(dst)))
    want, ec, _ = cpu.bfs_queue(cp, ri, 0)
    engine.upload_csc(cp.astype(ptr), ri, symmetric=True)
    w = np.zeros(1476, np.float32)
    w[-4:] = 1
    w[-4 + kind] = 0  # constant outputs, the smallest one's kind is taken
    before = engine.params
    try:
        engine.set_scheduler_weights(w)
        for wg in (64, 256, 1024):
            for hub in (0, 6):
                engine.set_params(llb_wg=wg, hub_degree=hub, mark_ratio_q10=0xFFFFFFFF)
                for spec in (1, 0, 1):
                    engine.set_params(speculate=spec)
                    lev, st = engine.run(0, "learned")
                    assert np.array_equal(lev, want), (wg, hub, spec)
                    assert st["edges_count"] == ec and st["reached"] == n
                    assert st["n_levels"] == depth + 1
                    # (the root's level runs LLB)
                    assert st["steps"][("llb", "glb", "slb")[kind]] == depth + (kind == 0)
    finally:
        engine.set_scheduler_weights(None)
        engine.set_params(**before)


# hubs gathered at the level end: fixed and changing kinds of step, bottom-up
# after bottom-up, after marking and bucketed steps and after thin ones, and
# trials of every kind from one state (whose walk then covers each level)
@pytest.mark.parametrize("scale", [9, 13, 16])
@pytest.mark.parametrize("bucket", [0, 0xFFFFFFFF])
def test_hubs_at_level_ends(engine, scale, bucket):
    say("hubs", scale, bucket)
    engine.generate_rmat(scale, 12, 0.57, 0.19, 0.19, 31 + scale, 41 + scale, 4)
    cp, ri = engine.download_csc()
    roots = engine.pick_roots(2, 9)
    before = engine.params
    try:
        engine.set_params(bucket_ratio_q10=bucket)
        engine.order_adjacency("pull_hub_first")
        want = [cpu.bfs_queue(cp, ri, int(r)) for r in roots]
        kinds = np.random.default_rng(scale)
        for r, (lv, ec, _) in zip(roots, want):
            for trial in range(6):
                w = np.zeros(1476, np.float32)
                w[:] = kinds.normal(0, 0.4, 1476)
                engine.set_scheduler_weights(w)
                for mark in (0, 4, 0xFFFFFFFF):
                    engine.set_params(mark_ratio_q10=mark)
                    lev, st = engine.run(int(r), "learned")
                    assert np.array_equal(lev, lv) and st["edges_count"] == ec, (trial, mark)
            for s in ("pull", "beamer"):
                lev, st = engine.run(int(r), s)
                assert np.array_equal(lev, lv) and st["edges_count"] == ec, s
        engine.set_params(mark_ratio_q10=4)
        X, _, _ = engine.sched_record(roots, repeats=2, epsilon=1.0, seed=3)
        sizes = [int((lv == d).sum()) for lv, _, _ in want for d in range(int(lv.max()) + 1)]
        got = np.rint(2.0 ** (X[:, 0].astype(np.float64) * 32) * (1 + len(cp) - 1) - 1).astype(int)
        assert len(got) == len(sizes)
        assert np.allclose(got, sizes, rtol=1e-3, atol=1)
    finally:
        engine.set_scheduler_weights(None)
        engine.set_params(**before)


# the histogram's two places to add: LDS up to 4096 levels, memory beyond
@pytest.mark.parametrize("depth", [4095, 4096, 4097])
@pytest.mark.parametrize("size", [1024, 4096, 4097, 9000])
def test_level_histogram_depths(engine, depth, size):
    say("histogram depths", depth, size)
    rng = np.random.default_rng(depth)
    # a path of `depth` vertices, some with leaves, the ids shuffled
    k = 3000
    at = rng.integers(0, depth - 1, k)
    at[:200] = 77
    name = rng.permutation(depth + k)
    src = name[np.concatenate([np.arange(depth - 1), at])]
    dst = name[np.concatenate([np.arange(1, depth), depth + np.arange(k)])]
    cp, ri = csc_from_edges(depth + k, *symmetrize(src, dst))
    engine.upload_csc(cp, ri, symmetric=True)
    lev, st = engine.run(int(name[0]), "llb")
    want, ec, _ = cpu.bfs_queue(cp, ri, int(name[0]))
    assert (lev == want).all() and st["n_levels"] == depth
    counts, edges = engine.level_histogram(size)
    deg = np.diff(cp.astype(np.int64))
    assert (counts == np.bincount(want)).all()
    assert (edges == np.bincount(want, weights=deg)).all()


# a list of more than 2^32 entries (17 GB of zeroes, so the edges are repeats
# of one) behind a level that one work-group's loop runs
def test_list_beyond_32_bits(engine):
    import bfsx
    length = 2 ** 32 + 5
    cp = np.array([0, 1, 1 + length, 2 + length, 3 + length, 3 + length, 3 + length], np.uint64)
    ri = np.zeros(length + 3, np.uint32)
    # 0 -> 1 -> {0 (often), 2, 3}, 2 -> 4, 3 -> 5
    ri[[0, 1001, length, 1 + length, 2 + length]] = [1, 2, 3, 4, 5]
    want = [0, 1, 2, 2, 3, 3]
    with bfsx.Engine(0) as eng:
        eng.upload_csc(cp, ri)
        del ri
        w = np.zeros(1476, np.float32)
        w[-3:] = 1  # constant outputs: LLB, the smallest, at every level
        eng.set_scheduler_weights(w)
        for s in ("llb", "slb", "learned"):
            say("long list", s)
            lev, st, par = eng.run(0, s, parents=True)
            assert lev.tolist() == want, s
            assert st["edges_count"] == length + 3 and st["reached"] == 6, s
            assert par[1:].tolist() == [0, 1, 1, 2, 3], s


# 4-byte offsets and a hub's list (17 GB) that ends less than a stride of the
# groups sharing it below 2^32
def test_hub_list_near_32_bits(engine):
    import bfsx
    length = 2 ** 32 - 3000
    cp = np.array([0, 1, 1 + length, 2 + length, 3 + length, 3 + length, 3 + length], np.uint32)
    ri = np.zeros(length + 3, np.uint32)
    ri[[0, 1001, length, 1 + length, 2 + length]] = [1, 2, 3, 4, 5]
    with bfsx.Engine(0) as eng:
        eng.upload_csc(cp, ri)
        del ri
        for s, mark in (("llb", 4), ("slb", 0xFFFFFFFF)):
            say("long hub", s, mark)
            eng.set_params(hub_degree=1024, mark_ratio_q10=mark)
            lev, st = eng.run(0, s)
            assert lev.tolist() == [0, 1, 2, 2, 3, 3], s
            assert st["edges_count"] == length + 3, s


# the ring wraps: more batches than it has slots, for levels of one byte (four
# pieces a batch) and of two (two), into destinations at any 4-byte offset
@pytest.mark.parametrize("depth", [200, 60000])
@pytest.mark.parametrize("offset", [0, 37])
def test_ring_wraps(engine, depth, offset):
    import ctypes as C
    import os
    import re

    import bfsx
    head = open(os.path.join(bfsx.HERE, "csrc", "bfsx_internal.hpp")).read()
    mib = int(re.search(r"RING_PIECE_BYTES = (\d+)u << 20", head).group(1))
    slots = int(re.search(r"RING_SLOTS = (\d+);", head).group(1))
    per_batch = 4 if depth < 255 else 2
    n = (slots * per_batch + 3 * per_batch // 2) * (mib << 20) // 4 + 4091
    say("ring wraps", depth, offset, n)
    # a path spread over all ids, its first vertex next to a third of the others
    step = n // (depth + 1)
    path = np.arange(depth + 1) * step
    leaf = np.arange(1, n, 3)
    leaf = leaf[(leaf % step != 0) | (leaf > path[-1])]
    deg = np.zeros(n, np.int64)
    deg[path[:-1]] = 1
    deg[0] += len(leaf)
    cp = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32)
    ri = np.concatenate([leaf, path[1:]]).astype(np.uint32)
    want = np.full(n, -1, np.int32)
    want[leaf] = 1
    want[path] = np.arange(depth + 1)
    engine.upload_csc(cp, ri)
    got_cp, got_ri = engine.download_csc()
    assert np.array_equal(got_cp, cp) and np.array_equal(got_ri, ri)
    room = np.full(n + offset + 100, 12345, np.int32)
    for _ in range(2):
        room[:] = 12345
        st = bfsx.RunStats()
        rc = bfsx.lib().bfsx_run(engine._h, 0, 0, 0, room[offset:].ctypes.data, None, C.byref(st))
        assert rc == 0 and st.max_level == depth
        assert np.array_equal(room[offset:offset + n], want)
        assert (room[:offset] == 12345).all() and (room[offset + n:] == 12345).all()


# the histogram that is added up in memory, on the same graphs as in LDS
@pytest.mark.parametrize("name", ["one", "3", "4", "257", "4096", "4099", "20001", "path2500",
                                  "star70001", "directed4099"])
def test_level_histogram_edges_in_memory(engine, name):
    say("histogram in memory", name)
    cp, ri, n_rows, sym, root = some_graph(name)
    engine.upload_csc(cp, ri, n_rows=n_rows, symmetric=sym)
    want, _, _ = cpu.bfs_queue(cp, ri, root, n_rows=n_rows)
    deg = np.where(np.arange(len(want)) < n_rows, np.diff(cp.astype(np.int64)), 0)
    engine.run(root, "llb")
    for size in (4097, 20000):
        counts, edges = engine.level_histogram(size)
        assert (counts == np.bincount(want[want >= 0])).all()
        assert (edges == np.bincount(want[want >= 0], weights=deg[want >= 0])).all()


# adjacency orders by runs of 256 edges (small graphs) up to 4096, the search
# for a run's columns over few and many of them
@pytest.mark.parametrize("m", [1, 255, 257, 65537, 131071, 300007, 1048575, 1048577, 1500001])
@pytest.mark.parametrize("n", [2, 64, 65, 66, 4097, 40011])
@pytest.mark.parametrize("ptr", [np.uint32, np.uint64])
def test_order_adjacency_run_lengths(engine, m, n, ptr):
    say("runs", m, n, ptr.__name__)
    rng = np.random.default_rng(m + n)
    col = np.sort((rng.random(m) ** 2 * n).astype(np.int64))
    ri = rng.integers(0, n, m).astype(np.uint32)
    deg = np.bincount(col, minlength=n)
    cp = np.concatenate([[0], np.cumsum(deg)]).astype(ptr)
    rank = np.empty(n, np.int64)
    rank[np.lexsort((np.arange(n), -deg))] = np.arange(n)
    for order in ("hub_first", "id"):
        engine.upload_csc(cp, ri)
        engine.order_adjacency(order)
        got_cp, got = engine.download_csc()
        key = rank[ri] if order == "hub_first" else ri
        assert np.array_equal(got_cp, cp) and np.array_equal(got, ri[np.lexsort((key, col))])


# arrays of up to 256 KB are checked on the host, larger ones on the card
@pytest.mark.parametrize("ptr", [np.uint32, np.uint64])
@pytest.mark.parametrize("nnz", [65535, 65536, 65537])
def test_refused_graphs_where_the_check_moves(engine, ptr, nnz):
    test_refused_graphs(engine, ptr, nnz)


# copies of up to 512 KB go whole, larger ones in pieces: levels, parents and
# graphs around that, small arrays of a graph together, destinations that
# straddle two of the ring's pages
@pytest.mark.parametrize("n", [3, 32766, 32767, 65535, 131071, 131072, 131073, 150001])
@pytest.mark.parametrize("ptr", [np.uint32, np.uint64])
def test_small_transfers(engine, n, ptr):
    import ctypes as C

    import bfsx
    say("small transfers", n, ptr.__name__)
    rng = np.random.default_rng(n)
    src, dst = rng.integers(0, n, n), rng.integers(0, n, n)
    cp, ri = csc_from_edges(n, *symmetrize(src, dst), dtype=ptr)
    engine.upload_csc(cp, ri, symmetric=True)
    got_cp, got_ri = engine.download_csc()
    assert np.array_equal(got_cp, cp) and np.array_equal(got_ri, ri)
    root = int(np.argmax(np.diff(cp.astype(np.int64))))
    want, ec, _ = cpu.bfs_queue(cp, ri, root)
    page = 2 << 20
    room = np.zeros(4 * page, np.uint8)
    edge = -room.ctypes.data % page + page  # (a page boundary inside)
    for at in (edge, edge - 4, edge - 2 * n // 4 * 4):
        lev = room[at:at + 4 * n].view(np.int32)
        par = np.empty(n + 1, np.uint32)[1:]
        st = bfsx.RunStats()
        room[:] = 7
        rc = bfsx.lib().bfsx_run(engine._h, root, 0, 0, lev.ctypes.data, par.ctypes.data, C.byref(st))
        assert rc == 0 and st.edges_count == ec and np.array_equal(lev, want)
        assert (room[:at] == 7).all() and (room[at + 4 * n:] == 7).all()
        assert cpu.check_parents(cp, ri, root, want, par) == 0


# contexts in turn and side by side, a thread each: a closed one's pinned ring
# goes to the next, and no two share one
def test_contexts_in_turn_and_side_by_side():
    import threading

    import bfsx
    rng = np.random.default_rng(5)
    graphs = []
    for n in (5, 3001, 300007, 900001):
        cp, ri = csc_from_edges(n, rng.integers(0, n, 3 * n), rng.integers(0, n, 3 * n))
        root = int(np.argmax(np.diff(cp.astype(np.int64))))
        graphs.append((cp, ri, root, cpu.bfs_queue(cp, ri, root)[0]))
    wrong = []

    def work(k):
        try:
            for i in range(6):
                cp, ri, root, want = graphs[(i + k) % len(graphs)]
                with bfsx.Engine(0) as eng:
                    eng.upload_csc(cp, ri)
                    got_cp, got_ri = eng.download_csc()
                    lev, _, par = eng.run(root, "llb", parents=True)
                    if not (np.array_equal(lev, want) and np.array_equal(got_ri, ri)
                            and np.array_equal(got_cp, cp)
                            and cpu.check_parents(cp, ri, root, want, par) == 0):
                        wrong.append((k, i))
        except Exception as e:  # (a thread's failure is the test's)
            wrong.append((k, repr(e)))

    for count in (1, 4):
        threads = [threading.Thread(target=work, args=(k,)) for k in range(count)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        say("contexts", count)
        assert not wrong
