"""BFS push levels over small frontiers run back to back in one workgroup
(gz_bfs_push_tail) against one launch per level (execution_bfs.c:146-169: the
host reads the vote after every level).

Bars: depths equal those of the paths, parents bit-exact against the
per-level launches, as many levels of each engine.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEFAULT_TAIL = 4096  # the library's default entry bound
DIRECT = 1 << 20


def _strands(V, lengths, seed):
    """Disjoint paths over random vertices, the last vertex among them;
    returns the edges and each path's vertices in order."""
    rng = np.random.default_rng(seed)
    ids = rng.choice(V, size=sum(lengths), replace=False).astype(np.uint64)
    if V - 1 not in ids:
        ids[-1] = V - 1
    paths = np.split(ids, np.cumsum(lengths)[:-1])
    pairs = np.concatenate([np.stack([p[:-1], p[1:]], axis=1) for p in paths])
    return pairs, paths


def _bfs(gz, opts, max_vote):
    gz.bfs_push_tail(max_vote)
    try:
        r = gz.run(opts)
        parents, depths = gz.bfs_result()
        return parents.copy(), depths.copy(), r
    finally:
        gz.bfs_push_tail(DEFAULT_TAIL)


@pytest.mark.parametrize("V", [65, 4097, DIRECT - 1, DIRECT, DIRECT + 1])
def test_bfs_tail_on_paths(gz, device, V):
    # every level is one or two vertices wide: the whole search is one launch
    n = min(V // 3, 400)
    pairs, paths = _strands(V, [n, n // 2, 2], V + 1)
    gz.load_pairs_device(V, pairs, symmetrize=True, relabel=True)
    for p, at in ((paths[0], n // 3), (paths[1], 0), (paths[2], 1)):
        p = p.astype(np.int64)
        want = np.full(V, 2**64 - 1, np.uint64)
        want[p] = np.abs(np.arange(len(p)) - at)
        for engine in ("push", "hybrid"):
            for cap in (0, 3, DEFAULT_TAIL):
                parents, depths, r = _bfs(gz, gz.options("bfs", engine=engine, root=int(p[at])), cap)
                assert np.array_equal(depths, want), (engine, cap)
                assert r.pull_iterations + r.push_iterations == r.iterations
                assert r.iterations == max(at, len(p) - 1 - at) + 1
                seen = np.nonzero(want != np.uint64(2**64 - 1))[0]
                up = seen[want[seen] > 0]
                assert np.all(want[parents[up]] + np.uint64(1) == want[up])


@pytest.mark.parametrize("stat", ["both", "outdeg", "count"])
@pytest.mark.parametrize("scale", [10, 13, 16])
def test_bfs_tail_equals_per_level(gz, device, scale, stat):
    # levels that leave the workgroup above the cap and come back below it:
    # the same depths, the same (smallest) parents among push levels, the
    # same number of levels
    gz.load_rmat_device(scale, 16 << scale, 5, relabel=True)
    deg = gz.outdegrees()[np.argsort(gz.original_ids())]
    for root in np.random.default_rng(scale).choice(np.nonzero(deg > 0)[0], 4, replace=False):
        for engine in ("push", "hybrid"):
            opts = gz.options("bfs", engine=engine, root=int(root), stat=stat)
            p0, d0, r0 = _bfs(gz, opts, 0)
            for cap in (16384, DEFAULT_TAIL, 100, 3):
                p, d, r = _bfs(gz, opts, cap)
                assert np.array_equal(d, d0), (engine, cap)
                assert r.iterations == r0.iterations
                assert (r.pull_iterations, r.push_iterations) == (r0.pull_iterations, r0.push_iterations)
                if engine == "push":
                    assert np.array_equal(p, p0), cap


@pytest.mark.parametrize("limit", [1, 2, 5, 40])
def test_bfs_tail_respects_max_iterations(gz, device, limit):
    V = 200
    pairs = np.stack([np.arange(V - 1), np.arange(1, V)], axis=1).astype(np.uint64)
    gz.load_pairs_device(V, pairs, symmetrize=True)
    _, depths, r = _bfs(gz, gz.options("bfs", engine="push", root=0, max_iterations=limit), DEFAULT_TAIL)
    assert r.iterations == limit
    reached = depths != np.uint64(2**64 - 1)
    assert np.array_equal(reached, np.arange(V) <= limit)


@pytest.mark.parametrize("V", [1 << 16, (1 << 20) - 1, 1 << 20, (1 << 20) + 77])
def test_bfs_push_in_parts_keeps_smallest_parents(gz, device, V):
    # large levels below the line of the parts: every parent is the smallest
    # in-neighbour one level up
    pairs = np.random.default_rng(V).integers(0, V, size=(5 * V, 2), dtype=np.uint64)
    pairs[:, 0] = pairs[:, 0] * pairs[:, 0] // np.uint64(V)  # skewed towards low ids
    gz.load_pairs_device(V, pairs)
    src, dst = pairs[:, 0].astype(np.int64), pairs[:, 1].astype(np.int64)
    for root in (int(src[0]), int(src[-1])):
        for stat in ("both", "outdeg"):
            gz.run(gz.options("bfs", engine="push", root=root, stat=stat))
            parents, depths = gz.bfs_result()
            depth = np.full(V, -1, np.int64)
            depth[root], level = 0, 0
            want = np.full(V, V, np.int64)
            while True:
                hit = (depth[src] == level) & ((depth[dst] < 0) | (depth[dst] == level + 1))
                if not hit.any():
                    break
                np.minimum.at(want, dst[hit], src[hit])
                depth[dst[hit]] = level + 1
                level += 1
            seen = depth >= 0
            assert np.array_equal(depths[seen].astype(np.int64), depth[seen])
            assert np.all(depths[~seen] == np.uint64(2**64 - 1))
            below = depth > 0
            assert np.array_equal(parents[below], want[below])


def _bits(gz, at):
    """HasInfo or WantsInfo (a device pointer) as booleans, and how to write them back."""
    n = (gz.num_vertices() + 63) // 64
    words = np.empty(n, np.uint64)
    gz.lib.gz_copy_to_host(words.ctypes.data_as(gz.vp), gz.vp(at), gz.C.c_size_t(8 * n))
    bits = np.unpackbits(words.view(np.uint8), bitorder="little").astype(bool)

    def write():
        w = np.packbits(bits, bitorder="little").view(np.uint64)
        gz.lib.gz_copy_to_device(gz.vp(at), w.ctypes.data_as(gz.vp), gz.C.c_size_t(8 * n))

    return bits, write


def _execute(gz, opts, max_vote):
    r = gz.RunResult()
    gz.bfs_push_tail(max_vote)
    try:
        gz.lib.gz_execution_run(gz.C.byref(opts), gz.C.byref(r))
    finally:
        gz.bfs_push_tail(DEFAULT_TAIL)
    return (*(x.copy() for x in gz.bfs_result()), r)


@pytest.mark.parametrize("extra", [2, 500])
@pytest.mark.parametrize("V", [5000, DIRECT, DIRECT + 1])
def test_bfs_tail_takes_the_frontier_it_is_given(gz, device, V, extra):
    # sources added to HasInfo after the start are searched from too, vertices
    # taken out of WantsInfo are not visited, and a run asked for another root
    # goes on from the prepared one
    edges = np.random.default_rng(V).integers(0, V, size=(2 * V, 2), dtype=np.uint64)
    gz.load_pairs_device(V, edges)
    src, dst = edges[:, 0].astype(np.int64), edges[:, 1].astype(np.int64)
    picked = np.random.default_rng(extra).choice(np.unique(src), extra + 40, replace=False)
    sources, barred = picked[:extra], picked[extra:]
    G = gz.phase_graph
    for engine in ("push", "hybrid"):
        depth = np.full(V, -1, np.int64)
        depth[sources], level = 0, 0
        depth[barred] = -2
        while True:
            hit = (depth[src] == level) & (depth[dst] == -1)
            if not hit.any():
                break
            level += 1
            depth[dst[hit]] = level
        want = np.where(depth > 0, depth.astype(np.uint64), np.uint64(2**64 - 1))
        want[sources[0]] = 0
        for cap in (0, 3, DEFAULT_TAIL):
            opts = gz.options("bfs", engine=engine, root=int(sources[0]))
            gz.lib.gz_execution_prepare(gz.C.byref(opts))
            has, put_has = _bits(gz, G.frontier_has_info)
            wants, put_wants = _bits(gz, G.frontier_wants_info)
            has[sources] = True
            wants[sources] = wants[barred] = False
            put_has()
            put_wants()
            opts.root = int(sources[-1])
            _, got, r = _execute(gz, opts, cap)
            assert np.array_equal(got, want), (engine, cap)
            assert r.iterations == level + 1
            left, _ = _bits(gz, G.frontier_wants_info)
            assert np.array_equal(left[:V], depth == -1), (engine, cap)


def test_bfs_tail_levels_beyond_the_words(gz, device):
    # a word holds 16 bits of level: from level 65,536 on a vertex of an
    # earlier level is told by WantsInfo alone
    V = 65536 + 300
    pairs = np.stack([np.arange(V - 1), np.arange(1, V)], axis=1).astype(np.uint64)
    gz.load_pairs_device(V, pairs, symmetrize=True)
    opts = gz.options("bfs", engine="push", root=0)
    parents, depths, r = _bfs(gz, opts, DEFAULT_TAIL)
    assert r.iterations == V
    assert np.array_equal(parents, np.arange(V) - 1)
    assert np.array_equal(depths, np.arange(V, dtype=np.uint64) % np.uint64(1 << 16))


def test_bfs_tail_frontier_past_its_list(gz, device):
    # a first frontier far beyond its root's statistic lists more vertices
    # than the workgroup holds: all of them reach the next level
    hubs, fan = 400, 100
    V = hubs * (fan + 1)
    hub = np.repeat(np.arange(hubs), fan)
    pairs = np.stack([hub, hubs + np.arange(hubs * fan)], axis=1).astype(np.uint64)
    gz.load_pairs_device(V, pairs)
    opts = gz.options("bfs", engine="push", root=0)
    gz.lib.gz_execution_prepare(gz.C.byref(opts))
    has, put = _bits(gz, gz.phase_graph.frontier_has_info)
    has[:hubs] = True
    put()
    parents, depths, r = _execute(gz, opts, DEFAULT_TAIL)
    assert r.iterations == 2
    assert np.all(depths[hubs:] == 1) and np.array_equal(parents[hubs:], hub)
    left, _ = _bits(gz, gz.phase_graph.frontier_wants_info)
    assert not left[hubs:V].any()


@pytest.mark.parametrize("V", [(1 << 24) - 1, 1 << 24, (1 << 24) + 77])
def test_bfs_push_in_parts(gz, device, V, tmp_path):
    # from 2^24 vertices, a level of at least a quarter of the vectors and at
    # most a fifth of the edges is pushed in parts (here the second, half a
    # million edges from 20,000 vertices with shared targets): depths, smallest
    # parents and edge counts as in one part, with and without the selector's
    # sums
    import selector_train as st

    rng = np.random.default_rng(V)
    ids = rng.choice(V, size=220001, replace=False)
    first, second = ids[1:20001], ids[20001:]
    src = np.concatenate([np.full(20000, ids[0]), np.repeat(first, 25), np.repeat(second, 14)])
    dst = np.concatenate([first, rng.choice(second, 20000 * 25), rng.integers(0, V, 200000 * 14)])
    gz.load_pairs_device(V, np.stack([src, dst], axis=1).astype(np.uint64))
    E = gz.num_edges()
    depth = np.full(V, -1, np.int64)
    depth[ids[0]], level = 0, 0
    want, out, walked = np.full(V, V, np.int64), gz.outdegrees(), []
    while True:
        walked.append(int(out[depth == level].sum()))
        hit = (depth[src] == level) & ((depth[dst] < 0) | (depth[dst] == level + 1))
        if not hit.any():
            break
        np.minimum.at(want, dst[hit], src[hit])
        depth[dst[hit]] = level + 1
        level += 1
    votes = [walked[i] + int((depth == i).sum()) for i in range(len(walked))]
    vectors = gz.lib.gz_graph_push_vector_count()
    assert any(vectors // 4 <= v <= E // 5 for v in votes[1:])
    params = np.zeros(gz.SEL_PARAMS, np.float32)
    params[-2:] = [10.0, -10.0]  # a model that always pushes
    st.save_weights(str(tmp_path / "push.bin"), params, np.zeros(8, np.float32), np.ones(8, np.float32))
    gz.selector_load(str(tmp_path / "push.bin"))
    gz.selector_set_trust(0.0)
    try:
        for engine in ("push", "learned"):
            for stats in (False, True):
                r = gz.run(gz.options("bfs", engine=engine, root=int(ids[0]), collect_stats=stats))
                assert r.push_iterations == r.iterations == len(walked)
                parents, depths = gz.bfs_result()
                seen, below = depth >= 0, depth > 0
                assert np.array_equal(depths[seen].astype(np.int64), depth[seen])
                assert np.all(depths[~seen] == np.uint64(2**64 - 1))
                assert np.array_equal(parents[below], want[below])
                if stats:
                    assert [x.edges for x in gz.records()] == walked
                    assert [x.frontier_stat for x in gz.records()] == votes
    finally:
        gz.selector_set_trust(gz.TRUST_ABOVE, gz.TRUST_BELOW)
        gz.selector_clear()
