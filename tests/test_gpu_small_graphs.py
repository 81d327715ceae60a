"""Work splits of the small-graph paths at the sizes where they change.

The scheduler-aware PageRank pull gives a chunk a workgroup of four
wavefronts on lists of at most 4096 chunks, and the sparse push gives a
wavefront 1, 4, 16 or 64 bitmap words by vertex count.  Bars as for every
other width: PageRank within 1e-12 of FP64 numpy (each sum is regrouped, and
2^-53 times the at most 20 iterations and a few thousand terms of a sum
stays below it; the oracle adds S over all edges in one chain, whose own
rounding passes that on the lists of millions of equal terms here), CC labels
and BFS words bit-exact with the oracle.
"""
import numpy as np
import pytest

import graphs

pytestmark = pytest.mark.gpu

PR_TOL = 1e-12


def _rel(a, b):
    return float(np.max(np.abs(a - b) / np.maximum(np.abs(b), 1e-300)))


def _ranks(g, iterations, damping=0.875):
    """PageRank in numpy: per-destination sums, S summed pairwise."""
    src, dst = g.pull[:, 0].astype(np.int64), g.pull[:, 1].astype(np.int64)
    nv = float(g.num_vertices)
    deg = np.bincount(src, minlength=g.num_vertices).astype(np.float64)
    deg[deg == 0] = nv
    props = 1.0 / nv / deg
    for _ in range(iterations):
        acc = np.bincount(dst, weights=props[src], minlength=g.num_vertices)
        props = ((acc + (1.0 - acc.sum()) / nv) * damping + (1.0 - damping) / nv) / deg
    return props * deg


def _line(gz, edges):
    """One destination per vector: vertex i + 1 from i, `edges` of them."""
    i = np.arange(edges, dtype=np.uint64)
    return gz.make_graph(np.stack([i, i + 1], axis=1), edges + 1)


def _fan(gz, width):
    """Every vertex into vertex 0: one run over all the list."""
    i = np.arange(1, width, dtype=np.uint64)
    return gz.make_graph(np.stack([i, np.zeros_like(i)], axis=1), width)


PULL_CASES = {
    "one_vector": lambda gz: _line(gz, 1),
    "quarter_and_one": lambda gz: _line(gz, 65),
    "chunk_less_one": lambda gz: _line(gz, 255),
    "chunk": lambda gz: _line(gz, 256),
    "chunk_and_one": lambda gz: _line(gz, 257),
    "one_run": lambda gz: _fan(gz, 9001),
    "hub": lambda gz: graphs.hub_graph(gz),
    "last_split_list": lambda gz: _line(gz, 256 * 4096),
    "first_unsplit_list": lambda gz: _line(gz, 256 * 4096 + 1),
    "8192_chunks": lambda gz: _line(gz, 256 * 8192),
    "8193_chunks": lambda gz: _line(gz, 256 * 8192 + 1),
}


@pytest.mark.parametrize("case", sorted(PULL_CASES))
@pytest.mark.parametrize("vpl", [1, 2])
def test_split_pull(gz, device, case, vpl):
    g = PULL_CASES[case](gz)
    ref = _ranks(g, 5)
    gz.set_chunk_vectors(256 * vpl)
    gz.set_vectors_per_lane(vpl)
    try:
        gz.load(g)
        gz.run(gz.options("pr", iterations=5))
        got = gz.pr_ranks()
        gz.run(gz.options("pr", iterations=1, collect_stats=True))
        stats = gz.records()[0]
    finally:
        gz.set_chunk_vectors(512)
        gz.set_vectors_per_lane(1)
    assert _rel(got, ref) <= PR_TOL
    assert stats.vectors == gz.pull_vector_count() and stats.edges == g.num_edges


# bitmap words at which a wavefront's share changes: 2048 wavefronts of 4, 16 and 64
@pytest.mark.parametrize("words", [1, 4 * 2048, 16 * 2048, 64 * 2048])
@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_sparse_push_widths(gz, orc, device, words, extra):
    n = 64 * words + extra
    core = gz.rmat_edges(10, 8 << 10, seed=words + 2)
    far = np.random.default_rng(words + extra).integers(0, n, size=(4000, 2), dtype=np.uint64)
    tail = np.array([[0, n - 1], [n - 1, n - 2], [n - 2, n // 2]], dtype=np.uint64)
    g = gz.make_graph(np.concatenate([core % np.uint64(n), far, tail]), n, symmetrize=True)
    G = orc.Graph(g.num_vertices, g.pull, g.push)
    gz.load(g)
    gz.run(gz.options("bfs", root=0))
    parents, depths = gz.bfs_result()
    ref = orc.bfs(G, orc.options(root=0))
    assert np.array_equal(parents, ref[0]) and np.array_equal(depths, ref[1])
    gz.cc_push_tail(0)
    try:
        gz.run(gz.options("cc", engine="push"))
        assert np.array_equal(gz.cc_labels(), orc.cc(G, orc.options())[0])
    finally:
        gz.cc_push_tail(4096)


def test_iteration_end_past_one_workgroup_sum(gz, orc, device):
    """More vote partials than one workgroup sums: the frontier words of the
    iteration's end have a launch of their own."""
    g = gz.rmat_graph(20, 16, seed=5)
    gz.set_chunk_vectors(64)
    try:
        gz.load(g)
        assert gz.pull_vector_count() > 64 * 65536
        gz.run(gz.options("cc"))
        got = gz.cc_labels()
    finally:
        gz.set_chunk_vectors(512)
    assert np.array_equal(got, orc.cc(orc.Graph(g.num_vertices, g.pull, g.push), orc.options(threads=8))[0])


@pytest.mark.parametrize("vpl", [1, 2, 4])
@pytest.mark.parametrize("edges", [3, 255, 256, 257, 4095, 70000, 1200000])
def test_cc_pull_runs_across_chunks(gz, device, edges, vpl):
    # one destination over many chunks, destinations of one vector, and lists
    # from a step to hundreds of chunks: a label written by the wrong unit
    # would stay too high
    rng = np.random.default_rng(edges + vpl)
    V = max(4, edges // 2)
    hubs = rng.choice(V, size=2, replace=False)
    half = edges // 2
    src = np.concatenate([rng.integers(0, V, size=half), rng.integers(0, V, size=edges - half)])
    dst = np.concatenate([hubs[rng.integers(0, 2, size=half)], rng.integers(0, V, size=edges - half)])
    pairs = np.stack([src, dst], axis=1).astype(np.uint64)
    want = np.arange(V)
    while True:  # smallest id of each component, by sweeps
        low = np.minimum(want[src], want[dst])
        new = want.copy()
        np.minimum.at(new, src, low)
        np.minimum.at(new, dst, low)
        new = new[new]
        if np.array_equal(new, want):
            break
        want = new
    gz.set_vectors_per_lane(vpl)
    try:
        gz.load_pairs_device(V, pairs, symmetrize=True)
        for engine in ("pull", "hybrid"):
            gz.run(gz.options("cc", engine=engine))
            assert np.array_equal(gz.cc_labels(), want.astype(np.uint64)), engine
    finally:
        gz.set_vectors_per_lane(1)


@pytest.mark.parametrize("chains", [39, 312])
def test_pull_passes_labels_along_a_chunk(gz, device, chains):
    # chains of 64 consecutive vertices hang off a spine of their first ones,
    # a vector each: a sweep's step holds one chain, so the smallest label
    # passes the spine by the chunk's eight steps in a sweep, then one vertex
    # of the last chain per sweep, whatever the list's length
    L = 64
    a = np.arange(chains * L, dtype=np.uint64).reshape(chains, L)
    pairs = np.concatenate([np.stack([a[:, :-1].ravel(), a[:, 1:].ravel()], axis=1),
                            np.stack([a[:-1, 0], a[1:, 0]], axis=1)])
    gz.load_pairs_device(chains * L, pairs, symmetrize=True)
    gz.set_chunk_vectors(512)
    r = gz.run(gz.options("cc", engine="pull"))
    assert not gz.cc_labels().any()
    assert r.iterations == r.pull_iterations <= (chains + 7) // 8 + L + 2


@pytest.mark.parametrize("chains", [64, 313, 341, 342])
def test_cc_sparse_push_on_both_sides_of_four_words(gz, device, chains):
    # the same graph: up to 341 chains its edges and vertices are within the
    # sparse push's bound of 2^16, a wavefront takes four chains, and a label
    # passes the spine by four of them an iteration
    L = 64
    a = np.arange(chains * L, dtype=np.uint64).reshape(chains, L)
    pairs = np.concatenate([np.stack([a[:, :-1].ravel(), a[:, 1:].ravel()], axis=1),
                            np.stack([a[:-1, 0], a[1:, 0]], axis=1)])
    gz.load_pairs_device(chains * L, pairs, symmetrize=True)
    within = gz.num_edges() + gz.num_vertices() <= 1 << 16
    assert within == (chains <= 341)
    for tail in (0, 4096):
        gz.cc_push_tail(tail)
        try:
            r = gz.run(gz.options("cc", engine="push"))
        finally:
            gz.cc_push_tail()
        assert not gz.cc_labels().any()
        assert r.iterations == r.push_iterations
        if within and tail == 0:
            assert r.iterations <= (chains + 3) // 4 + L + 2
