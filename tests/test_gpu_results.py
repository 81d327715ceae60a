"""Result getters formed on the device against the vertex words they come from.

Bars: bit-exact.  Ranks are the words times outdeg' (the vertex count for
sinks), one FP64 product; labels and BFS words are moved and decoded only.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("V", [1, 63, 64, 65, 257, 70001])
def test_getters_in_original_order(gz, device, V, relabel):
    rng = np.random.default_rng(V)
    pairs = rng.integers(0, V, size=(4 * V, 2), dtype=np.uint64)
    gz.load_pairs_device(V, pairs, relabel=relabel)
    old, deg = gz.original_ids().astype(np.int64), gz.outdegrees()
    deg = np.where(deg == 0, float(V), deg)
    words = np.empty(V, np.uint64)

    def device_words():
        gz.lib.gz_copy_to_host(words.ctypes.data_as(gz.vp), gz.vp(gz.phase_graph.vertex_props), gz.C.c_size_t(8 * V))
        return words

    gz.run(gz.options("pr", iterations=3))
    props = device_words().view(np.float64)
    assert np.array_equal(gz.pr_props()[old].view(np.uint64), words)
    assert np.array_equal(gz.pr_ranks()[old].view(np.uint64), (props * deg).view(np.uint64))
    gz.run(gz.options("cc"))
    device_words()
    assert np.array_equal(gz.cc_labels()[old], words)
    root = int(pairs[0, 0])
    gz.run(gz.options("bfs", root=root))
    device_words()
    parents, depths = gz.bfs_result()
    seen = words != np.uint64(2**64 - 1)
    assert np.array_equal(depths[old], np.where(seen, words >> np.uint64(48), np.uint64(2**64 - 1)))
    p = (words & np.uint64(2**48 - 1)).astype(np.int64)
    has = seen & (p != 2**48 - 1)
    assert np.array_equal(parents[old], np.where(has, old[np.where(has, p, 0)], -1))
    # the batch of searches has the same depths, and parents one level up
    gz.bfs_batch([root])
    batch_parents, batch_depths = gz.bfs_batch_result(0)
    assert np.array_equal(batch_depths, depths)
    up = batch_parents >= 0
    assert np.array_equal(up, parents >= 0)
    assert np.array_equal(depths[batch_parents[up]] + np.uint64(1), depths[up])


@pytest.mark.parametrize("relabel", [False, True])
def test_getters_leave_captures_valid(gz, device, relabel):
    # a run whose results are read between repeats is captured the second
    # time and replayed from then on: no getter allocates
    gz.load_rmat_device(12, 16 << 12, 9, relabel=relabel)
    root = int(gz.original_ids()[int(np.argmax(gz.outdegrees()))])
    gz.run(gz.options("bfs", root=root))  # the allocations of the runs below
    gz.run(gz.options("cc"))
    gz.bfs_batch([root])
    pr = gz.options("pr", iterations=6)
    gz.run(pr)
    (c0, l0), a0 = gz.graph_replay_counts(), gz.lib.gz_device_allocation_events()
    first = gz.pr_ranks().copy()
    for _ in range(3):
        gz.run(gz.options("bfs", root=root))
        gz.bfs_result()
        gz.run(gz.options("cc"))
        gz.cc_labels()
        gz.bfs_batch([root])
        gz.bfs_batch_result(0)
        gz.run(pr)
        gz.pr_props()
        assert np.array_equal(gz.pr_ranks().view(np.uint64), first.view(np.uint64))
    c1, l1 = gz.graph_replay_counts()
    assert (c1 - c0, l1 - l0) == (1, 3)
    assert gz.lib.gz_device_allocation_events() == a0
